// Decode attention for calls of few work items: attn_mfma's work with each of
// an item's W waves a workgroup of its own (decode_item<..., SPREAD>), so that
// the item's keys stream through W compute units instead of one.
//
// What bounds it: one wave alone on its SIMD, which issues one instruction at
// a time (per 16-key tile at head_dim 128 ~70 vector, ~57 scalar and 24 matrix
// instructions, ~1060 cycles; two tiles a step with the requests between the
// products ~950), behind a fixed ~9 us of launch and dependent round trips
// (arguments, record, page table and rows, first tiles; then the states'
// stores, the arrival and the merge's loads).  Each wave keeps 64 KiB of tiles
// in flight through LDS (32 KiB at head_dim 64).  One sequence of 2500 keys (8
// KV heads of 128, bf16, rotated): 27.7 -> 18.3 us per layer call; eight of 3000
// of f16 36.6 -> 23.1.
// States combined as the one-workgroup kernel combines them, so the results
// are the same bits.
#include "attn_decode.hpp"

namespace thb {
namespace {

template <int HD, bool F16, int W, int NB, bool FULL>
__global__ __launch_bounds__(64) void attn_spread(AttnArgs a) {
    __shared__ SpreadLds<HD, W> lds;
    // W workgroups per (item, KV head), one for each wave; KV head fastest.
    const uint32_t slot = blockIdx.x / a.n_kvh, kvh = blockIdx.x - slot * a.n_kvh;
    const uint32_t* G = a.items + static_cast<uint64_t>(slot / W) * kItemWords;
    decode_item<HD, F16, W, NB, FULL, true>(a, G, kvh, slot % W, lds, threadIdx.x);
}

// A device plan's launch of up to kSpreadMax rows x KV heads, whose records say
// which form each build chose from the rows' keys (dplan_kernel): a whole item
// per workgroup (attn_mfma), or one or two of an item's W waves, for which the
// workgroup's other waves end at once.  One kernel holds both forms, as a graph
// cannot choose its launches and a launch of each kind, of which one does
// nothing, would cost more.  Two waves of 256 registers (128 at head_dim 64) per
// SIMD bound it, which the spread form fits at head_dim 256 with the query's low
// halves in LDS (spilled, a reload waited for all tiles in flight: 64 us for 51).
// us per launch, one workgroup per item always / one per wave always / this (8
// KV heads of 128 x 4, rotated, f16, keys from HBM): one sequence of 200 keys
// 11.1 / 12.1 / 11.5, of 3000 35.2 / 21.0 / 22.2; eight of 200 11.5 / 13.3 / 11.6,
// of 3000 38.2 / 28.6 / 30.8; 2 KV heads of 64 x 7, eight of 200 9.8 / 11.1 /
// 10.0, of 3000 22.3 / 18.0 / 18.8.  (Plain loads in the latter two; non-temporal
// ones, as now, take 13 % less for eight of 3000, 4 % for one.)
template <int HD, bool F16, int W, bool FULL>
__global__ __launch_bounds__(64 * W, HD == 64 ? 4 : 2) void attn_pick(AttnArgs a) {
    __shared__ union {
        DecodeLds<HD, F16, W> item;
        SpreadLds<HD, W, HD == 256> wave[2];
    } lds;
    const uint32_t slot = blockIdx.x / a.n_kvh, kvh = blockIdx.x - slot * a.n_kvh;
    const uint32_t* G = a.items + static_cast<uint64_t>(slot) * kItemWords;
    const uint32_t part = G[kGroupWords], runs = part >> kRecRuns;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Each form reads the arguments through a pointer that the compiler must
    // take as new (an empty asm): those that both use, loaded in front of the
    // branch, would be waited for there and spilled (0.5 us of every launch).
    typedef const __attribute__((address_space(4))) AttnArgs* KArgs;
    KArgs kp = (KArgs)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(kp));
    if (runs == 0) {
        decode_item<HD, F16, W, ring_for(HD), FULL, false>(*(const AttnArgs*)kp, G, kvh, wave, lds.item, threadIdx.x);
    } else if (wave < runs) {
        asm volatile("" : "+s"(kp));
        decode_item<HD, F16, W, spread_ring(HD), FULL, true, HD == 256>(*(const AttnArgs*)kp, G, kvh,
                                                             (part >> kRecRun & 255u) + wave, lds.wave[wave],
                                                             threadIdx.x & 63u);
    }
}

template <int HD, bool F16>
void launch_pick_hd(dim3 grid, const AttnArgs& a, hipStream_t s) {
    constexpr int W = decode_waves(HD);
    if (a.full)
        hipLaunchKernelGGL((attn_pick<HD, F16, W, true>), grid, dim3(64 * W), 0, s, a);
    else
        hipLaunchKernelGGL((attn_pick<HD, F16, W, false>), grid, dim3(64 * W), 0, s, a);
}

template <int HD, bool F16>
void launch_spread_hd(dim3 grid, const AttnArgs& a, hipStream_t s) {
    constexpr int W = decode_waves(HD);
    if (a.full)
        hipLaunchKernelGGL((attn_spread<HD, F16, W, spread_ring(HD), true>), grid, dim3(64), 0, s, a);
    else
        hipLaunchKernelGGL((attn_spread<HD, F16, W, spread_ring(HD), false>), grid, dim3(64), 0, s, a);
}

}  // namespace

void launch_spread(uint32_t hd, bool f16, dim3 grid, const AttnArgs& a, hipStream_t s) {
    switch (hd) {
        case 64: f16 ? launch_spread_hd<64, true>(grid, a, s) : launch_spread_hd<64, false>(grid, a, s); break;
        case 128: f16 ? launch_spread_hd<128, true>(grid, a, s) : launch_spread_hd<128, false>(grid, a, s); break;
        default: f16 ? launch_spread_hd<256, true>(grid, a, s) : launch_spread_hd<256, false>(grid, a, s); break;
    }
}

void launch_pick(uint32_t hd, bool f16, dim3 grid, const AttnArgs& a, hipStream_t s) {
    switch (hd) {
        case 64: f16 ? launch_pick_hd<64, true>(grid, a, s) : launch_pick_hd<64, false>(grid, a, s); break;
        case 128: f16 ? launch_pick_hd<128, true>(grid, a, s) : launch_pick_hd<128, false>(grid, a, s); break;
        default: f16 ? launch_pick_hd<256, true>(grid, a, s) : launch_pick_hd<256, false>(grid, a, s); break;
    }
}

}  // namespace thb
