// Decode attention for calls of few work items: attn_mfma's work with each of
// an item's W waves a workgroup of its own (decode_wg<..., SPREAD>), so that
// the item's keys stream through W compute units instead of one.
//
// What bounds it: one wave alone on its SIMD, which issues one instruction at
// a time (per 16-key tile at head_dim 128 ~70 vector, ~57 scalar and 24 matrix
// instructions, ~1060 cycles; two tiles a step with the requests between the
// products ~950), behind a fixed ~9 us of launch and dependent round trips
// (arguments, record, page table and rows, first tiles; then the states'
// stores, the arrival and the merge's loads).  Each wave keeps 64 KiB of tiles
// in flight through LDS.  One sequence of 2500 keys (8 KV heads of 128, bf16,
// rotated): 27.7 -> 18.8 us per layer call; 4000 keys of f16 34.9 -> 21.7; a
// captured 32-layer step of 8 sequences of 300-3000 keys 1287 -> 970 us.
// States combined as the one-workgroup kernel combines them, so the results
// are the same bits.
#include "attn_decode.hpp"

namespace thb {
namespace {

template <int HD, bool F16, int W, int NB, bool FULL>
__global__ __launch_bounds__(64) void attn_spread(AttnArgs a) {
    __shared__ SpreadLds<HD, W> lds;
    decode_wg<HD, F16, W, NB, FULL, true>(a, blockIdx.x, lds, threadIdx.x);
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

}  // namespace thb
