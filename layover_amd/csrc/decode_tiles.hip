// Launches of decode_tiles.h's kernel (see there), in a translation unit of their own: one instance
// per pool format, query format and head_dim class.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "decode_tiles.h"
#include "host_common.h"

namespace lk {

template <int KV, int QF>
static void launch_tiles_dim(const DecodeArgs& a, uint32_t waves, uint32_t grid, hipStream_t stream) {
    const dim3 block(kWave * waves);
    const uint32_t lds = tiles_lds_bytes(a, KV, waves);
    if (a.head_dim <= 32) hipLaunchKernelGGL((decode_split_tiles<KV, QF, 32>), dim3(grid), block, lds, stream, a);
    else if (a.head_dim <= 64) hipLaunchKernelGGL((decode_split_tiles<KV, QF, 64>), dim3(grid), block, lds, stream, a);
    else if (a.head_dim <= 128) hipLaunchKernelGGL((decode_split_tiles<KV, QF, 128>), dim3(grid), block, lds, stream, a);
    else hipLaunchKernelGGL((decode_split_tiles<KV, QF, 256>), dim3(grid), block, lds, stream, a);
}

// Waves per workgroup: as decode_waves (kernels.hip), 4 when the grid gives every CU two workgroups,
// else 8, which the merge's LDS (at most 8 heads) and the registers (FP32 arithmetic on 256 dims
// keeps a wave at one per SIMD) must allow.
void launch_split_tiles(const DecodeArgs& a, int kv, int qf, hipStream_t stream) {
    const uint64_t grid = uint64_t(a.batch) * a.splits * a.kv_heads * ((a.groups + kMaxHeads - 1) / kMaxHeads);
    require(grid <= 0x7FFFFFFFull, "decode grid too large");
    const bool wide = a.head_dim > 128 && (kv == LK_F32 || qf == LK_F32);
    const uint32_t waves = grid >= 2ull * compute_units() || a.groups > 8 || wide ? 4 : 8;
    if (qf == LK_BF16) {
        if (kv == LK_BF16) launch_tiles_dim<LK_BF16, LK_BF16>(a, waves, uint32_t(grid), stream);
        else if (kv == LK_F32) launch_tiles_dim<LK_F32, LK_BF16>(a, waves, uint32_t(grid), stream);
        else launch_tiles_dim<LK_FP8_RECORD, LK_BF16>(a, waves, uint32_t(grid), stream);
    } else {
        if (kv == LK_BF16) launch_tiles_dim<LK_BF16, LK_F32>(a, waves, uint32_t(grid), stream);
        else if (kv == LK_F32) launch_tiles_dim<LK_F32, LK_F32>(a, waves, uint32_t(grid), stream);
        else launch_tiles_dim<LK_FP8_RECORD, LK_F32>(a, waves, uint32_t(grid), stream);
    }
}

}  // namespace lk
