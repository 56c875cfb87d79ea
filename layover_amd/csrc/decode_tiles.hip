// Launches of decode_tiles.h's kernel (see there), in a translation unit of their own: one instance
// per pool format, query format and head_dim class.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "decode_tiles.h"
#include "host_common.h"

namespace lk {

template <int KV, int QF>
static void launch_tiles_dim(const DecodeArgs& a, uint32_t waves, uint32_t grid, hipStream_t stream) {
    const dim3 block(kWave * waves);
    const uint32_t lds = tiles_lds_bytes(a, KV, waves);
    auto launch = [&](auto dim) {
        constexpr int kD = decltype(dim)::value;
        if (a.head_dim == kD) hipLaunchKernelGGL((decode_split_tiles<KV, QF, kD, true>), dim3(grid), block, lds, stream, a);
        else hipLaunchKernelGGL((decode_split_tiles<KV, QF, kD, false>), dim3(grid), block, lds, stream, a);
    };
    if (a.head_dim <= 32) launch(std::integral_constant<int, 32>{});
    else if (a.head_dim <= 64) launch(std::integral_constant<int, 64>{});
    else if (a.head_dim <= 128) launch(std::integral_constant<int, 128>{});
    else launch(std::integral_constant<int, 256>{});
}

void launch_split_tiles(const DecodeArgs& a, int kv, int qf, uint32_t waves, hipStream_t stream) {
    const uint64_t grid = uint64_t(a.batch) * a.splits * a.kv_heads * ((a.groups + kMaxHeads - 1) / kMaxHeads);
    require(grid <= 0x7FFFFFFFull, "decode grid too large");
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
