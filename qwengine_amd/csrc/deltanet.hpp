// Shapes shared by the Gated DeltaNet sources: deltanet.hip (decode / verify) and deltanet_rows.hip (prefill), which are
// built with different instruction schedulers.
#pragma once

#include "launch.hpp"
#include "qwattn_common.hpp"

namespace qwa {

constexpr int DN_CH = 10240;  // conv channels: q (16 x 128) | k (16 x 128) | v (48 x 128)
constexpr int DN_QK = 2048;
constexpr int DN_HD = 128;
constexpr int DN_KH = 16;
constexpr int DN_VH = 48;
constexpr int DN_VD = DN_VH * DN_HD;  // 6144
constexpr int DN_BA_LD = 64;          // row stride of the decode path's beta / alpha inputs

__device__ __forceinline__ float dn_silu(float x) { return x / (1.0f + __expf(-x)); }

}  // namespace qwa
