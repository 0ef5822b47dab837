// The model's attention shape (host and device code).
#pragma once

namespace qwa {

constexpr int NH = 24;     // query heads
constexpr int NKV = 4;     // KV heads
constexpr int HD = 256;    // head dim
constexpr int GRP = 6;     // query heads per KV head
constexpr int NROT = 64;   // rotary dims
constexpr int MAXQ = 8;    // queries per decode call
constexpr int MAX_POS = 262144;

}  // namespace qwa
