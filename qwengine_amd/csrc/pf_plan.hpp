// How a prefill pass is cut into row blocks and key splits, and the size of the scratch that follows from it (host code
// only, so that the sizes can be checked without a GPU, also for other tile shapes than the built one).
#pragma once

#include <algorithm>

#include "qwattn.h"
#include "shapes.hpp"

namespace qwa {

#ifndef QWA_PF_WAVES
#define QWA_PF_WAVES 8
#endif
constexpr int PF_WAVES = QWA_PF_WAVES;           // MFMA waves per workgroup
#ifndef QWA_PF_RT
#define QWA_PF_RT (16 / PF_WAVES > 0 ? 16 / PF_WAVES : 1)
#endif
constexpr int PF_RT = QWA_PF_RT;                 // 16-row MFMA tiles per wave
constexpr int PF_ROWS = PF_WAVES * PF_RT * 16;   // rows per workgroup
constexpr int PF_TILE = 32;                      // keys per tile
constexpr int PF_NS = PF_ROWS == 192 ? 6 : 8;    // key-range splits per row block (3 rounds of the chip for B = 1024)
constexpr int PF_MAXB = 1024;                    // tokens per pass
// row blocks of a pass of nb tokens (per KV head)
constexpr int pf_row_blocks(int nb) { return (GRP * nb + PF_ROWS - 1) / PF_ROWS; }
constexpr int PF_FEW = 12;  // row blocks up to which a pass takes the split count that fills one round of the chip
// splits of a pass of nb tokens whose keys end at npos.
// Up to PF_FEW row blocks (512 tokens): as many as make one round of the 256 CUs (64 / row blocks per KV head), each of
// at least one tile.  (Fewer splits for short key ranges, sqrt(c tiles / tokens) with c = 500 .. 2000 to weigh the
// partial states, measured the same or up to 3 us slower at contexts below 4000.)
// Measured, whole call, us, against 5 to 8 splits for every pass (Q8_0): 8 tokens at 20000 positions 153 -> 48, 77 at
// 20011 167 -> 84, 77 at 90000 648 -> 281, 128 at 32256 255 -> 152, 200 at 5000 69 -> 60, 256 at 32256 261 -> 235;
// 512 tokens unchanged (their 5 splits already make one round).  Odd counts, too: the next lower even one would let
// k_prefill number the row blocks that share a tile onto one XCD, but its longer splits cost more than that gives (whole
// call, us, the count / the even one: 21 / 20 splits, 128 tokens at 20000 F16 positions 99.5 / 102.5, Q8_0 103.1 / 103.0,
// at 149000 576 / 591; 9 / 8, 298 at 20000 174 / 178, at 149000 1067 / 1112; 7 / 6, 384 at 60000 551 / 595; 5 / 4, 512 at
// 60000 716 / 841).
// Above that (at most PF_NS): the count that fills the chip's 256 CUs in whole rounds best, i.e. the fewest rounds per
// split, ceil(workgroups / 256) / splits (1024 tokens: 8 splits, 3 rounds).
constexpr int pf_splits(int nb, int npos) {
    const int nrb = pf_row_blocks(nb);
    if (nrb <= PF_FEW) return std::min(256 / (NKV * nrb), (npos - 1) / PF_TILE + 1);
    const int groups = nrb * NKV;
    int best = PF_NS;
    for (int ns = PF_NS - 1; ns >= 6; ns--)  // 6 .. PF_NS: 5 splits are never the best of these passes
        if ((long)((groups * ns + 255) / 256) * best < (long)((groups * best + 255) / 256) * ns) best = ns;
    return best;
}
// Whether a call of nb tokens whose keys end at npos dequantises its KV range into fp16 images first (the results are the
// same bits either way).  Otherwise every workgroup converts its raw tiles in the loop: once more per row block, slower to
// start (a workgroup's first tile is converted before anything runs) and with 32-byte stores of its partial states, but
// without the image pass's launch and its 64 KB written and read per tile.  So the raw tiles win for the fewest row blocks
// and, with more of them, only from some length of the key range on; the cheaper the conversion, the earlier (F16: a copy).
// Whole call, us, images / raw tiles.  F16: 8 tokens at 200 positions 22.5 / 19.6, 36 at 0 23.6 / 24.4 and at 1500 34.6 /
// 34.4; 42 (1 block) at 2000 34.8 / 35.5, at 3500 38.3 / 37.4, at 60000 163 / 113; 64 (2) at 3200 39.1 / 39.9, at 5000
// 42.9 / 42.4, at 20000 83.7 / 73.2; 110 (3) at 5000 49.1 / 49.3, at 8192 60.5 / 59.4, at 20000 105 / 97; 150 (4) at 14336
// 93.8 / 94.5, at 20000 120 / 116; 171 (5) at 20000 140 / 144.  Q4_0: 8 at 200 24.6 / 21.9, 36 at 1500 39.6 / 38.9; 42 (1)
// at 2500 40.7 / 42.3, at 6500 47.0 / 46.4, at 60000 139 / 112; 64 (2) at 14336 67.8 / 68.3, at 20000 80.8 / 79.7, at 60000
// 182 / 171; 110 (3) at 60000 233 / 243.  Q8_0: 8 at 200 22.6 / 21.6, 20 at 1000 28.7 / 29.3 and at 3500 36.3 / 35.1; 42
// (1) at 2000 34.7 / 38.4, at 16384 60.1 / 60.0, at 60000 147 / 132; 64 (2) at 60000 188 / 196.
constexpr bool pf_use_image(int kvt, int nb, int npos) {
    constexpr int MAX_BLOCKS = 4, NEVER = MAX_POS + 1;
    const int nrb = pf_row_blocks(nb);
    if (nb <= (kvt == QWA_KV_Q8_0 ? 20 : 36)) return false;
    if (nrb > MAX_BLOCKS) return true;
    constexpr int f16[MAX_BLOCKS] = {2560, 4096, 6144, 16384}, q4[MAX_BLOCKS] = {4608, 18432, NEVER, NEVER},
                  q8[MAX_BLOCKS] = {16384, NEVER, NEVER, NEVER};
    return npos < (kvt == QWA_KV_F16 ? f16 : kvt == QWA_KV_Q4_0 ? q4 : q8)[nrb - 1];
}
// the most token-splits (splits x tokens) that a pass of up to PF_FEW row blocks takes (2728 of 256 rows, at 341 tokens),
// rounded up to a multiple of 16: the partial states start behind this many (m, l) rows, and 150 tokens at 0 Q8_0 positions
// take 29.8 us behind 2728 of them and 27.7 behind 2736 (their splits lie 1.8 MB apart, so the start decides how they share
// the memory channels)
constexpr int pf_few_token_splits() {
    int most = 0;
    for (int nrb = 1; nrb <= PF_FEW; nrb++)
        most = std::max(most, std::min(nrb * PF_ROWS / GRP, PF_MAXB) * (256 / (NKV * nrb)));
    return (most + 15) & ~15;
}
// token-splits that a workspace for passes of up to nb tokens has to hold: PF_NS per token, or what the shorter passes
// take, never decreasing in nb
constexpr int pf_token_splits(int nb) {
    return std::max(PF_NS * nb, std::min(256 / NKV * nb, pf_few_token_splits()));
}
#ifndef QWA_PF_UPW
#define QWA_PF_UPW 1
#endif
#ifndef QWA_PF_SEG_MAXPOS
#define QWA_PF_SEG_MAXPOS 81920
#endif
// (row block, KV head, split) units per workgroup of a pass of nb tokens whose keys end at npos: as many as make the
// units one round of the chip's 256 CUs, when the split count is 8 (so the workgroups of one XCD walk the splits in
// step, see k_prefill) and the pass's keys end within QWA_PF_SEG_MAXPOS; otherwise 1, the units running in rounds.
// Measured, whole call, 1024 tokens (in-process A/B against rounds): Q8_0 -31 us at p0 = 0, -30 at 8192, -43 at
// 32768, -43 at 49152, -23 at 65536, +19 at 100000 (Q4_0 -48 at 32768, -12 at 100000; F16 -41 at 32768).  Past
// ~80000 positions a workgroup's three splits are long enough for the row blocks sharing an XCD's L2 to drift apart.
// (QWA_PF_UPW = 0: always rounds.)
constexpr int pf_units_per_wg(int nb, int npos) {
    const int nrb = pf_row_blocks(nb), ns = pf_splits(nb, npos);
    if (!QWA_PF_UPW || nrb <= PF_FEW || ns != 8 || npos > QWA_PF_SEG_MAXPOS) return 1;
    const int units = nrb * NKV * ns;
    return (units + 255) / 256;
}

// ---- the ring of fp16 tile images in LDS, and the exchange of a short pass's partial states through it
constexpr int PF_IMG_K = PF_TILE * HD * 2;      // bytes of the K part of an image: [32 keys][256 dims] fp16
constexpr int PF_IMG_BYTES = 2 * PF_IMG_K;      // K part, then V^T part [256 dims][32 keys] fp16
constexpr int PF_IMG_NBUF = 3;                  // images in LDS: the one computed on and two in flight
constexpr int PF_XCH_BYTES = 16 * HD * 2;       // a wave's area: 16 rows of 256 16-bit values
constexpr bool PF_XCH_FITS = PF_WAVES * PF_XCH_BYTES <= PF_IMG_NBUF * PF_IMG_BYTES;

}  // namespace qwa
