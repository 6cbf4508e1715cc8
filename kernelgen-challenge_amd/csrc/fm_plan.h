// fm_plan.h -- host-side argument validation and launch planning of the gfx950
// fused_moe kernels. Plain C++ (no HIP): the same code is compiled into the HIP
// library and into a g++-built host test library.
#pragma once

#include <math.h>
#include <stddef.h>
#include <stdint.h>

#include "fused_moe.h"

namespace fm {

constexpr int kMaxExperts = 256;
constexpr int kMaxTopk = 32;
constexpr int kFusedTokens = 16;  // routing and plan in one launch up to this many tokens

constexpr int kTileRows = 256;    // pairs per tile of fm_gemm_kernel at most
constexpr int kTileCols = 256;    // weight rows per wide tile
constexpr int kNarrowCols = 64;   // weight rows per narrow tile
constexpr int kCus = 256;         // MI355X
constexpr int kXcds = 8;

struct Plan {
  int64_t P;            // pairs = M * topk
  int64_t nonempty;     // experts with a pair, at most
  bool gemm;            // fm_gemm_kernel (else fm_stream_kernel or fm_skinny_kernel)
  int tile_rows;        // pairs per tile
  int narrow_rows;      // gemm: tiles of at most this many pairs run as narrow ones
  int pb;               // not gemm: 16-pair blocks per tile (1, 2 or 4)
  int64_t max_tiles;    // upper bound on sum_e ceil(count_e / tile_rows)
  int tokens_per_wg, route_wgs;  // fm_route_kernel: at most 256 work-groups (0: fused)
  size_t ids_off, wts_off, hist_off, sorted_off, tiles_off, inter_off, y_off, bytes;
};

inline size_t round_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// The kernel and its tiles, from the average pairs per expert n (an expert's
// count spreads about sqrt(n) around it) and the launch's work items per CU.
// fm_gemm_kernel runs one work-group per CU, so what counts is how many rounds
// of items there are and how long one is. Measured whole calls (us), wide 256 /
// wide 128 / narrow, the chosen one in brackets:
//   K = 2048, N = 1024, E = 8, topk = 2: M = 256 57 / 56 / [39], M = 512
//   65 / 63 / [45], M = 700 74 / 61 / [51], M = 1024 89 / [65] / 87, M = 2048
//   [93] / 109 / 123, M = 3000 [104] / 122 / 162;
//   E = 64, topk = 6: M = 512 [198] / 198 / 211, M = 1024 [219] / 218 / 248;
//   K = 4096, N = 2048, E = 8, topk = 2, M = 700: 147 / [132] / 166.
//   Short last tiles narrow against wide: M = 4096, E = 8 [134] / 175; M =
//   1500, K = 2048, N = 1408, E = 16, topk = 4 169 / [164]; M = 4001, E = 64,
//   topk = 6 481 / [385].
// The streamed tiles win where the weights of many experts are the traffic
// (E = 64, topk = 6: M = 64 152 against 183, M = 8 94 against 122) and up to 12
// pairs per expert in general (E = 8, topk = 2, M = 16 29 against 30; K = 4096,
// N = 512, E = 32, topk = 4, M = 60 88 against 102). Past that they need two
// pair blocks per tile, and fm_gemm_kernel wins with at most one narrow item
// per CU (E = 8, topk = 2, M = 64 34 against 41) or short K loops in the down
// GEMM (N <= 512: E = 128, topk = 8, M = 200 97 against 117), and from 8
// pairs where N is not a multiple of 256 (E = 16, topk = 4, N = 1408, M = 60 79
// against 90).
inline void choose_tiles(const fm_args* a, Plan& p) {
  const double n = double(p.P) / double(a->E), sd = sqrt(n);
  auto tiles = [&](double pairs, int rows) { return double(p.nonempty) * ceil(pairs / rows); };
  const double cols = double(a->N) / (kTileCols / 2), narrow = double(a->N) / (kNarrowCols / 2);
  const bool one_round = tiles(n + 1.5 * sd, kTileRows) * narrow <= kCus;
  p.tile_rows = kTileRows;
  p.narrow_rows = 0;
  if (a->flags & (FM_FLAG_LARGE_TILES | FM_FLAG_BIG_TILES))
    p.gemm = true;
  else if (a->flags & FM_FLAG_SMALL_TILES)
    p.gemm = false;
  else
    p.gemm = n > 24.0 || (n > 12.0 && (one_round || a->N <= 512)) ||
             (a->N % 256 != 0 && n > 8.0);
  // 16 or 32 pairs per small tile (64 only when forced)
  p.pb = n > 24.0 && a->N % 256 == 0 ? 4 : n > 12.0 ? 2 : 1;
  if (!p.gemm) {
    p.tile_rows = 16 * p.pb;
  } else if (a->flags & FM_FLAG_LARGE_TILES) {
    p.tile_rows = 128;
  } else if (one_round && (a->flags & FM_FLAG_BIG_TILES) == 0) {
    p.narrow_rows = kTileRows;
  } else if (tiles(n + 0.5 * sd, 128) * cols <= kCus && (a->flags & FM_FLAG_BIG_TILES) == 0) {
    p.tile_rows = 128;
  } else {
    // an expert's last tile goes narrow when it has at most 128 pairs, if that
    // saves a round of wide items and is itself at most two rounds
    const double wide = double(p.nonempty) * floor((n + sd + 127.0) / kTileRows) * cols;
    if (ceil(tiles(n + sd, kTileRows) * cols / kCus) > ceil(wide / kCus) &&
        double(p.nonempty) * narrow <= 2 * kCus)
      p.narrow_rows = 128;
  }
}

inline Plan make_plan(const fm_args* a) {
  Plan p{};
  p.P = a->M * a->topk;
  p.nonempty = a->E < p.P ? a->E : p.P;
  choose_tiles(a, p);
  p.max_tiles = p.P / p.tile_rows + p.nonempty;
  p.tokens_per_wg = int((a->M + 4095) / 4096) * 16;
  p.route_wgs = a->M <= kFusedTokens ? 0 : int((a->M + p.tokens_per_wg - 1) / p.tokens_per_wg);
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off = round_up(off + bytes, 256);
    return o;
  };
  p.ids_off = take(size_t(p.P) * 4);
  p.wts_off = take(size_t(p.P) * 4);
  p.hist_off = take(size_t(p.route_wgs) * size_t(a->E) * 4);
  p.sorted_off = take(size_t(p.P) * 4);
  p.tiles_off = take(16 + size_t(p.max_tiles) * 16);  // count, then int4 per tile
  p.inter_off = take(size_t(p.P) * size_t(a->N) * 2);
  p.y_off = take(size_t(p.P) * size_t(a->K) * 2);
  p.bytes = off;
  return p;
}

inline int validate(const fm_args* a) {
  if (a == nullptr) return FM_EINVAL;
  if (a->M < 0 || a->K <= 0 || a->N <= 0 || a->E <= 0 || a->topk <= 0) return FM_EINVAL;
  if (a->topk > a->E) return FM_EINVAL;
  if (a->E > kMaxExperts || a->topk > kMaxTopk) return FM_EUNSUPPORTED;
  if (a->K % kTileCols != 0 || a->N % (kTileCols / 2) != 0) return FM_EUNSUPPORTED;
  const uint32_t tile_flags = a->flags & (FM_FLAG_LARGE_TILES | FM_FLAG_SMALL_TILES |
                                          FM_FLAG_BIG_TILES);
  if ((a->flags & ~(tile_flags | FM_FLAG_ORDERED_SUM)) != 0 ||
      (tile_flags & (tile_flags - 1)) != 0)
    return FM_EINVAL;  // unknown bits, or more than one tile choice
  if (a->M == 0) return FM_OK;
  if (!a->hidden || !a->w1 || !a->w2 || !a->score || !a->out) return FM_EINVAL;
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  if (!al16(a->hidden) || !al16(a->w1) || !al16(a->w2) || !al16(a->out)) return FM_EINVAL;
  if ((reinterpret_cast<uintptr_t>(a->score) & 1u) != 0) return FM_EINVAL;
  if (a->s_hidden < a->K || a->s_hidden % 8 != 0 || a->s_out < a->K || a->s_out % 8 != 0 ||
      a->s_score < a->E)
    return FM_EINVAL;
  // 32-bit byte offsets: rows of hidden, of one expert's weights and of the
  // intermediate buffers
  const int64_t lim = int64_t(UINT32_MAX) - 4096;
  if ((a->M - 1) * a->s_hidden * 2 + a->K * 2 > lim) return FM_EUNSUPPORTED;
  if (2 * a->N * a->K * 2 > lim) return FM_EUNSUPPORTED;
  if (a->M * a->topk * a->N * 2 > lim || a->M * a->topk * a->K * 2 > lim) return FM_EUNSUPPORTED;
  return FM_OK;
}

}  // namespace fm
