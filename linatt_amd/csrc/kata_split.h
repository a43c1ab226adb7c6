// Work split of the KATA attention passes for launches with few workgroups.
//
// Unsplit, one workgroup walks every key tile of its 128 queries (forward),
// a serial chain of up to T / 64 tiles: at B1 H12 T3001 that is 288 chains
// on 256 CUs, the longest 47 tiles.  The score has no softmax maximum, so the
// sums of disjoint key ranges simply add: the split gives every tile list
// longer than L to several workgroups of at most L tiles each, whose float32
// partial sums a second launch adds in order.
#pragma once

#include <hip/hip_runtime.h>

namespace linatt {

// pieces of a list of n tiles cut into runs of at most L (all but the last
// equally long, none empty)
__host__ __device__ inline int split_pieces(int n, int L) { return (n + L - 1) / L; }

// 64-key tiles of query tile qt (128 queries, causal)
__host__ __device__ inline int kata_key_tiles(int qt, int T) {
  const int s_end = 128 * qt + 128 < T ? 128 * qt + 128 : T;
  return (s_end + 63) / 64;
}
inline int kata_fwd_items(int T, int L) {
  int n = 0;
  for (int qt = 0; qt < (T + 127) / 128; ++qt) n += split_pieces(kata_key_tiles(qt, T), L);
  return n;
}

struct SplitRun {
  int tile, piece, pieces, lo, hi;  // tiles [lo, hi) of list `tile`
};
// item j of a head's (list, piece) pairs, longest lists first
__device__ __forceinline__ SplitRun kata_fwd_run(int j, int nqt, int T, int L) {
  SplitRun r;
  r.tile = nqt - 1;
  int n = kata_key_tiles(r.tile, T);
  r.pieces = split_pieces(n, L);
  while (j >= r.pieces) {
    j -= r.pieces;
    --r.tile;
    n = kata_key_tiles(r.tile, T);
    r.pieces = split_pieces(n, L);
  }
  r.piece = j;
  const int per = (n + r.pieces - 1) / r.pieces;
  r.lo = j * per;
  r.hi = r.lo + per < n ? r.lo + per : n;
  return r;
}

// floats of a partial block of 32 queries: 32 x 64 sums, a den per lane (float16:
// per lane of the lower half, the row scale in the upper)
constexpr int kFwdPart = 32 * 64 + 64;
// most pieces of one list (the partial blocks reserved for it)
constexpr int kMaxPieces = 16;

// A workgroup's time per tile alone on its CU and with the CU full (slots / 256
// workgroups sharing it), and what a split adds to the call: once, per piece of
// the longest list (the second launch adds a block's pieces one after another),
// and the part of a run that is left uneven at the end.  A split has to be
// modelled below `win` of the unsplit launch.
struct TileTime {
  double solo_us, full_us;
  int slots;
  double split_us, piece_us, tail, win;
};

// Tiles per workgroup with the least modelled time, 0 to leave the launch
// unsplit.  Modelled as the longer of the longest list at the solo rate and
// the whole work over all slots at the full rate; for a split the rate of its
// runs is 1.3 solo and `tail` of a run is left uneven at the end, and it adds
// split_us (the second launch, and the first tile's latency in every workgroup),
// piece_us per piece and the partial blocks written and read at 4.5 TB/s.
template <typename Lists>
inline int best_split(const Lists& lists, int64_t heads, int nlists, const TileTime& tt, double list_bytes) {
  int64_t units = 0;
  int longest = 0;
  for (int i = 0; i < nlists; ++i) {
    const int n = lists(i);
    units += n;
    if (n > longest) longest = n;
  }
  const double all = (double)(units * heads) * tt.full_us / tt.slots;
  auto longer = [](double a, double b) { return a > b ? a : b; };
  double best = tt.win * longer(longest * tt.solo_us, all);
  int L_best = 0;
  for (int L = 1; L < longest; L = L < 4 ? L + 1 : L + L / 4) {
    if (split_pieces(longest, L) > kMaxPieces) continue;
    int64_t part = 0;
    for (int i = 0; i < nlists; ++i) {
      const int p = split_pieces(lists(i), L);
      if (p > 1) part += p;
    }
    const double t = longer(1.3 * L * tt.solo_us, all + tt.tail * L * tt.solo_us) + tt.split_us +
                     split_pieces(longest, L) * tt.piece_us + (double)(part * heads) * list_bytes * (2. / 4.5e6);
    if (t < best) {
      best = t;
      L_best = L;
    }
  }
  return L_best;
}

// Forward, per 64-key tile of 128 queries (measured, B1 to B8, H = 12).  16-bit:
// three workgroups per CU at dk = 64, two at dk = 128; fp16 adds the row
// rescaling.  float32: 32 x 32 x 2 products, two workgroups per CU.
// Unsplit -> split, us: float32 B1 H4 T512 48 -> 17; fp16 M = 2 B1 H12 T3001
// 57 -> 38; bf16 B1 H12 T2048: sum M = 4 75 -> 39, decayed dk = 128 55 -> 31.
// The second launch costs 0.2 to 0.4 us per piece; without that term the rule took
// runs of one or two tiles that were slower than no split (bf16 M = 1 B1 H1 T1000:
// unsplit 13.3, 16 pieces 15.5, six 10.2; dk = 128 H8 T1000: 17.5, eight pieces
// 19.3, six 15.0).  Left unsplit: concat M = 4 at B2 T2048 (30 against 33 at the
// best run length), B4 (39 against 48); and, where the model is on the safe
// side, B1 H12 T2048 (28 against 23), M = 1 T1500 (18 against 17).
inline TileTime kata_fwd_tile_time(int elt_bytes, bool fp16, int dk, int M, bool sum, bool decay) {
  if (elt_bytes == 4) return {6., 14., 512, 8., 0., 0.5, 0.9};
  double solo = sum && M > 1 ? (M == 2 ? 1.3 : 2.4) : 0.85;
  if (dk == 128) solo *= decay ? 1.4 : 1.35;
  if (decay) solo *= 1.4;
  if (fp16) solo *= 1.4;
  const bool wide = dk == 128;
  return {solo, (wide ? 1.4 : 2.2) * solo, wide ? 512 : 768, 6.6, 0.2, 0.55, 0.92};
}
inline int kata_fwd_split(int64_t BH, int T, const TileTime& tt) {
  return best_split([&](int qt) { return kata_key_tiles(qt, T); }, BH, (T + 127) / 128, tt, 4. * kFwdPart * 4);
}
// partial blocks of a forward split by L, bytes
inline size_t kata_fwd_part_bytes(int64_t BH, int T, int L) {
  const int nqt = (T + 127) / 128;
  return (size_t)split_pieces(kata_key_tiles(nqt - 1, T), L) * BH * 4 * nqt * kFwdPart * sizeof(float);
}

// dk/dv (bf16, dk = 64, no decay): the list of key tile st (128 keys) is the
// query tiles of 64 at or after it, over the G query heads of its kv head.
__host__ __device__ inline int kata_query_tiles(int st, int T, int G) { return G * ((T + 63) / 64 - 2 * st); }
inline int kata_dkdv_items(int T, int G, int L) {
  int n = 0;
  for (int st = 0; st < (T + 127) / 128; ++st) n += split_pieces(kata_query_tiles(st, T, G), L);
  return n;
}
// item j of a kv head, longest lists (first key tiles) first
__device__ __forceinline__ SplitRun kata_dkdv_run(int j, int T, int G, int L) {
  SplitRun r;
  r.tile = 0;
  int n = kata_query_tiles(0, T, G);
  r.pieces = split_pieces(n, L);
  while (j >= r.pieces) {
    j -= r.pieces;
    ++r.tile;
    n = kata_query_tiles(r.tile, T, G);
    r.pieces = split_pieces(n, L);
  }
  r.piece = j;
  const int per = (n + r.pieces - 1) / r.pieces;
  r.lo = j * per;
  r.hi = r.lo + per < n ? r.lo + per : n;
  return r;
}
// floats of a wave's partial block: 32 keys x (64 dk + 64 dv)
constexpr int kDkdvPart = 32 * 128;
__host__ __device__ inline int64_t dkdv_part_offset(int piece, int nbk, int bh, int nkt, int blk) {
  return (((int64_t)piece * nbk + bh) * (4 * nkt) + blk) * kDkdvPart;
}
// Per 64-query tile of 128 keys, two workgroups per CU.  Whole backward (dq and
// dk/dv), unsplit -> split, us: sum M = 2 B6 T1403 HQ12 H4 175 -> 153; concat
// M = 4 B1 H12 T2048 103 -> 86, B2 HQ16 H8 T2048 161 -> 130, B1 H4 T1000 58 -> 42;
// M = 1 B1 HQ8 H4 T3000 152 -> 87; sum M = 4 B1 H12 T2048 261 -> 202; with the
// output norm B1 H12 T2048 concat M = 4 111 -> 93, sum M = 4 269 -> 210.  Left
// unsplit: concat M = 4 B4 T1024 (63 against 67 at the best run length), B8 T2048
// (240 against 262); and, where split_us is on the safe side (it was fitted to a
// second launch 5 to 10 us slower than this one), M = 1 B1 H8 T1500 (58 against 50),
// concat M = 4 B1 H8 T700 (44 against 36).
inline TileTime kata_dkdv_tile_time(int M, bool sum) {
  const double full = sum && M > 1 ? (M == 2 ? 3.2 : 7.0) : M == 1 ? 2.1 : M == 2 ? 2.3 : 2.8;
  return {full / 1.6, full, 512, 13., 0., 0.5, 0.9};
}
inline int kata_dkdv_split(int64_t BH, int T, int G, const TileTime& tt) {
  return best_split([&](int st) { return kata_query_tiles(st, T, G); }, BH, (T + 127) / 128, tt, 4. * kDkdvPart * 4);
}
inline size_t kata_dkdv_part_bytes(int64_t BH, int T, int G, int L) {
  const int nkt = (T + 127) / 128;
  return (size_t)split_pieces(kata_query_tiles(0, T, G), L) * BH * 4 * nkt * kDkdvPart * sizeof(float);
}

}  // namespace linatt
