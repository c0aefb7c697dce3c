// Launch rules of the plane GEMM (plane_gemm_impl.hpp).
#include "plane_gemm_impl.hpp"

#include <algorithm>
#include <cmath>

namespace hos {
namespace {

// The tiles of the launches: rows / 32, columns / 128, slab depth, workgroups that share a CU, and what a launch
// costs per workgroup on it, fitted on the MI355X to 5,000 launches (M 64-8192, 24 weight shapes from 576×576 to
// 16384×2048, 1-16 splits, weights out of the caches; the fit is within 10-15%, and the tile it picks on average
// 1.5% slower than the best): a slab takes its latency or the CU's shared rate, whichever is longer, and each
// workgroup a prologue and epilogue.
struct TileCost {
  int tm, tn, bk, occ;
  double t0, lat, us, epi;  // µs: launch, slab latency, slab at full rate, prologue and epilogue
};
const TileCost kTiles3[] = {{4, 2, 32, 2, 0.0, 0.0, 1.172, 8.4},
                            {4, 1, 32, 3, 0.0, 0.76, 0.682, 5.63},
                            {2, 1, 64, 3, 2.5, 0.838, 0.733, 2.46},
                            {1, 1, 64, 4, 1.0, 0.696, 0.520, 2.08}};
const TileCost kTiles1[] = {{4, 2, 64, 2, 0.19, 0.582, 0.927, 8.41},
                            {4, 1, 64, 3, 0.09, 0.65, 0.512, 5.58},
                            {2, 1, 64, 3, 1.32, 0.545, 0.323, 2.89},
                            {1, 1, 64, 4, 1.1, 0.551, 0.254, 1.88}};
// mode 5 (the 128×256 tile's scaling does not fit the registers)
const TileCost kTiles5[] = {{4, 1, 32, 3, 0.0, 0.686, 0.685, 5.43},
                            {2, 1, 64, 3, 1.83, 0.168, 0.739, 2.73},
                            {1, 1, 64, 4, 2.08, 0.483, 0.396, 1.53}};

struct Pick {
  int tm, tn, bk, splits;
};

Pick plane_pick(long long M, long long N, long long C, int products, bool codes, bool can_split, bool wide_only,
                size_t ws_bytes) {
  Pick best{4, codes ? 1 : 2, 32, 1};
  double bt = 1e30;
  const TileCost* t0 = codes ? kTiles5 : (products == 1 ? kTiles1 : kTiles3);
  const int nt = codes ? 3 : 4;
  for (int ti = 0; ti < nt; ti++) {
    const TileCost& t = t0[ti];
    if (wide_only && t.tn != 2) continue;
    const int bk = C % t.bk == 0 ? t.bk : 32;
    const double rel = (double)bk / t.bk, us = t.us * rel * (products == 2 && !codes ? 2.0 / 3.0 : 1.0), lat = t.lat * rel;
    const long long tiles = (long long)ceil_div(M, 32 * t.tm) * ceil_div(N, 128 * t.tn);
    for (int s = 1; s <= 16; s *= 2) {
      if (s > 1 && (!can_split || C / s < 192 || (size_t)s * M * N * 4 > ws_bytes)) break;
      const double slabs = (double)ceil_div(C / bk, s);
      const long long n = (tiles * s + 255) / 256, full = n / t.occ, rest = n % t.occ;
      auto batch = [&](double w) { return std::max(lat, w * us) * slabs + t.epi * std::sqrt(w); };
      double est = t.t0 + (double)full * batch(t.occ) + (rest ? batch((double)rest) : 0.0);
      if (s > 1) est += 3.5 + (s + 1.0) * M * N * 4e-6 / 4.5;  // the partials' reduction
      if (est < bt) {
        bt = est;
        best = Pick{t.tm, t.tn, bk, s};
      }
    }
  }
  return best;
}

template <int NP>
void plane_dispatch(const Pick& k, const PlaneArgs& p, int row_tiles, const GemmEpi& e, float* ws, hipStream_t st) {
  constexpr int W = NP == 1 ? 64 : 32;  // slab depth of the 128-row tiles: two planes of 64 do not fit the registers
#define HOS_PG(TM_, TN_, BK_)                                                      \
  if (k.tm == TM_ && k.tn == TN_ && k.bk == BK_) {                                 \
    plane_launch<TM_, TN_, NP, BK_>(p, row_tiles, k.splits, e, ws, st);            \
    return;                                                                        \
  }
  if constexpr (NP != 5) { HOS_PG(4, 2, W) }
  HOS_PG(4, 1, W) HOS_PG(2, 1, 64) HOS_PG(1, 1, 64) HOS_PG(2, 1, 32) HOS_PG(1, 1, 32)
  if constexpr (W != 32) { HOS_PG(4, 2, 32) HOS_PG(4, 1, 32) }
#undef HOS_PG
  throw Error(HOS_E_INVALID, "plane gemm: no kernel for the chosen tile");
}

// One-slab launches of few workgroups (plane_small_kernel): measured faster than every tile and split of the others up
// to a workgroup per CU and 36 steps of 32 (M 16-256, 576 × 576: 6.5-7.0 against 8.3 µs; 960 × 576: 6.6 against 8.4;
// 1152 × 896: 8.9 against 10.3; at 1536 columns of contraction 12.1 against 9.5).
bool plane_small(long long M, long long N, long long C) {
  return C <= 1152 && (long long)ceil_div(M, 32) * ceil_div(N, 32) <= 256;
}

// What a launch multiplies: the precision mode, with mode 5 its three-product form where the planes are not codes.
int plane_np(int passes, const WPlanes& pl) { return pl.scale ? 5 : (passes == 5 ? 3 : passes); }

void plane_run(int np, const Pick& k, const PlaneArgs& p, int row_tiles, const GemmEpi& e, float* ws, hipStream_t st) {
  switch (np) {
    case 1: plane_dispatch<1>(k, p, row_tiles, e, ws, st); break;
    case 2: plane_dispatch<2>(k, p, row_tiles, e, ws, st); break;
    case 4: plane_dispatch<4>(k, p, row_tiles, e, ws, st); break;
    case 5: plane_dispatch<5>(k, p, row_tiles, e, ws, st); break;
    default: plane_dispatch<3>(k, p, row_tiles, e, ws, st); break;
  }
  HOS_HIP_CHECK(hipGetLastError());
}
void plane_run_small(int np, const PlaneArgs& p, const GemmEpi& e, hipStream_t st) {
  switch (np) {
    case 1: plane_small_launch<1>(p, e, st); break;
    case 2: plane_small_launch<2>(p, e, st); break;
    case 4: plane_small_launch<4>(p, e, st); break;
    case 5: plane_small_launch<5>(p, e, st); break;
    default: plane_small_launch<3>(p, e, st); break;
  }
  HOS_HIP_CHECK(hipGetLastError());
}

template <int R>
void plane_chain_launch(int splits, const PlaneArgs& p, const GemmEpi& e, hipStream_t st) {
  const dim3 grid(p.N / 16, ceil_div(p.M, 16 * R));
  switch (splits) {
    case 1: plane_chain_kernel<1, R><<<grid, 256, 0, st>>>(p, e); break;
    case 2: plane_chain_kernel<2, R><<<grid, 512, 0, st>>>(p, e); break;
    default: plane_chain_kernel<4, R><<<grid, 1024, 0, st>>>(p, e); break;
  }
}
// The split of the dequantizing kernel's 64×64 tiles, whose sums plane_chain_kernel repeats.
int chain_splits(long long M, long long N, long long C, bool whole) {
  const long long tiles = (long long)ceil_div(M, 64) * ceil_div(N, 64), nslab = C / 64;
  int s = 1;
  while (!whole && tiles * s < 320 && nslab / (s * 2) >= 8) s *= 2;
  return ceil_div(nslab, ceil_div(nslab, s));
}

}  // namespace

// Up to 512 workgroups of 32×32 outputs (128 rows: a 3072-wide projection has 384), where that kernel takes 64×64 tiles
// of 64-deep slabs and at most four splits, all of them full.
bool plane_chain(long long M, long long N, long long C) {
  if (C % 64 != 0 || C >= 4096 || N % 32 != 0 || (long long)ceil_div(M, 32) * ceil_div(N, 32) > 512) return false;
  const int s = chain_splits(M, N, C, false);
  return s == 1 || s == 2 || s == 4;
}

bool plane_gemm_wanted(const QWeight& w, bool dx, int passes, long long M, int groups) {
  const long long C = dx ? w.rows / groups : w.cols;
  if (C % 32 != 0 || w.cols % 32 != 0) return false;
  if (groups > 1) return true;
  // The vocabulary-wide contraction of the head's dX re-reads its operands more than it multiplies, and the planes are
  // 3.6 times the Q8_0 weight: 1087 µs at best (mode 4, 2048 × 896 × 151936) against 1001 on the quantized weight.
  if (dx && C >= 32768) return false;  // (which also bounds the build's grid)
  // Few rows against a wide weight stream it: 4 bytes a weight against 0.7-1.1 (16-64 rows, 8192 × 2048: 15.8-16.9 µs at
  // one pass against 14.5-16.7); up to 4096 columns, and from 96 rows on, the planes are the faster (8-64 rows: 768²
  // 6.7-8.3 against 10.6-11.4, 2048 × 8192 three products 25-30 against 32-36).
  const long long N = dx ? w.cols : w.rows / groups;
  return M >= 96 || (M >= 8 && N <= 4096);
}

bool launch_plane_gemm(bool dx, const QWeight& w, H16 a, long long lda, long long M, GemmEpi epi, float* ws,
                       size_t ws_bytes, int passes, hipStream_t st) {
  const WPlanes& pl = w.pl[dx];
  if (!has_planes(pl, dx, passes) || !plane_gemm_wanted(w, dx, passes, M)) return false;
  const long long N = dx ? w.cols : w.rows, C = dx ? w.rows : w.cols;
  if (lda % 8 != 0 || lda >= (1 << 23) || epi.rank < 0 || epi.rank > 128) return false;
  if (epi.rank > 0 && epi.ustep > 0 && (epi.ub0 % 64 != 0 || (epi.ub1 < N && epi.ub1 % 64 != 0))) return false;
  if ((passes == 2 || passes == 3 || passes == 5) && !a.lo) return false;
  if (epi.rstat && (dx || pl.scale)) return false;
  if (epi.rank > 0 && !epi.Lf && !prepare_rank(epi, a.rinv, M, N, ws, &ws_bytes, st)) return false;
  const int np = plane_np(passes, pl), products = np == 1 ? 1 : (np == 3 ? 3 : 2);
  PlaneArgs p{a.data, a.lo, a.rinv, lda, (int)M, (int)N, (int)C, (int)C, pl.p, (C / 32) * 512LL * pl.planes, 512 * pl.planes,
              (int)((N + 15) / 16), 1, nullptr, 0, pl.scale};
  Pick k{1, 1, 32, 1};
  if (np == 3 && !epi.rstat && plane_chain(M, N, C)) {
    const int s = chain_splits(M, N, C, epi.rank > 32 || epi.ustep > 0);
    p.per = ceil_div(C / 64, s) * 64;
    if ((long long)ceil_div(M, 16) * (N / 16) <= (s == 4 ? 256 : 512))
      plane_chain_launch<1>(s, p, epi, st);
    else
      plane_chain_launch<2>(s, p, epi, st);
    HOS_HIP_CHECK(hipGetLastError());
  } else if (!epi.rstat && plane_small(M, N, C)) {
    plane_run_small(np, p, epi, st);
  } else {
    k = plane_pick(M, N, C, products, np == 5, !epi.rstat, epi.rstat != nullptr, ws_bytes);
    if (np != 1 && k.tm == 4) k.bk = 32;
    p.per = ceil_div(C / k.bk, k.splits) * k.bk;
    k.splits = ceil_div(C, p.per);
    const int row_tiles = ceil_div(M, 32 * k.tm);
    p.gm = std::min(row_tiles, 8);
    plane_run(np, k, p, row_tiles, epi, ws, st);
  }
  if (epi.defer) {
    HOS_REQUIRE(k.splits == 1 || (!epi.bias && !epi.accumulate), HOS_E_INVALID,
                "qgemm: a deferred reduction takes no bias and no accumulation");
    *epi.defer = k.splits;
  } else if (k.splits > 1) {
    launch_qgemm_split_reduce(ws, k.splits, M, (int)N, a.rinv, epi, st);
  }
  return true;
}

bool launch_plane_gemm_grouped(bool dx, const QWeight& w, GroupSched gs, H16 a, long long lda, GemmEpi epi, int passes,
                               hipStream_t st) {
  const WPlanes& pl = w.pl[dx];
  if (!has_planes(pl, dx, passes) || lda % 8 != 0 || lda >= (1 << 23) || epi.rank != 0 || epi.rstat) return false;
  if ((passes == 2 || passes == 3 || passes == 5) && !a.lo) return false;
  const long long er = w.rows / gs.n_experts, N = dx ? w.cols : er, C = dx ? er : w.cols;
  const long long nstride = (C / 32) * 512LL * pl.planes;
  const int nb = (int)((N + 15) / 16);
  PlaneArgs p{a.data, a.lo, a.rinv, lda, 0, (int)N, (int)C, (int)C, pl.p, nstride, 512 * pl.planes, nb, 1, gs.tiles,
              nb * nstride, pl.scale};
  static_assert(GROUP_BM == 128, "the schedule's row tiles are the kernel's");
  const int np = plane_np(passes, pl);
  plane_run(np, Pick{4, N >= 512 && np != 5 ? 2 : 1, np == 1 && C % 64 == 0 ? 64 : 32, 1}, p, gs.max_tiles, epi, nullptr, st);
  return true;
}

}  // namespace hos
