// GEMM of an fp16 row-scaled activation operand against a frozen weight kept as fp16 planes in MFMA fragment order
// (WPlanes, planes.hip): out[m][n] = Σ_c A[m][c]·B(n, c), in precision modes 1-4 of qgemm_impl.hpp, with the planes
// qgemm_impl.hpp forms in registers (the same fp16 values), so a launch computes the same products.
//
// What bounds it: with real operands the card's power limit, not the MFMA issue rate — 4096³ at three products ran 1080
// TFLOP/s on random values and 1500 on zeros — so the kernel is built to move few bytes per product:
//  - v_mfma_f32_16x16x32_f16 rather than 32x32x16: half the accumulator traffic per product (a register-only loop on
//    random values holds 1900 against 1660 TFLOP/s; this kernel 8192×8192×2048, three products: 617 against 716 µs).
//  - The four waves of a workgroup stand side by side along the columns: a wave's weight fragments go straight from L2 to
//    its registers (1 KB contiguous loads, no other wave needs them), only the activation tile goes through LDS
//    (double-buffered, read without bank conflicts). Dequantizing both planes and passing them through LDS in every
//    launch cost the former kernel its LDS bandwidth: 64×64 wave tiles at three products need all 128 B/clk.
//  - 128×256 tiles (wave tiles 128×64, 244 registers, two workgroups per CU) where the shape fills the chip with them;
//    smaller tiles and split contractions otherwise (plane_gemm.hip).
// Against the dequantizing kernel on the MI355X: forward 8192×8192×2048 Q4_K, three products and a rank-32 term 889 ->
// 640 µs; 4096³ dX one pass 178 -> 131 µs; Qwen2.5-0.5B's layer GEMMs (2048 rows) 610 -> 500 µs a layer.
#pragma once
#include "kernels.hpp"

namespace hos {
namespace {

struct PlaneArgs {
  const _Float16* A;
  const _Float16* Alo;
  const float* rinv;
  long long lda;
  int M, N, C, per;            // per: contraction length of one split
  const _Float16* W;           // fragment (nb, ks, plane) at W + nb·nstride + ks·kstride + plane·512
  long long nstride;           // halves per 16-column block
  int kstride, nb;             // halves per 32-deep step; 16-column blocks present
  int gm;                      // row tiles per group of the tile order
  const int* tiles;            // grouped launch: (expert, first row, rows) per row tile
  long long wexp;              // halves of one expert's planes
  const float* S = nullptr;    // mode 5: block scales, 16 columns of one 32-deep step together (nb, ks, column)
};

template <int TM, int TN, int NP, int BK>
struct PGeo {
  static constexpr int BM = 32 * TM, BN = 128 * TN, CH = BK / 8, KS = BK / 32;
  static constexpr int NA = (NP == 2 || NP == 3 || NP == 5) ? 2 : 1, NB = (NP == 3 || NP == 4) ? 2 : 1;
  static constexpr int AT = BM * BK;                     // halves of one staged A plane
  static constexpr int AV = (BM * CH + 255) / 256;       // 16-byte pieces per thread per plane
  static constexpr int BUF = NA * AT;
  static constexpr int TS = 40;                          // f32 row stride of a staged output tile
  static constexpr int SMEM = (2 * BUF * 2 > 4 * 32 * TS * 4) ? 2 * BUF : 4 * 32 * TS * 2;  // halves
};

// Position of 16-byte chunk c of row r in a staged A plane (rows BK halves long, unpadded): the chunks of a row are
// permuted so that any 16 (BK 32) or 8 (BK 64) consecutive rows' pieces of one chunk fall on different banks.
template <int BK>
__device__ __forceinline__ int a_pos(int r, int c) {
  if constexpr (BK == 32) return r * 32 + ((c ^ ((r >> 2) & 3)) << 3);
  else return r * 64 + ((c ^ ((r >> 1) & 7)) << 3);
}

template <int TM, int TN, int NP, int BK>
__global__ void __launch_bounds__(256, 2) plane_gemm_kernel(PlaneArgs p, GemmEpi epi, float* __restrict__ ws) {
  using G = PGeo<TM, TN, NP, BK>;
  constexpr bool ALO = G::NA == 2, BLO = G::NB == 2, CODES = NP == 5;
  __shared__ __attribute__((aligned(16))) _Float16 smem[G::SMEM];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  int mt, nt;
  if (p.tiles) {
    const int* tl = p.tiles + 3 * blockIdx.y;
    const int e = tl[0];
    if (e < 0) return;
    const long long r0 = tl[1];
    p.M = tl[2];
    p.A += r0 * p.lda;
    if (ALO) p.Alo += r0 * p.lda;
    p.rinv += r0;
    epi.out += r0 * epi.ldo;
    if (epi.resid) epi.resid += r0 * epi.ldo;
    p.W += e * p.wexp;
    if (CODES) p.S += e * (p.wexp / 32);
    mt = 0;
    nt = blockIdx.x;
  } else {
    // XCD runs (workgroup ids go round-robin over the 8 XCDs), each run walking groups of gm row tiles by all column
    // tiles, rows fastest: the tiles an XCD runs together form a near-square block of the output.
    const int X = gridDim.x, Y = gridDim.y, T = X * Y, full = T & ~7;
    int t = blockIdx.x + X * blockIdx.y;
    if (t < full) t = (t & 7) * (full >> 3) + (t >> 3);
    const int g = t / (p.gm * X), r0 = g * p.gm, gh = min(p.gm, Y - r0), u = t - r0 * X;
    mt = r0 + u % gh;
    nt = u / gh;
  }
  const int m0 = mt * G::BM, n0 = nt * G::BN + wave * 32 * TN;
  const int zsp = blockIdx.z;
  const int cbeg = zsp * p.per, cend = min(p.C, cbeg + p.per);
  const int nslab = (cend - cbeg) / BK;

  constexpr int TR = 2 * TM, TC = 2 * TN;  // 16×16 output tiles of a wave
  f4v acc[TR][TC];
#pragma unroll
  for (int i = 0; i < TR; i++)
#pragma unroll
    for (int j = 0; j < TC; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[i][j][r] = 0.0f;

  // this thread's 16-byte pieces of an A slab: byte offsets from the tile's first row (rows past M re-read row M-1:
  // they only feed output rows that are never stored)
  uint32_t aoff[G::AV];
#pragma unroll
  for (int v = 0; v < G::AV; v++) {
    const int idx = tid + 256 * v, row = min(idx / G::CH, min(G::BM, p.M - m0) - 1), cv = idx % G::CH;
    aoff[v] = (uint32_t)row * (uint32_t)p.lda * 2u + 16u * cv;
  }
  const char* abase = (const char*)(p.A + (long long)m0 * p.lda + cbeg);
  const char* albase = ALO ? (const char*)(p.Alo + (long long)m0 * p.lda + cbeg) : nullptr;
  // this wave's weight fragments, 1 KB each: lane l holds column l & 15, contraction 8·(l >> 4) .. +7
  const char* wbase[TC];
#pragma unroll
  for (int j = 0; j < TC; j++)
    wbase[j] = (const char*)(p.W + (long long)min(n0 / 16 + j, p.nb - 1) * p.nstride + (long long)(cbeg / 32) * p.kstride);
  const uint32_t loff = lane * 16;
  const float* sbase[CODES ? TC : 1];  // mode 5: this lane's column of the block scales
  if constexpr (CODES)
#pragma unroll
    for (int j = 0; j < TC; j++)
      sbase[j] = p.S + ((long long)min(n0 / 16 + j, p.nb - 1) * (p.C / 32) + cbeg / 32) * 16 + (lane & 15);

  // One slab in flight: this thread's pieces of A (to LDS later) and this wave's fragments.
  struct Slab {
    h8 a[G::AV], al[ALO ? G::AV : 1];
    h8 h[G::KS][TC], l[BLO ? G::KS : 1][BLO ? TC : 1];
    float d[CODES ? G::KS : 1][CODES ? TC : 1];
  };
  auto load = [&](Slab& S, int s) {
    s = min(s, nslab - 1);  // past the end: a harmless re-read of the last slab
    const char* a = abase + (long long)s * (BK * 2);
    const char* al = ALO ? albase + (long long)s * (BK * 2) : nullptr;
#pragma unroll
    for (int v = 0; v < G::AV; v++) {
      S.a[v] = *(const h8*)(a + aoff[v]);
      if constexpr (ALO) S.al[v] = *(const h8*)(al + aoff[v]);
    }
#pragma unroll
    for (int k = 0; k < G::KS; k++)
#pragma unroll
      for (int j = 0; j < TC; j++) {
        const char* w = wbase[j] + (long long)(s * G::KS + k) * p.kstride * 2;
        S.h[k][j] = *(const h8*)(w + loff);
        if constexpr (BLO) S.l[k][j] = *(const h8*)(w + 1024 + loff);
        if constexpr (CODES) S.d[k][j] = sbase[j][(s * G::KS + k) * 16];
      }
  };
  auto store_a = [&](const Slab& S, int buf) {
    _Float16* d = smem + buf * G::BUF;
#pragma unroll
    for (int v = 0; v < G::AV; v++) {
      const int idx = tid + 256 * v, row = idx / G::CH, cv = idx % G::CH;
      if (G::BM * G::CH % 256 == 0 || row < G::BM) {
        *(h8*)(d + a_pos<BK>(row, cv)) = S.a[v];
        if constexpr (ALO) *(h8*)(d + G::AT + a_pos<BK>(row, cv)) = S.al[v];
      }
    }
  };
  // The A fragments of IG 16-row blocks (read from LDS) are one group ahead of the products, which go pass by pass over
  // the group's tiles, so consecutive MFMAs go to different accumulators.
  constexpr int IG = TC >= 4 ? 1 : 2, NG = G::KS * TR / IG;
  struct AFrag {
    h8 h[IG], l[ALO ? IG : 1];
  };
  auto read_a = [&](AFrag& f, int g, int buf) {
    const _Float16* as = smem + buf * G::BUF;
    const int k = g / (TR / IG), i0 = g % (TR / IG) * IG;
#pragma unroll
    for (int i = 0; i < IG; i++) {
      const int o = a_pos<BK>(16 * (i0 + i) + (lane & 15), 4 * k + (lane >> 4));
      f.h[i] = *(const h8*)(as + o);
      if constexpr (ALO) f.l[i] = *(const h8*)(as + G::AT + o);
    }
  };
  auto scale_in = [&](const Slab& B, const f4v (&t)[IG][TC], int g) {
    const int k = g / (TR / IG), i0 = g % (TR / IG) * IG;
#pragma unroll
    for (int i = 0; i < IG; i++)
#pragma unroll
      for (int j = 0; j < TC; j++)
#pragma unroll
        for (int r = 0; r < 4; r++)
          acc[i0 + i][j][r] = __builtin_fmaf(B.d[CODES ? k : 0][CODES ? j : 0], t[i][j][r], acc[i0 + i][j][r]);
  };
  auto mul = [&](const Slab& B, int buf) {
    AFrag f[2];
    f4v t[CODES ? 2 : 1][IG][TC];
    read_a(f[0], 0, buf);
#pragma unroll
    for (int g = 0; g < NG; g++) {
      const int k = g / (TR / IG), i0 = g % (TR / IG) * IG;
      const AFrag& a = f[g & 1];
      if (g + 1 < NG) read_a(f[(g + 1) & 1], g + 1, buf);
      if constexpr (CODES) {
        // A 32-deep step is one scale block: its two products on their own, then into the accumulator times the scale —
        // one group later, beside the next group's products.
        const f4v z = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < IG; i++)
#pragma unroll
          for (int j = 0; j < TC; j++) t[g & 1][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.l[i], B.h[k][j], z, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < IG; i++)
#pragma unroll
          for (int j = 0; j < TC; j++) {
            f4v& u = t[g & 1][i][j];
            u = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.h[i], B.h[k][j], u, 0, 0, 0);
          }
        if (g > 0) scale_in(B, t[(g - 1) & 1], g - 1);
        __builtin_amdgcn_sched_barrier(0);
        if (g + 1 == NG) scale_in(B, t[g & 1], g);
        continue;
      }
      __builtin_amdgcn_s_setprio(1);
      if constexpr (BLO)
#pragma unroll
        for (int i = 0; i < IG; i++)
#pragma unroll
          for (int j = 0; j < TC; j++)
            acc[i0 + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.h[i], B.l[k][j], acc[i0 + i][j], 0, 0, 0);
      if constexpr (ALO)
#pragma unroll
        for (int i = 0; i < IG; i++)
#pragma unroll
          for (int j = 0; j < TC; j++)
            acc[i0 + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.l[i], B.h[k][j], acc[i0 + i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < IG; i++)
#pragma unroll
        for (int j = 0; j < TC; j++)
          acc[i0 + i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.h[i], B.h[k][j], acc[i0 + i][j], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
    }
  };
  // Multiply slab s (A in LDS buffer s & 1, fragments in S) while slab s + 1 is on its way to N, whose A pieces move to
  // the other buffer afterwards. (Two slabs of lead measured no faster at any tile, also with the weights out of the
  // caches; register copies between the slabs instead of the unrolled pair make the compiler wait for every load.)
  auto step = [&](const Slab& S, Slab& N, int s) {
    load(N, s + 1);
    __builtin_amdgcn_sched_barrier(0);
    mul(S, s & 1);
    __builtin_amdgcn_sched_barrier(0);
    store_a(N, (s & 1) ^ 1);
    __syncthreads();
  };
  if (nslab > 0) {
    Slab S0, S1;
    load(S0, 0);
    store_a(S0, 0);
    __syncthreads();
    for (int s = 0;; s += 2) {
      step(S0, S1, s);
      if (s + 1 >= nslab) break;
      step(S1, S0, s + 1);
      if (s + 2 >= nslab) break;
    }
  }

  // ---- epilogue ----
  const bool split = gridDim.z > 1;
  // Fused rank-r term s·U·L on bf16 MFMA (hi·hi + lo·hi + hi·lo), both factors already laid out as planes (GemmEpi::Uf /
  // Lf): formed here from the f32 factors, their scattered loads and splits took 59 µs of the 676 µs launch at
  // 8192 × 8192 × 2048, rank 32. The first split's partial carries the term.
  if (epi.rank > 0 && !(split && zsp != 0) && n0 < p.N) {
    const int seg = epi.ustep ? 32 * ((n0 >= epi.ub0) + (n0 >= epi.ub1)) : 0;
    const int nrs = (epi.rank + 31) >> 5;
    const __bf16* ub = epi.Uf + seg + 8 * (lane >> 4);
    for (int rs = 0; rs < nrs; rs++) {
      bf8 lh[TC], ll[TC];
#pragma unroll
      for (int j = 0; j < TC; j++) {
        const __bf16* lp = epi.Lf + ((long long)min(n0 / 16 + j, p.nb - 1) * nrs + rs) * 1024 + lane * 8;
        lh[j] = *(const bf8*)lp;
        ll[j] = *(const bf8*)(lp + 512);
      }
#pragma unroll
      for (int i = 0; i < TR; i++) {
        const __bf16* up = ub + (long long)min(m0 + 16 * i + (lane & 15), p.M - 1) * epi.ldf + 32 * rs;
        const bf8 uh = *(const bf8*)up, ul = *(const bf8*)(up + epi.ulo);
#pragma unroll
        for (int j = 0; j < TC; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ul, lh[j], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < TC; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uh, ll[j], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < TC; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uh, lh[j], acc[i][j], 0, 0, 0);
      }
    }
  }
  // Each 32×32 block goes through a per-wave LDS transpose and leaves as row-major float4 runs. (The loop's last
  // barrier has passed: no wave reads the slabs any more.)
  float* tb = reinterpret_cast<float*>(smem) + wave * 32 * G::TS;
  const bool stats = TN == 2 && epi.rstat != nullptr && !split;
  const int N = p.N, M = p.M;
  const bool vec = (N & 3) == 0 && (split || ((epi.ldo & 3) == 0 && ((uintptr_t)epi.out & 15) == 0 &&
                                              (!epi.resid || ((uintptr_t)epi.resid & 15) == 0) &&
                                              (!epi.bias || ((uintptr_t)epi.bias & 15) == 0)));
#pragma unroll
  for (int i = 0; i < TM; i++) {
    float smx[4], ssm[4];  // row statistics: one (max, exp-sum) per lane and pass, folded over the column tiles
#pragma unroll
    for (int pz = 0; pz < 4; pz++) {
      smx[pz] = -INFINITY;
      ssm[pz] = 0.0f;
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
#pragma unroll
      for (int q = 0; q < 4; q++)  // 16×16 tile: lane l, register r is row 4·(l >> 4) + r, column l & 15
#pragma unroll
        for (int r = 0; r < 4; r++)
          tb[(16 * (q >> 1) + 4 * (lane >> 4) + r) * G::TS + 16 * (q & 1) + (lane & 15)] = acc[2 * i + (q >> 1)][2 * j + (q & 1)][r];
#pragma unroll
      for (int pz = 0; pz < 4; pz++) {
        const int lr = 8 * pz + (lane >> 3), c4 = 4 * (lane & 7);
        const float4 t4 = *reinterpret_cast<const float4*>(tb + lr * G::TS + c4);
        const int row = m0 + 32 * i + lr, col = n0 + 32 * j + c4;
        if (row >= M || col >= N) continue;
        float v[4] = {t4.x, t4.y, t4.z, t4.w};
        if (split) {
          float* d = ws + ((long long)zsp * M + row) * N + col;
          if (vec) {
            *reinterpret_cast<float4*>(d) = t4;
          } else {
            for (int e = 0; e < 4 && col + e < N; e++) d[e] = v[e];
          }
          continue;
        }
        const float ri = p.rinv[row];
        const long long off = (long long)row * epi.ldo + col;
        float* o = epi.out + off;
        if (vec) {
          const float4 b4 = epi.bias ? *reinterpret_cast<const float4*>(epi.bias + col) : make_float4(0.f, 0.f, 0.f, 0.f);
          float4 y = make_float4(v[0] * ri + b4.x, v[1] * ri + b4.y, v[2] * ri + b4.z, v[3] * ri + b4.w);
          if (epi.accumulate || epi.resid) {
            const float4 q = *reinterpret_cast<const float4*>(epi.accumulate ? o : epi.resid + off);
            y = make_float4(q.x + y.x, q.y + y.y, q.z + y.z, q.w + y.w);
          }
          *reinterpret_cast<float4*>(o) = y;
          v[0] = y.x;
          v[1] = y.y;
          v[2] = y.z;
          v[3] = y.w;
        } else {
          for (int e = 0; e < 4 && col + e < N; e++) {
            float x = v[e] * ri;
            if (epi.bias) x += epi.bias[col + e];
            x = epi.accumulate ? o[e] + x : (epi.resid ? epi.resid[off + e] + x : x);
            o[e] = x;
            v[e] = x;
          }
        }
        if (stats) {
          float mx = smx[pz];
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (col + e < N) mx = fmaxf(mx, v[e]);
          float sm = smx[pz] == -INFINITY ? 0.0f : ssm[pz] * exp_rs(smx[pz] - mx);
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (col + e < N) sm += exp_rs(v[e] - mx);
          smx[pz] = mx;
          ssm[pz] = sm;
        }
      }
    }
    if (stats) {
      // the 8 lanes of a row (lane bits 0-2) merge in a fixed tree order; lane 8·k writes row 8·pz + k
#pragma unroll
      for (int pz = 0; pz < 4; pz++) {
        float m = smx[pz], sm = ssm[pz];
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) {
          const float m2 = __shfl_xor(m, o), s2 = __shfl_xor(sm, o), mn = fmaxf(m, m2);
          sm = (m == -INFINITY ? 0.0f : sm * exp_rs(m - mn)) + (m2 == -INFINITY ? 0.0f : s2 * exp_rs(m2 - mn));
          m = mn;
        }
        const int row = m0 + 32 * i + 8 * pz + (lane >> 3);
        if ((lane & 7) == 0 && row < M && n0 < N) epi.rstat[(long long)row * epi.rstat_ld + n0 / 64] = make_float2(m, sm);
      }
    }
  }
}

// The same product where the output has too few tiles to fill the chip: 32×32 outputs per workgroup, its 8 waves each on
// an eighth of the contraction (32-deep steps w, w + 8, …) with both operands straight from global memory, the partial
// tiles summed through LDS in wave order. Bound by memory latency, so a wave keeps two steps of loads in flight and
// nothing else is waited for before the one barrier. 128 rows, 576 × 576,
// three products: 6.9 against 8.3 µs with the smallest tile above (and 16.5 dequantizing).
constexpr int SW = 8;
template <int NP>
__global__ void __launch_bounds__(64 * SW) plane_small_kernel(PlaneArgs p, GemmEpi epi) {
  constexpr bool ALO = NP == 2 || NP == 3 || NP == 5, BLO = NP == 3 || NP == 4, CODES = NP == 5;
  constexpr int TS = 36;  // f32 row stride of a partial tile
  __shared__ __attribute__((aligned(16))) float part[SW][32 * TS];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32, KT = p.C / 32;
  const int lr = lane & 15, lc = lane >> 4;
  f4v acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
  const _Float16 *ar[2], *al[2], *wr[2];
  const float* sr[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const long long o = (long long)min(m0 + 16 * i + lr, p.M - 1) * p.lda + 8 * lc;
    ar[i] = p.A + o;
    al[i] = ALO ? p.Alo + o : nullptr;
    wr[i] = p.W + (long long)min(n0 / 16 + i, p.nb - 1) * p.nstride + lane * 8;
    sr[i] = CODES ? p.S + (long long)min(n0 / 16 + i, p.nb - 1) * KT * 16 + lr : nullptr;
  }
  struct Step {
    h8 a[2], al[2], b[2], bl[2];
    float d[2];
  };
  auto load = [&](Step& s, int k) {
    k = min(k, KT - 1);  // past the end: a harmless re-read, never multiplied
#pragma unroll
    for (int i = 0; i < 2; i++) {
      s.a[i] = *(const h8*)(ar[i] + 32 * k);
      if constexpr (ALO) s.al[i] = *(const h8*)(al[i] + 32 * k);
      const _Float16* w = wr[i] + (long long)k * p.kstride;
      s.b[i] = *(const h8*)w;
      if constexpr (BLO) s.bl[i] = *(const h8*)(w + 512);
      if constexpr (CODES) s.d[i] = sr[i][16 * k];
    }
  };
  auto mul = [&](const Step& s) {
    if constexpr (CODES) {
      f4v t[2][2];
      const f4v z = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) t[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(s.al[i], s.b[j], z, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
          t[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(s.a[i], s.b[j], t[i][j], 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; r++) acc[i][j][r] = __builtin_fmaf(s.d[j], t[i][j][r], acc[i][j][r]);
        }
      return;
    }
    if constexpr (BLO)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(s.a[i], s.bl[j], acc[i][j], 0, 0, 0);
    if constexpr (ALO)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(s.al[i], s.b[j], acc[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(s.a[i], s.b[j], acc[i][j], 0, 0, 0);
  };
  Step s0, s1, s2;
  load(s0, wave);
  load(s1, wave + SW);
  load(s2, wave + 2 * SW);
  // the rank-r term (see plane_gemm_kernel) goes to the wave with the fewest steps
  if (wave == SW - 1 && epi.rank > 0) {
    const int seg = epi.ustep ? 32 * ((n0 >= epi.ub0) + (n0 >= epi.ub1)) : 0, nrs = (epi.rank + 31) >> 5;
    for (int rs = 0; rs < nrs; rs++) {
      bf8 uh[2], ul[2], lh[2], ll[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const __bf16* up = epi.Uf + seg + 8 * lc + (long long)min(m0 + 16 * i + lr, p.M - 1) * epi.ldf + 32 * rs;
        const __bf16* lp = epi.Lf + ((long long)min(n0 / 16 + i, p.nb - 1) * nrs + rs) * 1024 + lane * 8;
        uh[i] = *(const bf8*)up;
        ul[i] = *(const bf8*)(up + epi.ulo);
        lh[i] = *(const bf8*)lp;
        ll[i] = *(const bf8*)(lp + 512);
      }
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ul[i], lh[j], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uh[i], ll[j], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uh[i], lh[j], acc[i][j], 0, 0, 0);
        }
    }
  }
  for (int k = wave; k < KT; k += 3 * SW) {
    mul(s0);
    load(s0, k + 3 * SW);
    if (k + SW >= KT) break;
    mul(s1);
    load(s1, k + 4 * SW);
    if (k + 2 * SW >= KT) break;
    mul(s2);
    load(s2, k + 5 * SW);
  }
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) part[wave][(16 * i + 4 * lc + r) * TS + 16 * j + lr] = acc[i][j][r];
  __syncthreads();
  if (tid >= 256) return;
  const int rr = tid >> 3, c4 = 4 * (tid & 7), row = m0 + rr, col = n0 + c4;
  if (row >= p.M || col >= p.N) return;
  float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int w = 0; w < SW; w++) {
    const float4 x = *reinterpret_cast<const float4*>(&part[w][rr * TS + c4]);
    t = make_float4(t.x + x.x, t.y + x.y, t.z + x.z, t.w + x.w);
  }
  const float ri = p.rinv[row], v[4] = {t.x * ri, t.y * ri, t.z * ri, t.w * ri};
  const long long off = (long long)row * epi.ldo + col;
  float* o = epi.out + off;
  for (int e = 0; e < 4 && col + e < p.N; e++) {
    float x = v[e];
    if (epi.bias) x += epi.bias[col + e];
    o[e] = epi.accumulate ? o[e] + x : (epi.resid ? epi.resid[off + e] + x : x);
  }
}

template <int NP>
void plane_small_launch(const PlaneArgs& p, const GemmEpi& epi, hipStream_t st) {
  plane_small_kernel<NP><<<dim3(ceil_div(p.N, 32), ceil_div(p.M, 32)), 64 * SW, 0, st>>>(p, epi);
}

// Three products for outputs of few tiles, in exactly the sums of the dequantizing kernel's 64×64×64 tiles
// (qgemm_impl.hpp: four accumulator chains a contraction slab's twelve products rotate over, split over the contraction
// by the same rule), bit for bit, without that kernel's partials and reduction launch: a training run's trajectory
// amplifies any rounding, so small models keep theirs. 16·R × 16 outputs per workgroup (the chip has 256 units for
// 128 × 576 outputs), a wave per chain and split. Two slabs at a time: their six products are three 16×16×32 instructions,
// whose upper 16 of the contraction are the chain's next product (the unit adds them after the lower 16, as the two
// instructions would). Bound by memory latency: A rows come in whole lines through LDS (its fragments straight from memory, 32 bytes
// a row, were address bound: 31.8 µs at 128 × 576 × 3072), B fragments straight, three pairs of slabs in flight
// (16 waves of two row tiles: two).
// 128 rows on the MI355X, against that kernel: 576 × 576 6.1 µs, 960 × 576 6.3, 3072 × 576 9.4, 576 × 1536 8.5, 576 × 3072
// 12.9; a 30-layer training step of those 7.55 -> 6.2 ms.
constexpr int CHAIN_LDA = 136;  // halves of an LDS row: 128 and a 16-byte skew
template <int S, int R>
__global__ void __launch_bounds__(256 * S) plane_chain_kernel(PlaneArgs p, GemmEpi epi) {
  constexpr int ROWS = 16 * R, TILE = ROWS * CHAIN_LDA, DEPTH = S == 4 && R == 2 ? 2 : 3;  // (pairs of registers there are)
  __shared__ __attribute__((aligned(16))) _Float16 sa[S][2][2][TILE];  // split, buffer, plane
  static_assert(sizeof(sa) >= sizeof(float) * 4 * S * R * 256);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int z = wave >> 2, c = wave & 3;
  const int m0 = blockIdx.y * ROWS, n0 = blockIdx.x * 16;
  const int lr = lane & 15, lc = lane >> 4, up = lane >> 5, lh = lc & 1;
  const int beg = z * p.per / 64, nslab = max(0, (min(p.C, (z + 1) * p.per) - z * p.per) / 64);
  const int npair = (p.per / 64 + 1) >> 1;  // (the same for every split: zeros past a split's end)
  // product g of a pair's six is number c + 4·(g % 3) of slab g / 3's twelve: 16-deep step number / 3, kind number % 3
  // (0 hi·hi, 1 lo·hi, 2 hi·lo); lanes 32-63 hold the odd ones
  int as[3], sub[3];
  const _Float16* wp[3];
  const _Float16* wcol = p.W + (long long)blockIdx.x * p.nstride + lr * 8;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const int g = 2 * i + up, q = c + 4 * (g % 3), t = q / 3, kind = q % 3;
    sub[i] = g / 3;
    as[i] = (kind == 1 ? TILE : 0) + lr * CHAIN_LDA + 64 * sub[i] + 16 * t + 8 * lh;
    wp[i] = wcol + (2LL * (beg + sub[i]) + (t >> 1)) * p.kstride + (kind == 2 ? 512 : 0) + (2 * (t & 1) + lh) * 128;
  }
  // a split's 256 threads stage its pair: 16 pieces of 8 halves to a row
  const int piece = tid & 15, srow = (tid & 255) >> 4;
  const int k0 = 64 * beg + 8 * piece, kend = 64 * (beg + nslab);
  struct Pair {
    h8 a[2][R], b[3];
  };
  const h8 zero = (h8)(_Float16)0;
  auto load = [&](Pair& x, int s) {
    const int k = k0 + 128 * s;
    const bool in = k < kend;
#pragma unroll
    for (int i = 0; i < R; i++) {
      const long long off = (long long)min(m0 + 16 * i + srow, p.M - 1) * p.lda + (in ? k : 0);
      x.a[0][i] = *(const h8*)(p.A + off);
      x.a[1][i] = *(const h8*)(p.Alo + off);
      if (!in) x.a[0][i] = x.a[1][i] = zero;
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const bool bin = 2 * s + sub[i] < nslab;
      x.b[i] = *(const h8*)(bin ? wp[i] + 4LL * s * p.kstride : p.W);
      if (!bin) x.b[i] = zero;
    }
  };
  f4v acc[R];
#pragma unroll
  for (int i = 0; i < R; i++) acc[i] = (f4v){0.f, 0.f, 0.f, 0.f};
  auto step = [&](Pair& x, int s) {
    _Float16* d = &sa[z][s & 1][0][0];
#pragma unroll
    for (int i = 0; i < R; i++) {
      *(h8*)(d + (16 * i + srow) * CHAIN_LDA + 8 * piece) = x.a[0][i];
      *(h8*)(d + TILE + (16 * i + srow) * CHAIN_LDA + 8 * piece) = x.a[1][i];
    }
    __syncthreads();  // (also: every wave is done with the buffer the next step writes)
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int r = 0; r < R; r++)
        acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(*(const h8*)(d + as[i] + 16 * r * CHAIN_LDA), x.b[i], acc[r], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);  // (the loads stay here: the compiler would move them down to their use)
    if (s + DEPTH < npair) load(x, s + DEPTH);
    __builtin_amdgcn_sched_barrier(0);
  };
  Pair q0, q1, q2;
  load(q0, 0);
  load(q1, 1);
  if constexpr (DEPTH > 2) load(q2, 2);
  __builtin_amdgcn_sched_barrier(0);
  for (int s = 0; s < npair; s += DEPTH) {
    step(q0, s);
    if (s + 1 >= npair) break;
    step(q1, s + 1);
    if constexpr (DEPTH > 2) {
      if (s + 2 >= npair) break;
      step(q2, s + 2);
    }
  }
  __syncthreads();
  float(*part)[R][256] = reinterpret_cast<float(*)[R][256]>(&sa[0][0][0][0]);
#pragma unroll
  for (int r = 0; r < R; r++) *(f4v*)(&part[wave][r][4 * lane]) = acc[r];
  __syncthreads();
  if (wave >= R) return;
  const int mt = m0 + 16 * wave, col = n0 + lr;  // one wave to a 16 × 16 output; register i of a lane: row 4·lc + i
  auto chains = [&](int zz) {
    f4v v = *(const f4v*)(&part[4 * zz][wave][4 * lane]);
#pragma unroll
    for (int k = 1; k < 4; k++) v += *(const f4v*)(&part[4 * zz + k][wave][4 * lane]);
    return v;
  };
  f4v v = chains(0);
  if (epi.rank > 0) {
    // the rank-r term goes into the first split's sum, 16 ranks at a time lo·hi, hi·lo, hi·hi: six products, in pairs, too.
    // (Fetched ahead of the slabs its fragments cost more in registers than they gain: 8.8 -> 9.6 µs.)
    const int seg = epi.ustep ? 32 * ((n0 >= epi.ub0) + (n0 >= epi.ub1)) : 0, nrs = (epi.rank + 31) >> 5;
    const __bf16* u = epi.Uf + seg + 8 * lh + (long long)min(mt + lr, p.M - 1) * epi.ldf;
    const __bf16* l = epi.Lf + (long long)blockIdx.x * nrs * 1024 + lr * 8;
    for (int rs = 0; rs < nrs; rs++)
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const int g = 2 * i + up, h = g / 3, kind = g % 3;
        const bf8 x = *(const bf8*)(u + 32 * rs + 16 * h + (kind == 0 ? epi.ulo : 0));
        const bf8 y = *(const bf8*)(l + rs * 1024 + (kind == 1 ? 512 : 0) + (2 * h + lh) * 128);
        v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, v, 0, 0, 0);
      }
  }
#pragma unroll
  for (int zz = 1; zz < S; zz++) v += chains(zz);
  if (col >= p.N) return;
  const float b = epi.bias ? epi.bias[col] : 0.0f;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int row = mt + 4 * lc + r;
    if (row >= p.M) break;
    const long long off = (long long)row * epi.ldo + col;
    float* o = epi.out + off;
    float y = v[r] * p.rinv[row] + b;
    if (epi.accumulate || epi.resid) y = (epi.accumulate ? *o : epi.resid[off]) + y;
    *o = y;
  }
}

template <int TM, int TN, int NP, int BK>
void plane_launch(const PlaneArgs& p, int row_tiles, int splits, const GemmEpi& epi, float* ws, hipStream_t st) {
  using G = PGeo<TM, TN, NP, BK>;
  dim3 grid(ceil_div(p.N, G::BN), row_tiles, splits);
  plane_gemm_kernel<TM, TN, NP, BK><<<grid, 256, 0, st>>>(p, epi, ws);
}

}  // namespace
}  // namespace hos
