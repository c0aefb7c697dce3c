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
};

template <int TM, int TN, int NP, int BK>
struct PGeo {
  static constexpr int BM = 32 * TM, BN = 128 * TN, CH = BK / 8, KS = BK / 32;
  static constexpr int NA = (NP == 2 || NP == 3) ? 2 : 1, NB = (NP == 3 || NP == 4) ? 2 : 1;
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
  constexpr bool ALO = G::NA == 2, BLO = G::NB == 2;
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
  // One slab in flight: this thread's pieces of A (to LDS later) and this wave's fragments.
  struct Slab {
    h8 a[G::AV], al[ALO ? G::AV : 1];
    h8 h[G::KS][TC], l[BLO ? G::KS : 1][BLO ? TC : 1];
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
  auto mul = [&](const Slab& B, int buf) {
    AFrag f[2];
    read_a(f[0], 0, buf);
#pragma unroll
    for (int g = 0; g < NG; g++) {
      const int k = g / (TR / IG), i0 = g % (TR / IG) * IG;
      const AFrag& a = f[g & 1];
      if (g + 1 < NG) read_a(f[(g + 1) & 1], g + 1, buf);
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

template <int TM, int TN, int NP, int BK>
void plane_launch(const PlaneArgs& p, int row_tiles, int splits, const GemmEpi& epi, float* ws, hipStream_t st) {
  using G = PGeo<TM, TN, NP, BK>;
  dim3 grid(ceil_div(p.N, G::BN), row_tiles, splits);
  plane_gemm_kernel<TM, TN, NP, BK><<<grid, 256, 0, st>>>(p, epi, ws);
}

}  // namespace
}  // namespace hos
