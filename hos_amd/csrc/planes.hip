// Frozen weights dequantized once into fp16 planes in MFMA fragment order (WPlanes, common.hpp), the form the plane
// GEMM (plane_gemm.hip) reads: the same hi / lo values the dequantizing GEMM forms in registers for every launch.
#include <algorithm>

#include "ctx.hpp"
#include "qgemm_impl.hpp"

namespace hos {
namespace {

// A 32-value run of one weight row per thread, dequantized by the GEMM's own run_load / run_store (so the planes are
// the values it forms), 8 halves per plane and 16-byte piece.
template <uint32_t QT>
__device__ __forceinline__ void run_planes(const QWeightView& w, long long e, _Float16 (&v)[64]) {
  Run<QT, 32> r;
  run_load<QT, 32>((const uint8_t*)w.q + run_qoff<QT>(e), w.s + run_soff<QT>(e), r);
  run_store<QT, 32, true>(r, v, 32);
}

// Forward: a run is one column n's share of a 32-deep step, four pieces of its fragment. A thread per (n, step), n
// fastest, so 16 threads write a fragment's 256-byte rows. 4096² Q4_K: 26 µs (a byte-wise version 65).
template <uint32_t QT>
__global__ void __launch_bounds__(256) build_fwd_kernel(QWeightView w, int planes, long long er, long long Np, int KT,
                                                        long long groups, _Float16* __restrict__ dst) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long n = i % Np, u = i / Np, ks = u % KT, g = u / KT;
  if (g >= groups) return;
  __attribute__((aligned(16))) _Float16 v[64];
  if (n < er) {
    run_planes<QT>(w, (g * er + n) * w.cols + 32 * ks, v);
  } else {
#pragma unroll
    for (int q = 0; q < 64; q++) v[q] = (_Float16)0.0f;
  }
  _Float16* d = dst + (((g * (Np >> 4) + (n >> 4)) * KT + ks) * planes) * 512 + (n & 15) * 8;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    *(h8*)(d + q * 128) = *(const h8*)(v + 8 * q);
    if (planes == 2) *(h8*)(d + 512 + q * 128) = *(const h8*)(v + 32 + 8 * q);
  }
}

// Mode 5's codes, laid out as the forward planes (one plane), and their scales.
__global__ void __launch_bounds__(256) build_codes_kernel(QWeightView w, long long er, long long Np, int KT, long long groups,
                                                          _Float16* __restrict__ dst, float* __restrict__ scale) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long n = i % Np, u = i / Np, ks = u % KT, g = u / KT;
  if (g >= groups) return;
  __attribute__((aligned(16))) _Float16 v[32];
  float sc = 0.0f;
  if (n < er) {
    const long long e = (g * er + n) * w.cols + 32 * ks;
    Run<GGUF_Q8_0, 32> r;
    run_load<GGUF_Q8_0, 32>((const uint8_t*)w.q + e, w.s + (e >> 5), r);
    sc = r.s[0].x;
    run_store<GGUF_Q8_0, 32, false, true>(r, v, 0);
  } else {
#pragma unroll
    for (int q = 0; q < 32; q++) v[q] = (_Float16)0.0f;
  }
  const long long f = (g * (Np >> 4) + (n >> 4)) * KT + ks;
  _Float16* d = dst + f * 512 + (n & 15) * 8;
#pragma unroll
  for (int q = 0; q < 4; q++) *(h8*)(d + q * 128) = *(const h8*)(v + 8 * q);
  scale[f * 16 + (n & 15)] = sc;
}

// dX: the contraction runs down the rows, so a workgroup turns 32 rows × 256 columns round in LDS: a thread per run in,
// then fragment pieces (8 rows of a column) out.
template <uint32_t QT>
__global__ void __launch_bounds__(256) build_dx_kernel(QWeightView w, int planes, long long er, int KT,
                                                       _Float16* __restrict__ dst) {
  constexpr int LD = 256 + 8;
  __shared__ __attribute__((aligned(16))) _Float16 t[2][32 * LD];
  const int ks = blockIdx.y % KT;
  const long long g = blockIdx.y / KT, n0 = 256LL * blockIdx.x;
  const int nb = (int)((w.cols + 15) / 16), row = threadIdx.x >> 3, c = 32 * (threadIdx.x & 7);
  if (n0 + c < w.cols) {
    __attribute__((aligned(16))) _Float16 v[64];
    run_planes<QT>(w, (g * er + 32 * ks + row) * w.cols + n0 + c, v);
#pragma unroll
    for (int q = 0; q < 4; q++) {
      *(h8*)(t[0] + row * LD + c + 8 * q) = *(const h8*)(v + 8 * q);
      *(h8*)(t[1] + row * LD + c + 8 * q) = *(const h8*)(v + 32 + 8 * q);
    }
  }
  __syncthreads();
  for (int f = threadIdx.x; f < 16 * 64; f += 256) {
    const int b = f >> 6, lane = f & 63, col = 16 * b + (lane & 15);
    if (n0 + col >= w.cols) break;
    for (int p = 0; p < planes; p++) {
      h8 x;
#pragma unroll
      for (int q = 0; q < 8; q++) x[q] = t[p][(8 * (lane >> 4) + q) * LD + col];
      *(h8*)(dst + (((g * nb + (n0 >> 4) + b) * KT + ks) * planes + p) * 512 + lane * 8) = x;
    }
  }
}

template <uint32_t QT>
void build_typed(const QWeight& w, bool dx, int planes, int groups, half_t* dst, hipStream_t st) {
  const long long er = w.rows / groups;
  if (dx) {
    const int KT = (int)(er / 32);
    build_dx_kernel<QT><<<dim3(ceil_div(w.cols, 256), (unsigned)(groups * KT)), 256, 0, st>>>(view(w), planes, er, KT, dst);
  } else {
    const long long Np = (er + 15) / 16 * 16, KT = w.cols / 32;
    build_fwd_kernel<QT><<<ceil_div(Np * KT * groups, 256), 256, 0, st>>>(view(w), planes, er, Np, (int)KT, groups, dst);
  }
  HOS_HIP_CHECK(hipGetLastError());
}

// 8 values to bf16 hi / lo, 16 bytes each.
__device__ __forceinline__ void put_split(const float (&v)[8], __bf16* hi, __bf16* lo) {
  bf8 h, l;
#pragma unroll
  for (int q = 0; q < 8; q++) split_bf(v[q], h, l, q);
  *(bf8*)hi = h;
  *(bf8*)lo = l;
}

// A wave per item: the fragments of 16 columns of a factor, every rank step (zero past the rank and the columns).
__global__ void __launch_bounds__(256) rank_frags_kernel(const RankItem* __restrict__ items, int n,
                                                         const float* __restrict__ src, __bf16* __restrict__ dst) {
  const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= n) return;
  const RankItem it = items[i];
  const int col = 16 * it.nb + (lane & 15);
  __bf16* d = dst + it.dst + lane * 8;
  for (int r0 = 0; r0 < it.rank; r0 += 32, d += 1024) {
    const int k0 = r0 + 8 * (lane >> 4);
    float v[8];
#pragma unroll
    for (int q = 0; q < 8; q++)
      v[q] = (k0 + q < it.rank && col < it.cols) ? src[it.off + (long long)(k0 + q) * it.ld + col] * it.scale : 0.0f;
    put_split(v, d, d + 512);
  }
}

// Both factors of one launch (GemmEpi U / L with their strides and segments): threads below nl make a lane of a
// fragment of L, the others 8 ranks of a row of U.
__global__ void __launch_bounds__(256) rank_prep_kernel(GemmEpi e, const float* __restrict__ rinv, int M, int N, int nseg,
                                                        long long nl, __bf16* uf, __bf16* lf) {
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  const int nrs = (e.rank + 31) >> 5;
  float v[8];
  if (t < nl) {
    const int lane = (int)(t & 63);
    const long long f = t >> 6;  // (nb, rs)
    const int nb = (int)(f / nrs), rs = (int)(f % nrs), col = 16 * nb + (lane & 15), k0 = 32 * rs + 8 * (lane >> 4);
#pragma unroll
    for (int q = 0; q < 8; q++)
      v[q] = (k0 + q < e.rank && col < N) ? e.L[(long long)(k0 + q) * e.slj + (long long)col * e.sln] * e.scale : 0.0f;
    __bf16* d = lf + f * 1024 + lane * 8;
    put_split(v, d, d + 512);
    return;
  }
  const long long u = t - nl;
  const int per = nseg * nrs * 4;  // 8-column runs per row
  const long long row = u / per;
  if (row >= M) return;
  const int c = (int)(u % per) * 8, seg = nseg > 1 ? c / 32 : 0, k0 = nseg > 1 ? c % 32 : c;
  const float inv = __uint_as_float((254u << 23) - __float_as_uint(rinv[row]));  // 1 / 2^-e
#pragma unroll
  for (int q = 0; q < 8; q++)
    v[q] = k0 + q < e.rank ? e.U[row * e.ldu + (long long)seg * e.ustep + k0 + q] * inv : 0.0f;
  __bf16* d = uf + row * e.ldf + c;
  put_split(v, d, d + e.ulo);
}

}  // namespace

void launch_rank_frags(const RankItem* items, int n, const float* src, __bf16* dst, hipStream_t st) {
  if (n <= 0) return;
  rank_frags_kernel<<<(n + 3) / 4, 256, 0, st>>>(items, n, src, dst);
  HOS_HIP_CHECK(hipGetLastError());
}

bool prepare_rank(GemmEpi& e, const float* rinv, long long M, long long N, float* ws, size_t* ws_bytes, hipStream_t st) {
  const int nrs = (e.rank + 31) / 32, nseg = e.ustep ? 1 + (e.ub0 < N) + (e.ub1 < N) : 1;
  if (nseg > 1 && nrs > 1) return false;
  e.ldf = 32LL * nseg * nrs;
  e.ulo = M * e.ldf;
  const long long nb = (N + 15) / 16;
  const size_t ub = (size_t)M * e.ldf * 4, lb = (size_t)nb * nrs * 2048, need = (ub + lb + 511) / 256 * 256;
  if (need > *ws_bytes) return false;
  char* base = (char*)ws + (*ws_bytes - need) / 256 * 256;
  *ws_bytes = (size_t)(base - (char*)ws);
  e.Uf = (const __bf16*)base;
  e.Lf = (const __bf16*)(base + (ub + 255) / 256 * 256);
  const long long nl = nb * nrs * 64, n = nl + M * nseg * nrs * 4;
  rank_prep_kernel<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(e, rinv, (int)M, (int)N, nseg, nl, (__bf16*)e.Uf,
                                                                (__bf16*)e.Lf);
  HOS_HIP_CHECK(hipGetLastError());
  return true;
}

static void plane_dims(const QWeight& w, bool dx, int groups, long long* er, long long* N, long long* C) {
  *er = w.rows / groups;
  *N = dx ? w.cols : *er;
  *C = dx ? *er : w.cols;
}

// 1 KB fragments of one plane.
static size_t plane_frags(const QWeight& w, bool dx, int groups) {
  long long er, N, C;
  plane_dims(w, dx, groups, &er, &N, &C);
  return (size_t)groups * ((N + 15) / 16) * (C / 32);
}

size_t planes_bytes(const QWeight& w, bool dx, int kind, int groups) {
  return plane_frags(w, dx, groups) * (kind == kPlaneCodes ? 1024 + 64 : 1024 * kind);
}

WPlanes build_planes(const QWeight& w, bool dx, int kind, int groups, half_t* dst, hipStream_t st) {
  long long er, N, C;
  plane_dims(w, dx, groups, &er, &N, &C);
  HOS_REQUIRE(w.rows % groups == 0 && C % 32 == 0 && w.cols % 32 == 0 && (!dx || groups * (er / 32) < 65536), HOS_E_INVALID,
              "planes: contraction must be a multiple of 32");
  if (kind == kPlaneCodes) {
    HOS_REQUIRE(!dx && w.type == GGUF_Q8_0, HOS_E_INVALID, "planes: integer codes are for forward Q8_0 weights");
    float* scale = (float*)(dst + plane_frags(w, dx, groups) * 512);
    const long long Np = (er + 15) / 16 * 16, KT = w.cols / 32;
    build_codes_kernel<<<ceil_div(Np * KT * groups, 256), 256, 0, st>>>(view(w), er, Np, (int)KT, groups, dst, scale);
    HOS_HIP_CHECK(hipGetLastError());
    return WPlanes{dst, 1, false, scale};
  }
  switch (w.type) {
    case GGUF_Q8_0: build_typed<GGUF_Q8_0>(w, dx, kind, groups, dst, st); break;
    case GGUF_Q4_K: build_typed<GGUF_Q4_K>(w, dx, kind, groups, dst, st); break;
    case GGUF_Q6_K: build_typed<GGUF_Q6_K>(w, dx, kind, groups, dst, st); break;
    case GGUF_Q5_K: build_typed<GGUF_Q5_K>(w, dx, kind, groups, dst, st); break;
    case GGUF_F16: build_typed<GGUF_F16>(w, dx, kind, groups, dst, st); break;
    case GGUF_BF16: build_typed<GGUF_BF16>(w, dx, kind, groups, dst, st); break;
    case GGUF_F32: build_typed<GGUF_F32>(w, dx, kind, groups, dst, st); break;
    default: throw Error(HOS_E_UNSUPPORTED_QUANT, "planes: unsupported quant type");
  }
  return WPlanes{dst, kind, false, nullptr};
}

// Planes a context may allocate between two looks at the free memory (a look costs as much as building small planes).
constexpr size_t kPlaneCredit = 256ull << 20;

bool planes_fit(size_t bytes) {
  size_t fr = 0, total = 0;
  HOS_HIP_CHECK(hipMemGetInfo(&fr, &total));
  return fr >= total / 2 && fr - total / 2 >= bytes;
}

void ensure_planes(QWeight& w, bool dx, int passes, long long M, size_t* credit, hipStream_t st) {
  WPlanes& p = w.pl[dx];
  const int want = plane_kind(w, dx, passes);
  if (has_planes(p, dx, passes) || !plane_gemm_wanted(w, dx, passes, M)) return;
  // A capture records the build without running it: later eager launches would read planes that are not there yet.
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  HOS_HIP_CHECK(hipStreamIsCapturing(st, &cs));
  if (cs != hipStreamCaptureStatusNone) return;
  const size_t bytes = planes_bytes(w, dx, want, 1);
  if (*credit < bytes) {
    const size_t ask = std::max(bytes, kPlaneCredit);
    if (!planes_fit(ask)) return;
    *credit = ask;
  }
  void* d = nullptr;
  if (hipMalloc(&d, bytes) != hipSuccess) {
    (void)hipGetLastError();  // no planes then: the launch runs on the quantized weight
    return;
  }
  if (p.owned) {  // another kind so far, and launches on the stream may still read it
    HOS_HIP_CHECK(hipStreamSynchronize(st));
    (void)hipFree(p.p);
  }
  *credit -= bytes;
  p = WPlanes{};
  WPlanes q{(half_t*)d, 0, true, nullptr};
  try {
    q = build_planes(w, dx, want, 1, (half_t*)d, st);
  } catch (...) {
    (void)hipFree(d);
    throw;
  }
  q.owned = true;
  p = q;
}

}  // namespace hos
