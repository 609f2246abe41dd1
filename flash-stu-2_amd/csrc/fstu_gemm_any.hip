// General dense contraction  C[m, n] = T( sum_k A[m, k] W[n, k] )  for what the bf16 prompt GEMM (fstu_gemm.hip) does
// not take: fp32 (the bit-parity path of the reference's fp32 configuration, flash_stu/model.py:108-205 with
// torch_dtype float32), bf16 shapes with K % 32 != 0 or unaligned rows, and operands with any pair of strides (the
// (K*d, T) slabs of the exact-mode operator in fp32, flash_stu/modules/stu.py:107-120; phi @ M_filters, stu.py:88).
// Accumulation in fp32 on the fp32 matrix instructions (bf16 inputs widen exactly), one rounding to the output dtype.
// Every global access is bounds-checked, so any M, N, K >= 1 works.  The order of the sums depends on M, N and K alone:
// strides and alignment only choose how a tile is read and how much of it ahead.
#include <algorithm>
#include "fstu_common.h"

namespace {

typedef float floatx16_t __attribute__((ext_vector_type(16)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

// Elements k..k+3 of a row, zero from K on.  VEC: k runs with stride 1, rows start on 4-element boundaries and K % 4 == 0;
// each operand for itself (with W alone transposed 4096 x 768 x 768 takes 67 us; 138 where both were read one by one).
// The loads are unconditional (an address beyond K is replaced by the row's start), so several stay in flight.
template <typename T, bool VEC>
__device__ __forceinline__ floatx4_t ga_load4(const T* __restrict__ row, long long sk, int k, int K) {
  floatx4_t v;
  if constexpr (VEC) {
    const T* p = row + (k < K ? k : 0);
    if constexpr (sizeof(T) == 4) {
      v = *reinterpret_cast<const floatx4_t*>(p);
    } else {
      const uint2 u = *reinterpret_cast<const uint2*>(p);
      v = floatx4_t{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                    __uint_as_float(u.y & 0xffff0000u)};
    }
    if (k >= K) v = floatx4_t{0.f, 0.f, 0.f, 0.f};
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = DT<T>::ld(row + (size_t)(k + e < K ? k + e : 0) * sk);
      v[e] = k + e < K ? x : 0.f;
    }
  }
  return v;
}

// Few output tiles: the NW waves of a workgroup share one tile of 16*TM rows x 16*TN features and take every NW-th group of
// 16 k, reading the fragments of v_mfma_f32_16x16x4_f32 from global memory (a lane holds 4 consecutive k, one matrix
// instruction per element); the NW partial tiles are added in wave order through LDS.  Bound by one or two trips to
// memory: a workgroup's k loop is K / (16 NW) trips where a tile of the staged kernel below takes K / 16 of them, one
// behind the other.
template <typename T, bool VA, bool VW, int TM, int TN, int NW, int U>
__global__ void __launch_bounds__(64 * NW)
gemm_any_split_kernel(const T* __restrict__ A, long long sam, long long sak, const T* __restrict__ W, long long swn, long long swk,
                      T* __restrict__ C, long long ldc, int M, int N, int K) {
  __shared__ float red[NW][TM * TN][256];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int m0 = blockIdx.x * 16 * TM, n0 = blockIdx.y * 16 * TN;
  const T *ar[TM], *wr[TN];
#pragma unroll
  for (int j = 0; j < TM; ++j) ar[j] = A + (size_t)min(m0 + 16 * j + r, M - 1) * sam;
#pragma unroll
  for (int i = 0; i < TN; ++i) wr[i] = W + (size_t)min(n0 + 16 * i + r, N - 1) * swn;
  floatx4_t acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 16 * w; k0 < K; k0 += 16 * NW * U) {
    floatx4_t av[U][TM], wv[U][TN];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 16 * NW * u;
      if (k >= K) break;
#pragma unroll
      for (int i = 0; i < TN; ++i) wv[u][i] = ga_load4<T, VW>(wr[i], swk, k + 4 * g, K);
#pragma unroll
      for (int j = 0; j < TM; ++j) av[u][j] = ga_load4<T, VA>(ar[j], sak, k + 4 * g, K);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k0 + 16 * NW * u >= K) break;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[u][i][e], av[u][j][e], acc[i][j], 0, 0, 0);
    }
  }
  // D: lane l holds row l % 16 and features 4*(l/16) + e of a 16 x 16 tile
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) *reinterpret_cast<floatx4_t*>(&red[w][i * TM + j][4 * lane]) = acc[i][j];
  __syncthreads();
  for (int idx = threadIdx.x; idx < TM * TN * 256; idx += 64 * NW) {
    const int f = idx % (16 * TN), mm = idx / (16 * TN);
    const int tile = (f >> 4) * TM + (mm >> 4), off = ((((f & 15) >> 2) << 4) + (mm & 15)) * 4 + (f & 3);
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < NW; ++q) s += red[q][tile][off];
    if (m0 + mm < M && n0 + f < N) DT<T>::st(C + (size_t)(m0 + mm) * ldc + n0 + f, s);
  }
}

// Many output tiles: a workgroup of 4 waves owns B rows x B features, B = 128 or 64, a wave B/2 x B/2 on v_mfma_f32_32x32x2_f32; K runs
// in tiles of 16 through two LDS buffers, the loads of the next two tiles in flight while one is multiplied; of one where the large tile
// reads an operand element by element, whose registers would cost it a workgroup on the compute unit (1000 x 12288 x 3072 with both
// so 811 us, two ahead 890).  A k step of a wave is B/32 LDS reads for (B/64)^2 matrix instructions of 64 cycles.  Bound by the fp32
// matrix rate.  Both sizes add in the same order.  fp32, us, one ahead / two: 16384 x 2048 x 2048 1154 / 1084 (127 TFLOP/s), 1000 x 12288 x
// 3072 675 / 612.
#define GA_BK 16
#define GA_LD (GA_BK + 1)

// a thread's share (B / 16 elements) of a B x 16 tile; threads run along the index whose stride is 1, so loads coalesce
template <typename T, bool VEC, int B>
__device__ __forceinline__ void ga_fetch(float (&v)[B / 16], const T* __restrict__ src, long long srow, long long sk, int row0,
                                         int nrows, int k0, int K) {
  if constexpr (VEC) {
#pragma unroll
    for (int i = 0; i < B / 64; ++i) {
      const int r = (threadIdx.x >> 2) + 64 * i, k = k0 + 4 * (threadIdx.x & 3);
      const floatx4_t t = ga_load4<T, true>(src + (size_t)min(row0 + r, nrows - 1) * srow, 1, k, K);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * i + e] = t[e];
    }
  } else {
#pragma unroll
    for (int i = 0; i < B / 16; ++i) {
      const int idx = threadIdx.x + 256 * i;
      const int r = sk == 1 ? idx / GA_BK : idx % B, k = k0 + (sk == 1 ? idx % GA_BK : idx / B);
      const float x = DT<T>::ld(src + (size_t)min(row0 + r, nrows - 1) * srow + (size_t)(k < K ? k : 0) * sk);
      v[i] = k < K ? x : 0.f;
    }
  }
}

template <bool VEC, int B>
__device__ __forceinline__ void ga_put(float (*dst)[GA_LD], const float (&v)[B / 16], long long sk) {
#pragma unroll
  for (int i = 0; i < B / 16; ++i) {
    if constexpr (VEC) {
      dst[(threadIdx.x >> 2) + 64 * (i >> 2)][4 * (threadIdx.x & 3) + (i & 3)] = v[i];
    } else {
      const int idx = threadIdx.x + 256 * i;
      if (sk == 1) dst[idx / GA_BK][idx % GA_BK] = v[i];
      else dst[idx % B][idx / B] = v[i];
    }
  }
}

template <typename T, bool VA, bool VW, int B>
__global__ void __launch_bounds__(256)
gemm_any_tile_kernel(const T* __restrict__ A, long long sam, long long sak, const T* __restrict__ W, long long swn, long long swk,
                     T* __restrict__ C, long long ldc, int M, int N, int K) {
  constexpr int Q = B / 64;
  constexpr bool AHEAD = B == 64 || (VA && VW);        // two tiles ahead, or one
  __shared__ float xs[2][B][GA_LD], ws[2][B][GA_LD];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = B / 2 * (w & 1), wn = B / 2 * (w >> 1);
  const int m0 = blockIdx.x * B, n0 = blockIdx.y * B;
  const int l32 = lane & 31, lh = lane >> 5;
  floatx16_t acc[Q][Q];
#pragma unroll
  for (int i = 0; i < Q; ++i)
#pragma unroll
    for (int j = 0; j < Q; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  struct Next { float a[B / 16], w[B / 16]; } n1, n2;
  auto fetch = [&](Next& v, int k0) __attribute__((always_inline)) {
    ga_fetch<T, VA, B>(v.a, A, sam, sak, m0, M, k0, K);
    ga_fetch<T, VW, B>(v.w, W, swn, swk, n0, N, k0, K);
  };
  auto put = [&](int b, const Next& v) __attribute__((always_inline)) {
    ga_put<VA, B>(xs[b], v.a, sak);
    ga_put<VW, B>(ws[b], v.w, swk);
  };
  auto multiply = [&](int b) __attribute__((always_inline)) {
    // weights as the A operand (lane: feature l % 32, k = l / 32), activations as the B operand (lane: row l % 32)
#pragma unroll
    for (int kk = 0; kk < GA_BK; kk += 2) {
      float x[Q], y[Q];
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        x[i] = xs[b][wm + 32 * i + l32][kk + lh];
        y[i] = ws[b][wn + 32 * i + l32][kk + lh];
      }
#pragma unroll
      for (int i = 0; i < Q; ++i)
#pragma unroll
        for (int j = 0; j < Q; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(y[i], x[j], acc[i][j], 0, 0, 0);
    }
  };
  fetch(n1, 0);
  if constexpr (AHEAD) {
    fetch(n2, GA_BK);
    put(0, n1);
    fetch(n1, 2 * GA_BK);
    __syncthreads();
    int k0 = 0;
    auto pass = [&](int b, Next& v) __attribute__((always_inline)) {      // v: the tile behind this one
      multiply(b);
      put(b ^ 1, v);       // the other buffer was last read before the barrier that ended the previous tile
      fetch(v, K - k0 > 3 * GA_BK ? k0 + 3 * GA_BK : K);                   // zeros from K on, and no sum beyond an int for the longest K
      __syncthreads();
      return (k0 += GA_BK) < K;
    };
    while (pass(0, n2) && pass(1, n1)) {
    }
  } else {
    put(0, n1);
    __syncthreads();
    for (int k0 = 0, b = 0; k0 < K; k0 += GA_BK, b ^= 1) {
      const bool more = k0 + GA_BK < K;
      if (more) fetch(n1, k0 + GA_BK);
      multiply(b);
      if (more) put(b ^ 1, n1);
      __syncthreads();
    }
  }
  // D: lane l holds row l % 32 and features 8*(e/4) + 4*(l/32) + e%4 of a 32 x 32 tile
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    const int m = m0 + wm + 32 * j + l32;
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < Q; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int f = n0 + wn + 32 * i + 8 * (e >> 2) + 4 * lh + (e & 3);
        if (f < N) DT<T>::st(C + (size_t)m * ldc + f, acc[i][j][e]);
      }
  }
}

// 0: 16 x 16 tiles, 16 waves along K; 1: 32 x 32 tiles, 8 waves along K; 4: the same with 64 rows; 2: 64 x 64 tiles; 3: 128 x 128 tiles.  Rows or features that fill at
// most half of a large tile stay on 1 (bf16, us on 1 / 2: 17 x 50257 x 256 17 / 41, 64 x 50257 x 256 31 / 46, 100000 x 16 x 768
// 68 / 227, 100000 x 64 x 256 54 / 89; 100 x 50257 x 768 143 / 128).  A large tile (2, 3) needs more
// than one workgroup per compute unit before its matrix rate counts (192 tiles: 2000 x 1536 x 1536 141 us on 1, 158 on 2;
// 512 tiles: 4096 x 2048 x 24 40 us on 1, 33 on 2; 1024: 16384 x 2048 x 2048 1885 on 1, 1153 on 2), the 32 x 32 tile half
// the chip (16 tiles: 64 x 256 x 3072 13 us on 0, 27 on 1; 80: 300 x 256 x 3072 25 and 30; 256: 1000 x 256 x 3072 49 and 31).
// One kernel of 64 x 64 tiles with no loads ahead took 228, 525, 500 us for the last three, 283 and 2860 for the first and
// third, 23 us for 200 x 256 x 256 (now 8), and its sums in one chain were 2.5 to 4 times further from float64 than those
// of the split kernels.  Of the two large tiles the one whose rounds over the compute units are shorter, four rounds of the smaller one
// against 3.5 of the larger (LDS and the operands' second reading: 16384 x 2048 x 2048 1276 us on 2, 1084 on 3; 1024 tiles of 16384 x 1024 x 1024
// 328 and 296; 378 of 8000 x 768 x 768 103 and 123; 320 of 2500 x 2048 x 2048 198 and 287; 314 of 20000 x 256 x 256 36 and 52).
// Tiles of 64 rows fetch three quarters of the bytes to a matrix instruction and need a round of workgroups and more than a few trips of K
// (4 / 1, fp32: 1000 x 1024 x 1024 28.0 / 32.2, 2000 x 1536 x 1536 106 / 131, 4000 x 512 x 512 31.8 / 32.4; 1000 x 768 x 768, 768 tiles of 32 x 32,
// 22.3 / 19.7; 8000 x 384 x 384 36.8 / 36.2, 8000 x 256 x 256 20.8 / 18.9, 64 x 50257 x 256 32.3 / 28.2), and no rows that are mostly behind the end.
static int ga_pick(int M, int N, int K) {
  const long long t128 = (long long)((M + 127) / 128) * ((N + 127) / 128);
  const long long t32 = (long long)((M + 31) / 32) * ((N + 31) / 32);
  if (t32 < 128) return 0;
  if (t128 <= 256 || (std::min(M, N) <= 64 && N <= 65535 * 32))
    return t32 >= 1024 && K >= 512 && 16 * ((M + 63) / 64) * (long long)((N + 31) / 32) <= 9 * t32 ? 4 : 1;
  const long long t64 = (long long)((M + 63) / 64) * ((N + 63) / 64), cus = fstu_cus();
  const long long r128 = (t128 + cus - 1) / cus, r64 = (t64 + cus - 1) / cus;
  return 115 * r64 < 400 * r128 && (N + 63) / 64 <= 65535 ? 2 : 3;
}

template <typename T, bool VA, bool VW>
static void ga_launch(const T* A, long long sam, long long sak, const T* W, long long swn, long long swk, T* C, long long ldc,
                      int M, int N, int K, hipStream_t s) {
  switch (ga_pick(M, N, K)) {
    case 0:
      hipLaunchKernelGGL((gemm_any_split_kernel<T, VA, VW, 1, 1, 16, 4>), dim3((M + 15) / 16, (N + 15) / 16), dim3(1024), 0, s, A, sam,
                         sak, W, swn, swk, C, ldc, M, N, K);
      break;
    case 1:        // one group of 16 k requested at a time: more waves on a compute unit cover a trip better than a second group (fp32, us, two / one:
                   // 1000 x 512 x 512 12.2 / 10.9, 300 x 768 x 768 10.2 / 9.3, 2400 x 256 x 3072 73 / 67, 64 x 50257 x 256 33.0 / 28.2),
                   // but not where both operands are read element by element and no compute unit has a second workgroup (128 x 1024 x 18432
                   // 135 / 145, 256 x 768 x 6144 49 / 51, with 520 workgroups 2080 x 256 x 6144 132 / 123)
      if constexpr (!VA && !VW) {
        if ((long long)((M + 31) / 32) * ((N + 31) / 32) <= fstu_cus()) {
          hipLaunchKernelGGL((gemm_any_split_kernel<T, VA, VW, 2, 2, 8, 2>), dim3((M + 31) / 32, (N + 31) / 32), dim3(512), 0, s, A, sam,
                             sak, W, swn, swk, C, ldc, M, N, K);
          break;
        }
      }
      hipLaunchKernelGGL((gemm_any_split_kernel<T, VA, VW, 2, 2, 8, 1>), dim3((M + 31) / 32, (N + 31) / 32), dim3(512), 0, s, A, sam,
                         sak, W, swn, swk, C, ldc, M, N, K);
      break;
    case 4:
      hipLaunchKernelGGL((gemm_any_split_kernel<T, VA, VW, 4, 2, 8, 1>), dim3((M + 63) / 64, (N + 31) / 32), dim3(512), 0, s, A, sam,
                         sak, W, swn, swk, C, ldc, M, N, K);
      break;
    case 2:
      hipLaunchKernelGGL((gemm_any_tile_kernel<T, VA, VW, 64>), dim3((M + 63) / 64, (N + 63) / 64), dim3(256), 0, s, A, sam, sak, W, swn, swk,
                         C, ldc, M, N, K);
      break;
    default:
      hipLaunchKernelGGL((gemm_any_tile_kernel<T, VA, VW, 128>), dim3((M + 127) / 128, (N + 127) / 128), dim3(256), 0, s, A, sam, sak, W, swn,
                         swk, C, ldc, M, N, K);
  }
}

}  // namespace

// C (M, N; row stride ldc) = T(A W^T) with A element (m, k) at A[m*sam + k*sak] and W element (n, k) at
// W[n*swn + k*swk] (strides in elements, any sign-free combination); fp32 accumulation, one rounding.
extern "C" int fstu_gemm_any(const void* A, int64_t sam, int64_t sak, const void* W, int64_t swn, int64_t swk, void* C,
                             int64_t ldc, int M, int N, int K, int dtype, void* stream) {
  FSTU_REQUIRE(A && W && C, FSTU_ENULL, "fstu_gemm_any: null pointer");
  FSTU_REQUIRE(M >= 1 && N >= 1 && K >= 1 && ldc >= N, FSTU_ESHAPE, "fstu_gemm_any: M=%d N=%d K=%d ldc=%lld", M, N, K, (long long)ldc);
  FSTU_REQUIRE(sam >= 0 && sak >= 0 && swn >= 0 && swk >= 0 && (sam > 0 || M == 1) && (sak > 0 || K == 1) && (swn > 0 || N == 1) &&
                   (swk > 0 || K == 1),
               FSTU_ESHAPE, "fstu_gemm_any: strides must be positive (sam=%lld sak=%lld swn=%lld swk=%lld)", (long long)sam,
               (long long)sak, (long long)swn, (long long)swk);
  FSTU_REQUIRE(N <= 65535 * 128, FSTU_ESHAPE, "fstu_gemm_any: N=%d too large", N);
  // four elements per load: k contiguous, rows on 4-element boundaries, K a whole number of fours
  const size_t quad = dtype == FSTU_BF16 ? 8 : 16;
  const bool va = sak == 1 && K % 4 == 0 && (sam % 4 == 0 || M == 1) && fstu_aligned(A, quad);
  const bool vw = swk == 1 && K % 4 == 0 && (swn % 4 == 0 || N == 1) && fstu_aligned(W, quad);
#define GA_GO(VA, VW) ga_launch<T, VA, VW>((const T*)A, sam, sak, (const T*)W, swn, swk, (T*)C, ldc, M, N, K, (hipStream_t)stream)
  FSTU_DISPATCH_DTYPE(dtype, "fstu_gemm_any",
                      if (va && vw) GA_GO(true, true); else if (va) GA_GO(true, false); else if (vw) GA_GO(false, true); else GA_GO(false, false));
#undef GA_GO
  FSTU_CHECK_LAUNCH("fstu_gemm_any");
  return FSTU_OK;
}
