// Packing of bf16 weights into MFMA-fragment order for the decode kernels.
//
// Packed layout (built once on the host side from the (N,K) row-major weight):
//   Wp[tile][kstep][lane][8]   tile = n/16, kstep = k/32, lane = 16*g + r,
//   element e of lane (r,g) is W[16*tile + r][32*kstep + 8*g + e]
// i.e. exactly the A-operand fragment of v_mfma_f32_16x16x32_bf16, so one wave
// load instruction (64 lanes x 16 B) reads 1 KB of contiguous memory and a wave
// that walks a K range streams one contiguous block.  Rows beyond N are zero.
#include "fstu_common.h"

template <int DUMMY>
__global__ void pack_rows_kernel(const bf16_t* __restrict__ W, bf16_t* __restrict__ Wp, int N, int K, int ntiles) {
  // one thread per packed 16-byte fragment
  const size_t nfrag = (size_t)ntiles * (K >> 5) * 64;
  for (size_t f = (size_t)blockIdx.x * blockDim.x + threadIdx.x; f < nfrag; f += (size_t)gridDim.x * blockDim.x) {
    const int lane = f & 63;
    const size_t ts = f >> 6;
    const int kstep = ts % (K >> 5);
    const int tile = ts / (K >> 5);
    const int r = lane & 15, g = lane >> 4;
    const int n = tile * 16 + r;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (n < N) v = *(const uint4*)(W + (size_t)n * K + kstep * 32 + g * 8);
    *(uint4*)(Wp + f * 8) = v;
  }
}

extern "C" int64_t fstu_packed_elems(int N, int K) { return (int64_t)((N + 15) / 16) * 16 * (int64_t)K; }

extern "C" int fstu_pack_rows(const void* W, void* Wp, int N, int K, void* stream) {
  FSTU_REQUIRE(W && Wp, FSTU_ENULL, "fstu_pack_rows: null pointer");
  FSTU_REQUIRE(N >= 1 && K >= 32 && K % 32 == 0, FSTU_ESHAPE, "fstu_pack_rows: N=%d K=%d (K must be a multiple of 32)", N, K);
  FSTU_REQUIRE(fstu_aligned(W, 16) && fstu_aligned(Wp, 16), FSTU_EALIGN, "fstu_pack_rows: pointers must be 16-byte aligned");
  const int ntiles = (N + 15) / 16;
  size_t nfrag = (size_t)ntiles * (K >> 5) * 64;
  unsigned blocks = (unsigned)((nfrag + 255) / 256 > 65535 ? 65535 : (nfrag + 255) / 256);
  hipLaunchKernelGGL(pack_rows_kernel<0>, dim3(blocks), dim3(256), 0, (hipStream_t)stream, (const bf16_t*)W, (bf16_t*)Wp, N,
                     K, ntiles);
  FSTU_CHECK_LAUNCH("fstu_pack_rows");
  return FSTU_OK;
}

// ---------------------------------------------------------------- transpose of the last two dimensions
// out[b][c][r] = in[b][r][c] through 64 x 64 tiles in LDS (rows padded by one 32-bit word so that the transposed reads
// fall into different banks): both the loads and the stores walk the contiguous dimension.  Used to hand a few long
// sequences to the spectral convolution time-major (flash_stu/modules/stu.py:89-98 of the reference convolves
// (B, L, d) tensors along L).
template <typename T>
__global__ void __launch_bounds__(256)
transpose_tiles_kernel(const T* __restrict__ in, T* __restrict__ out, int R, int C) {
  __shared__ T tile[64][64 + 4 / sizeof(T) * 1];
  const int b = blockIdx.z, r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  const int j = threadIdx.x & 63, i0 = threadIdx.x >> 6;
  const T* src = in + (size_t)b * R * C;
  T* dst = out + (size_t)b * R * C;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int i = i0 + 4 * k;
    if (r0 + i < R && c0 + j < C) tile[i][j] = src[(size_t)(r0 + i) * C + c0 + j];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const int i = i0 + 4 * k;
    if (c0 + i < C && r0 + j < R) dst[(size_t)(c0 + i) * R + r0 + j] = tile[j][i];
  }
}

// 16-bit elements, whole 16-byte pieces: a wave transposes 64 x 64 elements in registers, a lane an 8 x 8 block.  Lane (br, bc)
// reads 16 bytes of 8 rows and writes 16 bytes of 8 columns, so that both the loads and the stores of 8 lanes are 128 bytes in
// a row, all loads are in flight at once and there is no LDS between.  Rows R .. Rp of the input are zeros.  What bounds it is
// HBM; us, element by element through LDS -> now: 4096 x 2048 10.7 -> 7.6, 4 x 8192 x 1024 55 -> 28 (4.7 TB/s).
__global__ void __launch_bounds__(256)
transpose16_kernel(const bf16_t* __restrict__ in, size_t in_sb, size_t in_row, bf16_t* __restrict__ out, size_t out_sb, size_t out_row,
                   int R, int Rp, int C, int nx, int tiles) {
  const int lane = threadIdx.x & 63, tile = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tile >= tiles) return;
  const int r0 = tile / nx * 64 + (lane >> 3) * 8, c0 = tile % nx * 64 + (lane & 7) * 8;
  if (r0 >= Rp || c0 >= C) return;
  const bf16_t* src = in + (size_t)blockIdx.y * in_sb + (size_t)r0 * in_row + c0;
  bf16_t* dst = out + (size_t)blockIdx.y * out_sb + (size_t)c0 * out_row + r0;
  unsigned v[8][4];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    uint4 t = make_uint4(0, 0, 0, 0);
    if (r0 + k < R) t = *(const uint4*)(src + (size_t)k * in_row);
    v[k][0] = t.x; v[k][1] = t.y; v[k][2] = t.z; v[k][3] = t.w;
  }
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    unsigned o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o[j] = __builtin_amdgcn_perm(v[2 * j + 1][c >> 1], v[2 * j][c >> 1], (c & 1) ? 0x07060302 : 0x05040100);
    *(uint4*)(dst + (size_t)c * out_row) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// C a multiple of 8, Rp of 8 and >= R, all strides multiples of 8, 16-byte aligned: the caller's to check
int fstu_transpose16_launch(const void* in, size_t in_sb, size_t in_row, void* out, size_t out_sb, size_t out_row, int B, int R,
                            int Rp, int C, void* stream) {
  const int nx = (C + 63) / 64;
  const long long tiles = (long long)nx * ((Rp + 63) / 64);
  FSTU_REQUIRE(B >= 1 && B <= 65535 && tiles < (1ll << 30), FSTU_ESHAPE, "fstu_transpose: B=%d R=%d C=%d", B, Rp, C);
  hipLaunchKernelGGL(transpose16_kernel, dim3((unsigned)((tiles + 3) / 4), B), dim3(256), 0, (hipStream_t)stream, (const bf16_t*)in, in_sb,
                     in_row, (bf16_t*)out, out_sb, out_row, R, Rp, C, nx, (int)tiles);
  FSTU_CHECK_LAUNCH("fstu_transpose");
  return FSTU_OK;
}

extern "C" int fstu_transpose(const void* in, void* out, int B, int R, int C, int dtype, void* stream) {
  FSTU_REQUIRE(in && out && in != out, FSTU_ENULL, "fstu_transpose: null or aliased pointers");
  FSTU_REQUIRE(B >= 1 && B <= 65535 && R >= 1 && C >= 1 && (R + 63) / 64 <= 65535, FSTU_ESHAPE, "fstu_transpose: B=%d R=%d C=%d", B, R, C);
  if (dtype == FSTU_BF16 && R % 8 == 0 && C % 8 == 0 && fstu_aligned(in, 16) && fstu_aligned(out, 16))
    return fstu_transpose16_launch(in, (size_t)R * C, C, out, (size_t)R * C, R, B, R, R, C, stream);
  const dim3 grid((C + 63) / 64, (R + 63) / 64, B);
  FSTU_DISPATCH_DTYPE(dtype, "fstu_transpose",
                      hipLaunchKernelGGL(transpose_tiles_kernel<T>, grid, dim3(256), 0, (hipStream_t)stream, (const T*)in, (T*)out, R, C));
  FSTU_CHECK_LAUNCH("fstu_transpose");
  return FSTU_OK;
}
