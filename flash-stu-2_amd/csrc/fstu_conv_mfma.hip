// Spectral convolution of the STU as a Toeplitz product on the matrix cores (bf16, up to 4096 positions).
//
// Both operands of the convolution are bf16 (the projected inputs and phi_proj, flash_stu/modules/stu.py:88-98 of the
// reference), so every product x[u] f[t-u] is exact in fp32 and the sums are fp32: no transform, no twiddle rounding.  The two
// sign branches are plus = E + O and minus = E - O with E, O the sums over the even and odd lags (stu_utils.py:214-228); lags of
// one parity connect positions of fixed parities, so with x_p[m] = x[2m+p], fe[j] = f[2j], fo[j] = f[2j+1]
//   E_p[m] = sum_j fe[j] x_p[m-j],   O_1[m] = sum_j fo[j] x_0[m-j],   O_0[m+1] = W[m] = sum_j fo[j] x_1[m-j].
//
// One v_mfma_f32_16x16x32_bf16 forms 16 positions (rows i) of 16 columns, a column being a block of 64 positions of one
// parity of one sequence: D[i][col] += sum_k A[i][k] B[k][col] with B = 32 consecutive inputs of the column's own sequence, 32 s
// positions before the end of its block, and A[i][k] = f[16 a + i - k], a = 2s - 2 + row tile, the same for every column.  Four
// row tiles and the two filters share a B fragment, all tiles of columns share the filter fragments, and a fragment serves the
// row tiles of two successive steps from registers.
// A lane's 8 filter values start at any alignment, so the filter lies in LDS eight times, shifted by one element each; a wave
// expands 64 lags at a time into a ring of its own, from a time-major reversed copy (fstu_stu_conv_taps) read ahead.
//
// A workgroup has 8 channels (16 bytes of a row) of R sequences with R * NB = 8 blocks to a tile; the rows travel through LDS
// once, transposed 8 x 8 in registers, and a wave works on a channel by itself, so there are two barriers in all.  The result
// replaces the channel's inputs in LDS and leaves the way it came.
//
// us, transforms -> this: 8 x 512 x 768 16 -> 10.1, 32 x 300 x 2048 100 -> 47.5, 8 x 2048 x 768 61 -> 42, 1 x 4096 x 2048 56 (with a
// transpose) -> 43.6.  What bounds the longest two is the matrix cores: 2.36 and 2.62 M products of 16 x 16 x 32, which this card
// issues every 20 cycles on random operands, are 19 and 21 us; the rows' way in and out, 5 and 2 us, is not hidden behind them,
// because all workgroups that fit start together.  Blocks of 32 positions would save a sixth of the products, but the filter
// fragments then serve half as many each and the LDS becomes the bound (47 us).
#include "fstu_common.h"
#include <type_traits>
#include <algorithm>

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

constexpr int CM_RING = 4096;        // bytes of a wave's ring: 2 filters x 16 groups of 8 lags x 8 shifts x 16 bytes
// A 16-byte LDS read serves 16 lanes at a time, the lanes 0-3, 12-15, 20-27 of each half wave and then the others, from 64 banks.
// The 16-byte pieces of a block of 64 positions are permuted by the block's number, the parities lie whole multiples of 256
// bytes apart and the sequences NB blocks more, and in the ring the shifts of every other pair of groups are rotated by four:
// 16 different slots for every read of the products.
constexpr int cm_region(int HB) { return (128 * (1 + HB) + 255) & ~255; }      // a channel's parity, a block of zeros in front
constexpr int cm_row(int HB, int NB) { return 16 * cm_region(HB) + (NB < 8 ? 128 * NB : 0); }
__device__ __forceinline__ int ring_at(int n, int shift) { return (n & 15) * 128 + ((shift * 16) ^ (n & 2 ? 64 : 0)); }
__device__ __forceinline__ int piece_at(int block, int piece) { return 128 * block + ((piece ^ (block & 6)) * 16); }   // block -1: zeros

__device__ __forceinline__ bf16x8_t as_frag(uint4 v) { return __builtin_bit_cast(bf16x8_t, v); }

// LDS accesses of one wave are served in order: what one lane writes another lane reads once the compiler keeps the order too.
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The workgroup's 8 channels and first sequence.  The 8 workgroups that share the 128-byte lines of 64 channels run on one XCD
// (consecutive workgroups are dealt to the 8 XCDs in turn), so that a line is fetched into one L2.
__device__ __forceinline__ bool cm_place(int d, int rows, int R, int& c0, int& row0) {
  const int nu = (d + 63) >> 6, unit = (blockIdx.x >> 6) * 8 + (blockIdx.x & 7);
  c0 = unit % nu * 64 + ((blockIdx.x >> 3) & 7) * 8;
  row0 = unit / nu * R;
  return row0 < rows && c0 < d;
}

// M positions of one parity x 8 channels, dwords [position][channel pair] -> [channel][position pair], or N channels back
template <int M, int N>
__device__ __forceinline__ void transpose8(const unsigned (&v)[M][N / 2], unsigned (&o)[N][M / 2]) {
#pragma unroll
  for (int c = 0; c < N; ++c)
#pragma unroll
    for (int j = 0; j < M / 2; ++j)
      o[c][j] = __builtin_amdgcn_perm(v[2 * j + 1][c >> 1], v[2 * j][c >> 1], (c & 1) ? 0x07060302 : 0x05040100);
}

// 5 dwords of taps, loaded as they are stored: the last four are a write of their own.  Where the compiler loads the first four together it
// copies them to where the write wants them as soon as they are there, that is, waits for them one product after they were requested:
// us so / apart / apart and a channel's first taps with the inputs or in front of the results before, 4 x 4096 x 2048 164 / 155.6 / 153.4,
// 1 x 4096 x 2048 46.1 / 44.3 / 43.6, 32 x 300 x 2048 50.8 / 49.8 / 47.5, 8 x 2048 x 768 42.5 / 42.2 / 41.3, 8 x 1024 x 768 20.4 / 19.1,
// 3 x 777 x 768 12.0 / 11.1.
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef u32x4_t u32x4_a4_t __attribute__((aligned(4)));
struct Taps5 { unsigned first; u32x4_t rest; };

// NT tiles of NB = 1 << NBS blocks to a parity, NW waves, OCC of them to a SIMD
template <int NT, int NBS, int NW, int OCC>
__global__ void __launch_bounds__(NW * 64, OCC)
conv_mfma_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ taps, bf16_t* __restrict__ y, int B, int T, int d,
                 int single) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int NB = 1 << NBS, R = 8 >> NBS, HB = NB * NT;   // blocks of a tile, sequences, blocks of a parity
  constexpr int rg = cm_region(HB), rws = cm_row(HB, NB);
  int c0, row0;
  if (!cm_place(d, B, R, c0, row0)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // expansion: 5 dwords of the reversed taps give the shifts 2a and 2a+1 of a group of 8 lags
  const int xf = lane >> 5, xn = (lane >> 2) & 7, xa = lane & 3;
  constexpr int cap = 64 * HB, S = cap + 16;                 // HB pairs of steps
  constexpr int DEPTH = HB < 2 ? 1 : NT == 4 ? 4 : 2;        // groups of 64 taps on their way
  constexpr bool EARLY = NT > 1 || NBS < 3;                  // the next channel's are requested in front of this one's results, where registers are left
  unsigned one = 1;
  asm("" : "+v"(one));                                       // two loads: see Taps5
  const unsigned *tp, *tp1;
  Taps5 w[DEPTH], wf;
  auto fetch = [&](Taps5& r, int P) {
    r.first = *(tp - 32 * min(P, HB - 1));
    r.rest = *(const u32x4_a4_t*)(tp1 - 32 * min(P, HB - 1));
  };
  auto first_taps = [&](int ch) {
    tp = (const unsigned*)(taps + ((size_t)(c0 + ch) * 2 + xf) * S + cap - 8 * xn - 2 * xa - 2);
    tp1 = tp + one;
    fetch(wf, 0);
#pragma unroll
    for (int k = 0; k < DEPTH; ++k) fetch(w[k], k + 1);
  };
  if (EARLY) first_taps(wave);                               // with the inputs: one trip
  const int pieces = R * HB * 16;                           // (sequence, 8 positions of one parity)
  for (int v = tid; v < R * 128; v += NW * 64)               // the zeros in front of every region
    *(uint4*)(lds + (v >> 7) * rws + ((v >> 3) & 15) * rg + (v & 7) * 16) = make_uint4(0, 0, 0, 0);
  for (int v = tid; v < pieces; v += NW * 64) {
    const int mu = v & (HB * 8 - 1), p = (v / (HB * 8)) & 1, row = v / (HB * 16), t0 = 16 * mu + p;
    const bf16_t* src = x + ((size_t)(row0 + row) * T + t0) * d + c0;
    unsigned a[8][4], o[8][4];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      uint4 q = make_uint4(0, 0, 0, 0);
      if (t0 + 2 * e < T && row0 + row < B) q = *(const uint4*)(src + (size_t)(2 * e) * d);
      a[e][0] = q.x; a[e][1] = q.y; a[e][2] = q.z; a[e][3] = q.w;
    }
    transpose8<8, 8>(a, o);
    char* dst = lds + row * rws + p * rg + 128 + piece_at(mu >> 3, mu & 7);
#pragma unroll
    for (int c = 0; c < 8; ++c) *(uint4*)(dst + c * 2 * rg) = make_uint4(o[c][0], o[c][1], o[c][2], o[c][3]);
  }
  __syncthreads();

  const int col = lane & 15, g = lane >> 4;
  const int par = col >> 3, cc = col & 7, row = cc >> NBS, q = cc & (NB - 1);
  char* const ring = lds + R * rws + wave * CM_RING;
  char* const xdst = ring + xf * 2048 + ring_at(xn, 2 * xa);
  const int fh = (col >> 3) - g;                             // group of the lane's first filter value
  int fat[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) fat[k] = ring_at(fh + 2 * k, col & 7);

  for (int ch = wave; ch < 8; ch += NW) {
    auto expand = [&](const Taps5& r, bool odd) {
      char* dst = xdst + odd * 1024;
      *(u32x4_t*)dst = r.rest;
      *(uint4*)(dst + 16) = make_uint4(__builtin_amdgcn_alignbit(r.rest[0], r.first, 16), __builtin_amdgcn_alignbit(r.rest[1], r.rest[0], 16),
                                       __builtin_amdgcn_alignbit(r.rest[2], r.rest[1], 16), __builtin_amdgcn_alignbit(r.rest[3], r.rest[2], 16));
    };
    if (!EARLY) first_taps(ch);
    wave_order();
    if (lane < 48) *(uint4*)(ring + (lane / 24) * 2048 + 13 * 128 + (lane % 24) * 16) = make_uint4(0, 0, 0, 0);   // lags below 0
    expand(wf, false);
    wave_order();
    floatx4_t E[NT][4], O[NT][4];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) E[j][r] = O[j][r] = (floatx4_t){0.f, 0.f, 0.f, 0.f};
    char* const region = lds + row * rws + (ch * 2 + par) * rg + 128;
    uint4 fa[2][2], fb[2][2];                                 // [filter][a]: fragments of the row tiles 0, 1 and 2, 3
#pragma unroll
    for (int k = 0; k < 2; ++k) fa[k][0] = fa[k][1] = make_uint4(0, 0, 0, 0);
    // A pair of steps, 64 lags, for the tiles from J0 on; the next 64 lags are expanded behind the last reads of these.
    auto pair = [&](auto first, int P, bool odd, Taps5& r) {
      constexpr int J0 = decltype(first)::value;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        uint4 (&old)[2][2] = s ? fb : fa;
        uint4 (&now)[2][2] = s ? fa : fb;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const char* p = ring + (odd ? fat[2 * s + k] ^ 1024 : fat[2 * s + k]);
          now[0][k] = *(const uint4*)p;
          now[1][k] = *(const uint4*)(p + 2048);
        }
        uint4 b[NT];
#pragma unroll
        for (int j = J0; j < NT; ++j) b[j] = *(const uint4*)(region + piece_at(max(q + NB * j - P, -1), s ? g : g + 4));
        if (s == 1) {
          wave_order();
          expand(r, !odd);
          fetch(r, P + 1 + DEPTH);
          wave_order();
        }
#pragma unroll
        for (int j = J0; j < NT; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            E[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(i < 2 ? old[0][i] : now[0][i - 2]), as_frag(b[j]), E[j][i], 0, 0, 0);
            O[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(i < 2 ? old[1][i] : now[1][i - 2]), as_frag(b[j]), O[j][i], 0, 0, 0);
          }
      }
    };
    // tile j sees the lags of its own and all earlier blocks, j + 1 phases of NB pairs, as far as there are positions
    const int blocks = (T + 127) >> 7;
    auto phase = [&](auto first) {
      constexpr int J = decltype(first)::value;
      if constexpr (J < NT) {
#pragma unroll 1
        for (int P = J * NB; P < min((J + 1) * NB, blocks); P += DEPTH)
#pragma unroll
          for (int k = 0; k < DEPTH; ++k) pair(first, P + k, k & 1, w[k]);
      }
    };
    phase(std::integral_constant<int, 0>{});
    phase(std::integral_constant<int, 1>{});
    phase(std::integral_constant<int, 2>{});
    phase(std::integral_constant<int, 3>{});
    wave_order();

    if (EARLY && ch + NW < 8) first_taps(ch + NW);

    // Branches and rounding.  A lane of an x_0 column has E_0 and O_1, of an x_1 column E_1 and W = O_0 one position early.  The other
    // column's values cross over by a rotation within 16 lanes; W of the position before the lane's four comes from the lane 16
    // below, of the row tile or block before it where the lane has the first four.
    const int from = (g ? lane - 16 : lane + 48) * 4, from_block = (g ? lane - 16 : 48 + (col & 8) + (cc + 7) % 8) * 4;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      floatx4_t cross[4];
      const float tile_before = j ? fstu_dpp<0x128>(O[j ? j - 1 : 0][3][3]) : 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int k = 0; k < 4; ++k) cross[r][k] = fstu_dpp<0x128>(O[j][r][k]);          // row_ror:8
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float last;                                            // what this lane hands on
        if (r) {
          last = g == 3 ? cross[r - 1][3] : cross[r][3];
        } else {
          last = g != 3 ? cross[0][3] : q == NB - 1 ? tile_before : cross[3][3];
        }
        int src = r ? from : from_block;
        if (r == 0 && NB < 8 && g == 0 && q == 0) src = (48 + (col & 8) + cc + NB - 1) * 4;    // its own sequence's last block
        const float prev = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(last)));
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float o = par ? cross[r][k] : k ? cross[r][k ? k - 1 : 0] : prev;
          const float e = E[j][r][k];
          v[k] = single ? e + o : DT<bf16_t>::rnd(e + o) + DT<bf16_t>::rnd(e - o);
        }
        *(uint2*)(region + piece_at(q + NB * j, 2 * r + (g >> 1)) + (g & 1) * 8) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
      }
    }
    wave_order();
  }
  __syncthreads();

  for (int v = tid; v < pieces; v += NW * 64) {
    const int mu = v & (HB * 8 - 1), p = (v / (HB * 8)) & 1, rw = v / (HB * 16), t0 = 16 * mu + p;
    if (t0 >= T || row0 + rw >= B) continue;
    const char* src = lds + rw * rws + p * rg + 128 + piece_at(mu >> 3, mu & 7);
    unsigned a[8][4], o[8][4];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const uint4 t = *(const uint4*)(src + c * 2 * rg);
      a[c][0] = t.x; a[c][1] = t.y; a[c][2] = t.z; a[c][3] = t.w;
    }
    transpose8<8, 8>(a, o);
    bf16_t* dst = y + ((size_t)(row0 + rw) * T + t0) * d + c0;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (t0 + 2 * e < T) *(uint4*)(dst + (size_t)(2 * e) * d) = make_uint4(o[e][0], o[e][1], o[e][2], o[e][3]);
  }
}

// ---------------------------------------------------------------- gradients
// y = plus + minus = 2 E, so only the even lags have gradients: with g the gradient of y,
//   gx_p[m] = 2 sum_j fe[j] g_p[m+j],   gfe[j] = 2 sum_{rows, p, v} g_p[v] x_p[v-j].
// Both are products with the same Hankel matrix of g, A[i][k] = g_p[32 s + 16 r + i + k]: for block c of 64 positions (or lags)
// and row tile r, B[k][c] = fe[32 s + k - 64 c] gives gx_p[64 c + 16 r + i] and x_p[32 s + k - 64 c] gives gfe[64 c + 16 r + i].
// Eight of an MFMA's 16 columns are blocks of lags and eight of positions, so both come out of one pass over g, whose shifted
// copies a wave expands into its ring from g in LDS.  The parities of a row meet only in the filter's sums, so an item of work is one
// parity of one row: 70 KB of LDS at 2048 positions, and a second workgroup on the compute unit works while this one's operands come
// and its results go.  A workgroup has 8 channels, a wave each, and goes through R items: the sums of the filter's gradient stay in
// registers, and the next item is on its way while this one is worked on.  What it leaves are its items' fp32 sums, (chunks of
// items, lags, channels), added in the order of the items by conv_grad_finish_kernel.  Where the filter is phi @ M_filters, it leaves
// their product with the even rows of phi instead, phi_e (filters to whole tiles of 16, P lags), (chunks, filters, channels): a 42nd
// of the bytes at 1024 lags and 24 filters, and no product behind the launch.  Eight of an MFMA's columns are the channels' sums rounded to
// bf16, the other eight what that leaves of them, so a sum enters with 16 bits (8 as the gradient of the filter itself: 2.83e-3 off
// float64 after its rounding, 2.44e-3 so).  8 x 2048 x 768 with the launch behind it 56 + 5 + 17 us (sums, their join, the library's
// product) -> 60 + 5.
//
// us, transforms -> whole rows (106 KB, one workgroup to a compute unit) -> this, both launches: 8 x 512 x 768 29 -> 26 -> 22, 8 x 1024 x
// 768 51 -> 39 -> 32, 2 x 2048 x 768 42 -> 27 -> 25, 8 x 2048 x 768 117 -> 80 -> 62, 8 x 2048 x 2048 - -> 163 -> 128.  A row's products alone
// are 6.4 us of a compute unit, 11 with the LDS reads in front of them; the latter bound it now.
constexpr int cg_rows(int HB) { return 128 * HB + 256; }        // bytes of a channel of g: zeros behind it

template <int NT, bool PROJECT>
__global__ void __launch_bounds__(512, 4)
conv_grad_mfma_kernel(const bf16_t* __restrict__ gy, const bf16_t* __restrict__ x, const bf16_t* __restrict__ f, bf16_t* __restrict__ gx,
                      float* __restrict__ part, const bf16_t* __restrict__ phi_e, int K, int P, int B, int T, int L, int d, int R) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int HB = 8 * NT, cap = 64 * HB, rg = cm_region(HB), gg = cg_rows(HB), PC = HB * 16;
  char* const xl = lds;                                       // 8 regions as in the forward
  char* const fl = xl + 8 * rg;                               // 8 more: the even taps
  char* const gl = fl + 8 * rg;                               // 8 of g, in order
  char* const rings = gl + 8 * gg;
  int c0, item0;                                              // item 2 b + p: parity p of row b
  if (!cm_place(d, 2 * B, R, c0, item0)) return;
  const int tid = threadIdx.x, end = min(item0 + R, 2 * B);
  if (tid < 16 * 8) *(uint4*)(lds + (tid >> 3) * rg + (tid & 7) * 16) = make_uint4(0, 0, 0, 0);
  if (tid < 8 * 16) *(uint4*)(gl + (tid >> 4) * gg + 128 * HB + (tid & 15) * 16) = make_uint4(0, 0, 0, 0);
  if (tid < HB * 8) {
    unsigned a[8][4], o[8][4];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int t = 2 * (8 * tid + e);
      uint4 v = make_uint4(0, 0, 0, 0);
      if (t < L) v = *(const uint4*)(f + (size_t)t * d + c0);
      a[e][0] = v.x; a[e][1] = v.y; a[e][2] = v.z; a[e][3] = v.w;
    }
    transpose8<8, 8>(a, o);
#pragma unroll
    for (int c = 0; c < 8; ++c)
      *(uint4*)(fl + c * rg + 128 + piece_at(tid >> 3, tid & 7)) = make_uint4(o[c][0], o[c][1], o[c][2], o[c][3]);
  }
  // A thread's piece: 4 positions of the item's parity of x (the first PC threads) or of g
  const int mu = tid % PC;
  const bool has = tid < 2 * PC, is_g = tid >= PC;
  unsigned in[4][4];
  auto request = [&](int item) {
    const int t0 = 8 * mu + (item & 1);
    const bf16_t* src = (is_g ? gy : x) + ((size_t)(item >> 1) * T + t0) * d + c0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint4 v = make_uint4(0, 0, 0, 0);
      if (has && t0 + 2 * e < T) v = *(const uint4*)(src + (size_t)(2 * e) * d);
      in[e][0] = v.x; in[e][1] = v.y; in[e][2] = v.z; in[e][3] = v.w;
    }
  };
  request(item0);

  const int lane = tid & 63, ch = tid >> 6, col = lane & 15, g = lane >> 4, c = col & 7;
  char* const ring = rings + ch * 2048;
  const int xn = lane >> 3, xs = lane & 7, odd = (xs & 1) * 16;   // expansion: one shift of a group of 8
  const int xdst = ring_at(xn, xs);
  const int fh = (col >> 3) + g;
  int fat[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) fat[k] = ring_at(fh + 4 + 2 * k, col & 7);
  const int fat0 = ring_at(fh, col & 7), fat1 = ring_at(fh + 2, col & 7);
  const int blocks = (T + 127) >> 7;
  floatx4_t S[NT][4];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[j][r] = (floatx4_t){0.f, 0.f, 0.f, 0.f};

  for (int item = item0; item < end; ++item) {
    if (has) {
      unsigned o[8][2];
      transpose8<4, 8>(in, o);
      char* const dst = is_g ? gl + mu * 8 : xl + 128 + piece_at(mu >> 4, (mu >> 1) & 7) + (mu & 1) * 8;
#pragma unroll
      for (int k = 0; k < 8; ++k) *(uint2*)(dst + k * (is_g ? gg : rg)) = make_uint2(o[k][0], o[k][1]);
    }
    __syncthreads();
    if (item + 1 < end) request(item + 1);
    char* const own = gl + ch * gg;
    const char* const bl = (col < 8 ? xl : fl) + ch * rg + 128;
    const char* const win = own + xn * 16 + (xs >> 1) * 4;
    unsigned w[5];
    auto window = [&](int P) {
#pragma unroll
      for (int k = 0; k < 5; ++k) w[k] = *(const unsigned*)(win + 128 * min(P, HB) + 4 * k);
    };
    auto expand = [&](bool oddp) {
      *(uint4*)(ring + xdst + oddp * 1024) =
          make_uint4(__builtin_amdgcn_alignbit(w[1], w[0], odd), __builtin_amdgcn_alignbit(w[2], w[1], odd),
                     __builtin_amdgcn_alignbit(w[3], w[2], odd), __builtin_amdgcn_alignbit(w[4], w[3], odd));
    };
    wave_order();
    window(0);
    expand(false);
    window(1);
    expand(true);
    window(2);
    wave_order();
    uint4 fa[2], fb[2];
    fa[0] = *(const uint4*)(ring + fat0);
    fa[1] = *(const uint4*)(ring + fat1);
    // A pair of steps, 64 positions of g, for the tiles up to J1: fragments of row tiles 0, 1 from the step before, 2, 3 now
    auto pair = [&](auto last, int P, bool oddp) {
      constexpr int J1 = decltype(last)::value;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        uint4 (&old)[2] = s ? fb : fa;
        uint4 (&now)[2] = s ? fa : fb;
#pragma unroll
        for (int k = 0; k < 2; ++k) now[k] = *(const uint4*)(ring + (oddp ? fat[2 * s + k] ^ 1024 : fat[2 * s + k]));
        uint4 b[NT];
#pragma unroll
        for (int j = 0; j <= J1; ++j) b[j] = *(const uint4*)(bl + piece_at(max(P - c - 8 * j, -1), s ? g + 4 : g));
        if (s == 1) {
          wave_order();
          expand(oddp);
          window(P + 3);
          wave_order();
        }
#pragma unroll
        for (int j = 0; j <= J1; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            S[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(i < 2 ? old[i] : now[i - 2]), as_frag(b[j]), S[j][i], 0, 0, 0);
      }
    };
#pragma unroll 1
    for (int P = 0; P < min(8, blocks); P += 2) {
      pair(std::integral_constant<int, 0>{}, P, false);
      pair(std::integral_constant<int, 0>{}, P + 1, true);
    }
    if constexpr (NT == 2) {
#pragma unroll 1
      for (int P = 8; P < blocks; P += 2) {
        pair(std::integral_constant<int, 1>{}, P, false);
        pair(std::integral_constant<int, 1>{}, P + 1, true);
      }
    }
    // this parity's gradient of x takes g's place; its columns start from zero again
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (col >= 8) {
          *(uint2*)(own + ((c + 8 * j) * 64 + 16 * r + 4 * g) * 2) = make_uint2(pack2_bf16(2.f * S[j][r][0], 2.f * S[j][r][1]),
                                                                              pack2_bf16(2.f * S[j][r][2], 2.f * S[j][r][3]));
          S[j][r] = (floatx4_t){0.f, 0.f, 0.f, 0.f};
        }
    __syncthreads();
    const int t0 = 8 * mu + (item & 1);
    if (gx && tid < PC && t0 < T) {
      unsigned a[8][2], o[4][4];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint2 v = *(const uint2*)(gl + k * gg + mu * 8);
        a[k][0] = v.x; a[k][1] = v.y;
      }
      transpose8<8, 4>(a, o);
      bf16_t* dst = gx + ((size_t)(item >> 1) * T + t0) * d + c0;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (t0 + 2 * e < T) *(uint4*)(dst + (size_t)(2 * e) * d) = make_uint4(o[e][0], o[e][1], o[e][2], o[e][3]);
    }
    if (item + 1 < end) __syncthreads();
  }
  if (!part) return;
  constexpr int STEPS = cap / 256;
  const int lag0 = ch * (cap / 8) + 8 * g;
  uint4 ph[2][STEPS];
  auto rows_of_phi = [&](int k0) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int step = 0; step < STEPS; ++step) {
        ph[t][step] = make_uint4(0, 0, 0, 0);
        if (k0 + 16 * t < K && lag0 + 32 * step < P) ph[t][step] = *(const uint4*)(phi_e + (size_t)(k0 + 16 * t + col) * P + lag0 + 32 * step);
      }
  };
  if constexpr (PROJECT) rows_of_phi(0);
  // lags of a channel -> channels of a lag, through the space of x and the taps
  float* const fl32 = (float*)xl;
  if (col < 8) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) *(floatx4_t*)(fl32 + ch * (cap + 4) + (c + 8 * j) * 64 + 16 * r + 4 * g) = S[j][r];
  }
  __syncthreads();
  if constexpr (PROJECT) {
    // wave ch: an eighth of the lags; the waves' tiles of 2 x 16 filters x (8 channels, 8 remainders) meet in the space of g and the rings
    float* const red = (float*)gl;
    for (int k0 = 0; k0 < K; k0 += 32) {
      floatx4_t acc[2];
      acc[0] = acc[1] = (floatx4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int step = 0; step < STEPS; ++step) {
        const float* s = fl32 + c * (cap + 4) + lag0 + 32 * step;
        const float4 v0 = *(const float4*)s, v1 = *(const float4*)(s + 4);
        float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        if (col >= 8)
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float head = DT<bf16_t>::rnd(v[e]);
            v[e] = head == v[e] ? 0.f : v[e] - head;           // an infinite sum leaves nothing
          }
        const bf16x8_t b = as_frag(make_uint4(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]), pack2_bf16(v[4], v[5]), pack2_bf16(v[6], v[7])));
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(ph[t][step]), b, acc[t], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) red[ch * 512 + (16 * t + 4 * g + e) * 16 + col] = acc[t][e];
      __syncthreads();
      if (tid < 256 && k0 + (tid >> 3) < K) {
        float sum = 0.f;
#pragma unroll
        for (int w8 = 0; w8 < 8; ++w8) sum += red[w8 * 512 + (tid >> 3) * 16 + (tid & 7)] + red[w8 * 512 + (tid >> 3) * 16 + 8 + (tid & 7)];
        part[((size_t)(item0 / R) * K + k0 + (tid >> 3)) * d + c0 + (tid & 7)] = sum;
      }
      if (k0 + 32 < K) {
        rows_of_phi(k0 + 32);
        __syncthreads();
      }
    }
    return;
  }
  const int lags = min(cap, (min(L, T) + 1) >> 1);
  float* const out = part + (size_t)(item0 / R) * lags * d + c0;
  for (int v = tid; v < lags * 2; v += 512) {
    const float* s = fl32 + (v & 1) * 4 * (cap + 4) + (v >> 1);
    *(float4*)(out + (size_t)(v >> 1) * d + (v & 1) * 4) = make_float4(s[0], s[cap + 4], s[2 * (cap + 4)], s[3 * (cap + 4)]);
  }
}

// gf[2j][c] = 2 * (the chunks' sums in their order), zero at odd lags and beyond the input; 8 channels per thread
__global__ void __launch_bounds__(256) conv_grad_finish_kernel(const float* __restrict__ part, bf16_t* __restrict__ gf, int chunks, int lags,
                                                               int L, int d) {
  const int groups = d >> 3, v = blockIdx.x * 256 + threadIdx.x;
  if (v >= L * groups) return;
  const int s = v / groups, c0 = v % groups * 8;
  float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (!(s & 1) && (s >> 1) < lags)
    for (int k = 0; k < chunks; ++k) {
      const float* p = part + ((size_t)k * lags + (s >> 1)) * d + c0;
      const float4 u = *(const float4*)p, w = *(const float4*)(p + 4);
      a[0] += u.x; a[1] += u.y; a[2] += u.z; a[3] += u.w;
      a[4] += w.x; a[5] += w.y; a[6] += w.z; a[7] += w.w;
    }
  *(uint4*)(gf + (size_t)s * d + c0) = make_uint4(pack2_bf16(2.f * a[0], 2.f * a[1]), pack2_bf16(2.f * a[2], 2.f * a[3]),
                                                  pack2_bf16(2.f * a[4], 2.f * a[5]), pack2_bf16(2.f * a[6], 2.f * a[7]));
}

// gm[i] = 2 * (the chunks' products in their order)
__global__ void __launch_bounds__(256) conv_grad_join_kernel(const float* __restrict__ part, bf16_t* __restrict__ gm, int chunks, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float a = 0.f;
#pragma unroll 8
  for (int k = 0; k < chunks; ++k) a += part[(size_t)k * n + i];
  gm[i] = f32_to_bf16(2.f * a);
}

// taps[c][p][cap - j] = f[2j+p][c] for 0 <= j, zero where the filter has no such lag; 8 channels x 8 places per thread
__global__ void __launch_bounds__(256)
conv_taps_kernel(const bf16_t* __restrict__ f, bf16_t* __restrict__ taps, int L, int d, int cap) {
  const int S = cap + 16, places = S >> 3, groups = d >> 3;
  const int v = blockIdx.x * 256 + threadIdx.x;
  if (v >= 2 * places * groups) return;
  const int c0 = v % groups * 8, p = v / groups & 1, i0 = v / groups / 2 * 8;
  unsigned a[8][4], o[8][4];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int j = cap - i0 - e, s = 2 * j + p;
    uint4 t = make_uint4(0, 0, 0, 0);
    if (j >= 0 && s < L) t = *(const uint4*)(f + (size_t)s * d + c0);
    a[e][0] = t.x; a[e][1] = t.y; a[e][2] = t.z; a[e][3] = t.w;
  }
  transpose8<8, 8>(a, o);
#pragma unroll
  for (int c = 0; c < 8; ++c)
    *(uint4*)(taps + ((size_t)(c0 + c) * 2 + p) * S + i0) = make_uint4(o[c][0], o[c][1], o[c][2], o[c][3]);
}

// The same taps of f = T(phi @ m), and f's first Lf rows.  A workgroup forms 64 places of 128 channels, a whole line of a channel's
// taps, 8 places of 4 channels to a thread, from LDS: both operands come in one trip (2048 x 24 @ 24 x 768 8.8 us; with a trip
// for phi and three for m 11; the product and the taps in launches of their own 7.8 + 5.3).
__global__ void __launch_bounds__(256)
conv_taps_project_kernel(const bf16_t* __restrict__ phi, const bf16_t* __restrict__ m, bf16_t* __restrict__ f, bf16_t* __restrict__ taps, int L,
                         int Lf, int K, int d, int cap) {
  extern __shared__ __attribute__((aligned(16))) float rows[];      // [filter][place], then m's 128 channels, [filter][channel]
  const int tid = threadIdx.x, S = cap + 16, p = blockIdx.y & 1, i0 = (int)(blockIdx.y >> 1) * 64, j0 = cap - i0;
  bf16_t* const cols = (bf16_t*)(rows + 64 * K);
  const int place = tid & 63, s0 = 2 * (j0 - place) + p, piece = (tid & 15) * 8, cp = blockIdx.x * 128 + piece;
  const bool lag = j0 >= place && s0 < L;
  const bf16_t* const src = phi + (size_t)(lag ? s0 : 0) * K;
  for (int k0 = 0; k0 < K; k0 += 32) {
    bf16_t v[8];
    uint4 w[2];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = lag ? src[min(k0 + 4 * i + (tid >> 6), K - 1)] : 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = k0 + 16 * i + (tid >> 4);
      w[i] = make_uint4(0, 0, 0, 0);
      if (k < K && cp < d) w[i] = *(const uint4*)(m + (size_t)k * d + cp);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = k0 + 4 * i + (tid >> 6);
      if (k < K) rows[k * 64 + place] = bf16_to_f32(v[i]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = k0 + 16 * i + (tid >> 4);
      if (k < K) *(uint4*)(cols + k * 128 + piece) = w[i];
    }
  }
  __syncthreads();
  const int e0 = (tid & 7) * 8, c0 = blockIdx.x * 128 + (tid >> 3) * 4;
  if (c0 >= d || i0 + e0 >= S) return;
  float acc[4][8];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[c][e] = 0.f;
#pragma unroll 8
  for (int k = 0; k < K; ++k) {
    const uint2 w = *(const uint2*)(cols + k * 128 + (tid >> 3) * 4);
    const float wv[4] = {__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u), __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u)};
    const float4 r0 = *(const float4*)(rows + k * 64 + e0), r1 = *(const float4*)(rows + k * 64 + e0 + 4);
    const float r[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[c][e] = fmaf(r[e], wv[c], acc[c][e]);
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)
    *(uint4*)(taps + ((size_t)(c0 + c) * 2 + p) * S + i0 + e0) = make_uint4(pack2_bf16(acc[c][0], acc[c][1]), pack2_bf16(acc[c][2], acc[c][3]),
                                                                            pack2_bf16(acc[c][4], acc[c][5]), pack2_bf16(acc[c][6], acc[c][7]));
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int j = j0 - e0 - e, s = 2 * j + p;
    if (j >= 0 && s < Lf) *(uint2*)(f + (size_t)s * d + c0) = make_uint2(pack2_bf16(acc[0][e], acc[1][e]), pack2_bf16(acc[2][e], acc[3][e]));
  }
}

// log2 of the blocks of a tile and the tiles for T positions
void cm_shape(int T, int& nbs, int& nt) {
  nbs = T <= 128 ? 0 : T <= 256 ? 1 : T <= 512 ? 2 : 3;
  nt = T <= 1024 ? 1 : T <= 2048 ? 2 : 4;
}

// Items (a row's two parities) that a workgroup of the gradients goes through: the whole row, or more rows where there are more than
// two workgroups to a compute unit and the parts of the filter's gradient grow; one item where even those leave compute units idle.
// us with 1 / 2 / 4 / 8 items, rows x positions x channels: 1 x 2000 x 768 18 / 22 / - / -, 4 x 2048 x 256 21.5 / 23.4 / 33 / 60,
// 2 x 2048 x 768 28 / 25 / 37 / -, 8 x 2048 x 768 70 / 62 / 65 / 68, 8 x 2048 x 2048 206 / 159 / 133 / 124, 5 x 700 x 1024 27 / 25 / 22 /
// 28, 8 x 512 x 768 29 / 22.9 / 22.0 / 23.5, 64 x 300 x 256 80 / 56 / 44 / 38.
int cg_items(int B, int T, int d) {
  const int groups = (d + 7) / 8, cus = fstu_cus();
  if ((long long)groups * 2 * B <= cus) return 1;
  const int chunks = std::max(1, std::min(B, (T <= 1024 ? 2 : 3) * cus / groups));
  return 2 * ((B + chunks - 1) / chunks);
}

}  // namespace

extern "C" int fstu_stu_conv_taps_len(int T) {
  if (T < 1 || T > 4096) return 0;
  int nbs, nt;
  cm_shape(T, nbs, nt);
  return 64 * (nt << nbs) + 16;
}

// From the length and the width alone, so that a row has the same bits whatever stands beside it, and one layer's operand of a
// length is either taps or spectra.  us, product / best of the transforms' kernels: 8 x 100 x 768 7.1 / 7.7, 8 x 512 x 768 10.5 /
// 16, 32 x 300 x 2048 51 / 100, 1 x 2048 x 768 18 / 23, 8 x 2048 x 768 45 / 61.  Beyond 2048 positions a workgroup fills a compute
// unit, and its 38 us pay for themselves where a round of workgroups is filled by 70 % with any number of rows: 1 x 4096 x 2048
// 45 / 56, 4 x 4096 x 2048 167 / 204.  A width of 1024 would gain with two rows and lose with one (36 / 32), of 768 lose with three
// (75 / 63).  Beyond 4096 the product's operations, which grow with the square of the length, cost more than the transforms.
extern "C" int fstu_stu_conv_mfma_takes(int T, int d) {
  if (T < 32 || T > 4096 || d < 8 || d % 8 != 0 || d > 1 << 20) return 0;
  const int groups = d / 8, cus = fstu_cus();
  return T <= 2048 || 10 * groups >= 7 * cus * ((groups + cus - 1) / cus);
}

extern "C" int fstu_stu_conv_taps(const void* filt, void* taps, int L, int d, int S, void* stream) {
  FSTU_REQUIRE(filt && taps, FSTU_ENULL, "fstu_stu_conv_taps: null pointer");
  FSTU_REQUIRE(L >= 1 && d >= 8 && d % 8 == 0 && d <= 1 << 20 && S >= 80 && S <= 2064 && S % 64 == 16, FSTU_ESHAPE,
               "fstu_stu_conv_taps: L=%d d=%d S=%d (d a multiple of 8, S of fstu_stu_conv_taps_len)", L, d, S);
  FSTU_REQUIRE(fstu_aligned(filt, 16) && fstu_aligned(taps, 16), FSTU_EALIGN, "fstu_stu_conv_taps: pointers must be 16-byte aligned");
  const int n = 2 * (S / 8) * (d / 8);
  hipLaunchKernelGGL(conv_taps_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, (const bf16_t*)filt, (bf16_t*)taps, L, d,
                     S - 16);
  FSTU_CHECK_LAUNCH("fstu_stu_conv_taps");
  return FSTU_OK;
}

extern "C" int fstu_stu_conv_taps_project(const void* phi, const void* m, void* f, void* taps, int L, int K, int d, int S, void* stream) {
  FSTU_REQUIRE(phi && m && f && taps, FSTU_ENULL, "fstu_stu_conv_taps_project: null pointer");
  FSTU_REQUIRE(L >= 1 && K >= 1 && K <= 128 && d >= 8 && d % 8 == 0 && d <= 1 << 20 && S >= 80 && S <= 2064 && S % 64 == 16, FSTU_ESHAPE,
               "fstu_stu_conv_taps_project: L=%d K=%d d=%d S=%d (K up to 128, d a multiple of 8, S of fstu_stu_conv_taps_len)", L, K, d, S);
  FSTU_REQUIRE(fstu_aligned(phi, 2) && fstu_aligned(m, 16) && fstu_aligned(f, 16) && fstu_aligned(taps, 16), FSTU_EALIGN,
               "fstu_stu_conv_taps_project: m, f and taps must be 16-byte aligned");
  hipLaunchKernelGGL(conv_taps_project_kernel, dim3((d + 127) / 128, 2 * ((S + 63) / 64)), dim3(256), 512 * (size_t)K, (hipStream_t)stream, (const bf16_t*)phi,
                     (const bf16_t*)m, (bf16_t*)f, (bf16_t*)taps, L, std::min(L, 2 * (S - 16)), K, d, S - 16);
  FSTU_CHECK_LAUNCH("fstu_stu_conv_taps_project");
  return FSTU_OK;
}

extern "C" int fstu_stu_conv_mfma(const void* x, const void* taps, void* y, int B, int T, int d, int single_branch, void* stream) {
  FSTU_REQUIRE(x && taps && y, FSTU_ENULL, "fstu_stu_conv_mfma: null pointer");
  FSTU_REQUIRE(B >= 1 && B <= 65535 && T >= 1 && T <= 4096 && d >= 8 && d % 8 == 0 && d <= 1 << 20, FSTU_ESHAPE,
               "fstu_stu_conv_mfma: B=%d T=%d d=%d (T up to 4096, d a multiple of 8)", B, T, d);
  FSTU_REQUIRE(fstu_aligned(x, 16) && fstu_aligned(taps, 16) && fstu_aligned(y, 16), FSTU_EALIGN,
               "fstu_stu_conv_mfma: pointers must be 16-byte aligned");
  int nbs, nt;
  cm_shape(T, nbs, nt);
  const int R = 8 >> nbs;
  const long long units = (long long)((d + 63) / 64) * ((B + R - 1) / R);
  FSTU_REQUIRE(units < 1 << 24, FSTU_ESHAPE, "fstu_stu_conv_mfma: B=%d d=%d", B, d);
  const dim3 grid((unsigned)((units + 7) / 8 * 64));
#define CM_GO(NT, NBS, NW, OCC)                                                                                                     \
  do {                                                                                                                              \
    constexpr int lds__ = (8 >> NBS) * cm_row(NT << NBS, 1 << NBS) + NW * CM_RING;                                                  \
    static fstu_lds_limit most;                                                                                                     \
    const int rc__ = fstu_need_lds((const void*)conv_mfma_kernel<NT, NBS, NW, OCC>, most, lds__, "fstu_stu_conv_mfma");             \
    if (rc__) return rc__;                                                                                                          \
    hipLaunchKernelGGL((conv_mfma_kernel<NT, NBS, NW, OCC>), grid, dim3(NW * 64), lds__, (hipStream_t)stream, (const bf16_t*)x,     \
                       (const bf16_t*)taps, (bf16_t*)y, B, T, d, single_branch);                                                    \
  } while (0)
  if (nt == 4) CM_GO(4, 3, 8, 2);
  else if (nt == 2) CM_GO(2, 3, 4, 3);
  else if (nbs == 3) CM_GO(1, 3, 4, 4);
  else if (nbs == 2) CM_GO(1, 2, 4, 4);
  else if (nbs == 1) CM_GO(1, 1, 4, 4);
  else CM_GO(1, 0, 4, 4);
#undef CM_GO
  FSTU_CHECK_LAUNCH("fstu_stu_conv_mfma");
  return FSTU_OK;
}

// Up to 192 positions an item is latency (a workgroup's tiles are made for 1024), and from some rows on the transforms' launches are
// shorter.  GPU us of a whole training step with both directions as products / as transforms, rows x positions x channels: 8 x 64 x 768
// 79.5 / 78.3, 32 x 64 x 768 117 / 99, 8 x 100 x 768 73 / 76, 24 x 100 x 768 108 / 104, 16 x 128 x 1024 117 / 116, 64 x 128 x 2048 416 / 328,
// 4 x 200 x 512 63 / 76, 8 x 200 x 768 94 / 101, 16 x 200 x 1024 124 / 127, 64 x 256 x 1024 265 / 267, 8 x 300 x 768 100 / 113.
extern "C" int fstu_stu_conv_mfma_grad_takes(int B, int T, int d, int L) {
  if (B < 1 || T < 32 || T > 2048 || d < 8 || d % 8 != 0 || d > 1 << 20 || L < 1 || (int64_t)L * d >= 1ll << 31) return 0;
  return T > 192 || (long long)B * (d / 8) <= 4 * fstu_cus();
}

extern "C" int64_t fstu_stu_conv_mfma_grad_ws(int B, int T, int d, int L) {
  if (B < 1 || T < 1 || T > 2048 || d < 8 || L < 1) return 0;
  const int R = cg_items(B, T, d), lags = ((L < T ? L : T) + 1) / 2;
  return (int64_t)((2 * B + R - 1) / R) * lags * d;
}

namespace {

int cg_launch(const char* name, const void* gy, const void* x, const void* filt, void* gx, float* part, const void* phi_e, int K, int P, int B, int T,
              int d, int L, int R, hipStream_t s) {
  FSTU_REQUIRE(B >= 1 && B <= 65535 && T >= 1 && T <= 2048 && d >= 8 && d % 8 == 0 && d <= 1 << 20 && L >= 1 && (int64_t)L * d < 1ll << 31,
               FSTU_ESHAPE, "%s: B=%d T=%d d=%d L=%d (T up to 2048, d a multiple of 8)", name, B, T, d, L);
  FSTU_REQUIRE(fstu_aligned(gy, 16) && fstu_aligned(x, 16) && fstu_aligned(filt, 16) && fstu_aligned(gx, 16) && fstu_aligned(part, 16) &&
                   fstu_aligned(phi_e, 16), FSTU_EALIGN, "%s: pointers must be 16-byte aligned", name);
  const long long units = (long long)((d + 63) / 64) * ((2 * B + R - 1) / R);
  FSTU_REQUIRE(units < 1 << 24, FSTU_ESHAPE, "%s: B=%d d=%d", name, B, d);
  const dim3 grid((unsigned)((units + 7) / 8 * 64));
#define CG_GO(NT, PROJECT)                                                                                                          \
  do {                                                                                                                              \
    constexpr int lds__ = 16 * cm_region(8 * NT) + 8 * cg_rows(8 * NT) + 8 * 2048;                                                 \
    static fstu_lds_limit most;                                                                                                     \
    const int rc__ = fstu_need_lds((const void*)conv_grad_mfma_kernel<NT, PROJECT>, most, lds__, name);                             \
    if (rc__) return rc__;                                                                                                          \
    hipLaunchKernelGGL((conv_grad_mfma_kernel<NT, PROJECT>), grid, dim3(512), lds__, s, (const bf16_t*)gy, (const bf16_t*)x, (const bf16_t*)filt, \
                       (bf16_t*)gx, part, (const bf16_t*)phi_e, K, P, B, T, L, d, R);                                               \
  } while (0)
  if (phi_e) {
    if (T <= 1024) CG_GO(1, true);
    else CG_GO(2, true);
  } else {
    if (T <= 1024) CG_GO(1, false);
    else CG_GO(2, false);
  }
#undef CG_GO
  FSTU_CHECK_LAUNCH(name);
  return FSTU_OK;
}

}  // namespace

extern "C" int fstu_stu_conv_mfma_grad(const void* gy, const void* x, const void* filt, void* gx, void* gf, float* part, int B, int T, int d,
                                       int L, void* stream) {
  FSTU_REQUIRE(gy && x && filt && (gx || gf) && (!gf || part), FSTU_ENULL, "fstu_stu_conv_mfma_grad: null pointer");
  FSTU_REQUIRE(fstu_aligned(gf, 16), FSTU_EALIGN, "fstu_stu_conv_mfma_grad: pointers must be 16-byte aligned");
  const int R = cg_items(B, T, d), chunks = (2 * B + R - 1) / R, lags = ((L < T ? L : T) + 1) / 2;
  const int rc = cg_launch("fstu_stu_conv_mfma_grad", gy, x, filt, gx, gf ? part : nullptr, nullptr, 0, 0, B, T, d, L, R, (hipStream_t)stream);
  if (rc || !gf) return rc;
  hipLaunchKernelGGL(conv_grad_finish_kernel, dim3((unsigned)(((long long)L * (d / 8) + 255) / 256)), dim3(256), 0, (hipStream_t)stream, part,
                     (bf16_t*)gf, chunks, lags, L, d);
  FSTU_CHECK_LAUNCH("fstu_stu_conv_mfma_grad");
  return FSTU_OK;
}

extern "C" int64_t fstu_stu_conv_mfma_grad_project_ws(int B, int T, int d, int K) {
  if (B < 1 || T < 1 || T > 2048 || d < 8 || K < 1) return 0;
  const int R = cg_items(B, T, d);
  return (int64_t)((2 * B + R - 1) / R) * K * d;
}

extern "C" int fstu_stu_conv_mfma_grad_project(const void* gy, const void* x, const void* filt, const void* phi_e, int P, void* gx, void* gm,
                                               float* part, int B, int T, int d, int L, int K, void* stream) {
  FSTU_REQUIRE(gy && x && filt && phi_e && gm && part, FSTU_ENULL, "fstu_stu_conv_mfma_grad_project: null pointer");
  FSTU_REQUIRE(K >= 1 && K <= 128 && P >= 8 && P % 8 == 0 && T <= L && 2 * (int64_t)P >= L, FSTU_ESHAPE,
               "fstu_stu_conv_mfma_grad_project: K=%d P=%d T=%d L=%d (K up to 128, P a multiple of 8 of at least L / 2, T up to L)", K, P, T, L);
  const int R = cg_items(B, T, d), n = K * d;
  const int rc = cg_launch("fstu_stu_conv_mfma_grad_project", gy, x, filt, gx, part, phi_e, K, P, B, T, d, L, R, (hipStream_t)stream);
  if (rc) return rc;
  hipLaunchKernelGGL(conv_grad_join_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, part, (bf16_t*)gm, (2 * B + R - 1) / R, n);
  FSTU_CHECK_LAUNCH("fstu_stu_conv_mfma_grad_project");
  return FSTU_OK;
}
