// Dense LDS over a whole sequence on the matrix cores (bf16): the loop of mini_stu/lds.py:95-101,
//   h <- h * A + x_t @ B ;  y_t = T(h @ C),   t = 0 .. T-1, state h (Bt,S) fp32 carried,
// cut into blocks of 128 positions that run in parallel, x read ONCE.  x_t @ B does not depend on the state, so a
// workgroup (block, batch row) forms U = X_blk B with MFMA tiles and keeps it in LDS from then on:
//   1  scan U from zero: the block's end state E, published at once as tagged 64-bit words (value, tag of the call)
//   2  the state that enters the block: carry = h, then carry = E[j] + A^128 * carry over the blocks j in front of it,
//      read from what those blocks published (they are earlier in launch order, so they are resident or done, and
//      they publish before they wait for anything: the wait ends; it is bounded all the same and reports a
//      time-out through a status word instead of hanging).  The chain is the same fused multiply-adds in the same
//      order for every block, so splitting a sequence at a multiple of 128 gives bit-identical states and outputs.
//      The last block of a row also forms the state behind the sequence.
//   3  scan U again from the carry (now the true states H), Y = H C with H split into a bf16 head and a bf16
//      remainder so that the second product keeps the fp32 state's accuracy.
// Weights are given transposed (B^T (S,d_in), C^T (d_out,S)) so that every MFMA fragment is one 16-byte piece; both
// travel through LDS so that the four waves of a workgroup share one fetch.
#include "fstu_common.h"
#include <algorithm>
#include <type_traits>

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

#define LSQ_TB 128        // positions per block
#define LSQ_NTMAX 16      // state tiles of 16 (S <= 256)

template <typename V> __device__ __forceinline__ bf16x8_t as_bf16x8(V v) { return __builtin_bit_cast(bf16x8_t, v); }

#define LSQ_SPIN_LIMIT (1 << 18)   // polls of one batch of published states before the wait gives up
#define LSQ_LOOK 8                 // published states requested at a time

// the 16 bytes of lane r ^ 8 of the same 16 lanes (a rotation of 16 lanes by 8)
__device__ __forceinline__ uint4 swap8(uint4 v) {
  v.x = __builtin_amdgcn_mov_dpp(v.x, 0x128, 0xf, 0xf, false);
  v.y = __builtin_amdgcn_mov_dpp(v.y, 0x128, 0xf, 0xf, false);
  v.z = __builtin_amdgcn_mov_dpp(v.z, 0x128, 0xf, 0xf, false);
  v.w = __builtin_amdgcn_mov_dpp(v.w, 0x128, 0xf, 0xf, false);
  return v;
}
typedef unsigned uintx4_t __attribute__((ext_vector_type(4)));
typedef uintx4_t uintx4_a8_t __attribute__((aligned(8)));
// outputs are 8-byte aligned
template <bool PAST>
__device__ __forceinline__ void store16(bf16_t* p, uint4 v) {
  if constexpr (PAST) __builtin_nontemporal_store(__builtin_bit_cast(uintx4_t, v), (uintx4_a8_t*)p);
  else *(uintx4_a8_t*)p = __builtin_bit_cast(uintx4_t, v);
}

// Two workgroups share a compute unit up to S = 160 (a workgroup's life is a chain of short barrier-separated phases, so one
// alone leaves the unit idle most of the time): at most 256 registers, and U without padding, 128 x S floats = 80 KB at S = 160.
// Instead of a pad, the 16-byte slot of element (row, mode) is XOR-ed with bits 1..3 of the row, which keeps the 16 rows of a
// tile access on 16 different slots; the scan, one thread per mode, follows the same map.
//
// NT = S / 16 is exact and every load of the two products unconditional (rows and chunks behind the end are clamped to the last
// ones, whose results nobody reads): with the number of tiles in a register and loads under conditions the loops were made of
// branches, each fragment read was waited for by itself and every chunk for all loads in flight.  us, so / now: 64 rows x 4096 x
// 1024, state 160, 389 / 331 (state 128 355 / 301), 51 x 3262 x 256, 96, 91 / 71, 8 x 2048 x 512, 128, 53 / 38, 1 x 4096 x 1024,
// 160, 87 / 55, 64 x 300 x 1024, 160, 88 / 55.  (x, BmT and CmT carry no __restrict__: loads of memory that nothing may change are
// moved behind the barriers to where their values are used.)
// What bounds the first: its 1.07 GB, which a copy moves in 208 us, and too few waves to keep memory, matrix cores (busy 38 % of the time)
// and LDS (32 %) at work at once: two a SIMD, of up to 256 registers.  Without the stores of y it takes 246, without the trips of x to HBM 295, without either
// 208, with the weights from the compute unit's own cache besides 162.  No gain: x past the caches (360: a line comes in two
// halves), the blocks of a row side by side (351), the two lines of 128 features of a row stored together (337), another first
// group of features for every row (340), the scans left out (322).  With whole lines of x to a load (half a line of twice as many
// rows before) 327 / 322, state 128 304 / 298.
//
// Fewer blocks than compute units: a group of 64 output features takes 1.1 us, one behind the other (16 of the 38 us of a call on one block of
// 1024 features, state 128), so as many workgroups as there are compute units for form the same U and states and a slice of the features
// each; the first one publishes.  A second one on a compute unit loses more (three times).  us, one / slices: 128 x 1 x 1024, state 128, 37.9 / 22.5,
// 3000 x 1 x 1024, 160, 45.8 / 30.2, 3000 x 3 x 1024, 128, 41.2 / 32.0, 4096 x 4 x 1024, 160, 48.1 / 40.4, 1000 x 8 x 512, 64, 20.7 / 17.7; where
// there are no compute units for a second slice 4096 x 6 x 1024, 160, 47.5 / 52.4.
//
// PAST: the outputs leave past the L2s, where they are more than those hold (32 MB): what they would push out are the weights
// that every workgroup fetches again, and the next kernel would not find them there.
//
// SLICED: the features may be in slices.  A kernel of its own for those in one only beyond S = 160, where a few more values that live through
// the second product cost its LDS reads their overlap (4096 x 40 x 1024, state 256, 333 us; 316 so).
template <int NT, bool PAST, bool SLICED>
__global__ void __launch_bounds__(256, NT <= 10 ? 2 : 1)   // beyond S = 160 one workgroup fills the LDS anyway
lds_seq_kernel(const bf16_t* x, const float* __restrict__ A, const bf16_t* BmT, const bf16_t* CmT, bf16_t* y, const float* __restrict__ h0,
               float* __restrict__ hnew, unsigned long long* __restrict__ etag, unsigned* __restrict__ status, unsigned tag,
               int T, int Bt, int d_in, int d_out, int nblk, int slices, int width) {
  constexpr int S = 16 * NT;
  extern __shared__ __align__(16) float Us[];       // LSQ_TB x S
  auto uslot = [](int row, int slot) { return slot ^ ((row >> 1) & 7); };   // 16-byte slot of a row (S/4 slots, a multiple of 8)
  // rows of the batch first: the blocks in front of a workgroup's are then long through when it asks for their states
  const int blk = (int)(blockIdx.z * gridDim.y + blockIdx.y), b = SLICED ? blockIdx.x / slices : blockIdx.x, slice = SLICED ? blockIdx.x % slices : 0;
  if (blk >= nblk) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 15, g = lane >> 4;
  const int t0 = blk * LSQ_TB;
  const int nvalid = min(LSQ_TB, T - t0);
  constexpr int WPT = NT / 2;                       // 16-byte pieces of a chunk of weights per thread
  // ---- U = X_blk B: wave w owns positions 32w .. 32w+31 (two tiles of 16).  The four waves need the same weight
  // fragments: B^T travels through LDS in chunks of 64 k (S rows of 128 bytes, 16-byte pieces XOR-ed with bits of the
  // row so that the 16 rows of a fragment read fall into 16 different slots), double-buffered in the space that U
  // takes afterwards, so a workgroup fetches every weight once instead of once per wave.
  // Both are requested three chunks ahead, x into three sets of registers and the weights into two: one chunk's products
  // are shorter than a trip to memory.
  {
    unsigned char* wst = (unsigned char*)Us;                 // two stages of S * 128 bytes
    constexpr unsigned wstage = S * 128u;
    floatx4_t acc[2][NT];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m][n] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    const bf16_t* xr[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) xr[m] = x + ((size_t)min(t0 + 32 * w + 16 * m + r, T - 1) * Bt + b) * d_in + g * 8;
    // A chunk of a row is a line.  The first eight lanes of a row's sixteen have its first half, the others the second, of rows 0..7 of a
    // tile in one load and of rows 8..15 in another: whole lines; lanes r and r ^ 8 swap pieces in front of the products.  Beyond S = 160,
    // where the accumulators alone are most of the registers, the swaps cost more than the lines give (4096 x 40 x 1024, us, half lines / whole:
    // state 256 333 / 341, 224 284 / 292, 192 255 / 261): there a load has its own k step's halves of sixteen lines.
    constexpr bool LINES = NT <= 10;
    const bf16_t* xl[2][2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int h = 0; h < 2; ++h) xl[m][h] = x + ((size_t)min(t0 + 32 * w + 16 * m + 8 * h + (r & 7), T - 1) * Bt + b) * d_in + 32 * (r >> 3) + g * 8;
    const int swz = (r >> 1) & 7;                            // rows 16n + r and 32i + row share these bits
    const unsigned char* const wrd[2] = {wst + r * 128 + ((g ^ swz) << 4), wst + r * 128 + (((g + 4) ^ swz) << 4)};
    auto multiply = [&](int kk, unsigned stage, const uintx4_t (&xs)[2]) __attribute__((always_inline)) {
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const bf16x8_t wa = as_bf16x8(*(const uint4*)(wrd[kk] + stage + n * 2048));
        acc[0][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa, as_bf16x8(xs[0]), acc[0][n], 0, 0, 0);
        acc[1][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa, as_bf16x8(xs[1]), acc[1][n], 0, 0, 0);
      }
    };
    const int nk = d_in >> 6;                                // whole chunks; 32 k may be left
    if (nk) {
      const bf16_t* const wsrc = BmT + (size_t)(tid >> 3) * d_in + (tid & 7) * 8;       // piece i: 32 i rows further
      unsigned char* const wdst = wst + (tid >> 3) * 128 + (((tid & 7) ^ ((tid >> 4) & 7)) << 4);
      auto wload = [&](int c, uintx4_t (&v)[WPT]) {
        const bf16_t* src = wsrc + 64 * min(c, nk - 1);
#pragma unroll
        for (int i = 0; i < WPT; ++i) v[i] = *(const uintx4_t*)(src + (size_t)(32 * i) * d_in);
      };
      auto wstore = [&](unsigned stage, const uintx4_t (&v)[WPT]) {
#pragma unroll
        for (int i = 0; i < WPT; ++i) *(uintx4_t*)(wdst + stage + i * 4096) = v[i];
      };
      auto xload = [&](int c, uintx4_t (&v)[2][2]) {            // both halves (or k steps) of both position tiles
        const int k0 = 64 * min(c, nk - 1);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int m = 0; m < 2; ++m) v[h][m] = *(const uintx4_t*)(LINES ? xl[m][h] + k0 : xr[m] + k0 + 32 * h);
      };
      uintx4_t wa[WPT], wb[WPT], xa[2][2], xb[2][2], xc[2][2];
      wload(0, wa);
      xload(0, xa);
      wload(1, wb);
      xload(1, xb);
      wstore(0, wa);
      wload(2, wa);
      xload(2, xc);
      __syncthreads();
      int c = 0;
      unsigned stage = 0;
      auto pass = [&](uintx4_t (&xs)[2][2], uintx4_t (&wn)[WPT]) __attribute__((always_inline)) { // chunk c; wn: the weights of chunk c + 1
        if constexpr (LINES) {
          uintx4_t x0[2], x1[2];
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            const uintx4_t o = __builtin_bit_cast(uintx4_t, swap8(__builtin_bit_cast(uint4, r < 8 ? xs[1][m] : xs[0][m])));
            x0[m] = r < 8 ? xs[0][m] : o;
            x1[m] = r < 8 ? o : xs[1][m];
          }
          multiply(0, stage, x0);
          multiply(1, stage, x1);
        } else {
          multiply(0, stage, xs[0]);
          multiply(1, stage, xs[1]);
        }
        stage = wstage - stage;
        wstore(stage, wn);
        wload(c + 3, wn);
        xload(c + 3, xs);
        __syncthreads();
        return ++c < nk;
      };
      while (pass(xa, wb) && pass(xb, wa) && pass(xc, wb) && pass(xa, wa) && pass(xb, wb) && pass(xc, wa)) {
      }
    }
    if (d_in & 32) {
      uintx4_t xs[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) xs[m] = *(const uintx4_t*)(xr[m] + 64 * nk);
      for (int q = tid; q < S * 4; q += 256)
        *(uint4*)(wst + (q >> 2) * 128 + (((q & 3) ^ ((q >> 3) & 7)) << 4)) = *(const uint4*)(BmT + (size_t)(q >> 2) * d_in + 64 * nk + (q & 3) * 8);
      __syncthreads();
      multiply(0, 0, xs);
      __syncthreads();
    }
    // (behind the last barrier every wave is through with the weight stages, U may overwrite them)
    // D layout: lane (r, g) holds modes 16n + 4g + i of position r of the tile
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n)
        *(float4*)(Us + (32 * w + 16 * m + r) * S + 4 * uslot(32 * w + 16 * m + r, 4 * n + g)) = make_float4(acc[m][n][0], acc[m][n][1], acc[m][n][2], acc[m][n][3]);
  }
  __syncthreads();
  // ---- scan over the block's positions: thread = mode
  if (tid < S) {
    const float a = A[tid];
    // element (p, tid) sits at p * S + 4 * uslot(p, tid / 4) + tid % 4
    auto at = [&](int p_) { return Us + p_ * S + 4 * uslot(p_, tid >> 2) + (tid & 3); };
    // 1: the block's end state from zero, published as (tag, value)
    float e = 0.f;
    {
      int p = 0;
      for (; p + 16 <= nvalid; p += 16) {
        float u[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) u[i] = *at(p + i);
#pragma unroll
        for (int i = 0; i < 16; ++i) e = fmaf(a, e, u[i]);
      }
      for (; p < nvalid; ++p) e = fmaf(a, e, *at(p));
    }
    const size_t rowbase = (size_t)b * nblk * S;
    if (slice == 0) __hip_atomic_store(etag + rowbase + (size_t)blk * S + tid, ((unsigned long long)tag << 32) | __float_as_uint(e),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // 2: the state that enters this block (every block in front of it is a full one)
    const double ad = (double)a;
    const float ap_full = (float)pow(ad, (double)LSQ_TB);
    float h = h0[(size_t)b * S + tid];
    bool timed_out = false;
    for (int j0 = 0; j0 < blk; j0 += LSQ_LOOK) {
      unsigned long long wv[LSQ_LOOK];
      int spins = 0;
      bool ok;
      do {
        ok = true;
#pragma unroll
        for (int i = 0; i < LSQ_LOOK; ++i) {
          const int j = min(j0 + i, blk - 1);
          wv[i] = __hip_atomic_load(etag + rowbase + (size_t)j * S + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int i = 0; i < LSQ_LOOK; ++i) ok = ok && (unsigned)(wv[i] >> 32) == tag;
        if (!ok) __builtin_amdgcn_s_sleep(4);
      } while (!ok && ++spins < LSQ_SPIN_LIMIT);
      timed_out = timed_out || !ok;
#pragma unroll
      for (int i = 0; i < LSQ_LOOK; ++i)
        if (j0 + i < blk) h = fmaf(ap_full, h, __uint_as_float((unsigned)wv[i]));
    }
    if (timed_out) atomicOr(status, 1u);
    if (blk == nblk - 1 && slice == 0) {
      const float ap = nvalid == LSQ_TB ? ap_full : (float)pow(ad, (double)nvalid);
      hnew[(size_t)b * S + tid] = fmaf(ap, h, e);
    }
    // 3: the true states of the block's positions
    int p = 0;
    for (; p + 16 <= nvalid; p += 16) {
      float u[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) u[i] = *at(p + i);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        h = fmaf(a, h, u[i]);
        *at(p + i) = h;
      }
    }
    for (; p < nvalid; ++p) {
      h = fmaf(a, h, *at(p));
      *at(p) = h;
    }
  }
  __syncthreads();
  // ---- Y = H C: wave w, positions 32w .. 32w+31; H as bf16 head + remainder
  {
    constexpr int KS = NT / 2;         // k steps of 32 modes
    uint4 hb[2][KS], lb[2][KS];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int hrow = 32 * w + 16 * m + r;
      const float* hr = Us + hrow * S;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        const float4 v0 = *(const float4*)(hr + 4 * uslot(hrow, 8 * k + 2 * g)), v1 = *(const float4*)(hr + 4 * uslot(hrow, 8 * k + 2 * g + 1));
        const float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        unsigned hi[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          hi[i] = pack2_bf16(v[2 * i], v[2 * i + 1]);
          lo[i] = pack2_bf16(v[2 * i] - __uint_as_float(hi[i] << 16), v[2 * i + 1] - __uint_as_float(hi[i] & 0xffff0000u));
        }
        hb[m][k] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        lb[m][k] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      }
    }
    // A lane stores 16 bytes, the eight lanes of a line next to each other in one instruction (straight from the
    // accumulators an instruction covers 32 bytes of 16 rows): the rows of the two tiles of 32 features are dealt so
    // that lane (r, g) ends up with features 8g .. 8g+7 of position r, and lanes r and r ^ 8 swap pieces, so that
    // they hold the two halves of a line of 64 features.
    const int trow = t0 + 32 * w + (r & 7), fcol = 32 * (r >> 3) + 8 * g;
    const int of = SLICED ? slice * width : 0, dn = SLICED ? min(width, d_out - of) : d_out;   // the features of this workgroup's slice
    CmT += (size_t)of * S;
    y += of;
    bf16_t* yr[4];                                           // position trow + 8 q
#pragma unroll
    for (int q = 0; q < 4; ++q) yr[q] = y + ((size_t)min(trow + 8 * q, T - 1) * Bt + b) * d_out + fcol;
    // C^T travels through LDS like B^T above, 64 output features (4 tiles) at a time, double-buffered in the space of
    // U now that every wave holds its H fragments in registers.  Rows are S * 2 + 16 bytes: an odd number of 16-byte
    // slots, so the 16 rows of a fragment read fall into 16 different slots.  Feature 32p + 8g + 4h + i lies in row
    // 32p + 16h + 4g + i.
    __syncthreads();
    unsigned char* cst = (unsigned char*)Us;
    constexpr unsigned RS = S * 2u + 16u, cstage = 64u * RS;
    constexpr int PPR = S / 8;                               // 16-byte pieces per row; a stage's lie in memory one after the other
    const int npiece = dn * PPR;
    unsigned cdst[WPT];
#pragma unroll
    for (int i = 0; i < WPT; ++i) {
      const int q = tid + i * 256, row = q / PPR, c = q - row * PPR;
      cdst[i] = (unsigned)((row & 0x23) | ((row & 0x18) >> 1) | ((row & 4) << 2)) * RS + c * 16;
    }
    auto cload = [&](int o0, uintx4_t (&v)[WPT]) {
#pragma unroll
      for (int i = 0; i < WPT; ++i) v[i] = *(const uintx4_t*)(CmT + 8 * (size_t)min(o0 * PPR + tid + i * 256, npiece - 1));
    };
    auto cstore = [&](unsigned stage, const uintx4_t (&v)[WPT]) {
#pragma unroll
      for (int i = 0; i < WPT; ++i) *(uintx4_t*)(cst + stage + cdst[i]) = v[i];
    };
    const unsigned char* const crd = cst + r * RS + g * 16;
    uintx4_t ca[WPT], cb[WPT];                                  // the next groups of output features
    cload(0, ca);
    cload(64, cb);
    cstore(0, ca);
    cload(128, ca);
    __syncthreads();
    auto outputs = [&](auto whole) __attribute__((always_inline)) {                         // whole: no position and no feature is behind the end
      int o0 = 0;
      unsigned stage = 0;
      auto pass = [&](uintx4_t (&cn)[WPT]) __attribute__((always_inline)) {
        uint4 pc[2][2];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          floatx4_t acc[2][2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            floatx4_t a0 = {0.f, 0.f, 0.f, 0.f}, a1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KS; ++k) {
              const bf16x8_t wc = as_bf16x8(*(const uint4*)(crd + stage + (32 * p + 16 * h) * RS + 64 * k));
              a0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc, as_bf16x8(hb[0][k]), a0, 0, 0, 0);
              a1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc, as_bf16x8(hb[1][k]), a1, 0, 0, 0);
              a0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc, as_bf16x8(lb[0][k]), a0, 0, 0, 0);
              a1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc, as_bf16x8(lb[1][k]), a1, 0, 0, 0);
            }
            acc[0][h] = a0;
            acc[1][h] = a1;
          }
#pragma unroll
          for (int m = 0; m < 2; ++m)
            pc[m][p] = make_uint4(pack2_bf16(acc[m][0][0], acc[m][0][1]), pack2_bf16(acc[m][0][2], acc[m][0][3]),
                                  pack2_bf16(acc[m][1][0], acc[m][1][1]), pack2_bf16(acc[m][1][2], acc[m][1][3]));
        }
        stage = cstage - stage;
        cstore(stage, cn);
        cload(o0 + 192, cn);
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const uint4 other = swap8(r < 8 ? pc[m][1] : pc[m][0]);
          const uint4 lo = r < 8 ? pc[m][0] : other, hi = r < 8 ? other : pc[m][1];
          if (decltype(whole)::value || (o0 + fcol < dn && trow + 16 * m < T)) store16<PAST>(yr[2 * m] + o0, lo);
          if (decltype(whole)::value || (o0 + fcol < dn && trow + 16 * m + 8 < T)) store16<PAST>(yr[2 * m + 1] + o0, hi);
        }
        __syncthreads();
        return (o0 += 64) < dn;
      };
      while (pass(cb) && pass(ca)) {
      }
    };
    if (nvalid == LSQ_TB && dn % 64 == 0) outputs(std::true_type{});
    else outputs(std::false_type{});
  }
}

// What a call needs before its blocks start: the published states cleared, the state that enters copied (the last block of a row leaves
// the new one in its place while others still read it) and, where the weights come as they lie, Bm (d_in, S) and Cm (S, d_out) transposed, a tile
// of 32 x 32 to each of the first nt workgroups.  One launch of 4.3 to 5.9 us: two transposes, the clearing and a copy of the state at the end
// took launches of their own (5.4 + 5.4 + 5.4 + 5.2 by the profiler; behind each other they hide in part: 64 rows x 4096 x 1024, state 160,
// with the whole lines of x above 327 -> 322 us a call).
__global__ void __launch_bounds__(256)
lds_seq_prepare_kernel(unsigned long long* __restrict__ etag, size_t n, unsigned* __restrict__ status, const float* __restrict__ h, float* __restrict__ h0,
                       int nh, const bf16_t* __restrict__ Bm, const bf16_t* __restrict__ Cm, bf16_t* __restrict__ wt, int d_in, int S, int d_out, int nb, int nt) {
  __shared__ bf16_t tile[32][34];
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < nt) {
    const bool first = (int)blockIdx.x < nb;
    const int t = blockIdx.x - (first ? 0 : nb), rows = first ? d_in : S, cols = first ? S : d_out, across = (cols + 31) >> 5;
    const bf16_t* const src = first ? Bm : Cm;
    bf16_t* const dst = wt + (first ? 0 : (size_t)S * d_in);
    const int r0 = t / across * 32, c0 = t % across * 32, i = tid >> 5, j = tid & 31;
#pragma unroll
    for (int k = 0; k < 32; k += 8)
      if (c0 + j < cols) tile[i + k][j] = src[(size_t)(r0 + i + k) * cols + c0 + j];       // rows: a multiple of 32
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 32; k += 8)
      if (c0 + i + k < cols) dst[(size_t)(c0 + i + k) * rows + r0 + j] = tile[j][i + k];
    return;
  }
  const size_t first = (size_t)(blockIdx.x - nt) * 256 + tid, step = (size_t)(gridDim.x - nt) * 256;
  for (size_t i = first; i < n; i += step) etag[i] = 0ull;
  for (size_t i = first; i < (size_t)nh; i += step) h0[i] = h[i];
  if (first == 0) *status = 0u;
}

}  // namespace

// workspace: 64 floats of header (status word), the published block states (nblk * Bt * S 64-bit words), the state that enters
extern "C" size_t fstu_lds_sequence_ws_floats(int T, int Bt, int S) {
  if (T < 0 || Bt < 1 || S < 1) return 0;
  const size_t nblk = (size_t)(T + LSQ_TB - 1) / LSQ_TB;
  return 64 + (2 * nblk + 1) * (size_t)Bt * S;
}

// wt null: Bm and Cm are given transposed
static int lds_sequence(float* h, const void* x, const float* A, const void* Bm, const void* Cm, void* wt, void* y, float* ws, int T, int Bt,
                        int d_in, int S, int d_out, void* stream) {
  const void *const BmT = wt ? wt : Bm, *const CmT = wt ? (const void*)((const bf16_t*)wt + (size_t)S * d_in) : Cm;
  FSTU_REQUIRE(h && x && A && Bm && Cm && y && ws, FSTU_ENULL, "fstu_lds_sequence: null pointer");
  FSTU_REQUIRE(T >= 0 && Bt >= 1 && Bt <= 65535, FSTU_ESHAPE, "fstu_lds_sequence: T=%d Bt=%d", T, Bt);
  FSTU_REQUIRE(d_in >= 32 && d_in % 32 == 0 && S >= 32 && S % 32 == 0 && S <= 16 * LSQ_NTMAX && d_out >= 16 && d_out % 16 == 0,
               FSTU_ESHAPE, "fstu_lds_sequence: need d_in %% 32 == 0, S %% 32 == 0 (<= %d), d_out %% 16 == 0 (d_in=%d S=%d d_out=%d)",
               16 * LSQ_NTMAX, d_in, S, d_out);
  FSTU_REQUIRE(fstu_aligned(x, 16) && fstu_aligned(BmT, 16) && fstu_aligned(CmT, 16) && fstu_aligned(y, 8) && fstu_aligned(ws, 16),
               FSTU_EALIGN, "fstu_lds_sequence: pointers must be 16-byte aligned");
  if (T == 0) return FSTU_OK;
  const int nblk = (T + LSQ_TB - 1) / LSQ_TB;
  const size_t BtS = (size_t)Bt * S;
  unsigned* status = (unsigned*)ws;
  unsigned long long* etag = (unsigned long long*)(ws + 64);
  float* h0 = ws + 64 + 2 * (size_t)nblk * BtS;
  const int nb = wt ? d_in / 32 * (S / 32) : 0, nt = wt ? nb + S / 32 * ((d_out + 31) / 32) : 0;
  const size_t shm = (size_t)LSQ_TB * S * sizeof(float);
  hipStream_t s = (hipStream_t)stream;
  const unsigned ny = nblk < 32768 ? (unsigned)nblk : 32768u;
  // Slices of the output features where there are fewer blocks than compute units (see the kernel); not where y is written over x, which the
  // other slices of a block may still have to read.
  const size_t xb = (size_t)T * Bt * d_in * sizeof(bf16_t), yb = (size_t)T * Bt * d_out * sizeof(bf16_t);
  const bool apart = (const char*)y + yb <= (const char*)x || (const char*)x + xb <= (const char*)y;
  const long long most_slices = fstu_cus() / ((long long)nblk * Bt);
  const int groups = (d_out + 63) / 64, want = apart ? (int)std::min<long long>(std::max(most_slices, 1ll), groups) : 1;
  const int width = 64 * ((groups + want - 1) / want), slices = (d_out + width - 1) / width;
  const dim3 grid((unsigned)Bt * slices, ny, ((unsigned)nblk + ny - 1) / ny);
  const size_t nwords = (size_t)nblk * BtS;
  unsigned cgrid = (unsigned)((nwords + 255) / 256);
  if (cgrid > 1024u) cgrid = 1024u;
  const bool past = yb > (size_t)32 << 20;
  int rc = FSTU_OK;
  auto run = [&](auto which) {                          // (a type for each kernel: a record of its own)
    constexpr auto kernel = decltype(which)::value;
    static fstu_lds_limit most;
    if ((rc = fstu_need_lds((const void*)kernel, most, shm, "fstu_lds_sequence"))) return;
    hipLaunchKernelGGL(lds_seq_prepare_kernel, dim3(nt + cgrid), dim3(256), 0, s, etag, nwords, status, (const float*)h, h0, (int)BtS, (const bf16_t*)Bm,
                       (const bf16_t*)Cm, (bf16_t*)wt, d_in, S, d_out, nb, nt);
    hipLaunchKernelGGL(kernel, grid, dim3(256), shm, s, (const bf16_t*)x, A, (const bf16_t*)BmT, (const bf16_t*)CmT, (bf16_t*)y,
                       (const float*)h0, h, etag, status, 1u, T, Bt, d_in, d_out, nblk, slices, width);
  };
#define LSQ_RUN(...) run(std::integral_constant<decltype(&lds_seq_kernel<__VA_ARGS__>), lds_seq_kernel<__VA_ARGS__>>{})
#define LSQ_CASE(n)                                                                                 \
  case 32 * n:                                                                                      \
    if (n > 5 && slices == 1) past ? LSQ_RUN(2 * n, true, n <= 5) : LSQ_RUN(2 * n, false, n <= 5);  \
    else past ? LSQ_RUN(2 * n, true, true) : LSQ_RUN(2 * n, false, true);                           \
    break
  switch (S) {
    LSQ_CASE(1); LSQ_CASE(2); LSQ_CASE(3); LSQ_CASE(4); LSQ_CASE(5); LSQ_CASE(6); LSQ_CASE(7); LSQ_CASE(8);
  }
#undef LSQ_CASE
#undef LSQ_RUN
  if (rc) return rc;
  FSTU_CHECK_LAUNCH("fstu_lds_sequence");
  return FSTU_OK;
}

extern "C" int fstu_lds_sequence(float* h, const void* x, const float* A, const void* BmT, const void* CmT, void* y, float* ws,
                                 int T, int Bt, int d_in, int S, int d_out, void* stream) {
  return lds_sequence(h, x, A, BmT, CmT, nullptr, y, ws, T, Bt, d_in, S, d_out, stream);
}

extern "C" int fstu_lds_sequence_bc(float* h, const void* x, const float* A, const void* Bm, const void* Cm, void* wt, void* y, float* ws,
                                    int T, int Bt, int d_in, int S, int d_out, void* stream) {
  FSTU_REQUIRE(wt, FSTU_ENULL, "fstu_lds_sequence_bc: null pointer");
  return lds_sequence(h, x, A, Bm, Cm, wt, y, ws, T, Bt, d_in, S, d_out, stream);
}

// 0, or 1 when a wait of the last fstu_lds_sequence call on this workspace ran out (synchronous read of the status word)
extern "C" int fstu_lds_sequence_status(const float* ws, int* err_out) {
  FSTU_REQUIRE(ws && err_out, FSTU_ENULL, "fstu_lds_sequence_status: null pointer");
  unsigned v = 0;
  hipError_t e = hipMemcpy(&v, ws, sizeof(v), hipMemcpyDeviceToHost);
  if (e != hipSuccess) { fstu_set_error("fstu_lds_sequence_status: %s", hipGetErrorString(e)); return (int)e; }
  *err_out = (int)v;
  return FSTU_OK;
}
