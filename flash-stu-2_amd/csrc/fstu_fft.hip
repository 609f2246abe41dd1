// Spectral convolution of the STU prefill (flash_stu/utils/stu_utils.py:195-246: rfft -> product -> irfft, both sign
// branches), as in-LDS complex FFTs on gfx950, on the two parities of the sequence at once.
//
// With E and O the even- and odd-lag parts of the causal convolution of x with a filter f, the two branches are
// plus = E + O and minus = E - O.  Lags of one parity connect positions of fixed parities only, so with
//     z[m] = x[2m] + i x[2m+1],   fe[j] = f[2j],   fo[j] = f[2j+1]
// the convolution of the complex sequence z with the REAL filter fe holds E of both parities, E[2m] + i E[2m+1], and its
// convolution with fo holds Re[m] = O[2m+1] and Im[m] = O[2m+2].  One forward transform of z and one inverse per part
// replace a forward and an inverse transform of twice the length: for approx mode three transforms of n/2 points instead
// of two of n, for a bank of K filters 1 + 2K of n/2 instead of 1 + K of n, each one level shorter and in half the LDS,
// so that two workgroups share a compute unit where one filled it.
//
// A transform of N = n/2 points belongs to N/16 threads, 16 points each.  Forward: radix-2 stages grouped by four in
// registers, natural order in, bit-reversed out (twiddles depend on the block); the last group stays in registers, where
// the spectrum is multiplied; inverse: bit-reversed in, natural out (twiddles depend on the position).  Both directions
// multiply BEFORE they add, so a butterfly with its twiddle is six fused multiply-adds (u = a + w b, v = 2a - u) and a
// group of 16 points 192 instructions and 8 twiddles; a radix-16 butterfly followed by 15 twiddles took 228, and 44 more
// for the powers.  The upper half of z is zero and only the lower half of the results is wanted: the first stage copies
// and the last produces half.  The two innermost groups exchange among 16 threads of one wave, without a barrier.
//
// What bounds it: vector-ALU issue.  The exact-mode bank of 4 x 8192 x 1024 positions and channels and 24 filters issues 1.6 k
// instructions per thread and filter, takes 2.86 to 2.98 ms and keeps the vector ALUs busy for 90 % of its 5.5 M cycles
// (4.66 ms on transforms of 16384 points in 139 KB of LDS, one workgroup per compute unit; 3.77 ms while spectra and
// twiddles lay in position order, so that every load of a wave touched up to 64 lines).  bf16, before -> now, us: 8 x 512 x
// 768 24.5 -> 17.4, 32 x 300 x 2048 188 -> 105, 4 x 4096 x 2048 296 -> 218, one time-major sequence of 4096 x 2048 95 -> 50.
//
// Error.  A group that forms half of its twiddles from the others (turn32) rounds them twice more, and v = 2a - u carries u's
// roundings on.  Beside the rounding of bf16 results neither shows.  fp32 operands take their twiddles from the table, each
// rounded once, and where sums over all positions follow (filter spectra, gradients) butterflies of two rounded outputs each.
// Relative error of fp32 results against float64, transforms of the whole sequence in radix 16 / these with formed twiddles /
// now: 1000 positions 1.80e-7 / 2.03e-7 / 1.66e-7, filter's gradient 2.18e-7 / 2.60e-7 / 2.04e-7; 8000 positions 2.16e-7 /
// 2.50e-7 / 1.90e-7 and 2.54e-7 / 3.24e-7 / 2.35e-7.  us, formed / now: 8 x 2048 x 768 64 / 64, gradients 105 / 110 (of both
// branches 164 / 181); 4 x 4096 x 2048 210 / 210; 32 x 300 x 2048 106 / 104.
#include "fstu_common.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef float2 cpx;

// LDS index of element i of a column: one pad slot every 16 elements keeps the stride-16 accesses of the stride-1 group
// (and every other power-of-two stride) off a single bank.
__device__ __forceinline__ int phys(int i) { return i + (i >> 4); }

// ---------------------------------------------------------------- butterflies
// How exact a transform is (see the note above).  FORMED: half the twiddles formed by turn32; TABLE: all from the table;
// TABLE_STEPS: the same stage by stage, for the row pieces, whose other registers leave the scheduler no room to run stages
// into each other (8 x 2048 x 768 72 us without, 64 with; the bank of filters of 2 x 2048 x 256 122 without, 139 with); DIRECT:
// all from the table and both outputs of a butterfly formed from its inputs.
enum { FORMED, TABLE, TABLE_STEPS, DIRECT };
template <typename T, int HOW> __host__ __device__ constexpr int fine() { return sizeof(T) == 4 ? HOW : FORMED; }
// (a, b) <- (a + w r b, a - w r b), r = 1 or (ROT) the quarter turn of the direction (-i forward, +i inverse)
template <bool INV, bool ROT>
__device__ __forceinline__ cpx turn(cpx b) {
  if constexpr (!ROT) return b;
  return INV ? make_float2(-b.y, b.x) : make_float2(b.y, -b.x);
}
template <bool INV, bool ROT>
__device__ __forceinline__ void bfly1(cpx& a, cpx& b) {
  const cpx t = turn<INV, ROT>(b);
  b = make_float2(a.x - t.x, a.y - t.y);
  a = make_float2(a.x + t.x, a.y + t.y);
}
template <bool INV, bool ROT, int HOW>
__device__ __forceinline__ void bfly(cpx& a, cpx& b, cpx w) {
  const cpx t = turn<INV, ROT>(b);
  const cpx u = make_float2(fmaf(-w.y, t.y, fmaf(w.x, t.x, a.x)), fmaf(w.y, t.x, fmaf(w.x, t.y, a.y)));
  b = HOW == DIRECT ? make_float2(fmaf(w.y, t.y, fmaf(-w.x, t.x, a.x)), fmaf(-w.y, t.x, fmaf(-w.x, t.y, a.y)))
           : make_float2(fmaf(2.f, a.x, -u.x), fmaf(2.f, a.y, -u.y));
  a = u;
}
// a + w r b alone
template <bool INV, bool ROT>
__device__ __forceinline__ cpx bsum(cpx a, cpx b, cpx w) {
  const cpx t = turn<INV, ROT>(b);
  return make_float2(fmaf(-w.y, t.y, fmaf(w.x, t.x, a.x)), fmaf(w.y, t.x, fmaf(w.x, t.y, a.y)));
}
__device__ __forceinline__ cpx cmul(cpx a, cpx b) { return make_float2(fmaf(a.x, b.x, -a.y * b.y), fmaf(a.x, b.y, a.y * b.x)); }

// ---------------------------------------------------------------- groups of 2^G points in registers
// cos / sin of k/32 turns, k = 0 .. 7
__device__ __forceinline__ constexpr float cos32(int k) {
  constexpr float c[8] = {1.f, 0.98078528040323044f, 0.92387953251128674f, 0.83146961230254524f, 0.70710678118654752f, 0.55557023301960222f, 0.38268343236508977f, 0.19509032201612827f};
  return c[k];
}
__device__ __forceinline__ constexpr float sin32(int k) { return k == 0 ? 0.f : cos32(8 - k); }
// e^(+-2 pi i k / 32), k = 0 .. 7
template <bool INV> __device__ __forceinline__ cpx root32(int k) { return make_float2(cos32(k), INV ? sin32(k) : -sin32(k)); }
template <bool INV> __device__ __forceinline__ cpx turn32(cpx z, int k) {
  if (k == 0) return z;
  if (k == 4) return INV ? make_float2((z.x - z.y) * cos32(4), (z.x + z.y) * cos32(4)) : make_float2((z.x + z.y) * cos32(4), (z.y - z.x) * cos32(4));
  const float c = cos32(k), s = INV ? sin32(k) : -sin32(k);
  return make_float2(fmaf(c, z.x, -s * z.y), fmaf(c, z.y, s * z.x));
}
__host__ __device__ constexpr int brev_bits(int v, int bits) {
  int r = 0;
  for (int i = 0; i < bits; ++i) r |= ((v >> i) & 1) << (bits - 1 - i);
  return r;
}
// The twiddles of G stages: w^(2^i), which the first butterfly (block) of stage G-1-i uses; but for FORMED those of the others
// up to quarter turns too.
template <int G, int HOW> struct Powers { cpx w[HOW != FORMED ? 1 << (G - 1) : G]; };
// where the twiddle of stage s and q steps of 2^(4-s)/32 turns lies
__host__ __device__ constexpr int twiddle_at(int G, int s, int q) { return q == 0 ? G - 1 - s : s == 2 ? G : q == 2 ? 5 : q == 1 ? 6 : 7; }

// G forward stages on 2^G points a fixed distance apart, natural order in, bit-reversed out.  TW: times the block's
// twiddles t; HALF0: the upper half of the inputs is zero.
template <int G, bool TW, bool HALF0, int HOW>
__device__ __forceinline__ void fwd_stages(cpx* v, const Powers<G, HOW>& t) {
#pragma unroll
  for (int s = 0; s < G; ++s) {
    const int dist = 1 << (G - 1 - s);
    if constexpr (HOW == TABLE_STEPS) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < (1 << s); ++b) {
      const int k = brev_bits(b, s), quarter = s > 0 ? 1 << (s - 1) : 1;
      const bool rot = s > 0 && k >= quarter;
      const int q = rot ? k - quarter : k, kr = q << (4 - s);       // in 1/32 turns
#pragma unroll
      for (int j = 0; j < dist; ++j) {
        cpx &x = v[b * 2 * dist + j], &y = v[b * 2 * dist + j + dist];
        if (s == 0 && HALF0) { y = x; continue; }
        if (!TW && kr == 0) {
          if (rot) bfly1<false, true>(x, y); else bfly1<false, false>(x, y);
        } else {
          const cpx w = !TW ? root32<false>(kr) : HOW != FORMED ? t.w[twiddle_at(G, s, q)] : turn32<false>(t.w[G - 1 - s], kr);
          if (rot) bfly<false, true, HOW>(x, y, w); else bfly<false, false, HOW>(x, y, w);
        }
      }
    }
  }
}
// G inverse stages, bit-reversed in, natural out; t holds the conjugate twiddles of the position.  LOWER: only the lower
// half of the results is produced.
template <int G, bool TW, bool LOWER, int HOW>
__device__ __forceinline__ void inv_stages(cpx* v, const Powers<G, HOW>& t) {
#pragma unroll
  for (int s = 0; s < G; ++s) {
    const int dist = 1 << s;
    if constexpr (HOW == TABLE_STEPS) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < (1 << s); ++b) {
      const int quarter = s > 0 ? 1 << (s - 1) : 1;
      const bool rot = s > 0 && b >= quarter;
      const int q = rot ? b - quarter : b, kr = q << (4 - s);
#pragma unroll
      for (int g = 0; g < (1 << G); g += 2 * dist) {
        cpx &x = v[g + b], &y = v[g + b + dist];
        const cpx w = !TW ? root32<true>(kr) : HOW != FORMED ? t.w[twiddle_at(G, s, q)] : turn32<true>(t.w[G - 1 - s], kr);
        if (LOWER && s == G - 1) {
          if (rot) x = bsum<true, true>(x, y, w); else x = bsum<true, false>(x, y, w);
        } else if (!TW && kr == 0) {
          if (rot) bfly1<true, true>(x, y); else bfly1<true, false>(x, y);
        } else {
          if (rot) bfly<true, true, HOW>(x, y, w); else bfly<true, false, HOW>(x, y, w);
        }
      }
    }
  }
}

// ---------------------------------------------------------------- a transform on N/16 threads, 16 points each
// Groups of stages from the inside out: four at stride 1 (16 neighbours), four at stride 16 (16 neighbouring threads
// exchange: one wave), four at stride 256, and the LOGN mod 4 remaining ones outermost.  Natural order is held by the
// threads of the outermost group, in registers: point r + Q*m with r = u + i*G (i < NI), m < R; of the zero-padded input
// and of the results only the lower half, m < R/2, 8 points per thread.
template <int LOGN> struct Half {
  static constexpr int N = 1 << LOGN, G = N / 16, STRIDE = N + N / 16, REM = LOGN & 3, NF = LOGN / 4;
  static constexpr int GL = REM ? REM : 4, R = 1 << GL, Q = N / R, NI = 16 / R, H = R / 2;   // the outermost group
  static constexpr int MID = REM ? NF - 1 : NF - 2;                                        // groups between it and stride 1
  static constexpr bool ONE_WAVE = G <= 64;                                                // a column's threads are in one wave
};

// the exchange through LDS behind a group: among the threads of one wave, or of the workgroup
__device__ __forceinline__ void wave_sync() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_sched_barrier(0);   // the next group starts with its own registers
}
template <int LOGN> __device__ __forceinline__ void col_sync() {
  if constexpr (Half<LOGN>::ONE_WAVE) wave_sync();
  else __syncthreads();
}

// The twiddle table: for every group the powers 1, 2, 4, 8 of the twiddles of its positions (inverse, conjugated) or
// blocks (forward, in block order) and behind them what twiddle_at names, as planes of two each, so that the lanes of a wave
// read whole lines and a group's twiddles are at most four loads (FORMED: two).  All of it fits n entries.
template <int LOGN> struct Table {
  using W = Half<LOGN>;
  static constexpr int planes(int stages) { return 1 << (stages - 1); }                        // entries per position
  static constexpr int INV1 = 0;                                                   // stride 16: 16 positions
  static constexpr int INV2 = INV1 + (W::MID >= 1 ? 16 * 8 : 0);                   // stride 256
  static constexpr int OUTER = INV2 + (W::MID >= 2 ? 256 * 8 : 0);                 // outermost group: Q positions
  static constexpr int FWD2 = OUTER + W::Q * planes(W::GL);
  static constexpr int FWD1 = FWD2 + (W::MID >= 2 ? (W::N >> 12) * 8 : 0);         // stride 16: N / 256 blocks
  static constexpr int FWD0 = FWD1 + (W::MID >= 1 ? (W::N >> 8) * 8 : 0);          // stride 1: N / 16 blocks
  static constexpr int END = FWD0 + (W::N >> 4) * 8;
  static_assert(END <= 2 * W::N, "the table fits n entries");
};
// the twiddles of GS stages of entry i of a part of the table that has `count` entries
template <int GS, int HOW> __device__ __forceinline__ Powers<GS, HOW> powers(const cpx* __restrict__ part, int count, int i) {
  constexpr int NW = HOW != FORMED ? 1 << (GS - 1) : GS;
  Powers<GS, HOW> t;
  if constexpr (GS == 1) {
    t.w[0] = part[i];
  } else {
#pragma unroll
    for (int p = 0; p < (NW + 1) / 2; ++p) {
      const float4 a = ((const float4*)part)[p * count + i];
      t.w[2 * p] = make_float2(a.x, a.y);
      if (2 * p + 1 < NW) t.w[2 * p + 1] = make_float2(a.z, a.w);
    }
  }
  return t;
}
// position of the thread's k-th natural-order point (k < 8)
template <int LOGN> __device__ __forceinline__ int point(int u, int k) {
  using W = Half<LOGN>;
  return u + (k / W::H) * W::G + (k % W::H) * W::Q;
}

// LDS index of the thread's i-th butterfly of the outermost group
template <int LOGN> __device__ __forceinline__ int butterfly_at(int u, int i) {
  using W = Half<LOGN>;
  if constexpr (W::G >= 16) return phys(u) + i * (W::G + W::G / 16);
  return phys(u + i * W::G);
}

// four stages at stride 16^LEVEL, in place
template <int LOGN, int LEVEL, int HOW>
__device__ __forceinline__ void fwd_mid(cpx* __restrict__ col, const cpx* __restrict__ tw, int u) {
  constexpr int LQ = 4 * LEVEL, S = LOGN - 4 - LQ, ST = (1 << LQ) + (1 << LQ) / 16;
  const int blk = u >> LQ;
  const Powers<4, HOW> t = powers<4, HOW>(tw + (LEVEL == 1 ? Table<LOGN>::FWD1 : Table<LOGN>::FWD2), 1 << S, blk);
  cpx* p = col + phys((blk << (LQ + 4)) + (u & ((1 << LQ) - 1)));
  cpx v[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) v[m] = p[m * ST];
  fwd_stages<4, true, false, HOW>(v, t);
#pragma unroll
  for (int m = 0; m < 16; ++m) p[m * ST] = v[m];
}
template <int LOGN, int LEVEL, int HOW>
__device__ __forceinline__ void inv_mid(cpx* __restrict__ col, const cpx* __restrict__ tw, int u) {
  constexpr int LQ = 4 * LEVEL, ST = (1 << LQ) + (1 << LQ) / 16;
  const int r = u & ((1 << LQ) - 1);
  const Powers<4, HOW> t = powers<4, HOW>(tw + (LEVEL == 1 ? Table<LOGN>::INV1 : Table<LOGN>::INV2), 1 << LQ, r);
  cpx* p = col + phys(((u >> LQ) << (LQ + 4)) + r);
  cpx v[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) v[m] = p[m * ST];
  inv_stages<4, true, false, HOW>(v, t);
#pragma unroll
  for (int m = 0; m < 16; ++m) p[m * ST] = v[m];
}

// z: the thread's 8 points of the lower half -> xs: spectrum of positions 16u .. 16u+15 (bit-reversed order).  When it
// returns, a thread may overwrite its own 16 positions of the column.
template <int LOGN, int HOW>
__device__ __forceinline__ void fft_forward(cpx* __restrict__ col, const cpx* __restrict__ tw, int u, const cpx (&z)[8], cpx (&xs)[16]) {
  using W = Half<LOGN>;
#pragma unroll
  for (int i = 0; i < W::NI; ++i) {
    cpx v[W::R];
#pragma unroll
    for (int m = 0; m < W::H; ++m) v[m] = z[i * W::H + m];
    fwd_stages<W::GL, false, true, HOW>(v, Powers<W::GL, HOW>{});
    cpx* p = col + butterfly_at<LOGN>(u, i);
#pragma unroll
    for (int m = 0; m < W::R; ++m) p[m * (W::Q + W::Q / 16)] = v[m];
  }
  if constexpr (W::MID >= 2) { col_sync<LOGN>(); fwd_mid<LOGN, 2, HOW>(col, tw, u); }
  if constexpr (W::MID >= 1) { col_sync<LOGN>(); fwd_mid<LOGN, 1, HOW>(col, tw, u); }
  if constexpr (W::MID == 0) col_sync<LOGN>();
  else wave_sync();
  const Powers<4, HOW> t = powers<4, HOW>(tw + Table<LOGN>::FWD0, W::G, u);
#pragma unroll
  for (int m = 0; m < 16; ++m) xs[m] = col[17 * u + m];
  fwd_stages<4, true, false, HOW>(xs, t);
}

// v: spectrum of positions 16u .. 16u+15 -> r: the thread's 8 points of the lower half of the result.  The thread's own 16
// positions of the column must be free; when it returns, other threads may still read the column.
template <int LOGN, int HOW>
__device__ __forceinline__ void fft_inverse(cpx* __restrict__ col, const cpx* __restrict__ tw, int u, cpx (&v)[16], cpx (&r)[8]) {
  using W = Half<LOGN>;
  inv_stages<4, false, false, HOW>(v, Powers<4, HOW>{});
#pragma unroll
  for (int m = 0; m < 16; ++m) col[17 * u + m] = v[m];
  if constexpr (W::MID == 0) col_sync<LOGN>();
  else wave_sync();
  if constexpr (W::MID >= 1) { inv_mid<LOGN, 1, HOW>(col, tw, u); col_sync<LOGN>(); }
  if constexpr (W::MID >= 2) { inv_mid<LOGN, 2, HOW>(col, tw, u); col_sync<LOGN>(); }
#pragma unroll
  for (int i = 0; i < W::NI; ++i) {
    const int rr = u + i * W::G;
    const Powers<W::GL, HOW> t = powers<W::GL, HOW>(tw + Table<LOGN>::OUTER, W::Q, rr);
    const cpx* p = col + butterfly_at<LOGN>(u, i);
    cpx x[W::R];
#pragma unroll
    for (int m = 0; m < W::R; ++m) x[m] = p[m * (W::Q + W::Q / 16)];
    inv_stages<W::GL, true, true, HOW>(x, t);
#pragma unroll
    for (int m = 0; m < W::H; ++m) r[i * W::H + m] = x[m];
  }
}

// Im of the result one position earlier (0 in front of the first) for each of a thread's 8 results: the neighbouring
// lane's, and across the ends of the waves through rec, 8 floats per wave (or column, where a wave holds several) of the
// workgroup.  Contains the barrier behind which the column is free.
template <int LOGN>
__device__ __forceinline__ void earlier_im(const cpx (&r)[8], float (&prev)[8], float* rec, int u) {
  using W = Half<LOGN>;
  constexpr int SEG = W::G < 64 ? W::G : 64;           // threads of a column in one wave
  const int seg = threadIdx.x / SEG, in = u % SEG;
  if (in == SEG - 1) {
#pragma unroll
    for (int k = 0; k < 8; ++k) rec[seg * 8 + k] = r[k].y;
  }
  col_sync<LOGN>();
#pragma unroll
  for (int k = 0; k < 8; ++k) prev[k] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(r[k].y), 0x138, 0xf, 0xf, true));   // lane - 1
  if (in == 0) {
    // u > 0: the last thread of the wave in front; u == 0: the column's last thread, one butterfly (or, for the first of
    // them, one step of Q) earlier
    const float* q = rec + (u > 0 ? seg - 1 : seg + W::G / SEG - 1) * 8;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int wrap = k >= W::H ? k - W::H : (W::NI - 1) * W::H + k - 1;
      prev[k] = u > 0 ? q[k] : (k > 0 ? q[wrap] : 0.f);
    }
  }
}

// The thread's 16 spectrum values times x.  A spectrum lies in memory as the transform's threads hold it: the values of
// positions 16u + 2k and 16u + 2k + 1 at float4 k*G + u, so that the lanes of a load read whole lines (in position order
// every load of a wave would touch 64 of them, and the eight loads together more than the L1 holds).
template <int LOGN>
__device__ __forceinline__ void product16(const cpx* __restrict__ sp, const cpx (&x)[16], cpx (&v)[16]) {
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float4 s = ((const float4*)sp)[k * Half<LOGN>::G];
    v[2 * k] = cmul(x[2 * k], make_float2(s.x, s.y));
    v[2 * k + 1] = cmul(x[2 * k + 1], make_float2(s.z, s.w));
  }
}

// Inside a loop over filters or channels the twiddles and addresses of a transform are the same every time round; hoisted
// out of the loop they would not fit the registers.  Passing the table pointer and the thread's index through here keeps
// their loads and arithmetic where they are used.
__device__ __forceinline__ const cpx* here(const cpx* p) {
  asm volatile("" : "+s"(p));
  return p;
}
__device__ __forceinline__ int here(int i) {
  asm volatile("" : "+v"(i));
  return i;
}

// the outputs of pair m from the even-lag result e = E[2m] + i E[2m+1] and the odd-lag results O[2m] = Im[m-1], O[2m+1] = Re[m]
// (SUM: both branches rounded and added, else the plus branch)
template <typename T, bool SUM>
__device__ __forceinline__ float branch_sum(float e, float o) {
  return SUM ? DT<T>::rnd(e + o) + DT<T>::rnd(e - o) : e + o;
}
template <typename T>
__device__ __forceinline__ float branch_sum(float e, float o, int mode) {
  return mode == 0 ? branch_sum<T, true>(e, o) : branch_sum<T, false>(e, o);
}

// ---------------------------------------------------------------- twiddle table
template <int LOGN>
__global__ void __launch_bounds__(256) fft_twiddle_kernel(cpx* __restrict__ tw) {
  using W = Half<LOGN>;
  using B = Table<LOGN>;
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= 2 * W::N) return;
  // entry j: its part, its index there, its power and its angle in turns
  struct Part { int begin, count, entries, shift; bool fwd; };
  const Part parts[6] = {{B::INV1, 16, W::MID >= 1 ? 8 : 0, 8, false},
                         {B::INV2, 256, W::MID >= 2 ? 8 : 0, 12, false},
                         {B::OUTER, W::Q, B::planes(W::GL), LOGN, false},
                         {B::FWD2, W::N >> 12, W::MID >= 2 ? 8 : 0, 0, true},
                         {B::FWD1, W::N >> 8, W::MID >= 1 ? 8 : 0, 0, true},
                         {B::FWD0, W::N >> 4, 8, 0, true}};
  double turns = 0.0;
  for (int q = 0; q < 6; ++q) {
    const Part& p = parts[q];
    const int o = j - p.begin;
    if (p.entries == 0 || o < 0 || o >= p.count * p.entries) continue;
    int i = o, power = 0, steps = 0;                   // w^(2^power), `steps` of 1/32 turns further
    if (p.entries > 1) {
      i = (o >> 1) % p.count;
      const int at = 2 * ((o >> 1) / p.count) + (o & 1), G = p.entries == 8 ? 4 : p.entries == 4 ? 3 : 2;
      for (int st = 0; st < G; ++st)
        for (int k = 0; k < (st < 2 ? 1 : 1 << (st - 1)); ++k)
          if (twiddle_at(G, st, k) == at) {
            power = G - 1 - st;
            steps = k << (4 - st);
          }
    }
    if (p.fwd) {
      int lg = 0;
      while ((1 << lg) < p.count) ++lg;
      const double f = lg ? (double)(__brev((unsigned)i) >> (32 - lg)) : 0.0;
      turns = -f * (double)(1 << power) / (double)(p.count * 16) - steps / 32.0;
    } else {
      turns = (double)i * (double)(1 << power) / (double)(1 << p.shift) + steps / 32.0;
    }
  }
  double s, c;
  sincospi(2.0 * turns, &s, &c);
  tw[j] = make_float2((float)c, (float)s);
}

// Columns a workgroup transforms at a time: 512 threads (70 KB of LDS, two workgroups per compute unit) for the long
// transforms, at most 16 (32 at N = 32) columns for the short ones; a thread may hold 128 registers.
template <int LOGN> __host__ __device__ constexpr int fft_lcols() { return LOGN >= 13 ? 0 : LOGN == 12 ? 1 : LOGN == 11 ? 2 : LOGN >= 9 ? 3 : LOGN >= 6 ? 4 : 5; }
template <int LOGN> __host__ __device__ constexpr int fft_threads() { return (1 << (LOGN + fft_lcols<LOGN>())) / 16; }
template <int LOGN, int NT> __host__ __device__ constexpr size_t fft_lds_bytes() {      // columns, and earlier_im's record
  return (size_t)(NT / Half<LOGN>::G) * Half<LOGN>::STRIDE * sizeof(cpx) + (size_t)(NT / (Half<LOGN>::G < 64 ? Half<LOGN>::G : 64)) * 32;
}

// ---------------------------------------------------------------- pairs of positions
// Two consecutive positions of a channel as they lie in memory when time is contiguous, and staged in LDS.
template <typename T> struct Pair;
template <> struct Pair<bf16_t> {
  typedef unsigned type;
  typedef unsigned mem __attribute__((aligned(2)));    // at any element's address
  static __device__ __forceinline__ cpx get(type v) { return make_float2(__uint_as_float(v << 16), __uint_as_float(v & 0xffff0000u)); }
  static __device__ __forceinline__ type put(float a, float b) { return pack2_bf16(a, b); }
};
template <> struct Pair<float> {
  typedef float type __attribute__((ext_vector_type(2)));
  typedef float mem __attribute__((ext_vector_type(2), aligned(4)));
  static __device__ __forceinline__ cpx get(type v) { return make_float2(v[0], v[1]); }
  static __device__ __forceinline__ type put(float a, float b) { return type{a, b}; }
};

// ---------------------------------------------------------------- filter spectra
// Column j of the filter matrix (element (s, j) at filt[s*f_ls + j*f_cs], taps s < taps) -> Fe / N in spec[j*n ..] and
// Fo / N in spec[j*n + N ..], in the order of product16.  One transform of fe + i fo gives both: with G its
// spectrum, Fe[k] = (G[k] + conj G[-k]) / 2 and Fo[k] = (G[k] - conj G[-k]) / 2i.  Channel-contiguous filters go through
// LDS so that the lanes of a load run along the channels.
template <typename T, int LOGN>
__global__ void __launch_bounds__(fft_threads<LOGN>())
fft_filter_kernel(const T* __restrict__ filt, size_t f_ls, size_t f_cs, cpx* __restrict__ spec, const cpx* __restrict__ tw,
                  int taps, int ncol_total) {
  extern __shared__ cpx fft_lds[];
  using H = Half<LOGN>;
  constexpr int N = H::N, LC = fft_lcols<LOGN>(), COLS = 1 << LC, NT = fft_threads<LOGN>();
  const int c0 = blockIdx.x * COLS;
  for (int idx = threadIdx.x; idx < COLS * (N / 2); idx += NT) {
    const int colid = idx & (COLS - 1), m = idx >> LC;
    const T* f = filt + (size_t)(2 * m) * f_ls + (size_t)(c0 + colid) * f_cs;
    cpx g = make_float2(0.f, 0.f);
    if (c0 + colid < ncol_total) {
      if (2 * m < taps) g.x = DT<T>::ld(f);
      if (2 * m + 1 < taps) g.y = DT<T>::ld(f + f_ls);
    }
    fft_lds[(size_t)colid * H::STRIDE + phys(m)] = g;
  }
  __syncthreads();
  const int colid = threadIdx.x / H::G, u = threadIdx.x % H::G;
  cpx* col = fft_lds + (size_t)colid * H::STRIDE;
  cpx z[8], v[16];
#pragma unroll
  for (int k = 0; k < 8; ++k) z[k] = col[phys(point<LOGN>(u, k))];
  __syncthreads();
  fft_forward<LOGN, fine<T, DIRECT>()>(col, tw, u, z, v);
#pragma unroll
  for (int m = 0; m < 16; ++m) col[17 * u + m] = v[m];
  __syncthreads();
  if (c0 + colid >= ncol_total) return;
  const float sc = 0.5f / (float)N;
  float4* out = (float4*)(spec + (size_t)(c0 + colid) * (2 * N)) + u;
#pragma unroll
  for (int m = 0; m < 16; m += 2) {
    cpx h[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const unsigned k = __brev((unsigned)(16 * u + m + i)) >> (32 - LOGN), km = (N - k) & (N - 1);
      h[i] = col[phys((int)(__brev(km) >> (32 - LOGN)))];
    }
    out[(m / 2) * H::G] = make_float4((v[m].x + h[0].x) * sc, (v[m].y - h[0].y) * sc, (v[m + 1].x + h[1].x) * sc, (v[m + 1].y - h[1].y) * sc);
    out[N / 2 + (m / 2) * H::G] = make_float4((v[m].y + h[0].y) * sc, (h[0].x - v[m].x) * sc, (v[m + 1].y + h[1].y) * sc, (h[1].x - v[m + 1].x) * sc);
  }
}

// ---------------------------------------------------------------- convolution of time-major slabs, one filter or a bank
// Positions lie next to each other (the transposed activations of a few long sequences, the U+- slabs of the filter bank):
// neighbouring threads hold neighbouring pairs, which are read from and written to memory straight from registers.
// Channel c of x at x[b*x_sb + c*x_sc]; the K outputs of a channel (K = 1: per-channel spectra spec[c]; K > 1: a shared
// bank spec[k]) at y[b*y_sb + k*y_sk + c*y_sc] (and y2 likewise).
// mode 0: y = T(T(plus) + T(minus));  mode 1: y = T(plus);  mode 2: y = T(plus), y2 = T(minus).
// NT threads: as many columns as fill the longest transforms' workgroup or, for small grids, one wave or column.  A workgroup takes the
// filters of its slice of the bank, kper of them (bank_slice); the loop counts from 0, which keeps the registers of the whole bank's (4 x 8192
// x 1024 2.95 ms; 3.00 from k0 to k1).
template <typename T, int LOGN, int NT, bool SUM>
__global__ void __launch_bounds__(NT, 4)
fft_slab_kernel(const T* __restrict__ x, size_t x_sb, size_t x_sc, const cpx* __restrict__ spec, T* __restrict__ y,
                T* __restrict__ y2, size_t y_sb, size_t y_sk, size_t y_sc, const cpx* __restrict__ tw, int Tn, int d, int K,
                int kper, int xcd_remap) {
  extern __shared__ cpx fft_lds[];
  using W = Half<LOGN>;
  constexpr int N = W::N, COLS = NT / W::G;
  const int k0 = blockIdx.z * kper, nk = min(K - k0, kper);   // the filters of this workgroup's slice
  int bx = blockIdx.x;
  if (xcd_remap) bx = (bx & 7) * (gridDim.x >> 3) + (bx >> 3);
  const int b = blockIdx.y, mycol = threadIdx.x / W::G, u = threadIdx.x % W::G, c = bx * COLS + mycol;
  const bool live = c < d;
  cpx* col = fft_lds + (size_t)mycol * W::STRIDE;
  float* rec = (float*)(fft_lds + (size_t)COLS * W::STRIDE);
  const T* xp = x + (size_t)b * x_sb + (size_t)min(c, d - 1) * x_sc;
  cpx z[8], xs[16];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int t = 2 * point<LOGN>(u, k);
    z[k] = make_float2(0.f, 0.f);
    if (t + 1 < Tn) z[k] = Pair<T>::get(*(const typename Pair<T>::mem*)(xp + t));
    else if (t < Tn) z[k].x = DT<T>::ld(xp + t);
  }
  fft_forward<LOGN, fine<T, TABLE>()>(col, tw, u, z, xs);
  const cpx* sp = spec + (size_t)(K == 1 ? min(c, d - 1) : k0) * (2 * N) + 2 * u;
  T* yp = y + (size_t)b * y_sb + (size_t)k0 * y_sk + (size_t)c * y_sc;
  T* yp2 = y2 + (size_t)b * y_sb + (size_t)k0 * y_sk + (size_t)c * y_sc;
  for (int k = 0; k < nk; ++k, sp += 2 * N, yp += y_sk, yp2 += y_sk) {
    cpx v[16], e[8], o[8];
    float prev[8];
    product16<LOGN>(sp, xs, v);
    fft_inverse<LOGN, fine<T, TABLE>()>(col, here(tw), here(u), v, e);
    col_sync<LOGN>();
    product16<LOGN>(sp + N, xs, v);
    fft_inverse<LOGN, fine<T, TABLE>()>(col, here(tw), here(u), v, o);
    earlier_im<LOGN>(o, prev, rec, u);
    const int uo = here(u), tmax = live ? Tn - 1 : 0;  // pairs t, t + 1 <= tmax are stored
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int t = 2 * point<LOGN>(uo, i);
      if (t < tmax) *(typename Pair<T>::mem*)(yp + t) = Pair<T>::put(branch_sum<T, SUM>(e[i].x, prev[i]), branch_sum<T, SUM>(e[i].y, o[i].x));
    }
    if (!SUM && y2) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int t = 2 * point<LOGN>(uo, i);
        if (t < tmax) *(typename Pair<T>::mem*)(yp2 + t) = Pair<T>::put(e[i].x - prev[i], e[i].y - o[i].x);
      }
    }
    if (live && (Tn & 1)) {                            // an odd length's last position
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (2 * point<LOGN>(uo, i) == Tn - 1) {
          DT<T>::st(yp + Tn - 1, branch_sum<T, SUM>(e[i].x, prev[i]));
          if (!SUM && y2) DT<T>::st(yp2 + Tn - 1, e[i].x - prev[i]);
        }
    }
  }
}

// ---------------------------------------------------------------- any strides
// The same for operands of any strides: element (b, t, c) of x at x[b*x_sb + t*x_st + c*x_sc], of the k-th output at
// y[b*y_sb + t*y_st + k*y_sk + c*y_sc].  Pairs pass through the columns' LDS so that the lanes of a memory access run
// along the channels.  A workgroup takes the filters of its slice of the bank, kper of them: few channels and rows alone
// are too few workgroups for the chip, and a slice more costs one forward transform beside the two inverse ones of each
// of its filters.  24 filters into (B, T, K, d), both branches, us with the whole bank per workgroup / in slices (the call's
// host side is 38): fp32 1 x 64 x 256 132 / 38, 2 x 100 x 256 140 / 38, 1 x 1000 x 256 226 / 53, 1 x 2048 x 256 247 / 84.
template <typename T, int LOGN>
__global__ void __launch_bounds__(fft_threads<LOGN>(), 4)
fft_conv_kernel(const T* __restrict__ x, size_t x_sb, size_t x_st, size_t x_sc, const cpx* __restrict__ spec,
                T* __restrict__ y, T* __restrict__ y2, size_t y_sb, size_t y_st, size_t y_sk, size_t y_sc,
                const cpx* __restrict__ tw, int Tn, int d, int K, int kper, int mode, int xcd_remap) {
  extern __shared__ cpx fft_lds[];
  using W = Half<LOGN>;
  constexpr int N = W::N, LC = fft_lcols<LOGN>(), COLS = 1 << LC, NT = fft_threads<LOGN>();
  int bx = blockIdx.x;
  if (xcd_remap) bx = (bx & 7) * (gridDim.x >> 3) + (bx >> 3);   // consecutive channel groups share an XCD
  const int c0 = bx * COLS, b = blockIdx.y, ncol = min(COLS, d - c0);
  const int k0 = blockIdx.z * kper, k1 = min(K, k0 + kper);
  float* rec = (float*)(fft_lds + (size_t)COLS * W::STRIDE);
  const T* xb = x + (size_t)b * x_sb + (size_t)c0 * x_sc;
  for (int idx = threadIdx.x; idx < COLS * (N / 2); idx += NT) {
    const int colid = idx & (COLS - 1), m = idx >> LC;
    cpx z = make_float2(0.f, 0.f);
    if (colid < ncol) {
      const T* p = xb + (size_t)(2 * m) * x_st + (size_t)colid * x_sc;
      if (2 * m < Tn) z.x = DT<T>::ld(p);
      if (2 * m + 1 < Tn) z.y = DT<T>::ld(p + x_st);
    }
    fft_lds[(size_t)colid * W::STRIDE + phys(m)] = z;
  }
  __syncthreads();
  const int mycol = threadIdx.x / W::G, u = threadIdx.x % W::G;
  cpx* col = fft_lds + (size_t)mycol * W::STRIDE;
  cpx z[8], xs[16];
#pragma unroll
  for (int k = 0; k < 8; ++k) z[k] = col[phys(point<LOGN>(u, k))];
  __syncthreads();
  fft_forward<LOGN, fine<T, TABLE>()>(col, tw, u, z, xs);
  const cpx* sp = spec + (size_t)(K == 1 ? min(c0 + mycol, d - 1) : k0) * (2 * N) + 2 * u;
  for (int k = k0; k < k1; ++k, sp += 2 * N) {
    cpx v[16], e[8], o[8];
    float prev[8];
    product16<LOGN>(sp, xs, v);
    fft_inverse<LOGN, fine<T, TABLE>()>(col, here(tw), here(u), v, e);
    col_sync<LOGN>();
    product16<LOGN>(sp + N, xs, v);
    fft_inverse<LOGN, fine<T, TABLE>()>(col, here(tw), here(u), v, o);
    earlier_im<LOGN>(o, prev, rec, u);
    for (int br = 0; br < (mode == 2 ? 2 : 1); ++br) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 8; ++i)
        col[phys(point<LOGN>(here(u), i))] = br ? make_float2(e[i].x - prev[i], e[i].y - o[i].x)
                                               : make_float2(branch_sum<T>(e[i].x, prev[i], mode), branch_sum<T>(e[i].y, o[i].x, mode));
      __syncthreads();
      T* yb = (br ? y2 : y) + (size_t)b * y_sb + (size_t)k * y_sk + (size_t)c0 * y_sc;
      for (int idx = threadIdx.x; idx < COLS * (N / 2); idx += NT) {
        const int colid = idx & (COLS - 1), m = idx >> LC;
        if (colid >= ncol || 2 * m >= Tn) continue;
        const cpx r = fft_lds[(size_t)colid * W::STRIDE + phys(m)];
        T* q = yb + (size_t)(2 * m) * y_st + (size_t)colid * y_sc;
        DT<T>::st(q, r.x);
        if (2 * m + 1 < Tn) DT<T>::st(q + y_st, r.y);
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------- whole 16-byte row pieces per lane
// The same for channel-contiguous (B, T, d) operands with d a multiple of the workgroup's channel count: a workgroup owns
// CHW = max(COLS, 16 bytes' worth) neighbouring channels, reads pairs of rows as 16-byte pieces (all loads in flight at
// once, kept in registers), passes the pairs of COLS channels at a time through LDS to the threads of their transforms and
// the finished pairs back, and writes 16-byte pieces of the output rows.  A group takes the first COLS channels of the
// pieces and puts its results behind the last ones, so the loop over the groups is one copy of the code and every index
// into the registers is a constant.
template <typename T> struct RowVec;
template <> struct RowVec<bf16_t> {
  static constexpr int CH = 8;
  // channel e of two consecutive rows
  static __device__ __forceinline__ unsigned pair(const unsigned (&a)[4], const unsigned (&b)[4], int e) {
    return (e & 1) ? __builtin_amdgcn_perm(b[e >> 1], a[e >> 1], 0x07060302) : __builtin_amdgcn_perm(b[e >> 1], a[e >> 1], 0x05040100);
  }
  // the pairs r[0..NE) of the first NE channels go behind the others
  template <int NE> static __device__ __forceinline__ void rotate_in(unsigned (&a)[4], unsigned (&b)[4], const unsigned (&r)[NE]) {
    if constexpr (NE == 1) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        a[i] = __builtin_amdgcn_alignbit(a[i + 1], a[i], 16);
        b[i] = __builtin_amdgcn_alignbit(b[i + 1], b[i], 16);
      }
      a[3] = __builtin_amdgcn_alignbit(r[0], a[3], 16);
      b[3] = __builtin_amdgcn_alignbit(r[0] >> 16, b[3], 16);
    } else {
#pragma unroll
      for (int i = 0; i < 4 - NE / 2; ++i) { a[i] = a[i + NE / 2]; b[i] = b[i + NE / 2]; }
#pragma unroll
      for (int i = 0; i < NE / 2; ++i) {
        a[4 - NE / 2 + i] = __builtin_amdgcn_perm(r[2 * i + 1], r[2 * i], 0x05040100);
        b[4 - NE / 2 + i] = __builtin_amdgcn_perm(r[2 * i + 1], r[2 * i], 0x07060302);
      }
    }
  }
  static __device__ __forceinline__ unsigned cut(unsigned p, bool first, bool second) { return (first ? p & 0xffffu : 0u) | (second ? p & 0xffff0000u : 0u); }
};
template <> struct RowVec<float> {
  static constexpr int CH = 4;
  typedef Pair<float>::type pair_t;
  static __device__ __forceinline__ pair_t pair(const unsigned (&a)[4], const unsigned (&b)[4], int e) { return pair_t{__uint_as_float(a[e]), __uint_as_float(b[e])}; }
  template <int NE> static __device__ __forceinline__ void rotate_in(unsigned (&a)[4], unsigned (&b)[4], const pair_t (&r)[NE]) {
#pragma unroll
    for (int i = 0; i < 4 - NE; ++i) { a[i] = a[i + NE]; b[i] = b[i + NE]; }
#pragma unroll
    for (int i = 0; i < NE; ++i) { a[4 - NE + i] = __float_as_uint(r[i][0]); b[4 - NE + i] = __float_as_uint(r[i][1]); }
  }
  static __device__ __forceinline__ pair_t cut(pair_t p, bool first, bool second) { return pair_t{first ? p[0] : 0.f, second ? p[1] : 0.f}; }
};

template <typename T, int LOGN> struct RowCut {
  static constexpr int COLS = 1 << fft_lcols<LOGN>(), CH = RowVec<T>::CH, CHW = COLS > CH ? COLS : CH;
  static constexpr int VR = CHW / CH, NG = CHW / COLS, NE = COLS < CH ? COLS : CH;   // pieces per row, groups, channels per piece and group
  static constexpr int NT = fft_threads<LOGN>(), NV = (Half<LOGN>::N / 2) * VR / NT;
};

template <typename T, int LOGN>
__global__ void __launch_bounds__(fft_threads<LOGN>(), LOGN == 13 ? 2 : 4)
fft_conv_rows_kernel(const T* __restrict__ x, size_t x_sb, size_t x_st, const cpx* __restrict__ spec, T* __restrict__ y,
                     size_t y_sb, size_t y_st, const cpx* __restrict__ tw, int Tn, int mode, int xcd_remap) {
  extern __shared__ cpx fft_lds[];
  using W = Half<LOGN>;
  using R = RowCut<T, LOGN>;
  typedef typename Pair<T>::type pair_t;
  constexpr int N = W::N, COLS = R::COLS, CH = R::CH, CHW = R::CHW, VR = R::VR, NV = R::NV, NE = R::NE, NT = R::NT;
  constexpr int PST = N / 2 + 1;                       // staged pairs of a column (odd: neighbouring channels in different banks)
  static_assert(NV * NT == (N / 2) * VR && (size_t)PST * sizeof(pair_t) <= (size_t)W::STRIDE * sizeof(cpx), "whole pairs per thread");
  int bx = blockIdx.x;
  if (xcd_remap) bx = (bx & 7) * (gridDim.x >> 3) + (bx >> 3);   // consecutive channel groups share an XCD
  const int c0 = bx * CHW, b = blockIdx.y;
  const T* xb = x + (size_t)b * x_sb + c0;
  unsigned io[NV][2][4];
#pragma unroll
  for (int r = 0; r < NV; ++r) {
    const int q = threadIdx.x + r * NT, m = q / VR, part = q % VR;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // rows behind the sequence re-read its last row (no branch around the load) and are replaced by zeros below
      const uint4 v = *(const uint4*)(xb + (size_t)min(2 * m + h, Tn - 1) * x_st + part * CH);
      io[r][h][0] = v.x; io[r][h][1] = v.y; io[r][h][2] = v.z; io[r][h][3] = v.w;
    }
  }
  const int mycol = threadIdx.x / W::G, u = threadIdx.x % W::G;
  cpx* col = fft_lds + (size_t)mycol * W::STRIDE;
  float* rec = (float*)(fft_lds + (size_t)COLS * W::STRIDE);
  pair_t* stage = (pair_t*)fft_lds;                    // [column][pair], in the columns' place
  const cpx* sp = spec + (size_t)(c0 + mycol) * (2 * N) + 2 * u;
  // with the table's twiddles the inverse of 4096 points spills 23 registers, and the error is small enough without (3000 / 4096
  // positions 1.80e-7 / 1.99e-7, radix 16 2.04e-7 / 2.12e-7)
  constexpr int BACK = LOGN == 12 ? FORMED : TABLE_STEPS;
  for (int g = 0; g < R::NG; ++g, sp += (size_t)COLS * (2 * N)) {
    if (g > 0) __syncthreads();                        // the previous group's results have been collected
    const int tid = here((int)threadIdx.x), ug = here(u);
    const cpx* twg = here(tw);
#pragma unroll
    for (int r = 0; r < NV; ++r) {
      const int q = tid + r * NT, m = q / VR, part = q % VR;
#pragma unroll
      for (int e = 0; e < NE; ++e)
        stage[(VR > 1 ? part * CH + e : e) * PST + m] = RowVec<T>::cut(RowVec<T>::pair(io[r][0], io[r][1], e), 2 * m < Tn, 2 * m + 1 < Tn);
    }
    __syncthreads();
    cpx xs[16], v[16], e[8], o[8];
    float prev[8];
    {
      cpx z[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) z[k] = Pair<T>::get(stage[mycol * PST + point<LOGN>(ug, k)]);
      __syncthreads();
      fft_forward<LOGN, fine<T, TABLE_STEPS>()>(col, twg, ug, z, xs);
    }
    product16<LOGN>(sp, xs, v);
    fft_inverse<LOGN, fine<T, BACK>()>(col, here(tw), ug, v, e);
    col_sync<LOGN>();
    product16<LOGN>(sp + N, xs, v);
    fft_inverse<LOGN, fine<T, BACK>()>(col, here(tw), ug, v, o);
    earlier_im<LOGN>(o, prev, rec, ug);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i)
      stage[mycol * PST + point<LOGN>(ug, i)] = Pair<T>::put(branch_sum<T>(e[i].x, prev[i], mode), branch_sum<T>(e[i].y, o[i].x, mode));
    __syncthreads();
    const int tid_o = here((int)threadIdx.x);
#pragma unroll
    for (int r = 0; r < NV; ++r) {
      const int q = tid_o + r * NT, m = q / VR, part = q % VR;
      pair_t p[NE];
#pragma unroll
      for (int k = 0; k < NE; ++k) p[k] = stage[(VR > 1 ? part * CH + k : k) * PST + m];
      RowVec<T>::template rotate_in<NE>(io[r][0], io[r][1], p);
    }
  }
  T* yb = y + (size_t)b * y_sb + c0;
#pragma unroll
  for (int r = 0; r < NV; ++r) {
    const int q = threadIdx.x + r * NT, m = q / VR, part = q % VR;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (2 * m + h < Tn)
        *(uint4*)(yb + (size_t)(2 * m + h) * y_st + part * CH) = make_uint4(io[r][h][0], io[r][h][1], io[r][h][2], io[r][h][3]);
  }
}

// ---------------------------------------------------------------- gradients of the convolution
// With gE = g+ + g- and gO = g+ - g- (the gradients that reach the even- and the odd-lag part; g- = g+ where the branches
// are only ever added, then gO vanishes and so do all odd lags), zE[m] = gE[2m] + i gE[2m+1] and the shifted
// zS[m] = gO[2m+1] + i gO[2m+2]:
//   gradient of the input, both parities at once:  sum_j zE[m+j] fe[j] + zS[m+j] fo[j]      -> one inverse transform of
//                                                  ZE conj(Fe) + ZS conj(Fo)
//   gradient of the filter, one batch row's part:  gfe[j] = Re sum_m zE[m+j] conj z[m],  gfo[j] = Re sum_m zS[m+j] conj z[m]
// so that a column costs four transforms of n/2 points (six with odd lags) and its operands are read once.  Composed of
// the forward kernel on time-reversed fp32 copies the same took 18 n/2-point transforms per column, one launch and one
// filter transform per batch row, and flips, sums and casts in between.  Rows' parts of the filter gradient go to memory in
// fp32 and are added by fft_corr_finish_kernel in the order of the rows (no atomics: the same bits every time).
// The vector ALUs are busy for 44 % of it at 8 x 2048 x 768 bf16: the rest are the barriers and the staging between its
// transforms.  111 us there and 10 us for the sum over the rows, where the composed form took 0.95 ms; a training step at that
// size 1.69 -> 0.32 ms.
// A workgroup owns the COLS neighbouring channels that its threads transform and reads them as pieces of a row.
template <typename T, int LOGN> struct CorrCut {
  static constexpr int COLS = 1 << fft_lcols<LOGN>(), NE = COLS < RowVec<T>::CH ? COLS : RowVec<T>::CH, VR = COLS / NE;
  static constexpr int NT = fft_threads<LOGN>(), NV = (Half<LOGN>::N / 2) * VR / NT, PST = Half<LOGN>::N / 2 + 1;
};
template <typename E, int NE> struct alignas(NE * sizeof(E)) Piece { E e[NE]; };
// channels c .. c+NE-1 of a row: one access where rows and channels are whole pieces (vec), else element by element
template <typename T, int NE>
__device__ __forceinline__ void load_piece(const T* p, int c, int d, bool vec, float (&f)[NE]) {
  if (vec) {
    Piece<T, NE> v = {};
    if (c < d) v = *(const Piece<T, NE>*)p;
#pragma unroll
    for (int k = 0; k < NE; ++k) f[k] = DT<T>::ld(&v.e[k]);
  } else {
#pragma unroll
    for (int k = 0; k < NE; ++k) f[k] = c + k < d ? DT<T>::ld(p + k) : 0.f;
  }
}
template <typename T, int NE>
__device__ __forceinline__ void store_piece(T* p, int c, int d, bool vec, const float (&f)[NE]) {
  if (vec) {
    Piece<T, NE> v;
#pragma unroll
    for (int k = 0; k < NE; ++k) DT<T>::st(&v.e[k], f[k]);
    if (c < d) *(Piece<T, NE>*)p = v;
  } else {
#pragma unroll
    for (int k = 0; k < NE; ++k)
      if (c + k < d) DT<T>::st(p + k, f[k]);
  }
}
template <int LOGN>
__device__ __forceinline__ void conj_product16(const cpx* __restrict__ sp, const cpx (&x)[16], cpx (&v)[16], bool add) {
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float4 s = ((const float4*)sp)[k * Half<LOGN>::G];
    const cpx a = cmul(x[2 * k], make_float2(s.x, -s.y)), b = cmul(x[2 * k + 1], make_float2(s.z, -s.w));
    v[2 * k] = add ? make_float2(v[2 * k].x + a.x, v[2 * k].y + a.y) : a;
    v[2 * k + 1] = add ? make_float2(v[2 * k + 1].x + b.x, v[2 * k + 1].y + b.y) : b;
  }
}

// (both branches in fp32 at 2048 points: 155 registers are one workgroup per compute unit, 8 x 2048 x 768 212 us; held to 128, two, 181)
template <typename T, int LOGN, bool ODD>
__global__ void __launch_bounds__(fft_threads<LOGN>(), ODD && !(LOGN == 11 && sizeof(T) == 4) ? 2 : 4)
fft_corr_kernel(const T* __restrict__ g1, const T* __restrict__ g2, const T* __restrict__ x, const cpx* __restrict__ spec,
                T* __restrict__ gx, float* __restrict__ part, const cpx* __restrict__ tw, int Tn, int d, int lags, int vec,
                int xcd_remap) {
  extern __shared__ cpx fft_lds[];
  using W = Half<LOGN>;
  using R = CorrCut<T, LOGN>;
  constexpr int N = W::N, COLS = R::COLS, NE = R::NE, VR = R::VR, NV = R::NV, NT = R::NT, PST = R::PST;
  static_assert(NV * NT == (N / 2) * VR && PST <= W::STRIDE, "whole pieces per thread");
  int bx = blockIdx.x;
  if (xcd_remap) bx = (bx & 7) * (gridDim.x >> 3) + (bx >> 3);   // consecutive channel groups share an XCD
  const int c0 = bx * COLS, b = blockIdx.y;
  const size_t row0 = (size_t)b * Tn;
  const int mycol = threadIdx.x / W::G, u = threadIdx.x % W::G, c = min(c0 + mycol, d - 1);
  cpx* col = fft_lds + (size_t)mycol * W::STRIDE;
  cpx* stage = fft_lds;                                // [column][pair], in the columns' place
  // pairs of rows of one tensor (WHICH 0: x, 1: gE, 2: gO) -> stage
  auto put_stage = [&](auto which) {
    constexpr int WHICH = decltype(which)::value;
#pragma unroll
    for (int r = 0; r < NV; ++r) {
      const int q = threadIdx.x + r * NT, m = q / VR, cp = (q % VR) * NE;
      float f[2][NE];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int t = 2 * m + h;
#pragma unroll
        for (int k = 0; k < NE; ++k) f[h][k] = 0.f;
        if (t < Tn) {
          const size_t at = (row0 + t) * (size_t)d + c0 + cp;
          if constexpr (WHICH == 0) {
            load_piece<T, NE>(x + at, c0 + cp, d, vec, f[h]);
          } else {
            load_piece<T, NE>(g1 + at, c0 + cp, d, vec, f[h]);
            if constexpr (!ODD) {
#pragma unroll
              for (int k = 0; k < NE; ++k) f[h][k] *= 2.f;
            } else if (g2) {
              float s[NE];
              load_piece<T, NE>(g2 + at, c0 + cp, d, vec, s);
#pragma unroll
              for (int k = 0; k < NE; ++k) f[h][k] = WHICH == 1 ? f[h][k] + s[k] : f[h][k] - s[k];
            }
          }
        }
      }
#pragma unroll
      for (int k = 0; k < NE; ++k) stage[(cp + k) * PST + m] = make_float2(f[0][k], f[1][k]);
    }
    if (ODD && threadIdx.x < COLS) stage[threadIdx.x * PST + N / 2] = make_float2(0.f, 0.f);
  };
  auto take = [&](cpx (&z)[8]) {
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; ++k) z[k] = stage[mycol * PST + point<LOGN>(u, k)];
    __syncthreads();
  };
  // real parts of a correlation: lags 2j + ODDLAG of this row's part of the filter gradient
  auto put_part = [&](const cpx (&r)[8], int odd_lag) {
    __syncthreads();
    float* st = (float*)stage;
#pragma unroll
    for (int k = 0; k < 8; ++k) st[mycol * PST + point<LOGN>(u, k)] = r[k].x * (1.f / (float)N);
    __syncthreads();
    const int rows = ODD ? lags : (lags + 1) / 2;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int q = threadIdx.x + v * NT, m = q / VR, cp = (q % VR) * NE;
      if (2 * m + odd_lag >= lags) continue;
      float f[NE];
#pragma unroll
      for (int k = 0; k < NE; ++k) f[k] = st[(cp + k) * PST + m];
      const int row = ODD ? 2 * m + odd_lag : m;
      store_piece<float, NE>(part + ((size_t)b * rows + row) * d + c0 + cp, c0 + cp, d, vec, f);
    }
    __syncthreads();
  };
  const cpx* sp = spec + (size_t)c * (2 * N) + 2 * u;
  cpx zx[8], z[8], xe[16], w[16], r8[8];
  if (part) {
    put_stage(std::integral_constant<int, 0>{});
    take(zx);
  }
  put_stage(std::integral_constant<int, 1>{});
  take(z);
  fft_forward<LOGN, fine<T, DIRECT>()>(col, tw, u, z, xe);
  if (gx) conj_product16<LOGN>(sp, xe, w, false);
  if constexpr (ODD) {
    cpx xx[16];
    if (part) {
      __syncthreads();
      fft_forward<LOGN, fine<T, DIRECT>()>(col, here(tw), here(u), zx, xx);
#pragma unroll
      for (int k = 0; k < 16; ++k) xe[k] = cmul(xe[k], make_float2(xx[k].x, -xx[k].y));
      fft_inverse<LOGN, fine<T, DIRECT>()>(col, here(tw), here(u), xe, r8);
      put_part(r8, 0);
    } else {
      __syncthreads();
    }
    put_stage(std::integral_constant<int, 2>{});
    __syncthreads();
    {
      const float* st = (const float*)(stage + mycol * PST);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int m = point<LOGN>(u, k);
        z[k] = make_float2(st[2 * m + 1], st[2 * m + 2]);
      }
    }
    __syncthreads();
    fft_forward<LOGN, fine<T, DIRECT>()>(col, here(tw), here(u), z, xe);
    if (gx) conj_product16<LOGN>(sp + N, xe, w, true);
    if (part) {
#pragma unroll
      for (int k = 0; k < 16; ++k) xe[k] = cmul(xe[k], make_float2(xx[k].x, -xx[k].y));
      fft_inverse<LOGN, fine<T, DIRECT>()>(col, here(tw), here(u), xe, r8);
      put_part(r8, 1);
    }
  }
  if (gx) {
    if (ODD) __syncthreads();
    fft_inverse<LOGN, fine<T, DIRECT>()>(col, here(tw), here(u), w, r8);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; ++k) stage[mycol * PST + point<LOGN>(here(u), k)] = r8[k];
    __syncthreads();
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int q = here((int)threadIdx.x) + v * NT, m = q / VR, cp = (q % VR) * NE;
      float f[2][NE];
#pragma unroll
      for (int k = 0; k < NE; ++k) {
        const cpx s = stage[(cp + k) * PST + m];
        f[0][k] = s.x;
        f[1][k] = s.y;
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (2 * m + h < Tn) store_piece<T, NE>(gx + (row0 + 2 * m + h) * (size_t)d + c0 + cp, c0 + cp, d, vec, f[h]);
    }
  }
  if constexpr (!ODD) {
    if (part) {
      cpx xx[16];
      __syncthreads();
      fft_forward<LOGN, fine<T, DIRECT>()>(col, here(tw), here(u), zx, xx);
#pragma unroll
      for (int k = 0; k < 16; ++k) xe[k] = cmul(xe[k], make_float2(xx[k].x, -xx[k].y));
      fft_inverse<LOGN, fine<T, DIRECT>()>(col, here(tw), here(u), xe, r8);
      put_part(r8, 0);
    }
  }
}

// filter gradient (L, d): the rows' parts (B, rows, d) added in order; lags that have none are zero
template <typename T, bool ODD>
__global__ void __launch_bounds__(256) fft_corr_finish_kernel(const float* __restrict__ part, T* __restrict__ gf, int B, int lags, int L, int d) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)L * d) return;
  const int s = (int)(i / d), c = (int)(i - (size_t)s * d), rows = ODD ? lags : (lags + 1) / 2;
  float a = 0.f;
  if (s < lags && (ODD || !(s & 1)))
    for (int b = 0; b < B; ++b) a += part[((size_t)b * rows + (ODD ? s : s >> 1)) * d + c];
  DT<T>::st(gf + i, a);
}

int ilog2_exact(int n) {
  int l = 0;
  while ((1 << l) < n) ++l;
  return ((1 << l) == n) ? l : -1;
}

int fft_cols(int half_logn) { return half_logn >= 13 ? 1 : half_logn == 12 ? 2 : half_logn == 11 ? 4 : half_logn >= 9 ? 8 : half_logn >= 6 ? 16 : 32; }

}  // namespace

extern "C" int fstu_fft_length(int T_) {
  int n = 64;
  while (n < 2 * T_ && n < (1 << 14)) n <<= 1;
  return (n >= 2 * T_) ? n : 0;
}

// KERNEL: one of the launchers below, given LOGN of the half-length transform
#define FFT_GO(KERNEL, THREADS, SHM, GRID, NAME, ...)                                                  \
  do {                                                                                                 \
    static fstu_lds_limit most__;                                                                      \
    const int rc__ = fstu_need_lds(reinterpret_cast<const void*>(KERNEL), most__, SHM, NAME);          \
    if (rc__) return rc__;                                                                             \
    hipLaunchKernelGGL(KERNEL, GRID, dim3(THREADS), SHM, (hipStream_t)stream, __VA_ARGS__);            \
  } while (0)
#define FFT_TABLE(L, GRID, NAME, ...) FFT_GO((fft_twiddle_kernel<L>), 256, 0, GRID, NAME, __VA_ARGS__)
#define FFT_FILTER(L, GRID, NAME, ...) \
  FFT_GO((fft_filter_kernel<T, L>), fft_threads<L>(), (fft_lds_bytes<L, fft_threads<L>()>()), GRID, NAME, __VA_ARGS__)
#define FFT_PLAIN(L, GRID, NAME, ...) \
  FFT_GO((fft_conv_kernel<T, L>), fft_threads<L>(), (fft_lds_bytes<L, fft_threads<L>()>()), GRID, NAME, __VA_ARGS__)
#define FFT_ROWS(L, GRID, NAME, ...) \
  FFT_GO((fft_conv_rows_kernel<T, L>), fft_threads<L>(), (fft_lds_bytes<L, fft_threads<L>()>()), GRID, NAME, __VA_ARGS__)
#define FFT_CORR_SUM(L, GRID, NAME, ...) \
  FFT_GO((fft_corr_kernel<T, L, false>), fft_threads<L>(), (fft_lds_bytes<L, fft_threads<L>()>()), GRID, NAME, __VA_ARGS__)
#define FFT_CORR_ALL(L, GRID, NAME, ...) \
  FFT_GO((fft_corr_kernel<T, L, true>), fft_threads<L>(), (fft_lds_bytes<L, fft_threads<L>()>()), GRID, NAME, __VA_ARGS__)
#define FFT_SLAB(L, GRID, NAME, ...)                                                                                        \
  do {                                                                                                                      \
    constexpr int few__ = Half<L>::G > 64 ? Half<L>::G : 64;                                                                \
    if (narrow && mode == 0)                                                                                                \
      FFT_GO((fft_slab_kernel<T, L, few__, true>), few__, (fft_lds_bytes<L, few__>()), GRID, NAME, __VA_ARGS__);            \
    else if (narrow)                                                                                                        \
      FFT_GO((fft_slab_kernel<T, L, few__, false>), few__, (fft_lds_bytes<L, few__>()), GRID, NAME, __VA_ARGS__);           \
    else if (mode == 0)                                                                                                     \
      FFT_GO((fft_slab_kernel<T, L, 512, true>), 512, (fft_lds_bytes<L, 512>()), GRID, NAME, __VA_ARGS__);                  \
    else                                                                                                                    \
      FFT_GO((fft_slab_kernel<T, L, 512, false>), 512, (fft_lds_bytes<L, 512>()), GRID, NAME, __VA_ARGS__);                 \
  } while (0)

#define FFT_LAUNCH(LOGN, KERNEL, GRID, NAME, ...)             \
  do {                                                        \
    switch (LOGN) {                                           \
      case 5: KERNEL(5, GRID, NAME, __VA_ARGS__); break;      \
      case 6: KERNEL(6, GRID, NAME, __VA_ARGS__); break;      \
      case 7: KERNEL(7, GRID, NAME, __VA_ARGS__); break;      \
      case 8: KERNEL(8, GRID, NAME, __VA_ARGS__); break;      \
      case 9: KERNEL(9, GRID, NAME, __VA_ARGS__); break;      \
      case 10: KERNEL(10, GRID, NAME, __VA_ARGS__); break;    \
      case 11: KERNEL(11, GRID, NAME, __VA_ARGS__); break;    \
      case 12: KERNEL(12, GRID, NAME, __VA_ARGS__); break;    \
      default: KERNEL(13, GRID, NAME, __VA_ARGS__); break;    \
    }                                                         \
  } while (0)

extern "C" int fstu_fft_twiddles(float* tw, int n, void* stream) {
  FSTU_REQUIRE(tw, FSTU_ENULL, "fstu_fft_twiddles: null pointer");
  const int logn = ilog2_exact(n);
  FSTU_REQUIRE(logn >= 6 && logn <= 14, FSTU_ESHAPE, "fstu_fft_twiddles: n=%d is not a power of two in 64..16384", n);
  FSTU_REQUIRE(fstu_aligned(tw, 16), FSTU_EALIGN, "fstu_fft_twiddles: tw must be 16-byte aligned");
  FFT_LAUNCH(logn - 1, FFT_TABLE, dim3((n + 255) / 256), "fstu_fft_twiddles", (cpx*)tw);
  FSTU_CHECK_LAUNCH("fstu_fft_twiddles");
  return FSTU_OK;
}

extern "C" int fstu_stu_fft_filter(const void* filt, int64_t f_ls, int64_t f_cs, float* spec, const float* tw, int taps,
                                   int ncols, int n, int single_branch, int dtype, void* stream) {
  FSTU_REQUIRE(filt && spec && tw, FSTU_ENULL, "fstu_stu_fft_filter: null pointer");
  const int logn = ilog2_exact(n);
  FSTU_REQUIRE(logn >= 6 && logn <= 14, FSTU_ESHAPE, "fstu_stu_fft_filter: n=%d is not a power of two in 64..16384", n);
  FSTU_REQUIRE(taps >= 1 && 2 * taps <= n && ncols >= 1, FSTU_ESHAPE,
               "fstu_stu_fft_filter: taps=%d must satisfy 1 <= taps <= n/2=%d (ncols=%d)", taps, n / 2, ncols);
  FSTU_REQUIRE(fstu_aligned(spec, 16) && fstu_aligned(tw, 16), FSTU_EALIGN, "fstu_stu_fft_filter: spec and tw must be 16-byte aligned");
  (void)single_branch;      // both parts of the spectrum serve both forms of the convolution
  const int cols = fft_cols(logn - 1);
  dim3 grid((ncols + cols - 1) / cols);
  FSTU_DISPATCH_DTYPE(dtype, "fstu_stu_fft_filter",
                      FFT_LAUNCH(logn - 1, FFT_FILTER, grid, "fstu_stu_fft_filter", (const T*)filt, (size_t)f_ls,
                                 (size_t)f_cs, (cpx*)spec, (const cpx*)tw, taps, ncols));
  FSTU_CHECK_LAUNCH("fstu_stu_fft_filter");
  return FSTU_OK;
}

// Filters to a slice of a bank of time-major slabs, whose channels and rows alone make `waves` waves.  Below one round of the chip (1024
// SIMDs of four waves) a transform is bound by its own chain of exchanges: it takes 2.3 + 0.7 times the waves on its SIMD (in us: 1.8 at
// less than one, 2.8 at one, 5.2 at four, bf16), so slices that fill the SIMDs pay for their one forward transform beside the two inverse
// ones of each filter; a round and more gains nothing (4 x 2000 x 768 398 / 407 in one / two slices, 3 x 6000 x 768 1419 / 1452).  24
// filters, both branches, bf16, us with the whole bank to a workgroup / in slices: 1 x 64 x 256 68 / 7.8, 1 x 300 x 768 88 / 27, 4 x 250 x 1024
// 102 / 58, 1 x 1000 x 1024 138 / 67, 3 x 700 x 768 161 / 134, 1 x 4000 x 256 142 / 73, 2 x 2000 x 512 143 / 126, 1 x 8000 x 256 216 / 176.
static int bank_slice(int K, long long waves) {
  if (waves >= 4096) return K;
  int best = K;
  long long least = -1;
  for (int kper = (K + 65534) / 65535; kper <= K; ++kper) {
    const long long w = waves * ((K + kper - 1) / kper), rest = w % 4096;
    const long long cost = (2 * kper + 1) * (w / 4096 * 51 * 1024 + (rest ? 23 * 1024 + 7 * rest : 0));
    if (least < 0 || cost < least) { least = cost; best = kper; }
  }
  return best;
}

// Whether no byte between the first and the last one of y (strides b, t, k, c in elements) lies between those of x.  A bank whose slab is
// written over x takes no slices: a workgroup that has all filters of its channels reads them before it writes, another slice's may not
// have read them yet.
static bool bank_apart(const void* x, const int64_t (&xs)[3], const void* y, const int64_t (&ys)[4], int B, int T_, int K, int d, int esz) {
  if (!y) return true;
  const int64_t xn[3] = {B, T_, d}, yn[4] = {B, T_, K, d};
  int64_t x_lo = 0, x_hi = 1, y_lo = 0, y_hi = 1;
  for (int i = 0; i < 3; ++i) (xs[i] < 0 ? x_lo : x_hi) += (xn[i] - 1) * xs[i];
  for (int i = 0; i < 4; ++i) (ys[i] < 0 ? y_lo : y_hi) += (yn[i] - 1) * ys[i];
  const char *const xb = (const char*)x, *const yb = (const char*)y;
  return yb + y_hi * esz <= xb + x_lo * esz || xb + x_hi * esz <= yb + y_lo * esz;
}

static int conv_fft_launch(const char* name, const void* x, int64_t x_sb, int64_t x_st, int64_t x_sc, const float* spec,
                           void* y, void* y2, int64_t y_sb, int64_t y_st, int64_t y_sk, int64_t y_sc, const float* tw,
                           int B, int T_, int d, int K, int n, int mode, int dtype, void* stream) {
  const int logn = ilog2_exact(n);
  FSTU_REQUIRE(logn >= 6 && logn <= 14, FSTU_ESHAPE, "%s: n=%d is not a power of two in 64..16384", name, n);
  FSTU_REQUIRE(B >= 1 && B <= 65535 && T_ >= 1 && d >= 1 && K >= 1 && 2 * T_ <= n, FSTU_ESHAPE,
               "%s: bad shape B=%d T=%d d=%d K=%d n=%d (n >= 2T required)", name, B, T_, d, K, n);
  FSTU_REQUIRE(fstu_aligned(spec, 16) && fstu_aligned(tw, 16), FSTU_EALIGN, "%s: spec and tw must be 16-byte aligned", name);
  const int cols = fft_cols(logn - 1), esz = dtype == FSTU_BF16 ? 2 : 4, ch = 16 / esz, chw = cols > ch ? cols : ch;
  // Channel-contiguous operands whose rows split into whole 16-byte pieces per workgroup: the row-piece kernel.  The long
  // transforms take a workgroup's channels one after the other, so that few groups of them leave compute units idle, and the
  // one-column kernel, eight (fp32 four) times the workgroups but two bytes (four) of a line at a time, is the faster one.
  // us, one column / row pieces: 4096 positions, bf16, 128 groups 43 / 62, 256 75 / 67, 384 106 / 93, fp32 192 37 / 36, 384
  // 60 / 51; 2500 positions, bf16, 256 groups 62 / 64; 8192 positions, bf16, 96 groups 96 / 107, 128 112 / 108, 256 230 /
  // 138, fp32 64 groups 37 / 59, 192 91 / 67.
  const bool enough = logn < 13 || (long long)(d / chw) * B >= (logn == 13 ? 320 : 128);
  if (K == 1 && mode != 2 && enough && x_sc == 1 && y_sc == 1 && d % chw == 0 && x_st % ch == 0 && y_st % ch == 0 &&
      x_sb % ch == 0 && y_sb % ch == 0 && fstu_aligned(x, 16) && fstu_aligned(y, 16)) {
    const int gx = d / chw;
    dim3 grid(gx, B);
    const int remap = (gx % 8 == 0) ? 1 : 0;
    FSTU_DISPATCH_DTYPE(dtype, name,
                        FFT_LAUNCH(logn - 1, FFT_ROWS, grid, name, (const T*)x, (size_t)x_sb, (size_t)x_st,
                                   (const cpx*)spec, (T*)y, (size_t)y_sb, (size_t)y_st, (const cpx*)tw, T_, mode, remap));
    FSTU_CHECK_LAUNCH(name);
    return FSTU_OK;
  }
  const int64_t xs[3] = {x_sb, x_st, x_sc}, ys[4] = {y_sb, y_st, y_sk, y_sc};
  const bool apart = K > 1 && bank_apart(x, xs, y, ys, B, T_, K, d, esz) && bank_apart(x, xs, y2, ys, B, T_, K, d, esz);
  if (x_st == 1 && y_st == 1) {
    // as many columns per workgroup as fill 512 threads, or, where that leaves compute units idle, one wave (or column)
    const int g = n / 32, many = g >= 512 ? 1 : 512 / g, few = g >= 64 ? 1 : 64 / g;
    const bool narrow = (long long)((d + many - 1) / many) * B < 512;
    const int gx = narrow ? (d + few - 1) / few : (d + many - 1) / many;
    const int kper = apart ? bank_slice(K, (long long)gx * B * (narrow ? std::max(1, g / 64) : 8)) : K;
    dim3 grid(gx, B, (K + kper - 1) / kper);
    const int remap = (gx % 8 == 0) ? 1 : 0;
    FSTU_DISPATCH_DTYPE(dtype, name,
                        FFT_LAUNCH(logn - 1, FFT_SLAB, grid, name, (const T*)x, (size_t)x_sb, (size_t)x_sc, (const cpx*)spec, (T*)y,
                                   mode == 2 ? (T*)y2 : (T*)nullptr, (size_t)y_sb, (size_t)y_sk, (size_t)y_sc, (const cpx*)tw, T_,
                                   d, K, kper, remap));
    FSTU_CHECK_LAUNCH(name);
    return FSTU_OK;
  }
  // slices of the bank up to two workgroups per compute unit, where there is not one (fp32, 24 filters, both branches, us
  // one / two slices: 4 x 1000 x 768, 384 workgroups, 396 / 409, 1 x 4096 x 512, 256 workgroups, 413 / 529)
  const int gx = (d + cols - 1) / cols;
  const long long groups = (long long)gx * B;
  const int slices = groups >= 256 || !apart ? 1 : (int)(512 / groups), kper = slices >= K ? 1 : (K + slices - 1) / slices;
  dim3 grid(gx, B, (K + kper - 1) / kper);
  const int remap = (gx % 8 == 0) ? 1 : 0;
  FSTU_DISPATCH_DTYPE(dtype, name,
                      FFT_LAUNCH(logn - 1, FFT_PLAIN, grid, name, (const T*)x, (size_t)x_sb, (size_t)x_st,
                                 (size_t)x_sc, (const cpx*)spec, (T*)y, (T*)y2, (size_t)y_sb, (size_t)y_st, (size_t)y_sk,
                                 (size_t)y_sc, (const cpx*)tw, T_, d, K, kper, mode, remap));
  FSTU_CHECK_LAUNCH(name);
  return FSTU_OK;
}

extern "C" int fstu_stu_conv_fft(const void* xp, const float* spec, void* y, const float* tw, int B, int T_, int d, int n,
                                 int single_branch, int dtype, void* stream) {
  FSTU_REQUIRE(xp && spec && y && tw, FSTU_ENULL, "fstu_stu_conv_fft: null pointer");
  return conv_fft_launch("fstu_stu_conv_fft", xp, (int64_t)T_ * d, d, 1, spec, y, nullptr, (int64_t)T_ * d, d, 0, 1, tw, B,
                         T_, d, 1, n, single_branch ? 1 : 0, dtype, stream);
}

// The same convolution on strided operands: element (b, t, c) of x at x_strides[0]*b + x_strides[1]*t + x_strides[2]*c
// (elements), y likewise.  Time-major operands (a time stride of 1) make the loads and stores of the one-column
// kernel coalesce, which is what a few long sequences want (few channels x batch rows, transform length 8192 or more).
extern "C" int fstu_stu_conv_fft_strided(const void* xp, const int64_t* x_strides, const float* spec, void* y,
                                         const int64_t* y_strides, const float* tw, int B, int T_, int d, int n,
                                         int single_branch, int dtype, void* stream) {
  FSTU_REQUIRE(xp && x_strides && spec && y && y_strides && tw, FSTU_ENULL, "fstu_stu_conv_fft_strided: null pointer");
  return conv_fft_launch("fstu_stu_conv_fft_strided", xp, x_strides[0], x_strides[1], x_strides[2], spec, y, nullptr, y_strides[0],
                         y_strides[1], 0, y_strides[2], tw, B, T_, d, 1, n, single_branch ? 1 : 0, dtype, stream);
}

extern "C" int fstu_stu_conv_bank_fft(const void* x, const int64_t* x_strides, const float* spec, void* u_plus,
                                      void* u_minus, const int64_t* u_strides, const float* tw, int B, int T_, int d,
                                      int K, int n, int dtype, void* stream) {
  FSTU_REQUIRE(x && x_strides && spec && u_plus && u_strides && tw, FSTU_ENULL, "fstu_stu_conv_bank_fft: null pointer");
  FSTU_REQUIRE(K >= 2, FSTU_ESHAPE, "fstu_stu_conv_bank_fft: K=%d (a bank has at least two filters)", K);
  return conv_fft_launch("fstu_stu_conv_bank_fft", x, x_strides[0], x_strides[1], x_strides[2], spec, u_plus, u_minus,
                         u_strides[0], u_strides[1], u_strides[2], u_strides[3], tw, B, T_, d, K, n, u_minus ? 2 : 1,
                         dtype, stream);
}

// Gradients of the convolution above.  g1, g2 (B, T, d): the gradients of the plus and the minus branch, or with
// branches = 0 (sum) g1 alone for y = plus + minus, with branches = 1 g1 alone for the plus branch.  gx (B, T, d) and
// gf (L, d) may each be null; part: fp32 scratch of fstu_stu_conv_fft_grad_ws(...) elements, needed for gf.
extern "C" int64_t fstu_stu_conv_fft_grad_ws(int B, int T_, int d, int L, int branches) {
  const int64_t lags = L < T_ ? L : T_;
  return (int64_t)B * (branches == 0 ? (lags + 1) / 2 : lags) * d;
}
extern "C" int fstu_stu_conv_fft_grad(const void* g1, const void* g2, const void* x, const float* spec, void* gx, void* gf,
                                      float* part, const float* tw, int B, int T_, int d, int L, int n, int branches,
                                      int dtype, void* stream) {
  FSTU_REQUIRE(g1 && spec && tw && (gx || gf), FSTU_ENULL, "fstu_stu_conv_fft_grad: null pointer");
  FSTU_REQUIRE(!gf || (x && part), FSTU_ENULL, "fstu_stu_conv_fft_grad: gf needs x and part");
  FSTU_REQUIRE(branches >= 0 && branches <= 2 && (branches == 2) == (g2 != nullptr), FSTU_EARG,
               "fstu_stu_conv_fft_grad: branches=%d (0 sum, 1 plus, 2 both; g2 belongs to 2 alone)", branches);
  const int logn = ilog2_exact(n);
  FSTU_REQUIRE(logn >= 6 && logn <= 14, FSTU_ESHAPE, "fstu_stu_conv_fft_grad: n=%d is not a power of two in 64..16384", n);
  FSTU_REQUIRE(B >= 1 && B <= 65535 && T_ >= 1 && d >= 1 && L >= 1 && 2 * T_ <= n, FSTU_ESHAPE,
               "fstu_stu_conv_fft_grad: bad shape B=%d T=%d d=%d L=%d n=%d (n >= 2T required)", B, T_, d, L, n);
  FSTU_REQUIRE(fstu_aligned(spec, 16) && fstu_aligned(tw, 16), FSTU_EALIGN, "fstu_stu_conv_fft_grad: spec and tw must be 16-byte aligned");
  const int cols = fft_cols(logn - 1), esz = dtype == FSTU_BF16 ? 2 : 4, ch = 16 / esz, ne = cols < ch ? cols : ch;
  // rows of whole pieces: every piece of every tensor lies on its own size (the fp32 parts are pieces of ne * 4 bytes)
  const size_t al = (size_t)ne * esz;
  const int vec = d % ne == 0 && fstu_aligned(g1, al) && (!g2 || fstu_aligned(g2, al)) && (!x || fstu_aligned(x, al)) &&
                  (!gx || fstu_aligned(gx, al)) && (!gf || fstu_aligned(part, (size_t)ne * 4));
  const int gxb = (d + cols - 1) / cols, lags = L < T_ ? L : T_;
  dim3 grid(gxb, B);
  const int remap = (gxb % 8 == 0) ? 1 : 0;
  float* pt = gf ? part : nullptr;
  if (branches == 0) {
    FSTU_DISPATCH_DTYPE(dtype, "fstu_stu_conv_fft_grad",
                        FFT_LAUNCH(logn - 1, FFT_CORR_SUM, grid, "fstu_stu_conv_fft_grad", (const T*)g1, (const T*)nullptr, (const T*)x,
                                   (const cpx*)spec, (T*)gx, pt, (const cpx*)tw, T_, d, lags, vec, remap));
  } else {
    FSTU_DISPATCH_DTYPE(dtype, "fstu_stu_conv_fft_grad",
                        FFT_LAUNCH(logn - 1, FFT_CORR_ALL, grid, "fstu_stu_conv_fft_grad", (const T*)g1, (const T*)g2, (const T*)x,
                                   (const cpx*)spec, (T*)gx, pt, (const cpx*)tw, T_, d, lags, vec, remap));
  }
  FSTU_CHECK_LAUNCH("fstu_stu_conv_fft_grad");
  if (!gf) return FSTU_OK;
  const dim3 fg((unsigned)(((size_t)L * d + 255) / 256));
  FSTU_DISPATCH_DTYPE(dtype, "fstu_stu_conv_fft_grad", if (branches == 0) {
    hipLaunchKernelGGL((fft_corr_finish_kernel<T, false>), fg, dim3(256), 0, (hipStream_t)stream, part, (T*)gf, B, lags, L, d);
  } else {
    hipLaunchKernelGGL((fft_corr_finish_kernel<T, true>), fg, dim3(256), 0, (hipStream_t)stream, part, (T*)gf, B, lags, L, d);
  });
  FSTU_CHECK_LAUNCH("fstu_stu_conv_fft_grad");
  return FSTU_OK;
}
