// Prefill GEMMs on the matrix cores (bf16, fp32 accumulation):  C[m, n] = sum_k A[m, k] W[n, k]
// for activations A (M rows, K contiguous) and nn.Linear weights W (N, K) — the dense contractions of the prompt pass
// (c_attn / c_proj flash_stu/modules/attention.py:74,101; gate / up / down flash_stu/modules/swiglu.py:22-29;
// x @ M_inputs flash_stu/modules/stu.py:87), with the element-wise work that follows them as epilogues:
//   mode 0  C = T(acc), any feature count and row stride: the tied head's 50257 features go through here too (on the
//           general kernel of fstu_gemm_any.hip they took longer than all layers: logits of 4 x 4096 positions at 2048-d,
//           8 layers 103.7 -> 42.9 ms, of 3 x 777 positions at 768-d, 12 layers 6.06 -> 2.97 ms for the whole pass)
//   mode 1  GLU: C[m, i] = T( T(gelu_tanh(T(acc_gate))) * T(acc_up) ) from two weight matrices (swiglu.py:23-26),
//           so the gate and up activations never travel through HBM
//   mode 2  C = T( R + T(acc) ): the residual add behind c_proj / down_proj (attention_layer.py:57,62, stu_layer.py:96)
//   split-K C = fp32 partial sums per K slice (fstu_add_rmsnorm adds the slices): the down projection of a decode
//           step over 17..32 rows, whose 16 output tiles would leave most of the chip without weights to stream
//
// A workgroup is WFN x WTN waves; a wave owns FI x TJ MFMA tiles of 32 features x 32 rows
// (v_mfma_f32_32x32x16_bf16), the workgroup 32*FI*WFN features x 32*TJ*WTN rows.  K runs in tiles of BK through NS
// LDS stages that are filled straight from global memory (buffer_load_dwordx4 ... lds, no stop in registers) one or more
// tiles ahead of the multiplication.  LDS rows are BK*2 bytes with the 16-byte chunk index XOR-ed with bits of the
// row, so neither the fills nor the fragment reads meet bank conflicts.  The weights are the MFMA A operand and the
// activations the B operand, so a lane ends up with 4 consecutive features of one row: 8-byte stores.  In mode 1 a
// wave's feature tiles are half gate, half up rows of the same features.  Workgroup ids are dealt round-robin to the
// 8 XCDs; each XCD works through its own contiguous share of the tiles in panels of 8 feature tiles, so the workgroups
// resident on an XCD share a few weight and activation tiles in its L2.
#include <algorithm>
#include <type_traits>
#include "fstu_common.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16_t __attribute__((ext_vector_type(16)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

#define GM_PANEL 8     // feature tiles per panel of the tile order
// A workgroup addresses its tile through a buffer descriptor whose base is the tile's first row (64-bit arithmetic) and a
// 32-bit byte offset per lane of at most 256 rows * row stride * 2 bytes: row strides (lda, and K for the weights) stay
// below 2^22 elements so that this offset cannot wrap; what lies beyond a tile's rows is cut off by the descriptor's range
#define GM_MAX_LD (1 << 22)

__device__ __forceinline__ float rnd_bf16(float v) { return bf16_to_f32(f32_to_bf16(v)); }
// The tanh-approximated GELU on the hardware exp and reciprocal, x (1 + tanh t) / 2 = x / (1 + exp(-2 t)): five full-rate and two
// quarter-rate instructions (eleven and two as 1 - 2 / (exp(2 t) + 1), which also cancelled for negative x: off by 1.5e-3 of the
// value at x = -4, 4e-6 so).  Of the 26820 bf16 inputs between 1e-30 and 40 in size 72 leave it not correctly rounded, 106 the longer form, which
// the packed decode launches keep.
__device__ __forceinline__ float gelu_tanh_short(float x) {
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * fmaf(x * x, -0.10294324f, -2.3022082f)));
}

// 16 bytes per lane from global memory into LDS without a stop in registers: the 64 lanes fill 64 consecutive 16-byte
// slots from `l` (wave-uniform) on.  The source is a buffer descriptor (base and range in SGPRs), a 32-bit byte offset
// per lane and a scalar offset for the k tile: rows beyond the range read zeros, so ragged tiles need no clamping
// (measured 2-13 % faster than the same fills through 64-bit per-lane addresses).
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t make_rsrc(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (unsigned)bytes, 0x00020000);
}
__device__ __forceinline__ void buf_load16_to_lds(rsrc_t rs, unsigned voff, unsigned soff, void* l) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)l, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ unsigned lds_addr(const void* p) {
  return (unsigned)(size_t)(const __attribute__((address_space(3))) void*)p;
}

// Fragment reads are written as asm: the compiler orders every LDS read it knows of behind all outstanding
// global->LDS loads (s_waitcnt vmcnt(0)), which would serialise the next tile's fetch with this tile's reads.
template <int OFF>
__device__ __forceinline__ u32x4_t lds_read16(unsigned addr) {
  u32x4_t v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  return v;
}
template <int N, int STEP, int I = 0>
__device__ __forceinline__ void lds_read_rows(u32x4_t* f, unsigned addr) {   // N reads, 32 rows (STEP bytes) apart
  if constexpr (I < N) {
    f[I] = lds_read16<I * STEP>(addr);
    lds_read_rows<N, STEP, I + 1>(f, addr);
  }
}
// Waits until at most LEFT of the reads issued so far are outstanding; the fragments pass through the statement so
// that nothing that uses them is placed ahead of the wait.
template <int LEFT, int N>
__device__ __forceinline__ void lds_wait(u32x4_t (&f)[N]) {
  static_assert(N == 2 || N == 3 || N == 4 || N == 6 || N == 8, "fragment group");
  if constexpr (N == 2)
    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(f[0]), "+v"(f[1]) : "n"(LEFT));
  else if constexpr (N == 3)
    asm volatile("s_waitcnt lgkmcnt(%3)" : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]) : "n"(LEFT));
  else if constexpr (N == 4)
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]) : "n"(LEFT));
  else if constexpr (N == 6)
    asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]) : "n"(LEFT));
  else
    asm volatile("s_waitcnt lgkmcnt(%8)"
                 : "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7])
                 : "n"(LEFT));
}

// 4 consecutive features of one row.  RAGGED: any row stride and feature count, so the address may be only 2-byte aligned
// (a global store takes any alignment) and the last group of a row may hold fewer than 4 features.
typedef unsigned u32x2_any_t __attribute__((ext_vector_type(2), aligned(2)));
template <bool RAGGED>
__device__ __forceinline__ void store_feat4(bf16_t* p, int left, unsigned lo, unsigned hi) {
  if constexpr (!RAGGED) {
    *(uint2*)p = make_uint2(lo, hi);
  } else if (left >= 4) {
    u32x2_any_t v = {lo, hi};
    *(u32x2_any_t*)p = v;
  } else {
    p[0] = (bf16_t)lo;
    if (left > 1) p[1] = (bf16_t)(lo >> 16);
    if (left > 2) p[2] = (bf16_t)hi;
  }
}

int gemm_cus() { return fstu_cus(); }

template <int WFN_, int WTN_, int FI_, int TJ_, int BK_, int NS_>
struct GemmTile {
  static constexpr int WFN = WFN_, WTN = WTN_, FI = FI_, TJ = TJ_, BK = BK_, NS = NS_;
  static constexpr int NW = WFN * WTN, THREADS = 64 * NW;
  static constexpr int BF = 32 * FI * WFN, BT = 32 * TJ * WTN;   // LDS rows of the weight / activation tile
  static constexpr int RB = BK * 2, CPR = RB / 16;               // bytes and 16-byte chunks per LDS row
  static constexpr int KK = BK / 16;                             // MFMA k steps per tile
  static constexpr int WL = BF * CPR / (64 * NW), AL = BT * CPR / (64 * NW);   // fill instructions per wave and tile
  static constexpr unsigned STAGE = (unsigned)(BF + BT) * RB;
  static constexpr unsigned LDS = STAGE * NS;
  static constexpr int NFR = FI + TJ;                            // fragments per k step
  static_assert(BK == 32 || BK == 64, "k tile");
  static_assert((BF * CPR) % (64 * NW) == 0 && (BT * CPR) % (64 * NW) == 0, "fill split");
  // Byte offset of 16-byte chunk c of a row inside a tile.  A 16-byte fragment read is served 16 lanes (16 consecutive
  // rows, one chunk each) at a time and is free of bank conflicts when those 16 pieces fall into 16 different 16-byte
  // slots of a 256-byte window: the row's position inside the window supplies 1 (128-byte rows) or 2 (64-byte rows) of
  // the 4 slot bits, the XOR with the next higher row bits the other 3 or 2.
  __device__ static __forceinline__ unsigned swz(int row, int c) {
    return (unsigned)row * RB + (unsigned)((c ^ (BK == 64 ? ((row >> 1) & 7) : ((row >> 2) & 3))) << 4);
  }
};

template <class G, int MODE>
__global__ void __launch_bounds__(G::THREADS)
gemm_bf16_kernel(const bf16_t* __restrict__ A, long long lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2,
                 const bf16_t* __restrict__ R, long long ldr, bf16_t* __restrict__ C, long long ldc, int M, int N, int K,
                 int mt, int nt, int share, int ksplit) {
  constexpr int FI = G::FI, TJ = G::TJ, BF = G::BF, BT = G::BT, WL = G::WL, AL = G::AL, NS = G::NS, KK = G::KK, NFR = G::NFR;
  constexpr int NF = MODE == 1 ? BF / 2 : BF;         // output features per workgroup
  constexpr unsigned STAGE = G::STAGE;
  extern __shared__ __align__(16) unsigned char gm_smem[];   // NS stages of (weights BF rows, activations BT rows)
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wf = w % G::WFN, wt = w / G::WFN;
  // ---- tile of this workgroup
  int o = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= share || o >= mt * nt * ksplit) return;
  const int slice = o / (mt * nt);                    // MODE 3: K slice of this workgroup (slices outermost)
  o -= slice * (mt * nt);
  const int kbeg = slice * (K / ksplit);
  const int per_panel = mt * GM_PANEL;
  const int panel = o / per_panel, in_panel = o - panel * per_panel;
  const int pw = min(GM_PANEL, nt - panel * GM_PANEL);        // the last panel may be narrower
  const int bt = in_panel / pw, bf = panel * GM_PANEL + in_panel % pw;
  const int m0 = bt * BT, n0 = bf * NF;
  // ---- fills: the XOR of the layout is applied on the global side: the lane that owns slot s (row s / CPR, physical
  // chunk s % CPR) fetches the logical chunk that belongs there.  Addresses are a per-workgroup buffer descriptor (the
  // tile's first row, its valid rows as the range), a per-lane byte offset and the k tile as the scalar offset.
  const int wv = __builtin_amdgcn_readfirstlane(w);   // wave-uniform by construction; keeps descriptors and LDS bases scalar
  const int rows_w = min(NF, N - n0), rows_a = min(BT, M - m0);
  const rsrc_t rs_w = make_rsrc(W + (size_t)n0 * K, (size_t)rows_w * K * 2);
  const rsrc_t rs_w2 = make_rsrc(MODE == 1 ? W2 + (size_t)n0 * K : W, MODE == 1 ? (size_t)rows_w * K * 2 : 0);
  const rsrc_t rs_a = make_rsrc(A + (size_t)m0 * lda, ((size_t)(rows_a - 1) * lda + K) * 2);
  unsigned wvoff[WL], avoff[AL];
#pragma unroll
  for (int j = 0; j < WL; ++j) {
    const int slot = (wv * WL + j) * 64 + lane, row = slot / G::CPR;
    const int ch = (int)((G::swz(row, slot % G::CPR) - (unsigned)row * G::RB) >> 4);   // XOR is its own inverse
    int n = row;
    if (MODE == 1) {
      // LDS rows of wave column wf': gate rows first, then the up rows of the same features (a fill instruction
      // covers 64 / CPR whole rows, all of them gate or all of them up)
      constexpr int HALF = 16 * FI;
      n = (row / (2 * HALF)) * HALF + (row % HALF);
    }
    wvoff[j] = (unsigned)n * (unsigned)K * 2u + (unsigned)ch * 16u;
  }
#pragma unroll
  for (int j = 0; j < AL; ++j) {
    const int slot = (wv * AL + j) * 64 + lane, row = slot / G::CPR;
    const int ch = (int)((G::swz(row, slot % G::CPR) - (unsigned)row * G::RB) >> 4);
    avoff[j] = (unsigned)row * (unsigned)lda * 2u + (unsigned)ch * 16u;
  }
  const unsigned wslot = (unsigned)(wv * WL) * 1024u, aslot = (unsigned)BF * G::RB + (unsigned)(wv * AL) * 1024u;
#define GM_FETCH(stage_, k0)                                                                                 \
  {                                                                                                          \
    unsigned char* st_ = gm_smem + (unsigned)(stage_) * STAGE;                                               \
    const unsigned so_ = (unsigned)(kbeg + (k0)) * 2u;                                                       \
    _Pragma("unroll") for (int j = 0; j < WL; ++j) {                                                         \
      const bool up_ = MODE == 1 && (((wv * WL + j) * (64 / G::CPR)) % (32 * FI)) >= 16 * FI;                \
      buf_load16_to_lds(up_ ? rs_w2 : rs_w, wvoff[j], so_, st_ + wslot + j * 1024);                          \
    }                                                                                                        \
    _Pragma("unroll") for (int j = 0; j < AL; ++j) buf_load16_to_lds(rs_a, avoff[j], so_, st_ + aslot + j * 1024); \
  }
#define GM_MFMAS(f_)                                                                                         \
  _Pragma("unroll") for (int i = 0; i < FI; ++i)                                                             \
    _Pragma("unroll") for (int j = 0; j < TJ; ++j)                                                           \
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, f_[i]),               \
                                                          __builtin_bit_cast(bf16x8_t, f_[FI + j]), acc[i][j], 0, 0, 0);
  const int l32 = lane & 31, lh = lane >> 5;
  // fragment addresses inside a stage for the k steps of a tile (rows 32 apart share the XOR term)
  unsigned fw_off[KK], fa_off[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) {
    fw_off[kk] = G::swz(wf * (32 * FI) + l32, kk * 2 + lh);
    fa_off[kk] = (unsigned)BF * G::RB + G::swz(wt * (32 * TJ) + l32, kk * 2 + lh);
  }
  floatx16_t acc[FI][TJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  const int nkt = K / ksplit / G::BK;
  // Software pipeline over the k tiles.  NS-1 tiles are in flight ahead of the one being multiplied.  Within a tile the
  // fragments of k step kk+1 are read while step kk is multiplied; before the last step of tile kt the wave makes sure
  // its reads of the tile are complete, waits for its share of tile kt+1, meets the barrier (every wave's share has
  // landed, every wave has left the stage of tile kt), refills that stage with tile kt+NS and reads the first
  // fragments of tile kt+1 — so the MFMAs of the last step cover the barrier and those reads.  The compiler's own
  // schedule would wait for each fragment read in turn; the fences keep the order written here.
  constexpr int LPT = WL + AL;                        // fills per wave and tile
#pragma unroll
  for (int t = 0; t < NS - 1; ++t)
    if (t < nkt) GM_FETCH(t, t * G::BK)
  const unsigned smem0 = lds_addr(gm_smem);
  if (NS - 2 < nkt) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * LPT) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();   // bare: the fence of __syncthreads would wait for the tiles still in flight
  if (NS - 1 < nkt) GM_FETCH(NS - 1, (NS - 1) * G::BK)
  u32x4_t fa_[NFR], fb_[NFR];                         // the two fragment sets, used by alternate k steps
  lds_read_rows<FI, 32 * G::RB>(fa_, smem0 + fw_off[0]);
  lds_read_rows<TJ, 32 * G::RB>(fa_ + FI, smem0 + fa_off[0]);
  int cur = 0;                                        // stage of tile kt
  for (int kt = 0; kt < nkt; ++kt) {
    const unsigned cb = smem0 + (unsigned)cur * STAGE;
    const int nxt = cur + 1 == NS ? 0 : cur + 1;
    __builtin_amdgcn_sched_barrier(0);
    lds_read_rows<FI, 32 * G::RB>(fb_, cb + fw_off[1]);
    lds_read_rows<TJ, 32 * G::RB>(fb_ + FI, cb + fa_off[1]);
    lds_wait<NFR>(fa_);
    GM_MFMAS(fa_)
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (KK == 4) {
      lds_read_rows<FI, 32 * G::RB>(fa_, cb + fw_off[2]);
      lds_read_rows<TJ, 32 * G::RB>(fa_ + FI, cb + fa_off[2]);
      lds_wait<NFR>(fb_);
      GM_MFMAS(fb_)
      __builtin_amdgcn_sched_barrier(0);
      lds_read_rows<FI, 32 * G::RB>(fb_, cb + fw_off[3]);
      lds_read_rows<TJ, 32 * G::RB>(fb_ + FI, cb + fa_off[3]);
      lds_wait<NFR>(fa_);
      GM_MFMAS(fa_)
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_wait<0>(fb_);                                 // this wave has left the stage of tile kt
    if (kt + 1 < nkt) {
      if (kt + NS - 1 < nkt) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * LPT) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      if (kt + NS < nkt) GM_FETCH(cur, (kt + NS) * G::BK)
      const unsigned nb = smem0 + (unsigned)nxt * STAGE;
      lds_read_rows<FI, 32 * G::RB>(fa_, nb + fw_off[0]);
      lds_read_rows<TJ, 32 * G::RB>(fa_ + FI, nb + fa_off[0]);
    }
    __builtin_amdgcn_sched_barrier(0);
    GM_MFMAS(fb_)
    cur = nxt;
  }
#undef GM_FETCH
#undef GM_MFMAS
  // ---- epilogue.  D of a 32x32 tile: lane l holds row (token) l % 32 and features 8*(e/4) + 4*(l/32) + e%4
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const int m = m0 + wt * (32 * TJ) + j * 32 + l32;
    if (m >= M) continue;
    if (MODE == 1) {
#pragma unroll
      for (int i = 0; i < FI / 2; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int f = n0 + wf * (16 * FI) + i * 32 + q * 8 + lh * 4;
          if (f >= N) continue;
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[e] = rnd_bf16(gelu_tanh_short(rnd_bf16(acc[i][j][q * 4 + e]))) * rnd_bf16(acc[i + FI / 2][j][q * 4 + e]);
          *(uint2*)(C + (size_t)m * ldc + f) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
        }
    } else {
#pragma unroll
      for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int f = n0 + wf * (32 * FI) + i * 32 + q * 8 + lh * 4;
          if (f >= N) continue;
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = acc[i][j][q * 4 + e];
          if (MODE == 3) {
            *(float4*)((float*)C + ((size_t)slice * M + m) * ldc + f) = make_float4(v[0], v[1], v[2], v[3]);
            continue;
          }
          if (MODE == 2) {
            const uint2 rv = *(const uint2*)(R + (size_t)m * ldr + f);
            v[0] = __uint_as_float(rv.x << 16) + rnd_bf16(v[0]);
            v[1] = __uint_as_float(rv.x & 0xffff0000u) + rnd_bf16(v[1]);
            v[2] = __uint_as_float(rv.y << 16) + rnd_bf16(v[2]);
            v[3] = __uint_as_float(rv.y & 0xffff0000u) + rnd_bf16(v[3]);
          }
          store_feat4<MODE == 0>(C + (size_t)m * ldc + f, N - f, pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
        }
    }
  }
}

template <class G, int MODE>
int gemm_launch_tile(const void* A, long long lda, const void* W, const void* W2, const void* R, long long ldr, void* C,
                     long long ldc, int M, int N, int K, hipStream_t s, int ksplit = 1) {
  constexpr int NF = MODE == 1 ? G::BF / 2 : G::BF;
  static fstu_lds_limit most;
  if (const int rc = fstu_need_lds((const void*)gemm_bf16_kernel<G, MODE>, most, G::LDS, "fstu_gemm_bf16")) return rc;
  const int mt = (M + G::BT - 1) / G::BT, nt = (N + NF - 1) / NF;
  const long long tiles = (long long)mt * nt * ksplit;
  const int share = (int)((tiles + 7) / 8);
  hipLaunchKernelGGL((gemm_bf16_kernel<G, MODE>), dim3((unsigned)share * 8u), dim3(G::THREADS), G::LDS, s, (const bf16_t*)A, lda,
                     (const bf16_t*)W, (const bf16_t*)W2, (const bf16_t*)R, ldr, (bf16_t*)C, ldc, M, N, K, mt, nt, share, ksplit);
  return 0;
}

// ---------------------------------------------------------------- 256 x 256 tiles in two alternating wave groups
// Large contractions.  A workgroup of 8 waves owns 256 features x 256 rows (mode 1: 128 features, gate and up), K in tiles
// of 64 through two LDS stages.  Waves 0-3 and 4-7 (one of each on every SIMD) run the same program half a phase apart:
// while one group multiplies, the other reads its next fragments and requests the tiles to come, so a SIMD's matrix core
// always has one of its two waves to work for, and neither barriers nor LDS reads show.
// The halves of the weight tile (W0, W1: 128 features) and of the activation tile (X0, X1: 128 rows) are parts of 16 KB;
// a wave owns 32 features of each W half and 64 rows of each X half, and a k tile is two phases of 32
// v_mfma_f32_16x16x32_bf16 (512 cycles) each:
//   phase  fragments read      multiplied      parts requested
//   0      W0, W1, X0 of kt    (W0, W1) X0     X1 of kt + 1
//   1      X1 of kt            (W0, W1) X1     W0, W1, X0 of kt + 2
// A part is requested in the first phase after its last readers have left it (their reads are complete before the barrier
// that ends a memory phase) and waited for three phases later: vmcnt(8) at the end of a memory phase leaves the two
// youngest requests in flight, at 512 cycles a phase and group that is longer than a trip to the memory-side cache.
// The grid is one workgroup per compute unit, each walks its share of the tiles: the first k tiles of the next output tile
// are requested before this one is stored.  The W rows are dealt so that a lane ends up with 8 consecutive features of a row,
// 16 bytes: the gated pair (the four lanes of a row hold 64 bytes) and the fp32 sums (128) leave straight from the accumulators
// without a barrier, us, through LDS / so: 16384 x 2 x 24576 x 2048 2324 / 2268, 2331 x 2 x 9216 x 768 69.3 / 64.7, 4096 x 2 x 9216 x
// 768 113 / 107, 2500 x 2048 x 24576 in three slices 203 / 196.  Plain and residual rows pass 32 at a time through LDS beside the
// stages and leave 512 bytes in a row: straight from the accumulators 2331 x 50257 x 768, whose rows begin anywhere, takes 213 us,
// 167 so.  The stores of a whole tile are not waited for before the next tile's first products (16384 x 2048 x 2048 with the
// residual 112 / 104, 16384 x 768 x 768 21.7 / 20.8).
// What bounds it: the power the matrix cores draw.  A loop of nothing but v_mfma on random bf16 operands runs at 1.77
// PFLOP/s in the 32x32x16 form and 2.03 in the 16x16x32 form on this card (2.42 on zeros): hence the smaller instruction,
// although it reads the same operands twice as often (1.30 -> 1.33-1.42 PFLOP/s).  Measured against the kernel above
// (256 x 256 tile) and hipBLASLt, us: 16384 x 2048 x 24576 with the residual 1099 / 1395 / 1190 (1.50 PFLOP/s; on zeros 888), 16384 x
// 6144 x 2048 288 / 384 / 292, 16384 x 50257 x 2048 2570 / 3339 / 2510; gate+up 16384 x 2 x 24576 x 2048 2268 / 3148, 4096 x
// 2 x 9216 x 768 107 / 133 (84 on zeros).  What keeps K = 2048 below K = 24576: the epilogue (in mode 1 the GELU's 70 cycles per element).
#define PP_STAGE 65536u
#define PP_PART 16384u
#define PP_LDS(MODE) (2 * PP_STAGE + ((MODE) == 1 || (MODE) == 3 ? 0u : 32768u))   // + what the epilogue passes the rows through
typedef unsigned u32x4_any_t __attribute__((ext_vector_type(4), aligned(2)));
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));

// 8 consecutive features of one row (the last group of a row may hold fewer), any 2-byte alignment; MODE 2: the residual
// row's 8 features are added first
template <int MODE>
__device__ __forceinline__ void store_feat8(u32x4_t v, const bf16_t* rp, bf16_t* cp, int left) {
  if (left >= 8) {
    if (MODE == 2) {
      const u32x4_any_t rv = *(const u32x4_any_t*)rp;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = pack2_bf16(__uint_as_float(rv[e] << 16) + __uint_as_float(v[e] << 16),
                          __uint_as_float(rv[e] & 0xffff0000u) + __uint_as_float(v[e] & 0xffff0000u));
    }
    *(u32x4_any_t*)cp = v;
    return;
  }
  for (int e = 0; e < left; ++e) {
    bf16_t h = (bf16_t)(v[e >> 1] >> (16 * (e & 1)));
    if (MODE == 2) h = f32_to_bf16(bf16_to_f32(rp[e]) + bf16_to_f32(h));
    cp[e] = h;
  }
}

// (transposing read: in a block of 16 lanes, lane i supplies the address of 4 consecutive columns of row i/4 starting at column
// 4*(i%4), and receives column i of the 4 rows)
template <int OFF>
__device__ __forceinline__ u32x2_t lds_read_tr8(unsigned addr) {
  u32x2_t v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  return v;
}
struct Frag8 { u32x2_t lo, hi; };

// TA: the activations are slabs with the reduction index slowest (see gemm_ta_bf16_kernel), M a multiple of 256.  Rows of an
// X part are then 64 k of 128 columns, filled 16 bytes = 8 columns per lane and read with transposing reads, k and k + 4 of a
// fragment's half; the 32-byte pieces of a row are XOR-ed with bits 0, 1 and 3 of k so that the eight rows that two blocks of
// lanes read together lie in different banks.  `mts` row tiles per slab, slabs sa / sc / sr elements apart.
// MODE 3: slices of K, outermost, each into fp32 sums of its own (C: slices x nb slabs x M x N floats), straight from the
// accumulators.
template <int MODE, bool TA = false>
__global__ void __launch_bounds__(512)
gemm_pp_bf16_kernel(const bf16_t* __restrict__ A, long long lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ W2,
                    const bf16_t* __restrict__ R, long long ldr, bf16_t* __restrict__ C, long long ldc, int M, int N, int K,
                    int mt, int nt, int share, int mts, long long sa, long long sc, long long sr, int nb) {
  constexpr int NF = MODE == 1 ? 128 : 256;
  extern __shared__ __align__(16) unsigned char gm_smem[];   // stage: W0 | W1 | X0 | X1
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int per_panel = mt * GM_PANEL, xcd = (int)(blockIdx.x & 7) * share, tiles = mt * nt;
  int idx = (int)(blockIdx.x >> 3);                    // this workgroup's next tile in its XCD's share
  if (idx >= share || xcd + idx >= tiles) return;
  int m0, n0;
  size_t wbytes, abytes;
  const bf16_t *wb, *wb2, *ab, *rb = R;
  bf16_t* cb = C;
  float* part = nullptr;
  const int KS = MODE == 3 ? K / (mt / mts / nb) : K;       // MODE 3: this workgroup's share of K
#define PP_OPEN_TILE                                                                     \
  {                                                                                      \
    const int o_ = xcd + idx;                                                            \
    const int panel_ = o_ / per_panel, in_panel_ = o_ - panel_ * per_panel;              \
    const int pw_ = min(GM_PANEL, nt - panel_ * GM_PANEL);                               \
    int bm_ = in_panel_ / pw_;                                                           \
    ab = A;                                                                              \
    wb = W;                                                                              \
    if constexpr (MODE == 3) {                                                           \
      const int part_ = bm_ / mts, slice_ = part_ / nb;                                  \
      bm_ -= part_ * mts;                                                                \
      ab += TA ? (size_t)(part_ - slice_ * nb) * sa + (size_t)slice_ * KS * lda : (size_t)slice_ * KS; \
      wb += (size_t)slice_ * KS;                                                         \
      part = (float*)C + (size_t)part_ * M * N;                                          \
    } else if constexpr (TA) {                                                           \
      const int slab_ = bm_ / mts;                                                       \
      bm_ -= slab_ * mts;                                                                \
      ab += (size_t)slab_ * sa;                                                          \
      cb = C + (size_t)slab_ * sc;                                                       \
      if (MODE == 2) rb = R + (size_t)slab_ * sr;                                        \
    }                                                                                    \
    m0 = bm_ * 256;                                                                      \
    n0 = (panel_ * GM_PANEL + in_panel_ % pw_) * NF;                                     \
    wbytes = ((size_t)(min(NF, N - n0) - 1) * K + KS) * 2;                               \
    abytes = TA ? ((size_t)(KS - 1) * lda + 256) * 2 : ((size_t)(min(256, M - m0) - 1) * lda + KS) * 2; \
    wb += (size_t)n0 * K;                                                                \
    wb2 = MODE == 1 ? W2 + (size_t)n0 * K : wb;                                          \
    ab += TA ? (size_t)m0 : (size_t)m0 * lda;                                            \
  }
  const int wn = wv & 3, wm = wv >> 2;                 // 32-feature slice and 64-row slice of every half
  // ---- fills: part = 128 rows x 128 bytes; a wave fills rows 16 wv .. 16 wv + 15 of it with two instructions
  unsigned wvoff[2], avoff[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = wv * 16 + j * 8 + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7);
    const int feat = MODE == 1 ? row : (row & 31) + 2 * (row & 96);
    wvoff[j] = (unsigned)feat * (unsigned)K * 2u + (unsigned)((lane & 7) ^ (((row >> 1) & 1) | ((row >> 2) & 6))) * 16u;
    if constexpr (TA) {
      const int kr = wv * 8 + j * 4 + (lane >> 4);
      avoff[j] = (unsigned)kr * (unsigned)lda * 2u + (unsigned)((lane & 15) ^ (4 * (kr & 3)) ^ (2 * ((kr >> 3) & 1))) * 16u;
    } else {
      avoff[j] = (unsigned)row * (unsigned)lda * 2u + (unsigned)ch * 16u;
    }
  }
  const unsigned w1off = MODE == 1 ? 0u : 32u * (unsigned)K * 2u, x1off = TA ? 256u : 128u * (unsigned)lda * 2u;
  const int nkt = KS >> 6;
  unsigned char* fill0 = gm_smem + (unsigned)wv * 2048u;
  // requests part P (0 W0, 1 X0, 2 W1, 3 X1) of k tile kt_; beyond the last tile the descriptor is empty: nothing is fetched
#define PP_FETCH(P, kt_, stage_)                                                                                           \
  {                                                                                                                        \
    const bool in_ = (kt_) < nkt;                                                                                          \
    const unsigned so_ = (unsigned)(kt_) * (TA && ((P) & 1) ? 128u * (unsigned)lda : 128u);                                 \
    unsigned char* l_ = fill0 + (stage_) * PP_STAGE + ((P) == 0 ? 0u : (P) == 2 ? PP_PART : (P) == 1 ? 2 * PP_PART : 3 * PP_PART); \
    const rsrc_t rs_ = ((P) & 1) ? make_rsrc(ab, in_ ? abytes : 0) : make_rsrc((P) == 2 ? wb2 : wb, in_ ? wbytes : 0);     \
    _Pragma("unroll") for (int j = 0; j < 2; ++j)                                                                          \
      buf_load16_to_lds(rs_, (((P) & 1) ? avoff[j] : wvoff[j]) + ((P) == 2 ? w1off : (P) == 3 ? x1off : 0u), so_, l_ + j * 1024); \
  }
  const int l16 = lane & 15, lq = lane >> 4;
  unsigned fw_off[2], fx_off[2];                       // fragment addresses of the two k steps inside a part
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int rw = wn * 32 + 8 * (l16 >> 2) + (l16 & 3), rx = wm * 64 + l16, c = kk * 4 + lq;
    fw_off[kk] = (unsigned)rw * 128u + (unsigned)((c ^ (((rw >> 1) & 1) | ((rw >> 2) & 6))) << 4);
    fx_off[kk] = 2 * PP_PART + (unsigned)rx * 128u + (unsigned)((c ^ ((rx >> 1) & 7)) << 4);
  }
  const unsigned smem0 = lds_addr(gm_smem);
  unsigned ta[4];                                      // TA: this lane's address of row tile t in an X part
  if constexpr (TA) {
    const int key = l16 >> 2;
#pragma unroll
    for (int t = 0; t < 4; ++t)
      ta[t] = 2 * PP_PART + (unsigned)(8 * lq + key) * 256u + (unsigned)((wm * 8 + t * 2 + ((l16 & 3) >> 1)) ^ (4 * key) ^ (2 * (lq & 1))) * 16u +
              (unsigned)(l16 & 1) * 8u;
  }
  u32x2_t xt[16];                                      // TA: the halves of X fragments (k step, row tile, half)
  u32x4_t wa[8], xf[8];                                // fragments: W (k step, half, feature tile), X (k step, row tile)
  floatx4_t acc[2][2][2][4];                           // [W half][feature tile][X half][row tile]
#define PP_READ_W(stage_)                                                                              \
  _Pragma("unroll") for (int kk = 0; kk < 2; ++kk) {                                                   \
    wa[4 * kk] = lds_read16<0>(smem0 + (stage_) * PP_STAGE + fw_off[kk]);                              \
    wa[4 * kk + 1] = lds_read16<512>(smem0 + (stage_) * PP_STAGE + fw_off[kk]);                       \
    wa[4 * kk + 2] = lds_read16<16384>(smem0 + (stage_) * PP_STAGE + fw_off[kk]);                      \
    wa[4 * kk + 3] = lds_read16<16384 + 512>(smem0 + (stage_) * PP_STAGE + fw_off[kk]);               \
  }
#define PP_READ_X(stage_, H)                                                                           \
  if constexpr (TA) {                                                                                  \
    _Pragma("unroll") for (int t = 0; t < 4; ++t) {                                                    \
      const unsigned a_ = smem0 + (stage_) * PP_STAGE + (H) * 16384u + ta[t];                          \
      xt[2 * t] = lds_read_tr8<0>(a_);                                                                 \
      xt[2 * t + 1] = lds_read_tr8<1024>(a_);                                                          \
      xt[8 + 2 * t] = lds_read_tr8<8192>(a_);                                                          \
      xt[8 + 2 * t + 1] = lds_read_tr8<8192 + 1024>(a_);                                               \
    }                                                                                                  \
  } else {                                                                                             \
    _Pragma("unroll") for (int kk = 0; kk < 2; ++kk)                                                   \
      lds_read_rows<4, 2048>(xf + 4 * kk, smem0 + (stage_) * PP_STAGE + (H) * 16384u + fx_off[kk]);    \
  }
  // all but the 8 youngest fills have landed; the stores of the tile before count with them while they are younger than what is waited for
  constexpr int STORES = MODE == 1 ? 8 : MODE == 3 ? 32 : 16;
  bool young = false;
#define PP_LANDED                                                               \
  if (young) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + STORES) : "memory");  \
  else asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  // end of a memory phase: this wave's reads are complete, its share of the parts that the next phase reads has landed
#define PP_MEM_END                                                                                     \
  PP_LANDED                                                                                            \
  if constexpr (TA)                                                                                    \
    asm volatile("s_waitcnt lgkmcnt(0)"                                                                \
               : "+v"(xt[0]), "+v"(xt[1]), "+v"(xt[2]), "+v"(xt[3]), "+v"(xt[4]), "+v"(xt[5]), "+v"(xt[6]), "+v"(xt[7]), \
                 "+v"(xt[8]), "+v"(xt[9]), "+v"(xt[10]), "+v"(xt[11]), "+v"(xt[12]), "+v"(xt[13]), "+v"(xt[14]), "+v"(xt[15]), \
                 "+v"(wa[0]), "+v"(wa[1]), "+v"(wa[2]), "+v"(wa[3]), "+v"(wa[4]), "+v"(wa[5]), "+v"(wa[6]), "+v"(wa[7])::"memory"); \
  else                                                                                                 \
    asm volatile("s_waitcnt lgkmcnt(0)"                                                                \
               : "+v"(xf[0]), "+v"(xf[1]), "+v"(xf[2]), "+v"(xf[3]), "+v"(xf[4]), "+v"(xf[5]), "+v"(xf[6]), "+v"(xf[7]), \
                 "+v"(wa[0]), "+v"(wa[1]), "+v"(wa[2]), "+v"(wa[3]), "+v"(wa[4]), "+v"(wa[5]), "+v"(wa[6]), "+v"(wa[7])::"memory"); \
  __builtin_amdgcn_s_barrier();                                                                        \
  __builtin_amdgcn_sched_barrier(0);
#define PP_MUL(HX)                                                                                     \
  __builtin_amdgcn_s_setprio(1);                                                                       \
  _Pragma("unroll") for (int kk = 0; kk < 2; ++kk)                                                     \
    _Pragma("unroll") for (int i = 0; i < 4; ++i)                                                      \
      _Pragma("unroll") for (int j = 0; j < 4; ++j)                                                    \
        acc[i >> 1][i & 1][HX][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wa[4 * kk + i]), \
                                                                            TA ? __builtin_bit_cast(bf16x8_t, Frag8{xt[8 * kk + 2 * j], xt[8 * kk + 2 * j + 1]}) \
                                                                               : __builtin_bit_cast(bf16x8_t, xf[4 * kk + j]), \
                                                                            acc[i >> 1][i & 1][HX][j], 0, 0, 0); \
  __builtin_amdgcn_s_setprio(0);                                                                       \
  __builtin_amdgcn_sched_barrier(0);                                                                   \
  __builtin_amdgcn_s_barrier();                                                                        \
  __builtin_amdgcn_sched_barrier(0);
#define PP_TILE(S_)                                                                                    \
  PP_READ_W(S_) PP_READ_X(S_, 0) PP_FETCH(3, kt + 1, 1 - (S_)) PP_MEM_END PP_MUL(0)                    \
  PP_READ_X(S_, 1) PP_FETCH(0, kt + 2, S_) PP_FETCH(2, kt + 2, S_) PP_FETCH(1, kt + 2, S_) PP_MEM_END PP_MUL(1)
#define PP_FIRST                                                         \
  PP_FETCH(0, 0, 0) PP_FETCH(2, 0, 0) PP_FETCH(1, 0, 0) PP_FETCH(3, 0, 0) \
  PP_FETCH(0, 1, 1) PP_FETCH(2, 1, 1) PP_FETCH(1, 1, 1)
  const unsigned scratch = smem0 + 2 * PP_STAGE + (unsigned)wm * 16384u;   // modes 0 and 2: 16 KB a group
  const int gl = tid & 255;
  PP_OPEN_TILE
  PP_FIRST
  for (;;) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i >> 2][(i >> 1) & 1][i & 1][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    PP_LANDED                                          // W0, W1 and X0 of k tile 0
    __builtin_amdgcn_s_barrier();
    if (wm) __builtin_amdgcn_s_barrier();              // the second group runs half a phase later
    __builtin_amdgcn_sched_barrier(0);
    for (int kt = 0;; ++kt) {
      PP_TILE(0)
      young = false;
      if (++kt >= nkt) break;
      PP_TILE(1)
      if (kt + 1 >= nkt) break;
    }
    if (!wm) __builtin_amdgcn_s_barrier();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the empty fills behind the last k tile
    __builtin_amdgcn_s_barrier();
    // every wave has left the stages: the next tile's first k tiles are on their way while this one is stored
    const int em0 = m0, en0 = n0;
    bf16_t* const ec = TA ? cb : C;
    const bf16_t* const er = TA ? rb : R;
    float* const ep = part;
    idx += (int)(gridDim.x >> 3);
    const bool more = idx < share && xcd + idx < tiles;
    if (more) {
      PP_OPEN_TILE
      PP_FIRST
    }
    asm volatile("" ::: "memory");
    // D of a 16x16 tile: lane l holds row l % 16, and of the two feature tiles of a W half features 8*(l/16) .. + 7 of its 32.
    // whole: no row and no feature is behind the end
    auto leave = [&](auto whole) __attribute__((always_inline)) {
      auto put = [&](u32x4_t v, int m, int f) __attribute__((always_inline)) {
        if (decltype(whole)::value || (m < M && f < N))
          store_feat8<MODE>(v, MODE == 2 ? er + (size_t)m * ldr + f : nullptr, ec + (size_t)m * ldc + f, decltype(whole)::value ? 8 : N - f);
      };
#pragma unroll
      for (int hx = 0; hx < 2; ++hx) {
        const int mrow = em0 + hx * 128 + wm * 64;
        if constexpr (MODE == 1 || MODE == 3) {        // straight from the accumulators
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int m = mrow + j * 16 + l16, f = en0 + wn * (MODE == 1 ? 32 : 64) + 8 * lq;
            if constexpr (MODE == 3) {
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const int fq = f + (q >> 1) * 32 + (q & 1) * 4;
                if (decltype(whole)::value || (m < M && fq < N)) *(floatx4_t*)(ep + (size_t)m * N + fq) = acc[q >> 1][q & 1][hx][j];
              }
            } else {
              float v[8];
#pragma unroll
              for (int e = 0; e < 8; ++e)
                v[e] = rnd_bf16(gelu_tanh_short(rnd_bf16(acc[0][e >> 2][hx][j][e & 3]))) * rnd_bf16(acc[1][e >> 2][hx][j][e & 3]);
              put(u32x4_t{pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]), pack2_bf16(v[4], v[5]), pack2_bf16(v[6], v[7])}, m, f);
            }
          }
        } else {                                       // 32 rows at a time through LDS, chunks XOR-ed with the row
#pragma unroll
          for (int j = 0; j < 4; j += 2) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
              for (int hw = 0; hw < 2; ++hw) {
                const int r = t * 16 + l16, c = wn * 8 + hw * 4 + lq;
                const floatx4_t a = acc[hw][0][hx][j + t], b = acc[hw][1][hx][j + t];
                const u32x4_t v = {pack2_bf16(a[0], a[1]), pack2_bf16(a[2], a[3]), pack2_bf16(b[0], b[1]), pack2_bf16(b[2], b[3])};
                asm volatile("ds_write_b128 %0, %1" ::"v"(scratch + (unsigned)(r * 512 + ((c ^ r) << 4))), "v"(v) : "memory");
              }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            u32x4_t o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int r = i * 8 + (gl >> 5), c = gl & 31;
              o[i] = lds_read16<0>(scratch + (unsigned)(r * 512 + ((c ^ r) << 4)));
            }
            lds_wait<0>(o);
            __builtin_amdgcn_s_barrier();
#pragma unroll
            for (int i = 0; i < 4; ++i) put(o[i], mrow + j * 16 + i * 8 + (gl >> 5), en0 + (gl & 31) * 8);
          }
        }
      }
    };
    young = !TA && em0 + 256 <= M && en0 + NF <= N;    // with transposing reads the loop is 2 to 5 % slower for the other waits
    if (young) leave(std::true_type{});
    else leave(std::false_type{});
    if (!more) break;
  }
#undef PP_OPEN_TILE
#undef PP_FIRST
#undef PP_FETCH
#undef PP_READ_W
#undef PP_READ_X
#undef PP_MEM_END
#undef PP_MUL
#undef PP_TILE
}

template <int MODE, bool TA = false>
int gemm_pp_launch(const void* A, long long lda, const void* W, const void* W2, const void* R, long long ldr, void* C,
                   long long ldc, int M, int N, int K, hipStream_t s, int nbatch = 1, long long sa = 0, long long sc = 0, long long sr = 0, int nb = 1) {
  constexpr int NF = MODE == 1 ? 128 : 256;
  static fstu_lds_limit most;
  if (const int rc = fstu_need_lds((const void*)gemm_pp_bf16_kernel<MODE, TA>, most, PP_LDS(MODE), "fstu_gemm_bf16")) return rc;
  const int mts = (M + 255) / 256, mt = mts * nbatch, nt = (N + NF - 1) / NF;
  const int share = (int)(((long long)mt * nt + 7) / 8);
  hipLaunchKernelGGL((gemm_pp_bf16_kernel<MODE, TA>), dim3(8u * (unsigned)std::min(share, gemm_cus() / 8)), dim3(512), PP_LDS(MODE), s, (const bf16_t*)A, lda,
                     (const bf16_t*)W, (const bf16_t*)W2, (const bf16_t*)R, ldr, (bf16_t*)C, ldc, M, N, K, mt, nt, share, mts, sa, sc, sr, nb);
  return 0;
}

// ---------------------------------------------------------------- 256 rows x 128 features in two alternating wave groups
// Products whose 256 x 256 tiles leave half of the compute units idle, whole or in slices of K.  Waves 0-3 own rows 0..127, waves 4-7
// rows 128..255, a wave 64 features x 64 rows; a k tile of 64 is one phase of 32 v_mfma_f32_16x16x32_bf16.  The groups run half
// a phase apart as above.  Three stages of W | X0 | X1 (16 KB each); in its memory phase of k tile kt a group reads its 16 fragments
// and requests its share of kt + 2 into the stage that both groups left a phase ago, and waits for its share of kt + 1.
// What bounds it: 0.58 us a k tile in a nearly empty round, of which its products are 0.49; 0.65 to 0.9 in a full one (power, LDS).
// us, before (256 x 256 or 128 x 128 tiles) / so: 4096 x 2048 x 2048 36.6 / 30.4, 2331 x 2304 x 768 16.4 / 12.7, 8192 x 768 x 768 16.3 / 12.6,
// 1024 x 8192 x 4096 65.9 / 53.5; joined slices of K 2331 x 768 x 9216 43.2 / 40.2, 4096 x 768 x 9216 65.8 / 60.3, 1000 x 2048 x 24576 102.6 / 88.5.
#define PH_STAGE 49152u
#define PH_LDS (3 * PH_STAGE)
template <int MODE>
__global__ void __launch_bounds__(512)
gemm_half_bf16_kernel(const bf16_t* __restrict__ A, long long lda, const bf16_t* __restrict__ W, const bf16_t* __restrict__ R, long long ldr,
                      bf16_t* __restrict__ C, long long ldc, int M, int N, int K, int mt, int nt, int share, int ksplit) {
  extern __shared__ __align__(16) unsigned char gm_smem[];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  int o = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= share || o >= mt * nt * ksplit) return;
  const int slice = o / (mt * nt), nk = K >> 6;       // MODE 3: slices of K outermost, any number of k tiles to each
  o -= slice * (mt * nt);
  const int kt0 = MODE == 3 ? (int)((long long)nk * slice / ksplit) : 0, kt1 = MODE == 3 ? (int)((long long)nk * (slice + 1) / ksplit) : nk;
  const int per_panel = mt * GM_PANEL, panel = o / per_panel, in_panel = o - panel * per_panel;
  const int pw = min(GM_PANEL, nt - panel * GM_PANEL);
  const int m0 = in_panel / pw * 256, n0 = (panel * GM_PANEL + in_panel % pw) * 128;
  const rsrc_t rs_w = make_rsrc(W + (size_t)n0 * K, (size_t)min(128, N - n0) * K * 2);
  const rsrc_t rs_a = make_rsrc(A + (size_t)m0 * lda, ((size_t)(min(256, M - m0) - 1) * lda + K) * 2);
  // ---- fills: a part is 128 rows of 128 bytes; a wave fills rows 16 wv .. + 15 of each with two instructions
  unsigned wvoff[2], avoff[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = wv * 16 + j * 8 + (lane >> 3);
    wvoff[j] = (unsigned)row * (unsigned)K * 2u + (unsigned)((lane & 7) ^ (((row >> 1) & 1) | ((row >> 2) & 6))) * 16u;
    avoff[j] = (unsigned)row * (unsigned)lda * 2u + (unsigned)((lane & 7) ^ ((row >> 1) & 7)) * 16u;
  }
  const unsigned x1off = 128u * (unsigned)lda * 2u;
  unsigned char* const fill0 = gm_smem + (unsigned)wv * 2048u;
  auto fetch = [&](int kt, unsigned stage) __attribute__((always_inline)) {   // beyond the last k tile that one again, into a stage that nobody reads
    const unsigned so = (unsigned)min(kt, kt1 - 1) * 128u;
    unsigned char* const l = fill0 + stage;
#pragma unroll
    for (int j = 0; j < 2; ++j) buf_load16_to_lds(rs_w, wvoff[j], so, l + j * 1024);
#pragma unroll
    for (int j = 0; j < 2; ++j) buf_load16_to_lds(rs_a, avoff[j], so, l + PP_PART + j * 1024);
#pragma unroll
    for (int j = 0; j < 2; ++j) buf_load16_to_lds(rs_a, avoff[j] + x1off, so, l + 2 * PP_PART + j * 1024);
  };
  const int l16 = lane & 15, lq = lane >> 4, wf = wv & 1, wr = (wv >> 1) & 1, grp = wv >> 2;
  unsigned fw_off[2], fx_off[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int rw = wf * 64 + 8 * (l16 >> 2) + (l16 & 3), rx = wr * 64 + l16, c = kk * 4 + lq;
    fw_off[kk] = (unsigned)rw * 128u + (unsigned)((c ^ (((rw >> 1) & 1) | ((rw >> 2) & 6))) << 4);
    fx_off[kk] = (unsigned)(1 + grp) * PP_PART + (unsigned)rx * 128u + (unsigned)((c ^ ((rx >> 1) & 7)) << 4);
  }
  const unsigned smem0 = lds_addr(gm_smem);
  u32x4_t wa[8], xf[8];                                // (k step, feature tile), (k step, row tile)
  floatx4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  fetch(kt0, 0);
  fetch(kt0 + 1, PH_STAGE);
  asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  if (grp) __builtin_amdgcn_s_barrier();               // the second group runs half a phase later
  unsigned cur = 0, two = 2 * PH_STAGE;                // stages of k tiles kt and kt + 2
  __builtin_amdgcn_sched_barrier(0);
  for (int kt = kt0; kt < kt1; ++kt) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const unsigned a = smem0 + cur + fw_off[kk];
      wa[4 * kk] = lds_read16<0>(a);
      wa[4 * kk + 1] = lds_read16<512>(a);
      wa[4 * kk + 2] = lds_read16<4096>(a);
      wa[4 * kk + 3] = lds_read16<4096 + 512>(a);
      lds_read_rows<4, 2048>(xf + 4 * kk, smem0 + cur + fx_off[kk]);
    }
    fetch(kt + 2, two);
    asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)"
                 : "+v"(xf[0]), "+v"(xf[1]), "+v"(xf[2]), "+v"(xf[3]), "+v"(xf[4]), "+v"(xf[5]), "+v"(xf[6]), "+v"(xf[7]),
                   "+v"(wa[0]), "+v"(wa[1]), "+v"(wa[2]), "+v"(wa[3]), "+v"(wa[4]), "+v"(wa[5]), "+v"(wa[6]), "+v"(wa[7])::"memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wa[4 * kk + i]), __builtin_bit_cast(bf16x8_t, xf[4 * kk + j]),
                                                              acc[i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    cur = cur == 2 * PH_STAGE ? 0 : cur + PH_STAGE;
    two = two == 2 * PH_STAGE ? 0 : two + PH_STAGE;
  }
  if (!grp) __builtin_amdgcn_s_barrier();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the fills behind the last k tile
  // lane l holds row l % 16 and, of two feature tiles, features 8*(l/16) .. + 7
  if constexpr (MODE == 3) {
    float* const part = (float*)C + (size_t)slice * M * N;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + grp * 128 + wr * 64 + j * 16 + l16, f = n0 + wf * 64 + (i >> 1) * 32 + 8 * lq + (i & 1) * 4;
        if (m < M && f < N) *(floatx4_t*)(part + (size_t)m * N + f) = acc[i][j];
      }
  } else {
    __builtin_amdgcn_s_barrier();                      // every wave has left the stages: rows of 256 bytes, chunks XOR-ed with the row
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int r = grp * 128 + wr * 64 + j * 16 + l16, c = wf * 8 + p * 4 + lq;
        const floatx4_t a = acc[2 * p][j], b = acc[2 * p + 1][j];
        *(uint4*)(gm_smem + r * 256 + ((c ^ (r & 15)) << 4)) = make_uint4(pack2_bf16(a[0], a[1]), pack2_bf16(a[2], a[3]), pack2_bf16(b[0], b[1]), pack2_bf16(b[2], b[3]));
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = i * 32 + (tid >> 4), c = tid & 15, m = m0 + r, f = n0 + c * 8;
      const u32x4_t v = *(const u32x4_t*)(gm_smem + r * 256 + ((c ^ (r & 15)) << 4));
      if (m < M && f < N) store_feat8<MODE>(v, MODE == 2 ? R + (size_t)m * ldr + f : nullptr, C + (size_t)m * ldc + f, N - f);
    }
  }
}

template <int MODE>
int gemm_half_launch(const void* A, long long lda, const void* W, const void* R, long long ldr, void* C, long long ldc, int M, int N, int K,
                     hipStream_t s, int ksplit = 1) {
  static fstu_lds_limit most;
  if (const int rc = fstu_need_lds((const void*)gemm_half_bf16_kernel<MODE>, most, PH_LDS, "fstu_gemm_bf16")) return rc;
  const int mt = (M + 255) / 256, nt = (N + 127) / 128, share = (int)(((long long)mt * nt * ksplit + 7) / 8);
  hipLaunchKernelGGL((gemm_half_bf16_kernel<MODE>), dim3((unsigned)share * 8u), dim3(512), PH_LDS, s, (const bf16_t*)A, lda, (const bf16_t*)W,
                     (const bf16_t*)R, ldr, (bf16_t*)C, ldc, M, N, K, mt, nt, share, ksplit);
  return 0;
}

// ---------------------------------------------------------------- transposed activations
// C[b][m, n] = sum_k A[b][k, m] W[n, k]: the activations come as a slab with the REDUCTION index slowest (k rows of
// lda elements, m contiguous) — the time-major U+- of the exact-mode STU operator (flash_stu/modules/stu.py:107-120:
// tensordot of U (B, L, K, d) with M_phi (K, d, d) over (K, d); the filter-bank kernel writes U as (B, K*d, L) so
// that its stores are whole lines).  Same tiles, pipeline and epilogues as gemm_bf16_kernel (mode 0 and 2); what
// differs is the activation tile: LDS rows are k (BK rows of BT*2 bytes, filled 16 bytes = 8 consecutive m per lane),
// and the MFMA B fragment — 8 consecutive k of one m per lane — is gathered by two transposing reads
// (ds_read_b64_tr_b16: in a block of 16 lanes, lane i supplies the address of 4 consecutive m of row i/4 starting at
// column 4*(i%4), and receives column i of the 4 rows).  The 64-byte column groups of a row are XOR-ed with the row's
// low two bits, so the four rows of a read fall into different banks.  `nbatch` slabs run as one grid.
template <int N, int STEP, int I = 0>
__device__ __forceinline__ void lds_read_tr_cols(u32x2_t* f, const unsigned* addr) {   // N column tiles, rows k..k+3 and k+4..k+7
  if constexpr (I < N) {
    f[2 * I] = lds_read_tr8<0>(addr[I]);
    f[2 * I + 1] = lds_read_tr8<4 * STEP>(addr[I]);
    lds_read_tr_cols<N, STEP, I + 1>(f, addr);
  }
}
template <int LEFT>
__device__ __forceinline__ void lds_wait_n() { asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(LEFT)); }
template <int N> __device__ __forceinline__ void pin4(u32x4_t* f) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i]));
}
template <int N> __device__ __forceinline__ void pin2(u32x2_t* f) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i]));
}

template <bool TW, int FI> struct WeightFrags {
  u32x4_t f[FI];
  __device__ __forceinline__ bf16x8_t frag(int i) const { return __builtin_bit_cast(bf16x8_t, f[i]); }
  __device__ __forceinline__ void pin() { pin4<FI>(f); }
};
template <int FI> struct WeightFrags<true, FI> {
  u32x2_t f[2 * FI];
  __device__ __forceinline__ bf16x8_t frag(int i) const { return __builtin_bit_cast(bf16x8_t, (Frag8{f[2 * i], f[2 * i + 1]})); }
  __device__ __forceinline__ void pin() { pin2<2 * FI>(f); }
};

// TW: the weights come the same way, (K, N) with rows of ldw elements and N a multiple of the tile, and take the same way through
// LDS: the gradient of a weight, whose sum over all positions has both operands' reduction index slowest.  What bounds it is a
// workgroup's chain of k tiles, 0.6 us each alone on a compute unit (the fills, which four stages do not shorten: M = N = 768,
// K = 16384 in 7 slices 31.7 us with four, 32.3 with two; two workgroups to a unit 48 and 36 in 8).
template <class G, int MODE, bool TW = false>
__global__ void __launch_bounds__(G::THREADS)
gemm_ta_bf16_kernel(const bf16_t* __restrict__ A, long long lda, long long sa, const bf16_t* __restrict__ W, long long ldw,
                    const bf16_t* __restrict__ R, long long ldr, long long sr, bf16_t* __restrict__ C, long long ldc,
                    long long sc, int M, int N, int K, int mt, int nt, int share, int nbatch, int ksplit) {
  constexpr int FI = G::FI, TJ = G::TJ, BF = G::BF, BT = G::BT, WL = G::WL, AL = G::AL, NS = G::NS, KK = G::KK;
  constexpr unsigned STAGE = G::STAGE;
  constexpr int RBT = BT * 2, CPRT = BT / 8;              // bytes and 16-byte chunks of an activation row (one k)
  constexpr int RBW = BF * 2, CPRW = BF / 8;              // TW: the same of a weight row
  constexpr int NRD = (TW ? 2 : 1) * FI + 2 * TJ;         // LDS reads per k step
  static_assert(!TW || MODE == 0 || MODE == 3, "TW: plain or split-K epilogue");
  static_assert(G::BK == 64 && BT >= 128, "k tile of 64, at least 128 columns");
  static_assert((MODE == 0 || MODE == 2 || MODE == 3), "plain, residual or split-K epilogue");
  extern __shared__ __align__(16) unsigned char gm_smem[];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wf = w % G::WFN, wt = w / G::WFN;
  int o = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= share || o >= mt * nt * nbatch * ksplit) return;
  const int bs = o / (mt * nt), slice = bs / nbatch, batch = bs - slice * nbatch;    // MODE 3: slices of K outermost
  o -= bs * (mt * nt);
  const int nk = (K + G::BK - 1) / G::BK;              // TW: the last k tile may be ragged, rows behind the end are zeros
  const int kbeg = MODE == 3 ? (int)((long long)nk * slice / ksplit) * G::BK : 0;              // this workgroup's share of K
  const int KS = MODE == 3 ? min((int)((long long)nk * (slice + 1) / ksplit) * G::BK, K) - kbeg : K;
  const int per_panel = mt * GM_PANEL;
  const int panel = o / per_panel, in_panel = o - panel * per_panel;
  const int pw = min(GM_PANEL, nt - panel * GM_PANEL);
  const int bt = in_panel / pw, bf = panel * GM_PANEL + in_panel % pw;
  const int m0 = bt * BT, n0 = bf * BF;
  A += (size_t)batch * sa + (MODE == 3 ? (size_t)kbeg * lda : 0);
  if (MODE == 3) W += TW ? (size_t)kbeg * ldw : (size_t)kbeg;
  C += (size_t)batch * sc;
  if (MODE == 2) R += (size_t)batch * sr;
  const int wv = __builtin_amdgcn_readfirstlane(w);
  const int rows_w = min(BF, N - n0);
  const rsrc_t rs_w = TW ? make_rsrc(W + n0, ((size_t)(KS - 1) * ldw + BF) * 2)
                         : make_rsrc(W + (size_t)n0 * K, ((size_t)(rows_w - 1) * K + KS) * 2);
  const rsrc_t rs_a = make_rsrc(A + m0, ((size_t)(KS - 1) * lda + BT) * 2);    // M % BT == 0: whole rows of BT columns
  unsigned wvoff[WL], avoff[AL];
#pragma unroll
  for (int j = 0; j < WL; ++j) {
    const int slot = (wv * WL + j) * 64 + lane, row = slot / G::CPR;
    const int ch = (int)((G::swz(row, slot % G::CPR) - (unsigned)row * G::RB) >> 4);
    wvoff[j] = (unsigned)row * (unsigned)K * 2u + (unsigned)ch * 16u;
    if constexpr (TW) {
      const int kr = slot / CPRW;
      wvoff[j] = (unsigned)kr * (unsigned)ldw * 2u + (unsigned)((slot % CPRW) ^ (4 * (kr & 3))) * 16u;
    }
  }
#pragma unroll
  for (int j = 0; j < AL; ++j) {
    const int slot = (wv * AL + j) * 64 + lane, kr = slot / CPRT, pc = slot % CPRT;
    const int lc = pc ^ (4 * (kr & 3));                  // the XOR is its own inverse
    avoff[j] = (unsigned)kr * (unsigned)lda * 2u + (unsigned)lc * 16u;
  }
  const unsigned wslot = (unsigned)(wv * WL) * 1024u, aslot = (unsigned)BF * G::RB + (unsigned)(wv * AL) * 1024u;
#define GT_FETCH(stage_, k0)                                                                                 \
  {                                                                                                          \
    unsigned char* st_ = gm_smem + (unsigned)(stage_) * STAGE;                                               \
    const unsigned sw_ = TW ? (unsigned)((size_t)(k0) * (size_t)ldw * 2u) : (unsigned)(k0) * 2u;              \
    const unsigned sa_ = (unsigned)((size_t)(k0) * (size_t)lda * 2u);                                        \
    _Pragma("unroll") for (int j = 0; j < WL; ++j) buf_load16_to_lds(rs_w, wvoff[j], sw_, st_ + wslot + j * 1024); \
    _Pragma("unroll") for (int j = 0; j < AL; ++j) buf_load16_to_lds(rs_a, avoff[j], sa_, st_ + aslot + j * 1024); \
  }
#define GT_MFMAS(fw_, fx_)                                                                                   \
  _Pragma("unroll") for (int i = 0; i < FI; ++i)                                                             \
    _Pragma("unroll") for (int j = 0; j < TJ; ++j) {                                                         \
      const Frag8 b_ = {fx_[2 * j], fx_[2 * j + 1]};                                                         \
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw_.frag(i), __builtin_bit_cast(bf16x8_t, b_), acc[i][j], 0, 0, 0); \
    }
  const int l32 = lane & 31, lh = lane >> 5;
  unsigned fw_off[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) fw_off[kk] = G::swz(wf * (32 * FI) + l32, kk * 2 + lh);
  // transposing reads: this lane's address inside a stage for column tile j at k step 0, rows k..k+3
  const int blk = lane >> 4, i16 = lane & 15, key = i16 >> 2;
  unsigned ta_off[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j)
    ta_off[j] = (unsigned)BF * G::RB + (unsigned)(8 * (blk >> 1) + key) * RBT + (unsigned)(((wt * TJ + j) ^ key) << 6) +
                (unsigned)(2 * (blk & 1) + ((i16 & 3) >> 1)) * 16u + (unsigned)(i16 & 1) * 8u;
  unsigned tw_off[FI];                                    // TW: the same for the feature tiles
#pragma unroll
  for (int i = 0; i < FI; ++i)
    tw_off[i] = (unsigned)(8 * (blk >> 1) + key) * RBW + (unsigned)(((wf * FI + i) ^ key) << 6) +
                (unsigned)(2 * (blk & 1) + ((i16 & 3) >> 1)) * 16u + (unsigned)(i16 & 1) * 8u;
  floatx16_t acc[FI][TJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  const int nkt = TW ? (KS + G::BK - 1) / G::BK : KS / G::BK;
  constexpr int LPT = WL + AL;
#pragma unroll
  for (int t = 0; t < NS - 1; ++t)
    if (t < nkt) GT_FETCH(t, t * G::BK)
  const unsigned smem0 = lds_addr(gm_smem);
  if (NS - 2 < nkt) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * LPT) : "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  if (NS - 1 < nkt) GT_FETCH(NS - 1, (NS - 1) * G::BK)
  WeightFrags<TW, FI> wa_, wb_;                       // weight fragments of alternate k steps
  u32x2_t xa_[2 * TJ], xb_[2 * TJ];                   // activation fragments (two halves per column tile)
  unsigned ta[TJ], tw[FI];
#define GT_READ(fw_, fx_, base_, kk_)                                                                        \
  {                                                                                                          \
    if constexpr (TW) {                                                                                      \
      _Pragma("unroll") for (int i = 0; i < FI; ++i) tw[i] = (base_) + tw_off[i] + (unsigned)(kk_) * 16u * RBW; \
      lds_read_tr_cols<FI, RBW>(fw_.f, tw);                                                                  \
    } else {                                                                                                 \
      lds_read_rows<FI, 32 * G::RB>(fw_.f, (base_) + fw_off[kk_]);                                           \
    }                                                                                                        \
    _Pragma("unroll") for (int j = 0; j < TJ; ++j) ta[j] = (base_) + ta_off[j] + (unsigned)(kk_) * 16u * RBT; \
    lds_read_tr_cols<TJ, RBT>(fx_, ta);                                                                      \
  }
#define GT_WAIT(left_, fw_, fx_)                                                                             \
  {                                                                                                          \
    lds_wait_n<left_>();                                                                                     \
    fw_.pin();                                                                                               \
    pin2<2 * TJ>(fx_);                                                                                       \
  }
  GT_READ(wa_, xa_, smem0, 0)
  int cur = 0;
  for (int kt = 0; kt < nkt; ++kt) {
    const unsigned cb = smem0 + (unsigned)cur * STAGE;
    const int nxt = cur + 1 == NS ? 0 : cur + 1;
    __builtin_amdgcn_sched_barrier(0);
    GT_READ(wb_, xb_, cb, 1)
    GT_WAIT(NRD, wa_, xa_)
    GT_MFMAS(wa_, xa_)
    __builtin_amdgcn_sched_barrier(0);
    GT_READ(wa_, xa_, cb, 2)
    GT_WAIT(NRD, wb_, xb_)
    GT_MFMAS(wb_, xb_)
    __builtin_amdgcn_sched_barrier(0);
    GT_READ(wb_, xb_, cb, 3)
    GT_WAIT(NRD, wa_, xa_)
    GT_MFMAS(wa_, xa_)
    __builtin_amdgcn_sched_barrier(0);
    GT_WAIT(0, wb_, xb_)                              // this wave has left the stage of tile kt
    if (kt + 1 < nkt) {
      if (kt + NS - 1 < nkt) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * LPT) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      if (kt + NS < nkt) GT_FETCH(cur, (kt + NS) * G::BK)
      const unsigned nb = smem0 + (unsigned)nxt * STAGE;
      GT_READ(wa_, xa_, nb, 0)
    }
    __builtin_amdgcn_sched_barrier(0);
    GT_MFMAS(wb_, xb_)
    cur = nxt;
  }
#undef GT_FETCH
#undef GT_MFMAS
#undef GT_READ
#undef GT_WAIT
  // ---- epilogue: lane l holds row (position) l % 32 and features 8*(e/4) + 4*(l/32) + e%4 of a 32x32 tile
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const int m = m0 + wt * (32 * TJ) + j * 32 + l32;
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < FI; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int f = n0 + wf * (32 * FI) + i * 32 + q * 8 + lh * 4;
        if (f >= N) continue;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[i][j][q * 4 + e];
        if (MODE == 3) {
          *(float4*)((float*)R + (((size_t)slice * nbatch + batch) * M + m) * N + f) = make_float4(v[0], v[1], v[2], v[3]);
          continue;
        }
        if (MODE == 2) {
          const uint2 rv = *(const uint2*)(R + (size_t)m * ldr + f);
          v[0] = __uint_as_float(rv.x << 16) + rnd_bf16(v[0]);
          v[1] = __uint_as_float(rv.x & 0xffff0000u) + rnd_bf16(v[1]);
          v[2] = __uint_as_float(rv.y << 16) + rnd_bf16(v[2]);
          v[3] = __uint_as_float(rv.y & 0xffff0000u) + rnd_bf16(v[3]);
        }
        *(uint2*)(C + (size_t)m * ldc + f) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
      }
  }
}

template <class G, int MODE, bool TW = false>
int gemm_ta_launch_tile(const void* A, long long lda, long long sa, const void* W, const void* R, long long ldr, long long sr,
                        void* C, long long ldc, long long sc, int M, int N, int K, int nbatch, hipStream_t s, int ksplit = 1, long long ldw = 0) {
  static fstu_lds_limit most;
  if (const int rc = fstu_need_lds((const void*)gemm_ta_bf16_kernel<G, MODE, TW>, most, G::LDS, "fstu_gemm_bf16_ta")) return rc;
  const int mt = M / G::BT, nt = (N + G::BF - 1) / G::BF;
  const long long tiles = (long long)mt * nt * nbatch * ksplit;
  const int share = (int)((tiles + 7) / 8);
  hipLaunchKernelGGL((gemm_ta_bf16_kernel<G, MODE, TW>), dim3((unsigned)share * 8u), dim3(G::THREADS), G::LDS, s, (const bf16_t*)A, lda, sa,
                     (const bf16_t*)W, ldw, (const bf16_t*)R, ldr, sr, (bf16_t*)C, ldc, sc, M, N, K, mt, nt, share, nbatch, ksplit);
  return 0;
}


//                     waves  tiles  BK  stages
using TileSmall = GemmTile<2, 2, 2, 2, 64, 2>;   // 128 x 128, 4 waves, 64 KB: two workgroups per compute unit
using TileDeep = GemmTile<2, 2, 2, 2, 64, 4>;    // 128 x 128, 4 waves, 3 tiles in flight: one workgroup per compute unit
using TileRows32 = GemmTile<2, 1, 2, 1, 64, 4>;  // 128 features x 32 rows, 2 waves, 80 KB: weight streaming, two workgroups per compute unit
using Tile96 = GemmTile<1, 4, 3, 1, 64, 4>;      // 96 features x 128 rows, 4 waves, 112 KB: N = 768 or 2304 in whole tiles
using TileK32 = GemmTile<2, 2, 4, 2, 32, 3>;     // 256 x 128, 4 waves, 72 KB, k tiles of 32 for K % 64 != 0

// Whether a product (K % 64 == 0) of that many tiles of either size runs on 256 x 256 tiles: both sides' estimate in twentieths of
// a round of small tiles, two to a compute unit.  A last round of small tiles costs 0.4 of a full one however few they are, and
// their stores, a quarter of a line at a time, 0.2 more than the large tiles' do.  A round of large tiles, one to a compute
// unit, takes 1.15 of them, and in mode 1, whose GELU covers only half of its round's products, 1.4 where K is long and 1.55
// where it is short; where K is long and over three rounds, from K = 4096 on over two, 1.25.  us, large / small tiles.  Mode 0: 4096 x 2304 (144 large tiles, 576 small) K = 64 8.8 / 13.1, 768 17.8 / 25.9,
// 2048 37.9 / 53.0; 2048 x 4096 (128, 512) 8.8 / 12.2, 17.8 / 19.6, 35.7 / 37.1; 8192 x 2304 (288, 1152) K = 768 38.5 / 42.9, 2048
// 78.6 / 82.6; the line: 3840 x 2048 (120, 480) K = 256 10.7 / 11.4, 2048 39.0 / 35.4.  Mode 1: 4096 x 2 x 1152 (144, 576) K = 64
// 9.4 / 9.8, 768 18.9 / 23.2, 2048 36.7 / 50.9; 8192 x 2 x 2304 (576, 2304) 21.6 / 22.3, 57.4 / 62.6, 128 / 144; the line: 8192
// x 2 x 1152 (288, 1152) 15.7 / 14.2, 37.1 / 36.5, 81.6 / 80.6, 20000 x 2 x 512 (316, 1256) 15.7 / 14.2, 36.8 / 35.7, 80.5 / 81.1;
// of a long K 608 x 2 x 24576 x 2048 (576, 1920) 124 / 126, in a model's pass 128 / 138, x 4096 244 / 257, 2842 x 2 x 3072 x 5120 (288, 1104) 185 / 195, 342 x 2 x 50256 x 12288 (786, 2358) 1032 /
// 1088, 263 rows of it at K = 6144 531 / 500, 970 x 2 x 4096 x 5120 (128, 512) 81 / 76.
bool pp_takes(int mode, int K, long long big, long long small, bool slabs = false) {
  const long long cus = gemm_cus(), full = small / (2 * cus), rest = small % (2 * cus);
  const long long little = (mode == 1 ? 6 : 4) + 20 * full + (rest ? 8 + 6 * rest / cus : 0);
  return (mode != 1 ? (slabs && K < 8192 ? 25 : 23) : K >= 1536 && big > (K < 4096 ? 2 : 1) * cus ? 25 : K >= 1024 ? 28 : 31) * ((big + cus - 1) / cus) < little;
}
long long tiles_of(int side, int M, int N) { return (long long)((M + side - 1) / side) * (((long long)N + side - 1) / side); }

// One round of 256 x 128 tiles where 128 x 128 ones would be more than one to a compute unit.  us, 256 x 128 / the others, either side of the
// line, rows x features (256 x 128 tiles, 128 x 128 tiles): 2048 x 2304 (144, 288) K = 64 8.0 / 9.1, 256 8.3 / 11.0, 768 12.7 / 16.9, 2048 24.7 / 30.1,
// 4096 42.0 / 50.6; 1024 x 8192 (256, 512) 8.1 / 8.6, 9.8 / 11.2, 16.7 / 19.0, 32.4 / 37.4, 53.3 / 65.0; 300 x 12000 (188, 282) K = 768 12.3 /
// 15.2; 2048 x 2048 (128, 256) K = 768 12.2 / 12.1, 2048 27.0 / 22.8; 4096 x 2304 (288, 576) K = 768 24.1 / 20.1.
bool half_takes(int M, int N) {
  return (long long)((M + 255) / 256) * ((N + 127) / 128) <= gemm_cus() && tiles_of(128, M, N) > gemm_cus();
}

template <int MODE>
int gemm_launch(const void* A, long long lda, const void* W, const void* W2, const void* R, long long ldr, void* C, long long ldc,
                int M, int N, int K, hipStream_t s) {
  if (K % 64 != 0) return gemm_launch_tile<TileK32, MODE>(A, lda, W, W2, R, ldr, C, ldc, M, N, K, s);
  if (M <= 32) return gemm_launch_tile<TileRows32, MODE>(A, lda, W, W2, R, ldr, C, ldc, M, N, K, s);
  const int columns = MODE == 1 ? 2 * N : N;
  const long long small = tiles_of(128, M, columns);
  if constexpr (MODE != 1) {
    if (half_takes(M, N)) return gemm_half_launch<MODE>(A, lda, W, R, ldr, C, ldc, M, N, K, s);
  }
  if (pp_takes(MODE, K, tiles_of(256, M, columns), small))
    return gemm_pp_launch<MODE>(A, lda, W, W2, R, ldr, C, ldc, M, N, K, s);
  // A grid that leaves one workgroup per compute unit anyway gains from the deeper pipeline when K is long (M=4096, N=768,
  // K=9216: 83 us against 93 us).
  if constexpr (MODE != 1) {
    // A feature count that is a whole number of 96-wide tiles but leaves compute units idle (or nearly idle in a last
    // round) with 128-wide ones: the time follows the rounds a compute unit runs times the area of a tile
    // (N = 768, M = 4096: 192 tiles of 128 x 128 on 256 CUs against 256 tiles of 96 x 128).  Only where the 128-wide
    // grid does not fill the chip: with several rounds per compute unit two resident workgroups of 128 x 128 cover
    // each other's start and end (N = 2304, M = 4096: 28.5 us against 35.2 us for the 96-wide tile).
    const long long cus = gemm_cus(), t96 = (long long)((M + 127) / 128) * (N / 96);
    if (N % 96 == 0 && small <= cus && ((t96 + cus - 1) / cus) * 96 < ((small + cus - 1) / cus) * 128)
      return gemm_launch_tile<Tile96, MODE>(A, lda, W, W2, R, ldr, C, ldc, M, N, K, s);
  }
  if (K >= 2048 && small <= gemm_cus()) return gemm_launch_tile<TileDeep, MODE>(A, lda, W, W2, R, ldr, C, ldc, M, N, K, s);
  return gemm_launch_tile<TileSmall, MODE>(A, lda, W, W2, R, ldr, C, ldc, M, N, K, s);
}

}  // namespace

// Slices of K for a product of few output tiles (1: none).  A workgroup that has a compute unit to itself takes 0.41 us per k tile
// of 64 on the deep pipeline (0.9 with two stages, which is what slices that leave one to a unit ran on before), two to a unit 0.61
// each; joining costs a launch and the slices' bytes out and back at 4 TB/s.  The estimate only has to rank: us without / with the
// slices it picks, rows x features x K: 300 x 768 x 9216 60 / 17.7 (12), 1000 x 768 x 9216 60 / 27.5 (4; 31.4 with two stages), 1400
// 60 / 34.0 (3; 39.7), 2400 61 / 44.7 (4; 47.2 with two, which were picked before and took 53.8), 3000 63 / 53 (3), 700 x 2048 x
// 24576 180 / 85 (4), 1500 x 2048 x 24576 184 / 160 (2), 300 x 2048 x 2048 21.8 / 15.0 (4).  Slabs take 0.6 us a k tile alone on a
// compute unit and 0.86 each two to a unit, with four stages no less than with the two that they run on; the counts are the best or
// within 12 % of it all the same: without / picked / best, 1 x 1024 x 1024 x 24576 219 / 58.5 (8), 1 x 512 x 1024 x 24576 226 / 40.6 (8) / 37.1
// (16), 4 x 512 x 512 x 12288 112 / 40.7 (4) / 37.0 (8), 2 x 256 x 512 x 12288 119 / 19.7 (12), 1 x 128 x 256 x 6144 54 / 12.5 (12).  Where it picks none, without / with two: 4096 x 768 x 9216 66.6 / 68.8, 600 x 2048 x
// 2048 22.0 / 18.8, 300 x 6144 x 2048 20.5 / 23.8, 1000 x 768 x 768 10.5 / 12.7.  Below K = 2048 the GPU gains less than the second
// launch and the slices' allocation cost the host (calls of 300 x 384 x 1536 one behind the other 16.0 us with three slices, 13.2
// without).
extern "C" int fstu_gemm_bf16_slices(int M, int N, int K, int nbatch) {
  if (M <= 32 || N % 4 != 0 || K % 64 != 0 || K < 2048) return 1;
  const long long cus = gemm_cus(), tiles = (long long)((M + 127) / 128) * ((N + 127) / 128) * nbatch;
  const int nkt = K / 64;
  double least = 0.41 * nkt;
  int best = 1;
  for (int s = 2; s <= 32 && K / s >= 512 && tiles * s <= 2 * cus; ++s) {
    if (nkt % s != 0) continue;
    const double us = nkt / s * (tiles * s <= cus ? 0.41 : 0.61) + 3.0 + 8e-6 / 4.0 * s * nbatch * (double)M * N;
    if (us < least) { least = us; best = s; }
  }
  return best;
}

namespace {

// The same where the slices can also run on 256 x 256 tiles in the alternating-group kernel (rows, or slabs of whole tiles of them):
// half the operands' bytes through the LDS for a product, and every compute unit at work where M and N leave it idle.  A k tile of
// 64 takes those 1 us in a nearly empty round and 1.35 in a full one, which draws the matrix cores' power; 128 x 128 tiles 0.43 us alone on
// a compute unit and, two to a unit, 0.55 to 0.9 in slices and up to 1.05 over a whole long K.  us on small tiles / with the slices it picks
// (L: large tiles), rows x features x K: 1408 x 2048 x 24576 151 / 119 (L4), 2500 257 / 186 (L3), 4096 391 / 277 (L2), 5500 x 768 x 9216
// 95 / 75 (L3).  Slabs: 1 x 8192 x 1024 x 24576 451 / 309 (L2), 4 x 2048 454 / 303 (L2), 2 x 2048 242 / 159 (L4), 1 x 4096 x 768 x 18432 142
// / 111 (L4); those of 129 to 144 large tiles in three slices / whole 3 x 6144 x 512 x 12288 220 / 231, 4 x 2816 x 768 x 9216 165 / 149.
// Rows (not slabs) have 256 x 128 tiles between the two, in slices of any number of k tiles, where one round holds them all: without / with
// the slices it picks, 2331 x 768 x 9216 43.4 / 40.2 (4), 4096 66.1 / 60.5 (2), 3200 54.8 / 50.4 (3), 1800 38.9 / 35.7 (5), 1000 x 2048 x 24576
// 100 / 88 (4).  They are not asked for where slices on large tiles gain (400 x 4100 x 8192 47.9 in four of those, 41.2 in three of these).
// A product whose whole runs on large or half tiles takes no slices where these do not gain: both sides' estimates there are fitted to 220
// products of 256 to 12000 rows, 512 to 4096 features and K = 2048 to 24576 with every count on every tile (2 to 5 % off), and tried on 220
// others.  A k tile costs the more the fuller the round is, large tiles from 32 and half ones from 96 of them on.  Slices on large tiles /
// whole: on half tiles 7882 x 768 x 9216 108.9 / 92.2, 10660 130.7 / 112.3, 4963 x 1536 x 9216 120.2 / 108.7, at the line 8504 x 512 x 6144 59.3 /
// 60.9, 2063 x 2048 x 6144 59.9 / 59.8; on large ones 4054 x 2304 x 6144 116.6 / 100.2, 5903 x 1536 x 6144 115.0 / 101.1, at the line 2119 x 4096 x
// 12288 193.9 / 199.0, 12000 x 768 x 9216 168.6 / 165.5; beyond K = 12288, where the estimate of a long round is low, 3520 x 3072 x 24576 402 / 434.
// Half tiles read the rows twice as often as large ones: where these are more than the memory-side cache holds beside the rest, slices stay
// (200 MB of rows: 10660 x 768 x 9216, 197 MB, above; 12724 x 512 x 9216, 235 MB, 114.4 / 126.8, 10348 x 768 x 12288, 254 MB, 160 / 180).
enum TileKind { SMALL, LARGE, HALF };
struct SlicePlan { int count; TileKind on; };
SlicePlan slice_plan(int M, int N, int K, int nb, bool rows) {
  const int before = fstu_gemm_bf16_slices(M, N, K, nb);
  if (M < 256 || N % 4 != 0 || K % 64 != 0 || K < 2048) return {before, SMALL};
  const long long cus = gemm_cus();
  const long long small = tiles_of(128, M, N) * nb, big = tiles_of(256, M, N) * nb;
  const int nkt = K / 64;
  const auto join = [&](int s) { return s == 1 ? 0.0 : 3.0 + 8e-6 / 4.0 * s * nb * (double)M * N; };
  const auto large = [&](int s) {
    const long long rounds = (big * s + cus - 1) / cus;
    const double full = (double)(big * s) / (double)(rounds * cus);
    return rounds * (nkt / s) * (1.0 + 0.35 * full * full) + join(s);
  };
  const auto little = [&](int s) {
    if (small * s <= cus) return nkt / s * 0.43 + join(s);
    const long long rounds = (small * s + 2 * cus - 1) / (2 * cus);
    return rounds * (nkt / s) * (0.55 + (s == 1 ? 0.5 : 0.35) * (double)(small * s) / (double)(rounds * 2 * cus)) + join(s);
  };
  const bool half_whole = rows && half_takes(M, N), large_whole = !half_whole && pp_takes(0, K, big, small);
  double least = 0.95 * (!rows && before == 1 && 9 * ((big + cus - 1) / cus) * cus < 4 * small ? large(1) : little(before));
  SlicePlan best = {before, SMALL};
  for (int s = 2; s <= 32 && K / s >= 512 && big * s <= 2 * cus; ++s) {
    if (nkt % s != 0) continue;
    const double us = large(s);
    if (us < least) { least = us; best = {s, LARGE}; }
  }
  if (!rows) return best;
  const long long halves = (long long)((M + 255) / 256) * ((N + 127) / 128);
  if (best.on == SMALL && halves <= cus) {
    // (what the products that it is compared with take, a little closer than to rank them among each other)
    const double full = (double)(small * before) / (double)cus;
    least = 0.93 * (small * before > cus ? 0.93 * little(before) : 4.0 + nkt / before * (0.43 + 0.12 * full * full) + join(before));
    for (int s = half_whole ? 1 : 2; s <= 32 && (s == 1 || nkt / s >= 16) && halves * s <= cus; ++s) {
      const double f = (double)(halves * s) / (double)cus;
      const int n = (nkt + s - 1) / s;
      const double us = 5.0 + n * (0.55 + 0.11 * f + (n > 128 ? 0.25 * f * f * f * f : 0.0)) + (s == 1 ? 0.0 : 3.0 + 8e-6 / 6.0 * s * (double)M * N);
      if (us < least) { least = us; best = {s, HALF}; }
    }
  }
  if (best.on == SMALL || best.count == 1 || before > 1 || !(half_whole ? (long long)M * K <= 100 << 20 : large_whole)) return best;
  const auto beyond = [](int n, int from, int over) { return std::min(1.0, std::max(0, n - from) / (double)over); };
  const auto us = [&](TileKind on, int s) {
    const double joined = s == 1 ? 0.0 : 7.0 + (on == LARGE ? 1e-6 : 0.8e-6) * s * (double)M * N;
    const int n = (nkt + s - 1) / s;
    if (on == HALF) {
      const double f = (double)(halves * s) / (double)cus;
      return 4.0 + n * (0.53 + 0.09 * f + f * f * f * f * (0.08 + 0.12 * beyond(n, 96, 288))) + joined;
    }
    const long long rounds = (big * s + cus - 1) / cus;
    const double f = (double)(big * s) / (double)(rounds * cus);
    return 5.0 + rounds * n * (0.9 + f * f * (0.36 + 0.19 * f * f * beyond(n, 32, 96))) + joined;
  };
  const TileKind whole = half_whole ? HALF : LARGE;
  if (us(whole, 1) * (half_whole ? 1.02 : nkt <= 192 ? 0.94 : 0.97) <= us(best.on, best.count)) return {1, whole};
  return best;
}

}  // namespace

extern "C" int fstu_gemm_bf16_row_slices(int M, int N, int K) { return slice_plan(M, N, K, 1, true).count; }
extern "C" int fstu_gemm_bf16_slab_slices(int M, int N, int K, int nbatch) {
  return M % 256 == 0 ? slice_plan(M, N, K, nbatch, false).count : fstu_gemm_bf16_slices(M, N, K, nbatch);
}

// slices as fstu_gemm_bf16_row_slices plans them, which need not be of one length, or any number that divides K's tiles of 64
extern "C" int fstu_gemm_bf16_splitk(const void* A, int64_t lda, const void* W, float* partial, int M, int N, int K, int ksplit,
                                     void* stream) {
  FSTU_REQUIRE(A && W && partial, FSTU_ENULL, "fstu_gemm_bf16_splitk: null pointer");
  const SlicePlan plan = slice_plan(M, N, K, 1, true);
  const bool as_planned = plan.count == ksplit && M > 32, half = as_planned && plan.on == HALF;
  FSTU_REQUIRE(ksplit >= 1 && ksplit <= 64 && (half || K % (64 * ksplit) == 0), FSTU_ESHAPE,
               "fstu_gemm_bf16_splitk: K=%d must be a multiple of 64*ksplit (ksplit=%d, 1..64), or ksplit that of fstu_gemm_bf16_row_slices", K, ksplit);
  FSTU_REQUIRE(M >= 1 && N >= 4 && N % 4 == 0 && lda >= K && lda % 8 == 0, FSTU_ESHAPE,
               "fstu_gemm_bf16_splitk: M=%d N=%d (N %% 4 == 0) lda=%lld", M, N, (long long)lda);
  FSTU_REQUIRE(fstu_aligned(A, 16) && fstu_aligned(W, 16) && fstu_aligned(partial, 16), FSTU_EALIGN,
               "fstu_gemm_bf16_splitk: pointers must be 16-byte aligned");
  FSTU_REQUIRE(lda < GM_MAX_LD && K < GM_MAX_LD, FSTU_ESHAPE, "fstu_gemm_bf16_splitk: lda=%lld / K=%d beyond the 32-bit tile offsets",
               (long long)lda, K);
  int rc;
  if (M <= 32) rc = gemm_launch_tile<TileRows32, 3>(A, lda, W, nullptr, nullptr, 0, partial, N, M, N, K, (hipStream_t)stream, ksplit);
  else if (half) rc = gemm_half_launch<3>(A, lda, W, nullptr, 0, partial, N, M, N, K, (hipStream_t)stream, ksplit);
  else if (as_planned && plan.on == LARGE)
    rc = gemm_pp_launch<3>(A, lda, W, nullptr, nullptr, 0, partial, N, M, N, K, (hipStream_t)stream, ksplit);
  else if ((long long)((M + 127) / 128) * ((N + 127) / 128) * ksplit <= gemm_cus())
    rc = gemm_launch_tile<TileDeep, 3>(A, lda, W, nullptr, nullptr, 0, partial, N, M, N, K, (hipStream_t)stream, ksplit);
  else rc = gemm_launch_tile<TileSmall, 3>(A, lda, W, nullptr, nullptr, 0, partial, N, M, N, K, (hipStream_t)stream, ksplit);
  if (rc) return rc;
  FSTU_CHECK_LAUNCH("fstu_gemm_bf16_splitk");
  return FSTU_OK;
}

// fp32 slices (ns, nb, M, N) added in order -> C[b] = T(sum), or T(R[b] + T(sum)): bound by the slices' bytes
__global__ void __launch_bounds__(256)
join_slices_kernel(const float* __restrict__ part, int ns, const bf16_t* R, long long ldr, long long sr, bf16_t* C, long long ldc,
                   long long sc, int M, int n4, unsigned groups) {
  const unsigned i = blockIdx.x * 256u + threadIdx.x;
  if (i >= groups) return;
  const unsigned row = i / (unsigned)n4, c = (i - row * (unsigned)n4) * 4, b = row / (unsigned)M, m = row - b * (unsigned)M;
  const float4* p = (const float4*)part + i;
  uint2 rv = make_uint2(0, 0);
  if (R) rv = *(const uint2*)(R + (size_t)b * sr + (size_t)m * ldr + c);
  float4 t = p[0];
#pragma unroll 4
  for (int s = 1; s < ns; ++s) {
    const float4 v = p[(size_t)s * groups];
    t.x += v.x; t.y += v.y; t.z += v.z; t.w += v.w;
  }
  if (R) {
    t.x = __uint_as_float(rv.x << 16) + rnd_bf16(t.x);
    t.y = __uint_as_float(rv.x & 0xffff0000u) + rnd_bf16(t.y);
    t.z = __uint_as_float(rv.y << 16) + rnd_bf16(t.z);
    t.w = __uint_as_float(rv.y & 0xffff0000u) + rnd_bf16(t.w);
  }
  *(uint2*)(C + (size_t)b * sc + (size_t)m * ldc + c) = make_uint2(pack2_bf16(t.x, t.y), pack2_bf16(t.z, t.w));
}
static int fstu_join_slices(const float* part, int ns, const void* R, long long ldr, long long sr, void* C, long long ldc, long long sc,
                            int nb, int M, int N, void* stream) {
  const long long groups = (long long)nb * M * (N / 4);
  FSTU_REQUIRE(groups < (1ll << 31), FSTU_ESHAPE, "fstu_gemm: %lld groups of slices", groups);
  hipLaunchKernelGGL(join_slices_kernel, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, (hipStream_t)stream, part, ns, (const bf16_t*)R,
                     ldr, sr, (bf16_t*)C, ldc, sc, M, N / 4, (unsigned)groups);
  FSTU_CHECK_LAUNCH("fstu_gemm: slices");
  return FSTU_OK;
}

// Rows of a plain or residual product that whole rounds of 256 x 256 tiles take (0: no split).  A last round of few large tiles
// costs nearly what a full one does; its rows by themselves run in slices of K or on small tiles, of which the chip holds as many at
// once as there are compute units.  us in one launch / split, rows x features x K: 9600 x 2048 x 24576 970 / 687, 8500 x 2048 x 24576
// 1029 / 590, 10500 x 2048 x 24576 971 / 739, 13500 1024 / 959, 17000 1490 / 1152, 20480 1502 / 1369, 22500 x 768 x 9216 409 / 237, 3000 x 6144 x 2048 83 / 65, 10240 x 2048 x 2048 81 /
// 73, 22500 x 768 x 768 42 / 37, 33000 x 512 x 512 31 / 28.  The line: 14500 x 2048 x 24576 (no slices of the rest) 1041 / 1015, below K
// = 2048 26000 x 768 x 768 (204) 38.5 / 39.3, 18500 x 1024 x 1024 (136) 44.9 / 43.1.  The dearest rest are 1 to 32 rows of a long K, which
// take no slices: 8200 x 2048 x 24576 1021 / 641, of which the 8 rows alone 108, but 8232 573 and 22; 21768 x 768 x 9216 396 / 248.
extern "C" int fstu_gemm_bf16_head_rows(int M, int N, int K) {
  if (M <= 256 || N < 256 || N % 4 != 0 || K % 64 != 0 || K < 512) return 0;
  const long long cus = gemm_cus(), nt = (N + 255) / 256, tiles = (long long)((M + 255) / 256) * nt;
  const long long head = tiles / cus * cus / nt * 256;
  if (head <= 0 || head >= M) return 0;
  const long long left = (M - head + 127) / 128 * ((N + 127) / 128);
  const SlicePlan rest = slice_plan((int)(M - head), N, K, 1, true);
  // (a rest that is whole on large tiles takes a round either way: 9587 x 6144 x 6144 498 split, 481 in one launch; 11157 x 2304 x 12288 485, 502)
  if (left <= (K < 2048 ? cus / 2 : cus) || rest.on == HALF || (rest.on == LARGE && (rest.count > 1 || K >= 12288))) return (int)head;
  return 0;
}

extern "C" int fstu_gemm_bf16(const void* A, int64_t lda, const void* W, const void* W2, const void* R, int64_t ldr, void* C,
                              int64_t ldc, int M, int N, int K, int mode, void* stream) {
  return fstu_gemm_bf16_ws(A, lda, W, W2, R, ldr, C, ldc, M, N, K, mode, nullptr, 1, stream);
}
// modes 0 and 2 with K in ksplit slices (partial: ksplit * M * N fp32), which a second launch adds
extern "C" int fstu_gemm_bf16_ws(const void* A, int64_t lda, const void* W, const void* W2, const void* R, int64_t ldr, void* C,
                                 int64_t ldc, int M, int N, int K, int mode, float* partial, int ksplit, void* stream) {
  FSTU_REQUIRE(A && W && C, FSTU_ENULL, "fstu_gemm_bf16: null pointer");
  FSTU_REQUIRE(mode >= 0 && mode <= 2, FSTU_EARG, "fstu_gemm_bf16: mode %d", mode);
  FSTU_REQUIRE((mode != 1 || W2) && (mode != 2 || R), FSTU_ENULL, "fstu_gemm_bf16: mode %d needs its second operand", mode);
  FSTU_REQUIRE(M >= 1 && N >= 1 && (mode == 0 || N % 4 == 0) && K >= 32 && K % 32 == 0, FSTU_ESHAPE,
               "fstu_gemm_bf16: need K %% 32 == 0 and, in modes 1 and 2, N %% 4 == 0 (M=%d N=%d K=%d)", M, N, K);
  FSTU_REQUIRE(lda >= K && lda % 8 == 0 && ldc >= N && (mode == 0 || ldc % 4 == 0) && (mode != 2 || (ldr >= N && ldr % 4 == 0)), FSTU_ESHAPE,
               "fstu_gemm_bf16: row strides (lda=%lld ldc=%lld ldr=%lld)", (long long)lda, (long long)ldc, (long long)ldr);
  FSTU_REQUIRE(fstu_aligned(A, 16) && fstu_aligned(W, 16) && fstu_aligned(W2, 16) && fstu_aligned(C, mode == 0 ? 2 : 8) && fstu_aligned(R, 8),
               FSTU_EALIGN, "fstu_gemm_bf16: pointers must be 16-byte aligned (C, R: 8; C in mode 0: 2)");
  FSTU_REQUIRE(lda < GM_MAX_LD && K < GM_MAX_LD, FSTU_ESHAPE, "fstu_gemm_bf16: lda=%lld / K=%d beyond the 32-bit tile offsets",
               (long long)lda, K);
  int rc;
  if (ksplit > 1) {
    FSTU_REQUIRE(mode != 1 && ldc % 4 == 0 && fstu_aligned(C, 8), FSTU_ESHAPE, "fstu_gemm_bf16_ws: slices in modes 0 and 2, ldc %% 4 == 0");
    rc = fstu_gemm_bf16_splitk(A, lda, W, partial, M, N, K, ksplit, stream);
    if (rc) return rc;
    return fstu_join_slices(partial, ksplit, mode == 2 ? R : nullptr, ldr, 0, C, ldc, 0, 1, M, N, stream);
  }
  if (mode == 0) rc = gemm_launch<0>(A, lda, W, W2, R, ldr, C, ldc, M, N, K, (hipStream_t)stream);
  else if (mode == 1) rc = gemm_launch<1>(A, lda, W, W2, R, ldr, C, ldc, M, N, K, (hipStream_t)stream);
  else rc = gemm_launch<2>(A, lda, W, W2, R, ldr, C, ldc, M, N, K, (hipStream_t)stream);
  if (rc) return rc;
  FSTU_CHECK_LAUNCH("fstu_gemm_bf16");
  return FSTU_OK;
}

static int split_check(const char* name, int N, int K, int ksplit, const void* partial) {
  FSTU_REQUIRE(partial && fstu_aligned(partial, 16), FSTU_EALIGN, "%s: partial must be 16-byte aligned", name);
  FSTU_REQUIRE(ksplit >= 1 && ksplit <= 64 && K % (64 * ksplit) == 0 && N % 4 == 0, FSTU_ESHAPE,
               "%s: K=%d must be a multiple of 64*ksplit (ksplit=%d, 1..64), N=%d of 4", name, K, ksplit, N);
  return FSTU_OK;
}

// C[b] = T(A[b]^T W^T) (mode 0) or T(R[b] + T(A[b]^T W^T)) (mode 2) for nbatch slabs A[b] of shape (K, M) with row
// stride lda (elements; the reduction index slowest, M contiguous), W (N, K) row-major.  M must be a multiple of 128.
extern "C" int fstu_gemm_bf16_ta(const void* A, int64_t lda, int64_t batch_stride_a, const void* W, const void* R, int64_t ldr,
                                 int64_t batch_stride_r, void* C, int64_t ldc, int64_t batch_stride_c, int M, int N, int K,
                                 int nbatch, int mode, void* stream) {
  return fstu_gemm_bf16_ta_ws(A, lda, batch_stride_a, W, R, ldr, batch_stride_r, C, ldc, batch_stride_c, M, N, K, nbatch, mode, nullptr, 1,
                              stream);
}
// the same with K in ksplit slices (partial: ksplit * nbatch * M * N fp32), which a second launch adds
extern "C" int fstu_gemm_bf16_ta_ws(const void* A, int64_t lda, int64_t batch_stride_a, const void* W, const void* R, int64_t ldr,
                                    int64_t batch_stride_r, void* C, int64_t ldc, int64_t batch_stride_c, int M, int N, int K,
                                    int nbatch, int mode, float* partial, int ksplit, void* stream) {
  FSTU_REQUIRE(A && W && C, FSTU_ENULL, "fstu_gemm_bf16_ta: null pointer");
  FSTU_REQUIRE(mode == 0 || mode == 2, FSTU_EARG, "fstu_gemm_bf16_ta: mode %d (0: plain, 2: residual add)", mode);
  FSTU_REQUIRE(mode != 2 || R, FSTU_ENULL, "fstu_gemm_bf16_ta: mode 2 needs R");
  FSTU_REQUIRE(M >= 128 && M % 128 == 0 && N >= 4 && N % 4 == 0 && K >= 64 && K % 64 == 0 && nbatch >= 1, FSTU_ESHAPE,
               "fstu_gemm_bf16_ta: need M %% 128 == 0, N %% 4 == 0, K %% 64 == 0 (M=%d N=%d K=%d nbatch=%d)", M, N, K, nbatch);
  FSTU_REQUIRE(lda >= M && lda % 8 == 0 && ldc >= N && ldc % 4 == 0 && (mode != 2 || (ldr >= N && ldr % 4 == 0)), FSTU_ESHAPE,
               "fstu_gemm_bf16_ta: row strides (lda=%lld ldc=%lld ldr=%lld)", (long long)lda, (long long)ldc, (long long)ldr);
  // 32-bit byte offsets inside a slab (buffer addressing) and inside W
  FSTU_REQUIRE((unsigned long long)K * (unsigned long long)lda * 2ull < 0xfff00000ull && (unsigned long long)N * K * 2ull < 0xfff00000ull,
               FSTU_ESHAPE, "fstu_gemm_bf16_ta: a slab (K*lda) or W (N*K) exceeds 4 GB of 32-bit offsets");
  FSTU_REQUIRE(lda < GM_MAX_LD && K < GM_MAX_LD, FSTU_ESHAPE, "fstu_gemm_bf16_ta: lda=%lld / K=%d beyond the 32-bit tile offsets",
               (long long)lda, K);
  FSTU_REQUIRE(batch_stride_a % 8 == 0 && batch_stride_c % 4 == 0 && batch_stride_r % 4 == 0, FSTU_ESHAPE,
               "fstu_gemm_bf16_ta: batch strides must keep the alignment");
  FSTU_REQUIRE(fstu_aligned(A, 16) && fstu_aligned(W, 16) && fstu_aligned(C, 8) && fstu_aligned(R, 8), FSTU_EALIGN,
               "fstu_gemm_bf16_ta: pointers must be 16-byte aligned (C, R: 8)");
  hipStream_t s = (hipStream_t)stream;
  int rc;
  if (ksplit > 1) {
    if ((rc = split_check("fstu_gemm_bf16_ta_ws", N, K, ksplit, partial))) return rc;
    const SlicePlan plan = slice_plan(M, N, K, nbatch, false);
    if (M % 256 == 0 && plan.on == LARGE && plan.count == ksplit)
      rc = gemm_pp_launch<3, true>(A, lda, W, nullptr, nullptr, 0, partial, N, M, N, K, s, ksplit * nbatch, batch_stride_a, 0, 0, nbatch);
    else rc = gemm_ta_launch_tile<TileSmall, 3>(A, lda, batch_stride_a, W, partial, 0, 0, C, 0, 0, M, N, K, nbatch, s, ksplit);
    if (rc) return rc;
    FSTU_CHECK_LAUNCH("fstu_gemm_bf16_ta_ws");
    return fstu_join_slices(partial, ksplit, mode == 2 ? R : nullptr, ldr, batch_stride_r, C, ldc, batch_stride_c, nbatch, M, N, stream);
  }
#define TA_GO(TILE)                                                                                                              \
  (mode == 0 ? gemm_ta_launch_tile<TILE, 0>(A, lda, batch_stride_a, W, R, ldr, batch_stride_r, C, ldc, batch_stride_c, M, N, K,  \
                                            nbatch, s)                                                                           \
             : gemm_ta_launch_tile<TILE, 2>(A, lda, batch_stride_a, W, R, ldr, batch_stride_r, C, ldc, batch_stride_c, M, N, K,  \
                                            nbatch, s))
  // The line between the tiles is gemm_launch's, but that a round of large tiles, whose transposing reads cost the loop more, is 1.25 of the
  // small ones' up to a K of 8192: us, large / small, 128 large tiles and just one round of small ones, 4 x 4096 x 512 x 1024 24.1 / 22.1,
  // x 4096 68.3 / 67.0, x 12288 223 / 232; a few more, 1 x 5632 x 1536 x 1024 24.4 / 32.1.  Large / 128 x 128 tiles (or 256 x 256 tiles all in step, the form before), us,
  // K = 24 N: 4 x 8192 x 1024 (512 large tiles) 1155 / 1475, 2 x 8192 x 1024 (256) 547 / 833, 4 x 8192 x 768 (384) 758 / 880,
  // 4 x 8192 x 512 (256) 295 / 458, 4 x 2048 x 1024 (128) 432 / 453, 1 x 8192 x 1024 (128) 443 / 440, 1 x 4096 x 768 (48) 176 / 179.
  if (M % 256 == 0 && pp_takes(0, K, tiles_of(256, M, N) * nbatch, tiles_of(128, M, N) * nbatch, true))
    rc = mode == 0 ? gemm_pp_launch<0, true>(A, lda, W, nullptr, R, ldr, C, ldc, M, N, K, s, nbatch, batch_stride_a, batch_stride_c, batch_stride_r)
                   : gemm_pp_launch<2, true>(A, lda, W, nullptr, R, ldr, C, ldc, M, N, K, s, nbatch, batch_stride_a, batch_stride_c, batch_stride_r);
  else rc = TA_GO(TileSmall);
#undef TA_GO
  if (rc) return rc;
  FSTU_CHECK_LAUNCH("fstu_gemm_bf16_ta");
  return FSTU_OK;
}

// Slices of K for fstu_gemm_bf16_tt, any number of k tiles to each: the least of an estimate, a chain of k tiles at 0.6 us alone on a
// compute unit and 0.86 two to a unit, and the join as in fstu_gemm_bf16_slices.  us, joined, with the slices it picks / one fewer / one
// more (or the next tried) / the transpose and fstu_gemm_bf16_ta in slices of one length, rows x features x K: 768 x 768 x 16384 32.3 (7) /
// 34.2 / 36.4 / 50.5, x 8192 22.3 (7) / 23.1 / 26.3 / 34.1, 512 x 512 x 4096 15.7 (8) / 15.3 / 15.3 / 22.9, 256 x 256 x 16384 17.2 (32) / 16.7
// (28) / - / 24.3, 768 x 768 x 1024 12.3 (1) / - / 13.4 / 18.2, 1024 x 1024 x 16384 43.9 (8) / 45.1 / 53.1 (10) / 63.8, 2048 x 2048 x 16384
// 135.6 (2) / 166.6 / 143.8 / 138.1.
extern "C" int fstu_gemm_bf16_tt_slices(int M, int N, int K) {
  if (M % 128 != 0 || N % 128 != 0 || M < 1 || N < 1 || K < 1) return 1;
  const long long cus = gemm_cus(), tiles = (long long)(M / 128) * (N / 128);
  const int nkt = (K + 63) / 64;
  double least = 1e30;
  int best = 1;
  for (int s = 1; s <= 32 && s <= nkt && (s == 1 || tiles * s <= 2 * cus); ++s) {
    const double us = (nkt + s - 1) / s * (tiles * s <= cus ? 0.6 : 0.86 * (double)((tiles * s + 2 * cus - 1) / (2 * cus))) + (s == 1 ? 0.0 : 3.0 + 8e-6 / 4.0 * s * (double)M * N);
    if (us < least) { least = us; best = s; }
  }
  return best;
}

// C[m, n] = T(sum_k A[k, m] W[k, n]) for A (K, M) and W (K, N), rows of lda and ldw elements, M and N multiples of 128, in
// ksplit slices of K (partial: ksplit * M * N fp32), which a second launch adds
extern "C" int fstu_gemm_bf16_tt(const void* A, int64_t lda, const void* W, int64_t ldw, void* C, int64_t ldc, int M, int N, int K,
                                 float* partial, int ksplit, void* stream) {
  FSTU_REQUIRE(A && W && C, FSTU_ENULL, "fstu_gemm_bf16_tt: null pointer");
  FSTU_REQUIRE(M >= 128 && M % 128 == 0 && N >= 128 && N % 128 == 0 && K >= 1, FSTU_ESHAPE,
               "fstu_gemm_bf16_tt: need M %% 128 == 0, N %% 128 == 0 (M=%d N=%d K=%d)", M, N, K);
  FSTU_REQUIRE(lda >= M && lda % 8 == 0 && ldw >= N && ldw % 8 == 0 && ldc >= N && ldc % 4 == 0, FSTU_ESHAPE,
               "fstu_gemm_bf16_tt: row strides (lda=%lld ldw=%lld ldc=%lld)", (long long)lda, (long long)ldw, (long long)ldc);
  // 32-bit byte offsets inside both operands (buffer addressing)
  FSTU_REQUIRE(lda < GM_MAX_LD && ldw < GM_MAX_LD && (unsigned long long)K * (unsigned long long)std::max(lda, ldw) * 2ull < 0xfff00000ull,
               FSTU_ESHAPE, "fstu_gemm_bf16_tt: an operand exceeds 4 GB of 32-bit offsets");
  FSTU_REQUIRE(fstu_aligned(A, 16) && fstu_aligned(W, 16) && fstu_aligned(C, 8), FSTU_EALIGN,
               "fstu_gemm_bf16_tt: pointers must be 16-byte aligned (C: 8)");
  hipStream_t s = (hipStream_t)stream;
  int rc;
  if (ksplit > 1) {
    FSTU_REQUIRE(partial && fstu_aligned(partial, 16) && ksplit <= 64 && ksplit <= (K + 63) / 64, FSTU_ESHAPE, "fstu_gemm_bf16_tt: %d slices of K=%d", ksplit, K);
    rc = gemm_ta_launch_tile<TileSmall, 3, true>(A, lda, 0, W, partial, 0, 0, C, 0, 0, M, N, K, 1, s, ksplit, ldw);
    if (rc) return rc;
    FSTU_CHECK_LAUNCH("fstu_gemm_bf16_tt");
    return fstu_join_slices(partial, ksplit, nullptr, 0, 0, C, ldc, 0, 1, M, N, stream);
  }
  rc = gemm_ta_launch_tile<TileSmall, 0, true>(A, lda, 0, W, nullptr, 0, 0, C, ldc, 0, M, N, K, 1, s, 1, ldw);
  if (rc) return rc;
  FSTU_CHECK_LAUNCH("fstu_gemm_bf16_tt");
  return FSTU_OK;
}
