// Prefill on gfx950: the target forward over a long prompt chunk (hundreds to thousands of rows),
// where every projection is a compute-bound GEMM and attention is causal.
//
// The decode kernels stream each weight once per call and suit M <= 64 rows; a 4096-token prompt
// through them re-reads every weight 64 times. Here (reference ssd/engine/speculative.py:149-151,
// the target's forward over the prompt):
//
// * prefill_gemm4_kernel: Y = X W^T over the same packed weights as the decode GEMMs (16 x 32 MFMA
//   A-operand tiles, any tile grouping) with v_mfma_f32_16x16x32_bf16: 4-wave workgroups with output
//   tiles from 32 x 32 to 256 x 256 chosen by the call's M, N and K (pick_prefill_tile), accumulators
//   pinned to the accumulator registers, operands loaded straight into LDS rings, outputs staged
//   through LDS and stored as 16-byte pieces. The decode epilogues run on the staged tile: SwiGLU for
//   gate/up (gate / up rows r and r + 8 meet through one v_permlane32_swap), residual add for o and
//   down, RoPE + KV-cache write for q/k/v; the folded RMSNorm scale comes from a row-scale pass. The
//   launch is persistent and XCD-aware: the workgroups resident on one XCD sweep neighbouring output
//   tiles together, so the weight and activation tiles they share are fetched into that XCD's L2 once.
//   4096 rows of the 8B shapes, us (before the memory operations were spread between the MFMAs, the
//   addresses made scalar and X loaded by whole lines): gate/up 728 (875), down 359 (427), o 111 (132),
//   q/k/v 183 (227): 0.52 of the MFMA peak at gate/up and down. Taking the loads out of the loop gives
//   down 230 us: the loads' path through L2 bounds the large tiles; small ones are bound by a step's
//   chain of barrier, MFMAs and LDS reads.
// * prefill_attention_kernel: causal flash attention, one wave per (q head, 16 or 32 tokens), K/V read
//   in the cache's 64-slot MFMA-operand blocks; S^T = K Q^T and O^T = V^T P^T on MFMA with the
//   running max / sum rescaled per 64-key block.
// * ssd_prefill: the whole target forward for one chunk of prompt rows in one C call.
//
// Prefill rows are not required to be bit-identical to the same rows decoded one by one: greedy
// speculative decoding and greedy autoregressive decoding both start from the same prefill, and
// the decode kernels keep their batch invariance among themselves.
#include "gemm_epi.h"

#include <math.h>

#include <type_traits>

namespace ssd {

// Tile (nb, kb) of a packed weight with `group` row tiles per k-block group: 64 lanes x 16 B.
__device__ __forceinline__ size_t packed_tile(int nb, int kb, int kbt, int group) {
  return ((size_t)(nb / group) * kbt + kb) * group + nb % group;
}

// ------------------------------------------------------------------ the GEMM
// One workgroup of 4 waves owns a 32 XT (N) x 32 YT (M) output tile; wave (wn, wm) computes
// 16 XT x 16 YT of it, XT YT accumulator tiles held in the accumulator registers. Operands reach LDS
// by direct global-to-LDS loads, 16 bytes per lane: a packed W tile (one contiguous KiB), or 8 tokens
// x 64 k of X (eight whole 128-byte lines; the eight 16-byte pieces of token r's line land at
// positions p ^ (r & 7), so that the fragment reads, 16 tokens x one piece, hit every LDS bank
// equally). A step is KU k-blocks of 32; W is kept in a ring of NS step slots, X in a ring of XU units
// of 64 k, both loaded AHEAD = NS - 1 steps before their MFMAs. Step s: wait until this wave's loads
// for step s + 1 have landed (those of the AHEAD - 2 steps after it may still run) and pass one barrier;
// run step s's MFMAs on the fragments read one step earlier, and between them -- a few after every
// row of MFMAs, so that neither the LDS nor the address unit holds back the next MFMA -- read step
// s + 1's fragments and issue loads: W of step s + AHEAD into the slot that held step s - 1, and of X, with
// KU = 2, that step's unit, with KU = 1 (AHEAD = 3) half of unit s / 2 + 2, which replaces unit
// s / 2 - 1. A slot's last fragments were read in the step before its last MFMAs, which waited for
// them before this step's barrier. Waves' global addresses are
// scalar pointers plus one 32-bit lane offset, ring positions scalar offsets. The step body takes its
// LDS areas as restrict pointers, which lets the compiler see that the fragment reads do not touch
// the areas being loaded (otherwise it waits for every load in flight before each LDS read). Every
// output element is one chain of MFMAs over k in ascending order whatever the tile shape, so all
// shapes give the same bits.
typedef __attribute__((address_space(3))) u32x4_t lds_u32x4;
typedef __attribute__((address_space(3))) unsigned char lds_byte;
typedef __attribute__((address_space(3))) void lds_void;

// Sizes of one tile shape. LDS holds the two operand rings during the k loop and the staged output
// tile (BM rows of ROW bf16) plus the row scales after it.
template <int EPI, int XT, int YT, int KU, int NS>
struct P4 {
  static constexpr int BN = 32 * XT, BM = 32 * YT;
  static constexpr int LW = XT * KU / 2, LX = YT * KU / 2, PER = LW + LX;  // loads per wave and step
  static constexpr int WSLOT = 2 * XT * KU * 1024, XUNIT = BM * 128;
  static constexpr int AHEAD = NS - 1;
  static constexpr int XU = KU == 1 ? 3 : NS;  // X units: steps of one k-block load half a unit each
  static constexpr int X_OFF = NS * WSLOT, RING = X_OFF + XU * XUNIT;
  static constexpr int COLS = EPI == EPI_SWIGLU ? BN / 2 : BN;  // staged columns
  static constexpr int ROW = COLS + 8;
  static constexpr int RN_OFF = BM * ROW * 2;
  static constexpr int STAGE = RN_OFF + BM * 4;
  static constexpr int LDS = RING > STAGE ? RING : STAGE;
  static_assert(KU == 2 || (KU == 1 && NS == 4), "an X unit is two k-blocks");
  static_assert((AHEAD - 1) * PER < 64, "vmcnt");
  static_assert(XT * KU % 2 == 0 && YT * KU % 2 == 0, "each wave loads whole tiles");
  static_assert(LDS <= 163840, "160 KiB of LDS");
};

template <int XT, int YT, int KU>
struct P4Frag {
  u32x4_t a[KU][XT], b[KU][YT];
};

// The k loop's MFMAs are written as inline assembly with the accumulators bound to the accumulator
// registers ("a"): left to the register allocator, some of the accumulator values land in vector
// registers and are copied in and out around their MFMAs, which costs up to half the loop's rate
// depending on the epilogue compiled after it. The accumulators are zeroed ahead of the first
// barrier; p4_drain() puts the wait states before the epilogue reads them.
__device__ __forceinline__ void mfma_acc(f32x4_t& c, const u32x4_t& a, const u32x4_t& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

template <int XT, int YT>
__device__ __forceinline__ void p4_drain(f32x4_t (&acc)[XT][YT]) {
  // the epilogue's reads of every accumulator depend on these statements, which follow the wait
  // states (more than the 16x16x32 MFMA's write latency) in program order
  asm volatile("s_nop 15\n\ts_nop 15" : "+a"(acc[0][0]));
#pragma unroll
  for (int x = 0; x < XT; ++x)
#pragma unroll
    for (int y = 0; y < YT; ++y)
      if (x | y) asm volatile("" : "+a"(acc[x][y]));
}

// this wave's loads but the last LATER have landed, then the workgroup barrier (no wait for other
// memory operations)
template <int LATER>
__device__ __forceinline__ void p4_wait() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(LATER) : "memory");
}
// the same with min(later, N) steps of PER loads still running
template <int PER, int N>
__device__ __forceinline__ void p4_wait_steps(int later) {
  if constexpr (N == 0) {
    p4_wait<0>();
  } else {
    if (later >= N) p4_wait<N * PER>();
    else p4_wait_steps<PER, N - 1>(later);
  }
}

// Load i of this wave's LW + LX of one step, into its first W tile dW / X piece dX (1 KiB each).
template <int LW, int LX>
__device__ __forceinline__ void p4_load(const char* const (&wp)[LW], const char* const (&xp)[LX], uint32_t wlane,
                                        const uint32_t (&xlane)[LX], int i, lds_byte* dW, lds_byte* dX) {
  if (i < LW) __builtin_amdgcn_global_load_lds((const void*)(wp[i] + wlane), (lds_void*)(dW + i * 1024), 16, 0, 0);
  else __builtin_amdgcn_global_load_lds((const void*)(xp[i - LW] + xlane[i - LW]), (lds_void*)(dX + (i - LW) * 1024), 16, 0, 0);
}

// Read r of this wave's KU (XT + YT) fragments of a step: nW points at its first W tile, nX[u] at its
// first X tile (16 tokens, 2 KiB apart) for k-block u; lanes already added.
template <int XT, int YT, int KU>
__device__ __forceinline__ void p4_fetch(P4Frag<XT, YT, KU>& nf, const lds_byte* nW, const lds_byte* const (&nX)[KU], int r) {
  const int u = r / (XT + YT), i = r % (XT + YT);
  if (i < YT) nf.b[u][i] = *(const lds_u32x4*)(nX[u] + i * 2048);
  else nf.a[u][i - YT] = *(const lds_u32x4*)(nW + (u * 2 * XT + i - YT) * 1024);
}

// One step: MFMAs on `f`; `nf` <- the next step's fragments; this step's loads into dW / dX.
template <int XT, int YT, int KU, int LW, int LX>
__device__ __forceinline__ void p4_step(const char* const (&wp)[LW], const char* const (&xp)[LX], uint32_t wlane,
                                        const uint32_t (&xlane)[LX], bool load_w, bool load_x, lds_byte* __restrict__ dW,
                                        lds_byte* __restrict__ dX, const lds_byte* __restrict__ nW,
                                        const lds_byte* const (&nX)[KU], bool fetch,
                                        const P4Frag<XT, YT, KU>& f, P4Frag<XT, YT, KU>& nf, f32x4_t (&acc)[XT][YT]) {
  constexpr int G = KU * XT;             // rows of YT MFMAs
  constexpr int GM = G > 1 ? G - 1 : 1;  // memory operations follow all but the last row
  constexpr int R = KU * (XT + YT), L = LW + LX;
#pragma unroll
  for (int q = 0; q < G; ++q) {
    const int u = q / XT, x = q % XT;
#pragma unroll
    for (int y = 0; y < YT; ++y) mfma_acc(acc[x][y], f.a[u][x], f.b[u][y]);
    __builtin_amdgcn_sched_barrier(0);
    if (q < GM) {
      if (fetch) {
#pragma unroll
        for (int r = R * q / GM; r < R * (q + 1) / GM; ++r) p4_fetch<XT, YT, KU>(nf, nW, nX, r);
      }
#pragma unroll
      for (int i = L * q / GM; i < L * (q + 1) / GM; ++i)
        if (i < LW ? load_w : load_x) p4_load<LW, LX>(wp, xp, wlane, xlane, i, dW, dX);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// SiLU of the prefill's SwiGLU staging: x / (1 + 2^(-x log2 e)) through the hardware base-2 exponential and
// reciprocal, the quotient corrected by its residual. Both sides of the quotient carry a factor of 1/16, which
// keeps the reciprocal normal where the exponential is near 2^128 (exact for a bf16 x, subnormal ones too); the
// fixup gives the quotients by infinity (x < -88.7: -0; x = -inf: NaN). x is a rounded bf16 value and the result is
// rounded to bf16, so the whole range is 65280 finite inputs: every one gives silu_f's bf16 value, i.e. that of
// the decode kernels. Without the correction 5.9375 and -87.5 .. -88.5 did not (the last flushed to -0). The
// four instructions more cost nothing that is measured; silu_f's own division and exponential cost half of
// the gate/up tile's staging.
__device__ __forceinline__ float pf_silu(float x) {
  const float d = fmaf(__builtin_amdgcn_exp2f(x * -1.4426950408889634f), 0.0625f, 0.0625f), n = x * 0.0625f;
  const float r = __builtin_amdgcn_rcpf(d), q = n * r;
  return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, n), r, q), d, n);
}

// q/k/v write-out of one staged tile: rows of q and K-cache slots (RoPE applied here), then 8-slot
// runs of V^T. Staged column 16 t + i holds weight tile nb0 + t's row i: rotary dim p 8 + i
// (i < 8) or hd / 2 + p 8 + i - 8 (i >= 8) of its head -- both halves of each rotary pair. Thread
// t's q/k items are (token, weight tile) = divmod(t + 256 i, 2 XT), i < NI; their rotary cos / sin
// pieces are loaded by p4_qkv_rope() before the tile is staged (clamped addresses for items that
// are not q/k, so the loads are unconditional), so their latency overlaps the staging.
template <class C>
struct P4Rope {
  static constexpr int NWT = C::BN / 16, ITEMS = C::BM * NWT, NI = (ITEMS + 255) / 256;
  Pack8 cs[NI], sn[NI];
};

template <class C>
__device__ __forceinline__ void p4_qkv_rope(const GemmArgs& a, int nb0, int m0, int pos0, int t, P4Rope<C>& r) {
  constexpr int NWT = P4Rope<C>::NWT;
  const int half = a.head_dim >> 1;
#pragma unroll
  for (int i = 0; i < P4Rope<C>::NI; ++i) {
    const int it = t + 256 * i, row = it / NWT, tt = it % NWT;
    const QkvTile q = qkv_tile(a, nb0 + tt);
    const int pos = min(max(pos0 + m0 + row, 0), (int)a.rope_rows - 1);
    const size_t at = (size_t)pos * half + (q.p & (half / 8 - 1)) * 8;
    r.cs[i].u = *(const uint4*)(a.cos_tab + at);
    r.sn[i].u = *(const uint4*)(a.sin_tab + at);
  }
}

template <class C>
__device__ __forceinline__ void p4_qkv_out(const GemmArgs& a, const bf16_t* stage, int nb0, int m0, int pos0, int t,
                                           const P4Rope<C>& r) {
  constexpr int NWT = P4Rope<C>::NWT;  // weight tiles of the workgroup tile
  const int hd = a.head_dim, half = hd >> 1;
  const int n_wt = min(NWT, a.N / 16 - nb0);  // N is a multiple of 16 (q/k/v shape)
  const bool qvec = a.ldy % 8 == 0 && ((uintptr_t)a.Y & 15) == 0;
  // q and K: one (token, weight tile) per item, two 16-byte pieces (the pair's halves)
#pragma unroll
  for (int i = 0; i < P4Rope<C>::NI; ++i) {
    const int it = t + 256 * i, row = it / NWT, tt = it % NWT, m = m0 + row;
    if (it >= P4Rope<C>::ITEMS || tt >= n_wt || m >= a.M) continue;
    const QkvTile q = qkv_tile(a, nb0 + tt);
    if (q.region == 2) continue;
    Pack8 lo, hi, olo, ohi;
    lo.u = *(const uint4*)(stage + row * C::ROW + tt * 16);
    hi.u = *(const uint4*)(stage + row * C::ROW + tt * 16 + 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float xl = bf2f(lo.h[e]), xh = bf2f(hi.h[e]), c = bf2f(r.cs[i].h[e]), s = bf2f(r.sn[i].h[e]);
      olo.h[e] = f2bf(rbf(rbf(xl * c) - rbf(xh * s)));
      ohi.h[e] = f2bf(rbf(rbf(xh * c) + rbf(xl * s)));
    }
    if (q.region == 0) {
      bf16_t* qo = a.Y + (size_t)m * a.ldy + (size_t)q.head * hd + q.p * 8;
      if (qvec) {
        *(uint4*)qo = olo.u;
        *(uint4*)(qo + half) = ohi.u;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          qo[e] = olo.h[e];
          qo[half + e] = ohi.h[e];
        }
      }
    } else {
      const int slot = pos0 + m;  // inside the cache (checked on the host)
      bf16_t* kc = a.k_cache + (size_t)q.head * a.max_len * hd;
      *(uint4*)(kc + k_off(slot, q.p * 8, hd)) = olo.u;
      *(uint4*)(kc + k_off(slot, half + q.p * 8, hd)) = ohi.u;
    }
  }
  // V^T: one (8-slot run, staged column) per item; runs cut by the tile's first or last token, or by
  // M, are written element by element (the neighbouring tile writes the rest of such a run)
  const int s_lo = pos0 + m0, s_hi = pos0 + min(m0 + C::BM, a.M);  // slots [s_lo, s_hi)
  const int g_lo = s_lo >> 3, n_runs = ((s_hi + 7) >> 3) - g_lo;
  for (int it = t; it < n_runs * NWT * 16; it += 256) {
    const int run = it / (NWT * 16), c = it % (NWT * 16), tt = c >> 4, i = c & 15;
    if (tt >= n_wt) continue;
    const QkvTile q = qkv_tile(a, nb0 + tt);
    if (q.region != 2) continue;
    const int d = q.p * 8 + (i & 7) + (i >= 8 ? half : 0);
    const int s0 = (g_lo + run) * 8;
    bf16_t* vt = a.vt_cache + (size_t)q.head * hd * a.max_len;
    if (s0 >= s_lo && s0 + 8 <= s_hi) {
      Pack8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v.h[e] = stage[(s0 + e - s_lo) * C::ROW + c];
      *(uint4*)(vt + v_off(s0, d, hd)) = v.u;
    } else {
      for (int e = 0; e < 8; ++e) {
        const int s = s0 + e;
        if (s >= s_lo && s < s_hi) vt[v_off(s, d, hd)] = stage[(s - s_lo) * C::ROW + c];
      }
    }
  }
}

// OCC: workgroups per CU the registers are budgeted for.
template <int EPI, bool RS, int XT, int YT, int KU, int NS, int OCC>
__global__ __launch_bounds__(256, OCC) void prefill_gemm4_kernel(GemmArgs a, int group, int n_mt, int n_nt, int pos0,
                                                                 int band) {
  typedef P4<EPI, XT, YT, KU, NS> C;
  constexpr int LW = C::LW, LX = C::LX, PER = C::PER;
  __shared__ __align__(16) unsigned char smem[C::LDS];
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int wn = w & 1, wm = w >> 1;
  const int n_rt = (a.N + 127) / 128 * 8;
  const int kbt = a.kb_total, n_steps = kbt / KU;  // kbt is even (K % 64 == 0)
  float* rn_s = (float*)(smem + C::RN_OFF);
  bf16_t* stage = (bf16_t*)smem;  // [BM tokens][ROW] after the k loop
  // Persistent and XCD-aware: output tiles are ordered in bands of `band` row tiles, rows fastest,
  // and each XCD takes one contiguous run of that order, so the workgroups resident on it work on a
  // block of neighbouring tiles and fetch the weight and activation tiles they share into that XCD's
  // L2 once.
  const int tiles = n_mt * n_nt, xcd = blockIdx.x % 8, per_xcd = (tiles + 7) / 8;
  for (int it = blockIdx.x / 8; it < per_xcd; it += gridDim.x / 8) {
  const int tile = xcd * per_xcd + it;
  if (tile >= tiles) break;  // uniform per workgroup
  const int bnd = tile / (band * n_nt), in_band = tile - bnd * band * n_nt, hb = min(band, n_mt - bnd * band);
  const int nb0 = in_band / hb * 2 * XT, m0 = (bnd * band + in_band % hb) * C::BM;
  // Wave w loads W tiles LW w .. of every slot ([k-block][row tile]; row tiles past the weight's last
  // load that one) and 8-token pieces of X: with KU = 2, pieces LX w .. of the unit; with KU = 1,
  // pieces 2 LX w .. + LX - 1 in a unit's first step and the next LX in its second (tokens past M
  // load the last row: neither is stored).
  const char *wp[LW], *xp[KU == 1 ? 2 : 1][LX];
  uint32_t xlane[KU == 1 ? 2 : 1][LX];
#pragma unroll
  for (int r = 0; r < LW; ++r) {
    const int i = LW * w + r, nb = min(nb0 + i % (2 * XT), n_rt - 1);
    wp[r] = (const char*)a.W + (packed_tile(nb, 0, kbt, group) + (size_t)(i / (2 * XT)) * group) * 1024;
  }
  const int l8 = lane >> 3;
#pragma unroll
  for (int h = 0; h < (KU == 1 ? 2 : 1); ++h)
#pragma unroll
    for (int r = 0; r < LX; ++r) {
      const int row0 = min(m0 + 8 * (KU == 1 ? 2 * LX * w + h * LX + r : LX * w + r), a.M - 1);
      xp[h][r] = (const char*)(a.X + (size_t)row0 * a.ldx);
      xlane[h][r] = (uint32_t)(min(row0 + l8, a.M - 1) - row0) * (uint32_t)a.ldx * 2 + ((lane & 7) ^ l8) * 16;
    }
  const uint32_t wlane = lane * 16;
  const size_t wstep = (size_t)group * 1024 * KU;
  lds_byte* const lds = (lds_byte*)smem;
  lds_byte* const dw0 = lds + w * LW * 1024;                                        // this wave's load areas
  lds_byte* const dx0 = lds + C::X_OFF + w * (KU == 1 ? 2 : 1) * LX * 1024;
  // and fragments: W tiles wn XT .., X tiles wm YT .. (k-block u's piece of token j sits at
  // position (4 u + g) ^ (j & 7))
  const lds_byte* const rw0 = lds + wn * XT * 1024 + lane * 16;
  const lds_byte* const rx0 = lds + C::X_OFF + wm * YT * 2048 + j * 128;
  const uint32_t px[2] = {(uint32_t)((g ^ (j & 7)) * 16), (uint32_t)(((4 + g) ^ (j & 7)) * 16)};

  f32x4_t acc[XT][YT];
#pragma unroll
  for (int x = 0; x < XT; ++x)
#pragma unroll
    for (int y = 0; y < YT; ++y) {
      acc[x][y] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+a"(acc[x][y]));  // here, not in each path of the k loop
    }

  // Prologue: KU = 2: W and X of steps 0 .. AHEAD - 1. KU = 1: X unit 0 and W 0, then what step 0 and step 1
  // wait for one step's worth of loads after another: W 1, half of unit 1; W 2, its other half.
  auto load_x_half = [&](int h, uint32_t off) {
#pragma unroll
    for (int i = LW; i < PER; ++i)
      p4_load<LW, LX>(wp, xp[KU == 1 ? h : 0], wlane, xlane[KU == 1 ? h : 0], i, dw0,
                      dx0 + off + (KU == 1 ? h * LX * 1024 : 0));
  };
  auto load_w_step = [&](uint32_t off) {
#pragma unroll
    for (int i = 0; i < LW; ++i) p4_load<LW, LX>(wp, xp[0], wlane, xlane[0], i, dw0 + off, dx0);
#pragma unroll
    for (int r = 0; r < LW; ++r) wp[r] += wstep;
  };
  auto next_unit = [&](int h) {
#pragma unroll
    for (int r = 0; r < LX; ++r) xp[KU == 1 ? h : 0][r] += 128;
  };
  P4Frag<XT, YT, KU> f0, f1;
  if constexpr (KU == 1) {
    load_x_half(0, 0);
    load_x_half(1, 0);
    next_unit(0);
    next_unit(1);
    load_w_step(0);
    load_w_step(C::WSLOT);  // kbt is even
    if (n_steps > 2) {
      load_x_half(0, C::XUNIT);
      load_w_step(2 * C::WSLOT);
      load_x_half(1, C::XUNIT);
      next_unit(0);
      next_unit(1);
    }
    if (n_steps > 2) p4_wait<2 * PER>();
    else p4_wait<0>();
  } else {
#pragma unroll
    for (int p = 0; p < C::AHEAD; ++p)
      if (p < n_steps) {
        load_w_step(p * C::WSLOT);
        load_x_half(0, p * C::XUNIT);
        next_unit(0);
      }
    p4_wait_steps<PER, C::AHEAD - 1>(n_steps - 1);
  }
  {
    const lds_byte* nx[KU];
#pragma unroll
    for (int u = 0; u < KU; ++u) nx[u] = rx0 + px[u];
#pragma unroll
    for (int r = 0; r < KU * (XT + YT); ++r) p4_fetch<XT, YT, KU>(f0, rw0, nx, r);
  }

  // ring positions (bytes): W slots of steps s + 1 (read) and s + AHEAD (loaded); X unit of step s + 1 and
  // the one being loaded
  uint32_t wr = C::WSLOT, ww = C::AHEAD * C::WSLOT, xr = KU == 1 ? 0 : C::XUNIT,
           xw = (KU == 1 ? 2 : C::AHEAD) * C::XUNIT;
  auto next_w = [](uint32_t x) {
    x += C::WSLOT;
    return x == NS * C::WSLOT ? 0u : x;
  };
  auto next_x = [](uint32_t x) {
    x += C::XUNIT;
    return x == C::XU * C::XUNIT ? 0u : x;
  };
  // step s, H = s % 2
  auto step = [&](auto full, auto half, int s, const P4Frag<XT, YT, KU>& f, P4Frag<XT, YT, KU>& nf) {
    constexpr bool FULL = decltype(full)::value;
    constexpr int H = decltype(half)::value, HX = KU == 1 ? H : 0;
    if constexpr (FULL) p4_wait<(C::AHEAD - 2) * PER>();
    else p4_wait_steps<PER, KU == 1 ? 0 : C::AHEAD - 2>(n_steps - 2 - s);
    const lds_byte* nx[KU];
    if constexpr (KU == 1) {
      if (H == 1) xr = next_x(xr);  // step s + 1 starts a unit
      nx[0] = rx0 + xr + px[1 - H];
    } else {
      nx[0] = rx0 + xr + px[0];
      nx[KU - 1] = rx0 + xr + px[1];
    }
    // KU = 1: X unit s / 2 + 2 (its first k-block is step 2 (s / 2) + 4); KU = 2: unit s + AHEAD
    const bool load_w = FULL || s + C::AHEAD < n_steps;
    const bool load_x = FULL || (KU == 1 ? s - H + 4 < n_steps : s + C::AHEAD < n_steps);
    // the lane offsets pass through an empty asm statement, so that the addresses stay a scalar pointer
    // plus a 32-bit offset (otherwise they become a pair of vector registers for every load)
    uint32_t wl = wlane, xl[LX];
    asm volatile("" : "+v"(wl));
#pragma unroll
    for (int r = 0; r < LX; ++r) {
      xl[r] = xlane[HX][r];
      asm volatile("" : "+v"(xl[r]));
    }
    p4_step<XT, YT, KU, LW, LX>(wp, xp[HX], wl, xl, load_w, load_x, dw0 + ww,
                                dx0 + xw + HX * LX * 1024, rw0 + wr, nx, FULL || s + 1 < n_steps, f, nf, acc);
#pragma unroll
    for (int r = 0; r < LW; ++r) wp[r] += wstep;
#pragma unroll
    for (int r = 0; r < LX; ++r) xp[HX][r] += 128;
    wr = next_w(wr);
    ww = next_w(ww);
    if (KU == 2) xr = next_x(xr);
    if (KU == 2 || H == 1) xw = next_x(xw);
  };
  using yes_t = std::integral_constant<bool, true>;
  using no_t = std::integral_constant<bool, false>;
  using even_t = std::integral_constant<int, 0>;
  using odd_t = std::integral_constant<int, 1>;
  int s = 0;
  for (; s + NS < n_steps; s += 2) {
    step(yes_t{}, even_t{}, s, f0, f1);
    step(yes_t{}, odd_t{}, s + 1, f1, f0);
  }
  for (; s < n_steps; s += 2) {  // the last steps
    step(no_t{}, even_t{}, s, f0, f1);
    if (s + 1 >= n_steps) break;
    step(no_t{}, odd_t{}, s + 1, f1, f0);
  }
  p4_drain<XT, YT>(acc);
  __syncthreads();  // every wave is done with the slots: the staged tile and the scales reuse LDS

  {
    // the epilogue's thread indices pass through an empty asm statement, so that nothing computed
    // from them is hoisted above the k loop and kept live (spilled) across it
    int te = t;
    asm volatile("" : "+v"(te));
    if constexpr (RS) {
      if (te < C::BM) rn_s[te] = a.row_scale[min(m0 + te, a.M - 1)];
      __syncthreads();
    }
    const int je = te & 15, ge = (te >> 4) & 3, we = te >> 6, wne = we & 1, wme = we >> 1;
    constexpr int NIT = C::COLS / 8;              // write-out items (16 bytes) per row
    constexpr int NTH = (C::BM * NIT + 255) / 256;  // and per thread
    const int n_out = EPI == EPI_SWIGLU ? a.N / 2 : a.N;
    const int c0 = (EPI == EPI_SWIGLU ? nb0 * 8 : nb0 * 16);
    // The residual joins in the staging: lane (g, j)'s four columns of tile (x, y) are one 8-byte
    // residual piece, loaded two token tiles ahead (clamped addresses, so the loads are
    // unconditional; columns past N are never stored). The rotary tables of the q/k/v write-out are
    // loaded before the staging. Either way the loads' latency overlaps the staging.
    const bool res = EPI == EPI_STORE && a.residual && a.ldr % 4 == 0 && ((uintptr_t)a.residual & 7) == 0 &&
                     n_out % 4 == 0;  // uniform
    // 16-byte stores of staged rows (with a residual, only when the staging added it)
    const bool vec = a.ldy % 8 == 0 && ((uintptr_t)a.Y & 15) == 0 && (!a.residual || res);
    [[maybe_unused]] uint2 rq[3][EPI == EPI_STORE ? XT : 1];
    auto load_res = [&](int y, uint2 (&dst)[EPI == EPI_STORE ? XT : 1]) {
      if constexpr (EPI == EPI_STORE) {
        const int m = min(m0 + (wme * YT + y) * 16 + je, a.M - 1);
#pragma unroll
        for (int x = 0; x < XT; ++x) {
          const int n = min(c0 + (wne * XT + x) * 16 + 4 * ge, n_out - 4);
          dst[x] = *(const uint2*)(a.residual + (size_t)m * a.ldr + n);
        }
      }
    };
    [[maybe_unused]] P4Rope<C> rope;
    if constexpr (EPI == EPI_STORE) {
      if (res) {
        load_res(0, rq[0]);
        if (YT > 1) load_res(1, rq[1]);
      }
    } else if constexpr (EPI == EPI_QKV) {
      p4_qkv_rope<C>(a, nb0, m0, pos0, te, rope);
    }
    // stage: lane (g, j) of tile (x, y) holds output rows 16 (wn XT + x) + 4 g + e of token
    // 16 (wm YT + y) + j -- four consecutive columns (plain, q/k/v). For SwiGLU, rows r (gate) and
    // r + 8 (up) meet through a lane swap, after which lanes g and g + 2 hold the same four pairs:
    // lanes g < 2 finish pairs 0, 1 and lanes g >= 2 pairs 2, 3 of them (intermediate columns
    // 8 (wn XT + x) + 4 (g & 1) + 2 (g >> 1) + 0, 1).
#pragma unroll
    for (int y = 0; y < YT; ++y) {
      // one row at a time: its accumulators are first read here
#pragma unroll
      for (int x = 0; x < XT; ++x) asm volatile("" : "+a"(acc[x][y])::"memory");
      const int mr = (wme * YT + y) * 16 + je;
      const float sc = RS ? rn_s[mr] : 1.f;
      if constexpr (EPI == EPI_STORE) {
        __builtin_amdgcn_sched_barrier(0);  // keep each row's loads two rows ahead (not all hoisted)
        if (res && y + 2 < YT) load_res(y + 2, rq[(y + 2) % 3]);
      }
#pragma unroll
      for (int x = 0; x < XT; ++x) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[x][y][e] * sc;
        if constexpr (EPI == EPI_SWIGLU) {
          float gt[4], up[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[e]), __float_as_uint(v[e]), false, false);
            gt[e] = __uint_as_float(p[0]);
            up[e] = __uint_as_float(p[1]);
          }
          const bool hi = ge >= 2;
          const float g0 = hi ? gt[2] : gt[0], g1 = hi ? gt[3] : gt[1];
          const float u0 = hi ? up[2] : up[0], u1 = hi ? up[3] : up[1];
          const float o0 = rbf(pf_silu(rbf(g0))) * rbf(u0), o1 = rbf(pf_silu(rbf(g1))) * rbf(u1);
          const int col = (wne * XT + x) * 8 + 4 * (ge & 1) + 2 * (ge >> 1);
          *(uint32_t*)(stage + mr * C::ROW + col) = pack_bf16x2(o0, o1);
        } else {
          if constexpr (EPI == EPI_STORE) {
            if (res) {
              // out = bf16(residual + bf16(acc sc)), the order of the decode epilogue
              const uint2 r = rq[y % 3][x];
              const uint32_t rw[2] = {r.x, r.y};
#pragma unroll
              for (int e = 0; e < 4; ++e) v[e] = bf2f((bf16_t)(rw[e >> 1] >> (16 * (e & 1)))) + rbf(v[e]);
            }
          }
          const int col = (wne * XT + x) * 16 + 4 * ge;
          *(uint2*)(stage + mr * C::ROW + col) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
        }
      }
    }
    __syncthreads();
    if constexpr (EPI == EPI_QKV) {
      p4_qkv_out<C>(a, stage, nb0, m0, pos0, te, rope);
    } else {
      // write out: 8 columns (16 bytes) per item, a row's items on consecutive threads
      if (vec && n_out % 8 == 0) {  // uniform: every item is one whole 16-byte piece
        for (int i = 0; i < NTH; ++i) {
          const int it = te + 256 * i, row = it / NIT, c8 = (it % NIT) * 8;
          const int m = m0 + row, n = c0 + c8;
          if ((NTH * 256 != C::BM * NIT && it >= C::BM * NIT) || m >= a.M || n >= n_out) continue;
          *(uint4*)(a.Y + (size_t)m * a.ldy + n) = *(const uint4*)(stage + row * C::ROW + c8);
        }
      } else {  // element by element (unaligned output or residual, or N not a multiple of 8)
        for (int i = 0; i < NTH; ++i) {
          const int it = te + 256 * i, row = it / NIT, c8 = (it % NIT) * 8;
          const int m = m0 + row, n = c0 + c8;
          if ((NTH * 256 != C::BM * NIT && it >= C::BM * NIT) || m >= a.M || n >= n_out) continue;
          Pack8 v;
          v.u = *(const uint4*)(stage + row * C::ROW + c8);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            if (n + e >= n_out) continue;
            float r = bf2f(v.h[e]);  // the staged value already holds the residual when res
            if (EPI == EPI_STORE && a.residual && !res) r = rbf(bf2f(a.residual[(size_t)m * a.ldr + n + e]) + r);
            a.Y[(size_t)m * a.ldy + n + e] = f2bf(r);
          }
        }
      }
    }
  }
  __syncthreads();  // the next tile's loads reuse LDS
  }  // tile loop
}

// ------------------------------------------------------------------ causal flash attention
// Row (token t, q head h) at position pos0 + t attends cache slots [0, pos0 + t] (the prompt rows
// before it and itself, whose K/V the q/k/v GEMM of this chunk already wrote).
__device__ __forceinline__ int pf_perm_key(int kt, int i) {
  return (kt >> 1) * 32 + (i >> 2) * 8 + (kt & 1) * 4 + (i & 3);
}

__device__ __forceinline__ float pf_max_lanes(float v) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pf_sum_lanes(float v) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Per-wave state of the causal attention: the query fragments of NT 16-row tiles (16 NT tokens), their
// running max / sum and output accumulators, and each lane's last attended key.
template <int HD, int NT>
struct PfAttnState {
  static constexpr int KS = HD / 32, DT = HD / 16;
  u32x4_t qf[NT][KS];
  float m_run[NT], l_run[NT];
  f32x4_t o[NT][DT];
  int lim[NT];
};

// One 64-key block b for the wave's row tiles. K / V fragments come from `ck` / `cv` (the block in LDS,
// SHARED) or from the cache rows `kb` / `vb`; with SHARED the copy of block b + 1 into `nk` / `nv`
// is issued first. The LDS pointers are restrict, so the compiler sees that the fragment reads do
// not touch the buffer being filled and does not wait for that copy before them. MASKED: the block may
// hold keys past a row's own or past the tile's last (the one or two last blocks of a tile; the other
// blocks need 200 vector instructions without the masks, 340 with them: 32 heads of 4096 tokens 173 -> 143 us).
template <int HD, bool SHARED, int NT, bool MASKED>
__device__ __forceinline__ void pf_attend_block(PfAttnState<HD, NT>& st, int b, int n_blk, int last,
                                                float scale_log2, int lane, int w, const bf16_t* kb, const bf16_t* vb,
                                                const char* ksrc, const char* vsrc,
                                                const lds_u32x4* __restrict__ ck, const lds_u32x4* __restrict__ cv,
                                                lds_u32x4* __restrict__ nk, lds_u32x4* __restrict__ nv) {
  constexpr int KS = HD / 32, DT = HD / 16;
  constexpr int PIECES = 64 * HD / 8;  // 16-byte pieces of one block's K (and of its V^T)
  const int g = lane >> 4;
  if constexpr (SHARED) {
    // this block's copy landed (the only loads in flight: an explicit wait, since a workgroup
    // barrier does not wait for global-to-LDS loads) and every wave is done with the buffer the next
    // copy overwrites (it held block b - 1). The barrier is __syncthreads (not inline assembly) so
    // the compiler sees it and places its own wait for the copy there, not before the fragment reads.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (b + 1 < n_blk) {
      // wave w, load i copies pieces 256 i + 64 w + lane of block b + 1's K and V^T (scalar pointer plus
      // a 32-bit lane offset)
      const size_t off = ((size_t)(b + 1) * PIECES + 64 * w) * 16;
      const uint32_t l16 = lane * 16;
#pragma unroll
      for (int i = 0; i < PIECES / 256; ++i) {
        __builtin_amdgcn_global_load_lds((const void*)(ksrc + off + 4096 * i + l16), (lds_void*)(nk + 256 * i + 64 * w), 16,
                                         0, 0);
        __builtin_amdgcn_global_load_lds((const void*)(vsrc + off + 4096 * i + l16), (lds_void*)(nv + 256 * i + 64 * w), 16,
                                         0, 0);
      }
    }
  }
  // K first: the scores of both row tiles; V is read while the softmax runs (K and V are not live
  // together, which keeps the wave inside 256 registers)
  u32x4_t kf[4][KS];
#pragma unroll
  for (int kt = 0; kt < 4; ++kt)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if constexpr (SHARED) kf[kt][ks] = ck[(kt * KS + ks) * 64 + lane];
      else kf[kt][ks] = *(const u32x4_t*)(kb + (size_t)b * 64 * HD + (kt * KS + ks) * 512);
    }
  // k-step outer: consecutive MFMAs go to different accumulators (each sum keeps its ks order)
  f32x4_t s[NT][4];
#pragma unroll
  for (int rt = 0; rt < NT; ++rt)
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) s[rt][kt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
#pragma unroll
    for (int rt = 0; rt < NT; ++rt)
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) s[rt][kt] = mfma16x16x32(bits_bf16x8(kf[kt][ks]), bits_bf16x8(st.qf[rt][ks]), s[rt][kt]);
  u32x4_t vf[DT][2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    if constexpr (SHARED) {
      vf[dt][0] = cv[(dt * 2) * 64 + lane];
      vf[dt][1] = cv[(dt * 2 + 1) * 64 + lane];
    } else {
      vf[dt][0] = *(const u32x4_t*)(vb + (size_t)b * 64 * HD + (dt * 2) * 512);
      vf[dt][1] = *(const u32x4_t*)(vb + (size_t)b * 64 * HD + (dt * 2 + 1) * 512);
    }
  }
  if (MASKED && b == n_blk - 1) {
    // slots past the tile's last key hold whatever the cache held (not yet written): their
    // probabilities are 0, and 0 * V must stay 0, so V is zeroed there. Lane (g, i) of V tile
    // (dt, c) holds slots 64 b + 32 c + 8 g .. + 8.
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int s0 = b * 64 + c * 32 + g * 8;
      u32x4_t keep;
#pragma unroll
      for (int w2 = 0; w2 < 4; ++w2)
        keep[w2] = (s0 + 2 * w2 <= last ? 0x0000ffffu : 0u) | (s0 + 2 * w2 + 1 <= last ? 0xffff0000u : 0u);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) vf[dt][c] &= keep;
    }
  }
#pragma unroll
  for (int rt = 0; rt < NT; ++rt) {
    // Softmax in base 2 with the score scale folded into the exponent: p = 2^(s c - m), m a running
    // reference in scaled units. The reference only moves up when a block's maximum exceeds it by
    // more than 8 (so p <= 2^8 stays exact enough in fp32 and in the bf16 P operand); otherwise O
    // and l keep their scale and O is not rescaled -- for the whole wave when no row of it moved.
    // Every row attends key 0, so the first block sets a finite reference.
    float sv[16], mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = s[rt][kt][e];
        if (MASKED && b * 64 + pf_perm_key(kt, 4 * g + e) > st.lim[rt]) v = -INFINITY;
        sv[kt * 4 + e] = v;
        mx = fmaxf(mx, v);
      }
    mx = pf_max_lanes(mx) * scale_log2;
    const bool grow = mx > st.m_run[rt] + 8.f;  // true in the first block (m_run = -inf)
    const float m_use = grow ? mx : st.m_run[rt];
    const float alpha = grow ? __builtin_amdgcn_exp2f(st.m_run[rt] - mx) : 1.f;
    float l = 0.f;
    uint32_t pw[2][4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(sv[kt * 4 + e], scale_log2, -m_use));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(sv[kt * 4 + e + 1], scale_log2, -m_use));
        l += p0 + p1;
        pw[kt >> 1][(kt & 1) * 2 + e / 2] = pack_bf16x2(p0, p1);
      }
    l = pf_sum_lanes(l);
    st.l_run[rt] = fmaf(st.l_run[rt], alpha, l);  // spelled out: the masked and the plain instance must agree
    st.m_run[rt] = m_use;
    if (__builtin_amdgcn_ballot_w64(grow)) {  // wave-uniform: multiplying by alpha = 1 is exact
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) st.o[rt][dt] = st.o[rt][dt] * alpha;
    }
    const u32x4_t pb0 = {pw[0][0], pw[0][1], pw[0][2], pw[0][3]};
    const u32x4_t pb1 = {pw[1][0], pw[1][1], pw[1][2], pw[1][3]};
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) st.o[rt][dt] = mfma16x16x32(bits_bf16x8(vf[dt][0]), bits_bf16x8(pb0), st.o[rt][dt]);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) st.o[rt][dt] = mfma16x16x32(bits_bf16x8(vf[dt][1]), bits_bf16x8(pb1), st.o[rt][dt]);
  }
}

// SHARED: the workgroup's four waves are four q heads of one kv head, so each 64-key block of K and
// V^T is copied once per workgroup into LDS (direct global-to-LDS loads, 16 bytes per lane, the
// cache layout kept) one block ahead of its use, and the waves read their MFMA fragments from there;
// otherwise every wave loads its block's K and V straight into registers when it needs them. The
// fragments and their order are the same either way, so the outputs are bit-identical.
// NT: 16-row tiles per wave. Two halve the K / V fragment reads per row; one gives a short prompt twice
// the workgroups, each with half the work per block (a block then takes its chain of barrier, LDS reads,
// MFMAs and softmax, not its throughput): 32 heads of 512 tokens 18.3 us with two, 11.0 with one; 100
// tokens 8.1 and 5.6.
template <int HD, bool SHARED, int NT>
__global__ __launch_bounds__(256, 2) void prefill_attention_kernel(const bf16_t* __restrict__ Q, int64_t ldq, int M,
                                                                   int pos0, int heads, int kv_heads,
                                                                   const bf16_t* __restrict__ Kc,
                                                                   const bf16_t* __restrict__ Vt, int64_t max_len,
                                                                   float scale_log2, bf16_t* __restrict__ out,
                                                                   int64_t ldo, int n_tt) {
  constexpr int KS = HD / 32, DT = HD / 16, TOK = 16 * NT;
  constexpr int PIECES = 64 * HD / 8;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, g = lane >> 4;
  const int n_hg = (heads + 3) / 4;
  // the longest token tiles first (their rows attend the most keys)
  const int tt = n_tt - 1 - (int)blockIdx.x / n_hg;
  const int h = ((int)blockIdx.x % n_hg) * 4 + w;
  if (!SHARED && h >= heads) return;  // SHARED launches have heads % 4 == 0 (no wave leaves early)
  const int kvh = h / (heads / kv_heads);
  const int t0 = tt * TOK;
  const bf16_t* kb = Kc + (size_t)kvh * max_len * HD + lane * 8;
  const bf16_t* vb = Vt + (size_t)kvh * max_len * HD + lane * 8;
  // this kv head's blocks for the LDS copies
  const char* ksrc = (const char*)(Kc + (size_t)kvh * max_len * HD);
  const char* vsrc = (const char*)(Vt + (size_t)kvh * max_len * HD);

  PfAttnState<HD, NT> st;
#pragma unroll
  for (int rt = 0; rt < NT; ++rt) {
    const int tok = min(t0 + rt * 16 + j, M - 1);
    st.lim[rt] = pos0 + t0 + rt * 16 + j;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      st.qf[rt][ks] = *(const u32x4_t*)(Q + (size_t)tok * ldq + (size_t)h * HD + ks * 32 + g * 8);
    st.m_run[rt] = -INFINITY;
    st.l_run[rt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) st.o[rt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  const int last = pos0 + min(t0 + TOK, M) - 1;  // the tile's last attended key
  const int n_blk = last / 64 + 1;
  const int full_blk = min((pos0 + t0) / 64, n_blk - 1);  // blocks every row of the tile attends entirely

  // two K / V^T buffers (SHARED): blocks alternate between them
  constexpr int BUF = SHARED ? PIECES : 1;
  [[maybe_unused]] __shared__ __align__(16) u32x4_t kA[BUF], vA[BUF], kB[BUF], vB[BUF];
  typedef __attribute__((address_space(3))) u32x4_t* lp;
  if constexpr (SHARED) {
#pragma unroll
    for (int i = 0; i < PIECES / 256; ++i) {
      const size_t off = (size_t)(256 * i + 64 * w) * 16;
      __builtin_amdgcn_global_load_lds((const void*)(ksrc + off + (uint32_t)lane * 16),
                                       (lds_void*)((lp)kA + 256 * i + 64 * w), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const void*)(vsrc + off + (uint32_t)lane * 16),
                                       (lds_void*)((lp)vA + 256 * i + 64 * w), 16, 0, 0);
    }
  }
  // each instance of the body reads one buffer and fills the other
  auto even = [&](auto masked, int b) {
    pf_attend_block<HD, SHARED, NT, decltype(masked)::value>(st, b, n_blk, last, scale_log2, lane, w, kb, vb, ksrc, vsrc,
                                                             (lp)kA, (lp)vA, (lp)kB, (lp)vB);
  };
  auto odd = [&](auto masked, int b) {
    pf_attend_block<HD, SHARED, NT, decltype(masked)::value>(st, b, n_blk, last, scale_log2, lane, w, kb, vb, ksrc, vsrc,
                                                             (lp)kB, (lp)vB, (lp)kA, (lp)vA);
  };
  using yes_t = std::integral_constant<bool, true>;
  using no_t = std::integral_constant<bool, false>;
  int b = 0;
  for (; b + 1 < full_blk; b += 2) {
    even(no_t{}, b);
    odd(no_t{}, b + 1);
  }
  for (; b < n_blk; b += 2) {  // at most one block more that every row attends entirely, then the masked ones
    even(yes_t{}, b);
    if (b + 1 < n_blk) odd(yes_t{}, b + 1);
  }
  // lane (g, j) of o[rt][dt] holds dims 16 dt + 4 g + e of row j
#pragma unroll
  for (int rt = 0; rt < NT; ++rt) {
    const int tok = t0 + rt * 16 + j;
    if (tok >= M) continue;
    const float inv = 1.f / st.l_run[rt];
    bf16_t* dst = out + (size_t)tok * ldo + (size_t)h * HD;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const uint32_t lo = pack_bf16x2(st.o[rt][dt][0] * inv, st.o[rt][dt][1] * inv);
      const uint32_t hi = pack_bf16x2(st.o[rt][dt][2] * inv, st.o[rt][dt][3] * inv);
      *(uint2*)(dst + dt * 16 + 4 * g) = make_uint2(lo, hi);
    }
  }
}

// Row scales of the folded RMSNorm, rn[m] = rsqrt(mean(X[m, :K]^2) + eps), one wave per row: lane l
// sums its 8-element pieces l, l + 64, ... of the row in order, then a fixed butterfly (the order
// depends only on K, so a row's scale does not depend on M or on the chunking).
__global__ __launch_bounds__(256) void prefill_rowscale_kernel(const bf16_t* __restrict__ X, int64_t ldx, int M,
                                                               int K, float eps, float* __restrict__ rn) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  const bf16_t* x = X + (size_t)row * ldx;
  float acc = 0.f;
  for (int c = lane * 8; c < K; c += 512) acc += sumsq8(*(const u32x4_t*)(x + c));
  for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off);
  if (lane == 0) rn[row] = rsqrtf(acc / (float)K + eps);
}

// The tile shapes, largest first, and what a call with each costs: fixed + K / 64 * per-64-k cost *
// tiles of the busiest CU (two tiles share a CU's time where two workgroups fit). The costs are a
// least-squares fit (relative error) to the times of q/k/v, o, gate/up and down of the 1B, 8B and 70B shapes
// at 23 M from 24 to 4096 with every shape (us, this card; the five shapes of 96, 160 and 192 tokens at
// 24 M, 1B and 8B); the rule's choice is within 1.2 % of the fastest shape on average. Large tiles move the fewest operand bytes per MFMA;
// small ones put a short prompt's few rows on all CUs (M = 512, N = 4096, K = 14336: 32 tiles of 256
// x 256 279 us, 256 of 128 x 64 90 us).
// The shapes of 96, 160 and 192 tokens are for the row counts that 64, 128 and 256 pad the most: gate/up
// at N = 28672, K = 4096 -- 160 rows 71 us on 128-token tiles, 54 on 160; 350 rows 110 on 256, 84 on 192;
// down at 1150 rows 176 on 128, 134 on 160. Over 200 calls of the 1B and 8B shapes at 24 M from 66 to 4096
// the choice among all is 3.8 % faster (geometric mean) than among the other nine, at worst 2 % slower.
struct PrefillTile {
  int xt, yt, occ;
  double fixed, one, two;  // us; per 64 k with one tile on a CU, with two side by side (occ 2)
};
constexpr PrefillTile PREFILL_TILES[] = {
    {8, 8, 1, 14.2, 1.275, 0}, {6, 8, 1, 10.5, 1.032, 0},         {8, 6, 1, 11.3, 1.03, 0},
    {8, 4, 1, 3.0, 0.876, 0},  {6, 4, 1, 1.9, 0.746, 0},          {4, 6, 1, 7.8, 0.701, 0},
    {4, 5, 1, 4.0, 0.627, 0},  {4, 4, 1, 4.0, 0.509, 0},          {4, 3, 1, 6.3, 0.424, 0},
    {4, 2, 1, 2.9, 0.364, 0},  {2, 3, 2, 3.5, 0.299, 0.509},      {2, 2, 2, 2.7, 0.233, 0.418},
    {1, 2, 2, 3.1, 0.178, 0.294}, {1, 1, 2, 4.2, 0.121, 0.208},
};
constexpr int N_PREFILL_TILES = sizeof(PREFILL_TILES) / sizeof(PREFILL_TILES[0]);

static int pick_prefill_tile(int first, int M, int N, int K, int cus) {
  int best = first;
  double best_t = 0;
  for (int i = first; i < N_PREFILL_TILES; ++i) {
    const PrefillTile& p = PREFILL_TILES[i];
    const int64_t tiles = ((int64_t)M + 32 * p.yt - 1) / (32 * p.yt) * (((int64_t)N + 32 * p.xt - 1) / (32 * p.xt));
    const int64_t q = (tiles + cus - 1) / cus;  // tiles of the busiest CU
    const double t = p.fixed + K / 64 * (p.occ == 2 ? q / 2 * p.two + q % 2 * p.one : q * p.one);
    if (i == first || t < best_t) {
      best = i;
      best_t = t;
    }
  }
  return best;
}

template <int EPI, int XT, int YT, int KU, int NS, int OCC>
static int launch_prefill_tile(const GemmArgs& a, int group, int pos0, int cus, hipStream_t s) {
  const int n_mt = (a.M + 32 * YT - 1) / (32 * YT), n_nt = (a.N + 32 * XT - 1) / (32 * XT);
  const int per_xcd = (n_mt * n_nt + 7) / 8, resident = max(cus / 8, 1) * OCC;
  const int grid = 8 * min(per_xcd, resident);
  const int band = min(n_mt, 4);
  if (a.row_scale)
    SSD_LAUNCH((prefill_gemm4_kernel<EPI, true, XT, YT, KU, NS, OCC>), dim3(grid), dim3(256), 0, s, a, group, n_mt, n_nt,
               pos0, band);
  else
    SSD_LAUNCH((prefill_gemm4_kernel<EPI, false, XT, YT, KU, NS, OCC>), dim3(grid), dim3(256), 0, s, a, group, n_mt, n_nt,
               pos0, band);
  return check_launch("prefill_gemm4");
}

// Ring depth: as many steps as fit LDS beside the other workgroup; short steps need the depth to cover
// the memory latency (M = 100, N = 4096, K = 14336 on 32 x 64 tiles: 72 us with 4 slots, 44 with 6).
template <int EPI>
static int launch_prefill_gemm4(const GemmArgs& a, int group, int pos0, int cus, hipStream_t s) {
  // (the largest tile's q/k/v write-out would spill registers across the k loop: not offered there)
  switch (pick_prefill_tile(EPI == EPI_QKV ? 1 : 0, a.M, a.N, a.kb_total * 32, cus)) {
    case 0:
      if constexpr (EPI != EPI_QKV) return launch_prefill_tile<EPI, 8, 8, 1, 4, 1>(a, group, pos0, cus, s);
    case 1: return launch_prefill_tile<EPI, 6, 8, 1, 4, 1>(a, group, pos0, cus, s);
    case 2: return launch_prefill_tile<EPI, 8, 6, 1, 4, 1>(a, group, pos0, cus, s);
    case 3: return launch_prefill_tile<EPI, 8, 4, 1, 4, 1>(a, group, pos0, cus, s);
    case 4: return launch_prefill_tile<EPI, 6, 4, 1, 4, 1>(a, group, pos0, cus, s);
    case 5: return launch_prefill_tile<EPI, 4, 6, 1, 4, 1>(a, group, pos0, cus, s);
    case 6: return launch_prefill_tile<EPI, 4, 5, 2, 4, 1>(a, group, pos0, cus, s);
    case 7: return launch_prefill_tile<EPI, 4, 4, 2, 5, 1>(a, group, pos0, cus, s);
    case 8: return launch_prefill_tile<EPI, 4, 3, 2, 5, 1>(a, group, pos0, cus, s);
    case 9: return launch_prefill_tile<EPI, 4, 2, 2, 6, 1>(a, group, pos0, cus, s);
    case 10: return launch_prefill_tile<EPI, 2, 3, 2, 4, 2>(a, group, pos0, cus, s);
    case 11: return launch_prefill_tile<EPI, 2, 2, 2, 5, 2>(a, group, pos0, cus, s);
    case 12: return launch_prefill_tile<EPI, 1, 2, 2, 6, 2>(a, group, pos0, cus, s);
    default: return launch_prefill_tile<EPI, 1, 1, 2, 8, 2>(a, group, pos0, cus, s);
  }
}

static int launch_prefill_gemm(GemmArgs a, int group, int pos0, int epi, hipStream_t s) {
  static int cus_of[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return set_error(SSD_EHIP, "prefill gemm: no current device");
  int cus = dev >= 0 && dev < 64 ? cus_of[dev] : 0;
  if (cus <= 0) {
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    if (dev >= 0 && dev < 64) cus_of[dev] = cus;
  }
  // the kernel's lane offsets into X are 32 bits over at most 8 rows: rows further apart than that go
  // one by one
  if (a.ldx >= (int64_t)1 << 27 && a.M > 1) {
    for (int m = 0; m < a.M; ++m) {
      GemmArgs r = a;
      r.M = 1;
      r.X += (size_t)m * a.ldx;
      r.Y += (size_t)m * a.ldy;
      if (a.residual) r.residual += (size_t)m * a.ldr;
      if (a.row_scale) r.row_scale += m;
      const int rc = launch_prefill_gemm(r, group, pos0 + m, epi, s);
      if (rc) return rc;
    }
    return SSD_OK;
  }
  if (epi == EPI_SWIGLU) return launch_prefill_gemm4<EPI_SWIGLU>(a, group, pos0, cus, s);
  if (epi == EPI_QKV) return launch_prefill_gemm4<EPI_QKV>(a, group, pos0, cus, s);
  return launch_prefill_gemm4<EPI_STORE>(a, group, pos0, cus, s);
}

static int check_packed(int N, int K, int group) {
  if (N <= 0 || K <= 0 || K % 64) return set_error(SSD_EINVAL, "prefill gemm: N=%d K=%d (K %% 64 == 0)", N, K);
  const int tiles = (N + 127) / 128 * 8;  // packed row tiles (rows padded to 128)
  if (group < 1 || group > 16 || tiles % group)
    return set_error(SSD_EINVAL, "prefill gemm: group %d does not divide the %d row tiles", group, tiles);
  return SSD_OK;
}

}  // namespace ssd

using namespace ssd;

static int launch_row_scale(const uint16_t* X, int64_t ldx, int M, int K, float eps, float* rs, hipStream_t s) {
  SSD_LAUNCH(prefill_rowscale_kernel, dim3((M + 3) / 4), dim3(256), 0, s, (const bf16_t*)X, ldx, M, K, eps, rs);
  return check_launch("prefill_row_scale");
}

// Row scales of the RMSNorm folded into a prefill GEMM's packed weight: rs[m] = rsqrt(mean(X[m, :K]^2)
// + eps), one wave per row in a fixed order (a row's scale does not depend on M).
SSD_API int ssd_prefill_row_scale_bf16(const uint16_t* X, int64_t ldx, int M, int K, float eps, float* row_scale,
                                       hipStream_t stream) {
  if (!X || !row_scale) return set_error(SSD_EINVAL, "prefill row scale: null pointer");
  if (M <= 0 || K <= 0 || K % 8 || ldx < K || ldx % 8 || ((uintptr_t)X & 15) || !(eps > 0.f))
    return set_error(SSD_EINVAL, "prefill row scale: M=%d K=%d ldx=%lld eps=%g (16-byte rows, eps > 0)", M, K,
                     (long long)ldx, (double)eps);
  return launch_row_scale(X, ldx, M, K, eps, row_scale, stream);
}

// Y = epilogue(X W^T) with the folded RMSNorm's row scales (row_scale, [M] floats from
// ssd_prefill_row_scale_bf16) applied to the products, or none (row_scale null).
SSD_API int ssd_prefill_gemm_bf16(const uint16_t* X, int64_t ldx, int M, const uint16_t* W_packed, int group, int N,
                                  int K, const float* row_scale, int epi, uint16_t* Y, int64_t ldy,
                                  const uint16_t* residual, int64_t ldr, const SsdQkvEpilogue* qkv,
                                  hipStream_t stream) {
  if (!X || !W_packed || !Y) return set_error(SSD_EINVAL, "prefill gemm: null pointer");
  if (M <= 0) return set_error(SSD_EINVAL, "prefill gemm: M=%d", M);
  int rc = check_packed(N, K, group);
  if (rc) return rc;
  if (ldx < K || ldx % 8 || ((uintptr_t)X & 15)) return set_error(SSD_EINVAL, "prefill gemm: X rows must be 16-byte aligned");
  if (epi != SSD_EPI_STORE && epi != SSD_EPI_SWIGLU && epi != SSD_EPI_QKV)
    return set_error(SSD_EINVAL, "prefill gemm: epilogue %d", epi);
  if (epi == SSD_EPI_STORE && ldy < N) return set_error(SSD_EINVAL, "prefill gemm: ldy %lld < N", (long long)ldy);
  if (epi == SSD_EPI_SWIGLU && (N % 16 || ldy < N / 2)) return set_error(SSD_EINVAL, "prefill gemm: swiglu N=%d", N);
  if (epi != SSD_EPI_STORE && residual) return set_error(SSD_EINVAL, "prefill gemm: residual only with a plain store");
  GemmArgs a{};
  a.X = X; a.ldx = ldx; a.M = M; a.W = (const uint4*)W_packed; a.N = N; a.kb_total = K / 32;
  a.Y = Y; a.ldy = ldy; a.residual = residual; a.ldr = ldr;
  a.row_scale = row_scale;
  int pos0 = 0;
  if (epi == SSD_EPI_QKV) {
    if (!qkv || !qkv->cos || !qkv->sin || !qkv->k_cache || !qkv->vt_cache)
      return set_error(SSD_EINVAL, "prefill gemm: q/k/v epilogue needs rotary tables and the cache");
    const int hd = qkv->head_dim;
    if ((hd != 32 && hd != 64 && hd != 128) || qkv->heads <= 0 || qkv->kv_heads <= 0 ||
        N != (qkv->heads + 2 * qkv->kv_heads) * hd || ldy < (int64_t)qkv->heads * hd)
      return set_error(SSD_EINVAL, "prefill gemm: q/k/v shape N=%d heads=%d kv=%d hd=%d", N, qkv->heads,
                       qkv->kv_heads, hd);
    if (((uintptr_t)qkv->k_cache & 15) || ((uintptr_t)qkv->vt_cache & 15) || ((uintptr_t)qkv->cos & 15) ||
        ((uintptr_t)qkv->sin & 15))
      return set_error(SSD_EINVAL, "prefill gemm: caches and rotary tables must be 16-byte aligned");
    if (qkv->pos0 < 0 || qkv->pos0 + M > qkv->max_len || qkv->pos0 + M > qkv->rope_rows || qkv->max_len % 64)
      return set_error(SSD_EINVAL, "prefill gemm: rows [%d, %d) outside the cache (%lld) or rotary table (%lld)",
                       qkv->pos0, qkv->pos0 + M, (long long)qkv->max_len, (long long)qkv->rope_rows);
    a.heads = qkv->heads; a.kv_heads = qkv->kv_heads; a.head_dim = hd;
    a.cos_tab = qkv->cos; a.sin_tab = qkv->sin; a.rope_rows = qkv->rope_rows;
    a.k_cache = qkv->k_cache; a.vt_cache = qkv->vt_cache; a.max_len = qkv->max_len;
    pos0 = qkv->pos0;
  }
  return launch_prefill_gemm(a, group, pos0, epi, stream);
}

SSD_API int ssd_prefill_attention_bf16(const uint16_t* q, int64_t ldq, int M, int pos0, int heads, int kv_heads,
                                       int head_dim, const uint16_t* k_cache, const uint16_t* vt_cache,
                                       int64_t max_len, float scale, uint16_t* out, int64_t ldo,
                                       hipStream_t stream) {
  if (!q || !k_cache || !vt_cache || !out) return set_error(SSD_EINVAL, "prefill attention: null pointer");
  if (M <= 0 || pos0 < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads)
    return set_error(SSD_EINVAL, "prefill attention: M=%d pos0=%d heads=%d kv_heads=%d", M, pos0, heads, kv_heads);
  if (pos0 + M > max_len || max_len % 64 || ldq % 8 || ((uintptr_t)q & 15) || ((uintptr_t)k_cache & 15) ||
      ((uintptr_t)vt_cache & 15) || ldo % 4 || ((uintptr_t)out & 7))
    return set_error(SSD_EINVAL, "prefill attention: rows [%d, %d) vs cache %lld, or misaligned operands", pos0,
                     pos0 + M, (long long)max_len);
  // a workgroup's four waves share one kv head's K/V when 4 divides the q heads per kv head
  const bool shared = (heads / kv_heads) % 4 == 0;
  // One 16-row tile per wave while that leaves at most two workgroups per CU, or one where the waves read K / V for
  // themselves, at head_dim 128 and after a past of more than 2048 keys: two such workgroups on a CU then fetch twice
  // what one of 32 rows does (us, one tile / two: 24 q heads on 8 kv heads, 704 rows after 1000 keys 51 / 50,
  // 8000 292 / 208, 32000 1148 / 759; at head_dim 64 one tile stays the faster).
  const int n_hg = (heads + 3) / 4;
  const int most = shared || head_dim == 64 || pos0 <= 2048 ? 512 : 256;
  const bool small = (int64_t)((M + 15) / 16) * n_hg <= most;
  const int tok = small ? 16 : 32, n_tt = (M + tok - 1) / tok;
  const dim3 grid((unsigned)(n_tt * n_hg)), block(256);
  const float sl2 = scale * 1.4426950408889634f;
#define PF_ATT_NT(D, SH, NT)                                                                                       \
  SSD_LAUNCH((prefill_attention_kernel<D, SH, NT>), grid, block, 0, stream, (const bf16_t*)q, ldq, M, pos0, heads, \
             kv_heads, (const bf16_t*)k_cache, (const bf16_t*)vt_cache, max_len, sl2, (bf16_t*)out, ldo, n_tt)
#define PF_ATT(D, SH)               \
  if (small) PF_ATT_NT(D, SH, 1);   \
  else PF_ATT_NT(D, SH, 2)
  switch (head_dim) {
    case 64:
      if (shared) { PF_ATT(64, true); }
      else { PF_ATT(64, false); }
      break;
    case 128:
      if (shared) { PF_ATT(128, true); }
      else { PF_ATT(128, false); }
      break;
    default:
      return set_error(SSD_EINVAL, "prefill attention: head_dim %d unsupported (64, 128)", head_dim);
  }
#undef PF_ATT
#undef PF_ATT_NT
  return check_launch("prefill_attention");
}

// The target forward over prompt rows [pos0, pos0 + m): embed -> per layer q/k/v (+RoPE, KV
// write) -> causal attention -> o_proj + residual -> gate/up + SwiGLU -> down + residual; then the
// full-vocabulary head (head_w, final norm folded; NULL = none) on the last row. Buffers are
// [m_cap] rows.
SSD_API int ssd_prefill(const SsdModel* md, const uint16_t* head_w, const SsdPrefillBuffers* pb, const int32_t* ids,
                        int m, int pos0, hipStream_t s) {
  if (!md || !pb || !ids) return set_error(SSD_EINVAL, "prefill: null descriptor");
  if (m <= 0 || m > pb->m_cap) return set_error(SSD_EINVAL, "prefill: m=%d outside [1, %d]", m, pb->m_cap);
  if (!md->layers) return set_error(SSD_EINVAL, "prefill: null layer table");
  if (!(md->eps > 0.f)) return set_error(SSD_EINVAL, "prefill: norm eps must be > 0");
  if (pos0 < 0 || pos0 + m > pb->cache_cap)
    return set_error(SSD_EINVAL, "prefill: rows [%d, %d) beyond the cache (%lld)", pos0, pos0 + m,
                     (long long)pb->cache_cap);
  if (head_w && !pb->logits) return set_error(SSD_EINVAL, "prefill: no logits buffer");
  const int d = md->hidden, hd = md->head_dim, H = md->heads, KV = md->kv_heads, I = md->inter;
  const int64_t qdim = (int64_t)H * hd;
  const int nqkv = (H + 2 * KV) * hd;
  const size_t layer_elems = (size_t)KV * pb->cache_cap * hd;
  const int g_qkv = ssd_gemm_weight_group(nqkv, d), g_o = ssd_gemm_residual_group(d, (int)qdim);
  const int g_gu = md->mlp_fused ? ssd_mlp_group(I, d) : ssd_gemm_weight_group(2 * I, d);
  const int g_d = ssd_gemm_residual_group(d, I);
  if (g_qkv < 1 || g_o < 1 || g_gu < 1 || g_d < 1) return set_error(SSD_EINVAL, "prefill: no packing plan for this shape");
  int rc = ssd_embed_bf16(ids, m, md->embed, md->vocab, d, pb->h, d, s);
  if (rc) return rc;
  for (int li = 0; li < md->n_layers; ++li) {
    const SsdLayerW& L = md->layers[li];
    SsdQkvEpilogue qe{H, KV, hd, md->cos, md->sin, md->rope_rows, pos0, pb->k_arena + li * layer_elems,
                      pb->vt_arena + li * layer_elems, pb->cache_cap};
    // the input norm's row scales, computed once per row into the attention buffer (free until the
    // attention writes it)
    float* rs_qkv = (float*)pb->attn;
    if ((rc = launch_row_scale(pb->h, d, m, d, md->eps, rs_qkv, s))) return rc;
    if ((rc = ssd_prefill_gemm_bf16(pb->h, d, m, L.wqkv, g_qkv, nqkv, d, rs_qkv, SSD_EPI_QKV, pb->q, qdim, nullptr, 0,
                                    &qe, s)))
      return rc;
    if ((rc = ssd_prefill_attention_bf16(pb->q, qdim, m, pos0, H, KV, hd, qe.k_cache, qe.vt_cache, pb->cache_cap,
                                         md->attn_scale, pb->attn, qdim, s)))
      return rc;
    if ((rc = ssd_prefill_gemm_bf16(pb->attn, qdim, m, L.wo, g_o, d, (int)qdim, nullptr, SSD_EPI_STORE, pb->h, d, pb->h,
                                    d, nullptr, s)))
      return rc;
    // gate/up's norm scales computed once per row into the q buffer (free after the attention)
    float* rs = (float*)pb->q;
    if ((rc = launch_row_scale(pb->h, d, m, d, md->eps, rs, s))) return rc;
    if ((rc = ssd_prefill_gemm_bf16(pb->h, d, m, L.wgu, g_gu, 2 * I, d, rs, SSD_EPI_SWIGLU, pb->act, I, nullptr, 0,
                                    nullptr, s)))
      return rc;
    if ((rc = ssd_prefill_gemm_bf16(pb->act, I, m, L.wd, g_d, d, I, nullptr, SSD_EPI_STORE, pb->h, d, pb->h, d, nullptr,
                                    s)))
      return rc;
  }
  if (head_w)
    return ssd_gemm_bf16(pb->h + (size_t)(m - 1) * d, d, 1, head_w, md->vocab, d, md->eps, pb->logits, md->vocab,
                         nullptr, 0, nullptr, 0, s);
  return SSD_OK;
}
