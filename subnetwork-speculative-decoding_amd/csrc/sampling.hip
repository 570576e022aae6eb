// Sampling path: temperature + nucleus warp, Gumbel top-k draft proposals,
// speculative-sampling acceptance over the verify tree, and categorical draws.
//
// Reference semantics (restated, not transcribed):
// * warp_probs  ssd/engine/tree_drafter.py:34-45: p = softmax(logits / T); with
//   top_p < 1 an entry survives when the mass of the entries sorted before it is
//   <= top_p; survivors are renormalised.
// * _propose    ssd/engine/tree_drafter.py:124-145 (sampling branch): q is the warped
//   draft distribution over the full vocabulary (zero outside a draft-vocab subset);
//   children are min(k, |support|) draws without replacement, in draw order, via the
//   Gumbel top-k trick; their log-probs are log q.
// * sample_verify ssd/engine/verify.py:60-95: walk root -> children in rank order;
//   accept child x with probability min(1, p(x) / q(x)); on rejection
//   p <- (p - q)+ / sum (when the sum is positive), q(x) <- 0, q <- q / sum(q), stop when
//   q has no mass left; the bonus token is drawn from the final p.
// * torch.multinomial (ssd/engine/speculative.py:81-84, verify.py:94): one categorical
//   draw, here as argmax_y p(y) / E(y) with E(y) ~ Exp(1) (the Gumbel-max trick).
//
// Randomness: Philox4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as
// easy as 1, 2, 3", SC 2011). Key = 64-bit seed; counter = (element / 4 or step index,
// row | level << 16, round counter low word, round counter high bits << 8 | purpose tag),
// so every draw of a generation has its own counter and no result depends on launch
// shapes or on how many rows share a launch.
//
// Work layout: a row is cut into chunks of 4096 columns, one 1024-thread workgroup per
// (chunk, row), 4 consecutive columns per thread. Cross-chunk results go through a
// caller-provided workspace between launches: integer histograms built with atomics
// (order-independent), or per-chunk partials combined afterwards in chunk order, so every
// result is deterministic.
//
// Nucleus cut: the order of a row's probabilities is the order of its bf16 logits, so the
// cut is searched over the 16-bit logit keys: a 256-bin mass histogram of the key's high
// byte (mass = round(p * 2^52), exact integer sums), then a 256-bin count histogram of the
// low byte inside the cut bin, which fixes the cut key; equal logits rank lower column first
// (per-chunk counts of the cut key give each tie its column rank).
#include "common.h"

#include <math.h>

namespace ssd {

constexpr int SMP_THREADS = 1024;
constexpr int SMP_CHUNK = 4096;
constexpr int SMP_MAXK = 16;      // children per node / draws per row
constexpr int SMP_MAXC = 256;     // chunks per row (rows up to 1M columns)
constexpr int SMP_MAXDEPTH = 32;  // tree depth (matches the tree kernels)

enum SmpTag { TAG_PROPOSE = 1, TAG_ACCEPT = 2, TAG_BONUS = 3, TAG_DRAW = 4, TAG_TOP64 = 5 };

struct Rng {
  uint32_t k0, k1;       // key: seed
  uint32_t c2, c3_base;  // counter words 2 and 3 (round counter; tag is or-ed into c3)
};

static Rng make_rng(uint64_t seed, uint64_t ctr) {
  return Rng{(uint32_t)seed, (uint32_t)(seed >> 32), (uint32_t)ctr, (uint32_t)((ctr >> 32) << 8)};
}

struct U4 {
  uint32_t x, y, z, w;
};

// Philox4x32 with 10 rounds: multipliers 0xD2511F53 / 0xCD9E8D57, Weyl key increments
// 0x9E3779B9 / 0xBB67AE85 (the published constants of the generator).
__device__ __forceinline__ U4 philox(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint32_t lo0 = 0xD2511F53u * c0, hi0 = __umulhi(0xD2511F53u, c0);
    const uint32_t lo1 = 0xCD9E8D57u * c2, hi1 = __umulhi(0xCD9E8D57u, c2);
    c0 = hi1 ^ c1 ^ k0;
    c1 = lo1;
    c2 = hi0 ^ c3 ^ k1;
    c3 = lo0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return U4{c0, c1, c2, c3};
}

__device__ __forceinline__ U4 rng_block(const Rng& g, uint32_t c0, uint32_t c1, int tag) {
  return philox(c0, c1, g.c2, g.c3_base | (uint32_t)tag, g.k0, g.k1);
}

// Standard exponential -log(U) from 32 random bits, U = (b + 1/2) / 2^32 in (0, 1). The lower
// half of U is taken directly and the upper half through 1 - U, so both tails keep 24 bits.
__device__ __forceinline__ float exp1_from_bits(uint32_t b) {
  if (b < 0x80000000u) return -logf(((float)b + 0.5f) * 0x1p-32f);
  return -log1pf(-(((float)(~b) + 0.5f) * 0x1p-32f));
}

__device__ __forceinline__ double uniform_from_bits(uint32_t b) { return ((double)b + 0.5) * 0x1p-32; }

__device__ __forceinline__ uint32_t u4_get(const U4& r, int e) {
  return e == 0 ? r.x : e == 1 ? r.y : e == 2 ? r.z : r.w;
}

// ----------------------------------------------------------- reductions
// Workgroup reductions put the 16 waves' partials into `sh` and pass one barrier; `sh` belongs to that
// one reduction, so that none of them needs a second barrier before it is used again.
//
// Inside a wave, values move between lanes by DPP and the permlane swaps (VALU) rather than by shuffles,
// which all go through LDS: with 32 waves on a CU the ~60 exchanges of an acceptance pass cost more there
// than its loads. Steps 1, 2, 4, 8 pair lanes by quad permutation and the mirrors of 8 and 16 lanes (the
// lanes of each half hold one value by then, so a mirror reaches the same partner value as an xor),
// steps 16 and 32 by the swaps: every lane ends with the same value, and a sum adds the same pairs in
// the same order as a butterfly of xor shuffles.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140;

template <typename T>
struct Words {
  static constexpr int N = sizeof(T) / 4;
  uint32_t w[N];
};

// r0 and r1 of each lane: its own value and its partner's at the given step (in either order).
template <int STEP, typename T>
__device__ __forceinline__ void wave_pair(T v, T& r0, T& r1) {
  const Words<T> x = __builtin_bit_cast(Words<T>, v);
  Words<T> a, b;
#pragma unroll
  for (int i = 0; i < Words<T>::N; ++i) {
    a.w[i] = x.w[i];
    if constexpr (STEP == 1) b.w[i] = dpp<DPP_XOR1>(x.w[i]);
    else if constexpr (STEP == 2) b.w[i] = dpp<DPP_XOR2>(x.w[i]);
    else if constexpr (STEP == 4) b.w[i] = dpp<DPP_HALF_MIRROR>(x.w[i]);
    else if constexpr (STEP == 8) b.w[i] = dpp<DPP_MIRROR>(x.w[i]);
    else {
      const auto p = STEP == 16 ? __builtin_amdgcn_permlane16_swap(x.w[i], x.w[i], false, false)
                                : __builtin_amdgcn_permlane32_swap(x.w[i], x.w[i], false, false);
      a.w[i] = p[0];
      b.w[i] = p[1];
    }
  }
  r0 = __builtin_bit_cast(T, a);
  r1 = __builtin_bit_cast(T, b);
}

// All 64 lanes reduced by a commutative `op`.
template <typename T, class Op>
__device__ __forceinline__ T wave_reduce(T v, Op op) {
  T a, b;
  wave_pair<1>(v, a, b);
  wave_pair<2>(op(a, b), a, b);
  wave_pair<4>(op(a, b), a, b);
  wave_pair<8>(op(a, b), a, b);
  wave_pair<16>(op(a, b), a, b);
  wave_pair<32>(op(a, b), a, b);
  return op(a, b);
}

__device__ __forceinline__ float wave_max(float v) {
  return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  return wave_reduce(v, [](T a, T b) { return a + b; });
}

// Inclusive prefix sum over the lanes: DPP shifts inside each row of 16, then the rows' last lanes
// broadcast to the rows above (CTRL 0x142 / 0x143: lane 15 of each row, lane 31).
template <int CTRL, int ROWS>
__device__ __forceinline__ uint64_t dpp64(uint64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROWS, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, ROWS, 0xf, false);
  return (uint64_t)hi << 32 | lo;
}
__device__ __forceinline__ uint64_t wave_scan(uint64_t v) {
  v += dpp64<0x111, 0xf>(v);
  v += dpp64<0x112, 0xf>(v);
  v += dpp64<0x114, 0xf>(v);
  v += dpp64<0x118, 0xf>(v);
  v += dpp64<0x142, 0xa>(v);
  v += dpp64<0x143, 0xc>(v);
  return v;
}

__device__ __forceinline__ float block_max(float v, float* sh) {
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = sh[0];
#pragma unroll
  for (int i = 1; i < 16; ++i) r = fmaxf(r, sh[i]);
  return r;
}

// The waves' sums in order, once they are all in `sh`.
template <typename T>
__device__ __forceinline__ T sum16(const T* sh) {
  T r = sh[0];
#pragma unroll
  for (int i = 1; i < 16; ++i) r += sh[i];
  return r;
}

struct KeyIdx {
  float key;
  int idx;
};

__device__ __forceinline__ bool better(float ka, int ia, float kb, int ib) {
  return ka > kb || (ka == kb && ia < ib);
}

constexpr int NO_IDX = 0x7fffffff;

// Largest key, lowest index among equal keys (a strict order, so any order of merging gives the same).
__device__ __forceinline__ KeyIdx wave_argmax(float k, int i) {
  return wave_reduce(KeyIdx{k, i}, [](KeyIdx a, KeyIdx b) { return better(a.key, a.idx, b.key, b.idx) ? a : b; });
}

// f(e) for every set bit e of the lanes' 4-bit masks, all lanes taking their next one together. The
// columns of a nucleus are few (2 % of 128256 at T 0.7 and top_p 0.9), so a wave that looked at its lanes'
// four columns one after another would run the logarithms of a draw four times, mostly for a lane or two.
template <class F>
__device__ __forceinline__ void for_active(uint32_t mask, F f) {
  while (__ballot(mask != 0)) {
    if (mask) {
      f(__ffs((int)mask) - 1);
      mask &= mask - 1;
    }
  }
}
__device__ __forceinline__ float get4(const float (&v)[4], int e) {
  return e == 0 ? v[0] : e == 1 ? v[1] : e == 2 ? v[2] : v[3];
}

// The best of the 16 waves' records in `sh`, by one wave.
__device__ __forceinline__ KeyIdx argmax16(const KeyIdx* sh) {
  const int lane = threadIdx.x & 63;
  const KeyIdx v = lane < 16 ? sh[lane] : KeyIdx{-1.f, NO_IDX};
  return wave_argmax(v.key, v.idx);
}

// Inclusive prefix sum over the 1024 threads (thread order).
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* sh) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t n = __shfl_up(v, o);
    if (lane >= o) v += n;
  }
  if (lane == 63) sh[w] = v;
  __syncthreads();
  uint32_t add = 0;
  for (int i = 0; i < w; ++i) add += sh[i];
  __syncthreads();
  return v + add;
}

// ------------------------------------------------------------------------ workspace
// One caller-provided buffer, carved per (rows, chunks). Histograms are cleared by the first
// launch of each warp; every other array is fully written before it is read.
struct NodeKids {  // children of a verify node that the acceptance considers, in rank order
  int n;
  int kid[SMP_MAXK];
  int tok[SMP_MAXK];
};

struct SmpWs {
  float2* stats;      // [rows][C] chunk (max, sum exp) of logits / T
  uint64_t* coarse;   // [rows][256] mass by key high byte
  uint32_t* fine;     // [rows][256] count by key low byte inside the cut bin
  uint32_t* finec;    // [rows][C][256] the same per chunk (column rank of ties)
  KeyIdx* cand;       // [rows][C][SMP_MAXK] per-chunk Gumbel top-k candidates
  int* csupp;         // [rows][C] per-chunk support size
  KeyIdx* arg;        // [rows][C] per-chunk categorical draw
  double* zr;         // [rows][SMP_MAXK + 1][C] residual mass partials per rejection state
  KeyIdx* bon;        // [rows][SMP_MAXK + 1][C] bonus draw partials per rejection state
  double* s0;         // [rows][C] mass of q0 per chunk
  int* supp;          // [rows][C] support of q0 per chunk
  NodeKids* kids;     // [rows] each verify row's children, written by the first acceptance pass
  int C;
};

static int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

static int64_t smp_layout(int rows, int C, char* base, SmpWs* ws) {
  int64_t off = 0;
  auto take = [&](int64_t bytes) -> char* {
    char* p = base ? base + off : nullptr;
    off += align256(bytes);
    return p;
  };
  const int64_t R = rows, CC = C;
  SmpWs w;
  w.stats = (float2*)take(R * CC * sizeof(float2));
  w.coarse = (uint64_t*)take(R * 256 * 8);
  w.fine = (uint32_t*)take(R * 256 * 4);
  w.finec = (uint32_t*)take(R * CC * 256 * 4);
  w.cand = (KeyIdx*)take(R * CC * SMP_MAXK * sizeof(KeyIdx));
  w.csupp = (int*)take(R * CC * 4);
  w.arg = (KeyIdx*)take(R * CC * sizeof(KeyIdx));
  w.zr = (double*)take(R * (SMP_MAXK + 1) * CC * 8);
  w.bon = (KeyIdx*)take(R * (SMP_MAXK + 1) * CC * sizeof(KeyIdx));
  w.s0 = (double*)take(R * CC * 8);
  w.supp = (int*)take(R * CC * 4);
  w.kids = (NodeKids*)take(R * (int64_t)sizeof(NodeKids));
  w.C = C;
  if (ws) *ws = w;
  return off;
}

static int chunks_of(int n) { return (n + SMP_CHUNK - 1) / SMP_CHUNK; }

// ------------------------------------------------------------------------ warp
struct WarpArgs {
  const bf16_t* logits;
  int64_t ld;
  int rows, n;        // logit rows and columns
  const int* vocab;   // column -> token (draft-vocab subset), or null (column = token)
  const int* inv;     // token -> column or -1 (with vocab), length V
  int V;              // output row length (full vocabulary)
  float temp, top_p;
  uint64_t T;         // top_p in units of 2^-52
  const int* meta;    // tree meta: rows are the frontier proposing `level`; null: plain rows
  int level;
  float* out;
  int64_t ldo;
  SmpWs ws;
};

// Frontier size and first output row of a proposal step (tree meta layout: [0] nodes,
// [1 + d] start of level d, [1 + SMP_MAXDEPTH + d] its size). Level 0 proposes the root's
// children (q row 0); level d > 0 proposes children of level d - 1, whose node i keeps its
// q in row 1 + i.
__device__ __forceinline__ void frontier_rows(const int* meta, int level, int rows, int& F, int& base) {
  if (!meta) {
    F = rows;
    base = 0;
  } else if (level == 0) {
    F = 1;
    base = 0;
  } else {
    F = min(rows, meta[1 + SMP_MAXDEPTH + level - 1]);
    base = 1 + meta[1 + level - 1];
  }
}

// Monotone 16-bit key of a bf16 value (ascending key = ascending value) and its inverse.
__device__ __forceinline__ uint32_t bf_key(uint32_t h) { return h ^ ((h & 0x8000u) ? 0xffffu : 0x8000u); }
__device__ __forceinline__ uint32_t key_bf(uint32_t k) { return k ^ ((k & 0x8000u) ? 0x8000u : 0xffffu); }

// The probability of a logit and its fixed-point mass: one code path for every use, so a
// value and the mass accumulated for it always agree bit for bit.
__device__ __forceinline__ float scaled_of(uint32_t h, float temp) { return bf2f((bf16_t)h) / temp; }
__device__ __forceinline__ float prob_scaled(float x, float M, float S) { return expf(x - M) / S; }
__device__ __forceinline__ float prob_of(uint32_t h, float temp, float M, float S) {
  return prob_scaled(scaled_of(h, temp), M, S);
}
__device__ __forceinline__ uint64_t mass_of(float p) { return __double2ull_rn((double)p * 0x1p52); }

__device__ __forceinline__ void load4_bf16(const bf16_t* row, int i, int n, uint32_t h[4]) {
  if (i + 3 < n) {
    const uint2 raw = *(const uint2*)(row + i);
    h[0] = raw.x & 0xffff;
    h[1] = raw.x >> 16;
    h[2] = raw.y & 0xffff;
    h[3] = raw.y >> 16;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = i + e < n ? row[i + e] : 0xff80u;  // -inf pads
  }
}

// Row max and sum exp from the chunk partials, by one wave (C <= 256). The sum's order is that of a
// 1024-thread workgroup over the chunk index: a butterfly per 64 chunks, then those in order.
__device__ __forceinline__ void row_stats(const float2* st, int C, float& M, float& S) {
  const int lane = threadIdx.x & 63;
  float2 v[SMP_MAXC / 64];
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < SMP_MAXC / 64; ++u) {
    v[u] = make_float2(-INFINITY, 0.f);
    if (64 * u < C && lane + 64 * u < C) v[u] = st[lane + 64 * u];
    m = fmaxf(m, v[u].x);
  }
  M = wave_max(m);
  S = 0.f;
#pragma unroll
  for (int u = 0; u < SMP_MAXC / 64; ++u)
    if (u == 0 || 64 * u < C) {
      const float e = wave_sum(lane + 64 * u < C && v[u].x != -INFINITY ? v[u].y * expf(v[u].x - M) : 0.f);
      S = u == 0 ? e : S + e;
    }
}

// Scan of a 256-bin histogram from the largest key down, by one wave: lane l holds the masses of bins
// 255 - 4 l - e. cut: the bin with the first entry whose preceding mass exceeds T (-1 when the whole
// histogram fits under T); above: the mass of the bins over it, plus `base`; total: base plus all.
struct Cut {
  int bin;
  uint64_t above, total;
};

__device__ __forceinline__ Cut wave_cut(const uint64_t (&v)[4], uint64_t base, uint64_t T) {
  const int lane = threadIdx.x & 63;
  const uint64_t sum = v[0] + v[1] + v[2] + v[3];
  const uint64_t incl = wave_scan(sum);
  Cut r{-1, 0, base + __shfl(incl, 63)};
  uint64_t before = base + incl - sum;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (v[e] > 0 && before <= T && T < before + v[e]) {
      r.bin = 255 - 4 * lane - e;
      r.above = before;
    }
    before += v[e];
  }
  const uint64_t found = __ballot(r.bin >= 0);
  if (found) {
    const int src = __ffsll((unsigned long long)found) - 1;
    r.bin = __shfl(r.bin, src);
    r.above = __shfl(r.above, src);
  }
  return r;
}

// This lane's four bins of a histogram, in wave_cut's order.
template <typename T>
__device__ __forceinline__ void load_bins(const T* hist, T (&v)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = hist[255 - 4 * (threadIdx.x & 63) - e];
}

// The four launches of a warp are chains of memory round trips and reductions rather than bytes (16 rows
// of 128256: 11 MB). What concerns the whole row -- its statistics, the cut -- is therefore done by the
// first wave of each workgroup while the others load their logits, with one barrier behind it; scanning
// the histograms with all 1024 threads took two barriers and a serial pass over the 16 waves each
// (us for 16 rows, before / after: stats 5.6 / 4.9, coarse 8.2 / 6.2, fine 5.4 / 3.9, final
// 16.3 / 10.0).

// L0: chunk max / sum exp; the first chunk of each row clears the row's histograms.
__global__ __launch_bounds__(SMP_THREADS) void warp_stats_kernel(WarpArgs a) {
  __shared__ float red_m[16], red_s[16];
  int F, base;
  frontier_rows(a.meta, a.level, a.rows, F, base);
  const int f = blockIdx.y, c = blockIdx.x, t = threadIdx.x;
  if (f >= F) return;
  if (c == 0 && a.top_p < 1.f) {
    if (t < 256) a.ws.coarse[(size_t)f * 256 + t] = 0;
    if (t < 256) a.ws.fine[(size_t)f * 256 + t] = 0;
  }
  const int i = c * SMP_CHUNK + t * 4;
  uint32_t h[4];
  load4_bf16(a.logits + (size_t)f * a.ld, i, a.n, h);
  float x[4], m = -INFINITY;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[e] = i + e < a.n ? scaled_of(h[e], a.temp) : -INFINITY;
    m = fmaxf(m, x[e]);
  }
  const float M = block_max(m, red_m);
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) s += i + e < a.n ? expf(x[e] - M) : 0.f;
  s = wave_sum(s);
  if ((t & 63) == 0) red_s[t >> 6] = s;
  __syncthreads();
  if (t == 0) a.ws.stats[(size_t)f * a.ws.C + c] = make_float2(M, sum16(red_s));
}

// L1: mass histogram of the key high byte. A row's logits fall into few of the 256 bins (sign and
// exponent), so each bin has HCOPY counters side by side, picked by the thread.
constexpr int HCOPY = 8;
__global__ __launch_bounds__(SMP_THREADS) void warp_coarse_kernel(WarpArgs a) {
  __shared__ uint64_t hist[256 * HCOPY];
  __shared__ float M_sh, S_sh;
  int F, base;
  frontier_rows(a.meta, a.level, a.rows, F, base);
  const int f = blockIdx.y, c = blockIdx.x, t = threadIdx.x;
  if (f >= F) return;
  const int i = c * SMP_CHUNK + t * 4;
  uint32_t h[4];
  load4_bf16(a.logits + (size_t)f * a.ld, i, a.n, h);
  if (t < 64) {
    float M, S;
    row_stats(a.ws.stats + (size_t)f * a.ws.C, a.ws.C, M, S);
    if (t == 0) {
      M_sh = M;
      S_sh = S;
    }
  }
  for (int b = t; b < 256 * HCOPY; b += SMP_THREADS) hist[b] = 0;
  __syncthreads();
  const float M = M_sh, S = S_sh;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (i + e >= a.n) continue;
    const uint64_t w = mass_of(prob_of(h[e], a.temp, M, S));
    if (w) atomicAdd((unsigned long long*)&hist[(bf_key(h[e]) >> 8) * HCOPY + t % HCOPY], (unsigned long long)w);
  }
  __syncthreads();
  if (t < 256) {
    uint64_t w = 0;
#pragma unroll
    for (int u = 0; u < HCOPY; ++u) w += hist[t * HCOPY + u];
    if (w) atomicAdd((unsigned long long*)&a.ws.coarse[(size_t)f * 256 + t], (unsigned long long)w);
  }
}

// L2: inside the coarse cut bin, count histogram of the key low byte (row total and per chunk).
__global__ __launch_bounds__(SMP_THREADS) void warp_fine_kernel(WarpArgs a) {
  __shared__ uint32_t hist[256];
  __shared__ int cut_sh;
  int F, base;
  frontier_rows(a.meta, a.level, a.rows, F, base);
  const int f = blockIdx.y, c = blockIdx.x, t = threadIdx.x;
  if (f >= F) return;
  const int i = c * SMP_CHUNK + t * 4;
  uint32_t h[4];
  load4_bf16(a.logits + (size_t)f * a.ld, i, a.n, h);
  if (t < 64) {
    uint64_t v[4];
    load_bins(a.ws.coarse + (size_t)f * 256, v);
    const Cut cut = wave_cut(v, 0ull, a.T);
    if (t == 0) cut_sh = cut.bin;
  }
  if (t < 256) hist[t] = 0;
  __syncthreads();
  const int cut = cut_sh;
  if (cut < 0) return;  // everything fits under top_p (uniform per block)
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t k = bf_key(h[e]);
    if (i + e < a.n && (int)(k >> 8) == cut) atomicAdd(&hist[k & 255], 1u);
  }
  __syncthreads();
  if (t < 256) {
    const uint32_t v = hist[t];
    a.ws.finec[((size_t)f * a.ws.C + c) * 256 + t] = v;
    if (v) atomicAdd(&a.ws.fine[(size_t)f * 256 + t], v);
  }
}

// L3: probabilities out (renormalised survivors when top_p < 1); zeros outside a subset.
__global__ __launch_bounds__(SMP_THREADS) void warp_final_kernel(WarpArgs a) {
  __shared__ float M_sh, S_sh, scale_sh;
  __shared__ uint32_t cut_key_sh, c_keep_sh, prefix_sh, ties_sh[16];
  int F, base;
  frontier_rows(a.meta, a.level, a.rows, F, base);
  const int f = blockIdx.y, c = blockIdx.x, t = threadIdx.x, lane = t & 63;
  if (f >= F) return;
  float* out = a.out + (size_t)(base + f) * a.ldo;
  if (a.vocab) {  // tokens outside the subset have probability 0
    const int y0 = c * SMP_CHUNK + t * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (y0 + e < a.V && a.inv[y0 + e] < 0) out[y0 + e] = 0.f;
  }
  if (c * SMP_CHUNK >= a.n) return;  // a zero-fill-only chunk (uniform per block)
  const int i = c * SMP_CHUNK + t * 4;
  uint32_t h[4];
  load4_bf16(a.logits + (size_t)f * a.ld, i, a.n, h);
  if (t < 64) {  // the row's statistics and cut
    float M, S, scale = 1.f;
    uint64_t cm[4];
    uint32_t fn[4];
    if (a.top_p < 1.f) {  // loaded beside the statistics; the fine histogram is all zeros without a cut
      load_bins(a.ws.coarse + (size_t)f * 256, cm);
      load_bins(a.ws.fine + (size_t)f * 256, fn);
    }
    row_stats(a.ws.stats + (size_t)f * a.ws.C, a.ws.C, M, S);
    uint32_t key = 0, c_keep = 0xffffffffu, prefix = 0;
    if (a.top_p < 1.f) {
      const Cut cc = wave_cut(cm, 0ull, a.T);
      if (cc.bin < 0) {  // keep all: renormalise by the total mass
        scale = (float)(1.0 / ((double)cc.total * 0x1p-52));
      } else {
        const uint32_t* fine = a.ws.fine + (size_t)f * 256;
        // mass of fine bin b = count * mass of that exact logit
        uint64_t v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t b = 255 - 4 * lane - e, n = fn[e];
          v[e] = n ? (uint64_t)n * mass_of(prob_of(key_bf(((uint32_t)cc.bin << 8) | b), a.temp, M, S)) : 0ull;
        }
        const Cut fc = wave_cut(v, cc.above, a.T);
        const int fb = fc.bin < 0 ? 0 : fc.bin;  // always found: the coarse bin's mass straddles T
        key = ((uint32_t)cc.bin << 8) | (uint32_t)fb;
        // ties of the cut key in earlier chunks
        uint32_t n_before = 0;
        for (int u = lane; u < c; u += 64) n_before += a.ws.finec[((size_t)f * a.ws.C + u) * 256 + fb];
        const uint32_t n_t = fine[fb];
        const uint64_t w = mass_of(prob_of(key_bf(key), a.temp, M, S));
        const uint64_t C3 = fc.bin < 0 ? cc.above : fc.above;
        uint64_t keep = n_t;
        if (w > 0 && a.T >= C3) keep = min((uint64_t)n_t, (a.T - C3) / w + 1ull);
        c_keep = (uint32_t)keep;
        scale = (float)(1.0 / ((double)(C3 + keep * w) * 0x1p-52));
        prefix = wave_sum(n_before);
      }
    }
    if (t == 0) {
      M_sh = M;
      S_sh = S;
      scale_sh = scale;
      cut_key_sh = key;
      c_keep_sh = c_keep;
      prefix_sh = prefix;
    }
  }
  float x[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = scaled_of(h[e], a.temp);
  __syncthreads();
  const float M = M_sh, S = S_sh, scale = scale_sh;
  const uint32_t cut_key = cut_key_sh, c_keep = c_keep_sh;
  // column rank of this thread's ties of the cut key (columns ascend with the thread, then e)
  uint32_t rank = 0;
  const bool cut = a.top_p < 1.f && c_keep != 0xffffffffu;  // uniform per block
  if (cut) {
    uint32_t in_wave = 0, before = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint64_t m = __ballot(i + e < a.n && bf_key(h[e]) == cut_key);
      in_wave += __popcll(m);
      before += __popcll(m & ((1ull << lane) - 1));
    }
    if (lane == 0) ties_sh[t >> 6] = in_wave;
    __syncthreads();
    rank = prefix_sh + before;
    for (int w = 0; w < t >> 6; ++w) rank += ties_sh[w];
  }
  float p[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t k = bf_key(h[e]);
    bool keep = true;
    if (cut) {
      keep = k > cut_key;
      if (k == cut_key && i + e < a.n) keep = rank++ < c_keep;
    }
    const float pv = prob_scaled(x[e], M, S);
    p[e] = keep ? (a.top_p < 1.f ? pv * scale : pv) : 0.f;
  }
  if (!a.vocab && i + 3 < a.n) {
    *(float4*)(out + i) = make_float4(p[0], p[1], p[2], p[3]);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (i + e < a.n) out[a.vocab ? a.vocab[i + e] : i + e] = p[e];
  }
}

// ------------------------------------------------------------------- Gumbel top-k
struct TopkArgs {
  const float* q;
  int64_t ldq;
  int rows, V, k;
  const int* meta;
  int level;
  Rng rng;
  int* out_tok;   // [rows][k], -1 past min(k, support)
  float* out_lp;  // log q of each drawn token
  SmpWs ws;
};

__device__ __forceinline__ void load4_f32(const float* row, int i, int n, float v[4]) {
  if (i + 3 < n) {
    const float4 q = *(const float4*)(row + i);
    v[0] = q.x;
    v[1] = q.y;
    v[2] = q.z;
    v[3] = q.w;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = i + e < n ? row[i + e] : 0.f;
  }
}

// The k best of the records each lane holds 4 of, best first: out[r] from lane 0.
__device__ __forceinline__ void wave_topk(float (&kk)[4], int (&ki)[4], int k, KeyIdx* out) {
  for (int r = 0; r < k; ++r) {
    float bk = kk[0];
    int bi = ki[0];
#pragma unroll
    for (int e = 1; e < 4; ++e)
      if (better(kk[e], ki[e], bk, bi)) {
        bk = kk[e];
        bi = ki[e];
      }
    const KeyIdx w = wave_argmax(bk, bi);
    if ((threadIdx.x & 63) == 0) out[r] = w;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (ki[e] == w.idx) {
        kk[e] = -1.f;
        ki[e] = NO_IDX;
      }
  }
}

// Per chunk: the k largest keys q(y) / E(y) (E ~ Exp(1) from the PROPOSE stream) and the
// support size. Every wave takes the k best of its 256 columns, then the first wave the k best of the
// 16 lists: one barrier however large k is (a workgroup-wide maximum per draw took two each: 9.4 us for
// 6 rows of 128256 and k = 2, now 7.0).
__global__ __launch_bounds__(SMP_THREADS) void gumbel_chunk_kernel(TopkArgs a) {
  __shared__ KeyIdx list[16][SMP_MAXK];
  __shared__ int red_i[16];
  int F, base;
  frontier_rows(a.meta, a.level, a.rows, F, base);
  const int f = blockIdx.y, c = blockIdx.x, t = threadIdx.x, lane = t & 63;
  if (f >= F) return;
  const float* q = a.q + (size_t)(base + f) * a.ldq;
  const int i = c * SMP_CHUNK + t * 4;
  float v[4];
  load4_f32(q, i, a.V, v);
  const U4 r = rng_block(a.rng, (uint32_t)(i >> 2), (uint32_t)f | ((uint32_t)a.level << 16), TAG_PROPOSE);
  float kk[4];
  int ki[4];
  uint32_t on = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    on |= (uint32_t)(i + e < a.V && v[e] > 0.f) << e;
    kk[e] = -1.f;
    ki[e] = NO_IDX;
  }
  int supp = __popc(on);
  for_active(on, [&](int e) {
    const float key = get4(v, e) / exp1_from_bits(u4_get(r, e));
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (u == e) {
        kk[u] = key;
        ki[u] = i + u;
      }
  });
  wave_topk(kk, ki, a.k, list[t >> 6]);
  supp = wave_sum(supp);
  if (lane == 0) red_i[t >> 6] = supp;
  __syncthreads();
  if (t >= 64) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) {  // 16 k <= 256 records, 4 a lane
    const int j = lane + 64 * e;
    const bool on = j < 16 * a.k;
    kk[e] = on ? list[j / a.k][j % a.k].key : -1.f;
    ki[e] = on ? list[j / a.k][j % a.k].idx : NO_IDX;
  }
  wave_topk(kk, ki, a.k, a.ws.cand + ((size_t)f * a.ws.C + c) * SMP_MAXK);
  if (t == 0) a.ws.csupp[(size_t)f * a.ws.C + c] = sum16(red_i);
}

// Per row: merge the chunks' candidates; write min(k, support) tokens in draw order and log q of each.
// Wave w takes records 256 w .. of the row's C k (<= 4096), so up to 256 records need the first wave alone.
__global__ __launch_bounds__(SMP_THREADS) void gumbel_merge_kernel(TopkArgs a) {
  __shared__ KeyIdx list[16][SMP_MAXK];
  __shared__ KeyIdx best[SMP_MAXK];
  int F, base;
  frontier_rows(a.meta, a.level, a.rows, F, base);
  const int f = blockIdx.x, t = threadIdx.x, lane = t & 63, w = t >> 6;
  if (f >= F) return;
  const int C = a.ws.C;
  const int total = C * a.k;
  const float* q = a.q + (size_t)(base + f) * a.ldq;
  const int waves = (total + 255) / 256;  // <= 16: the launch has this many
  float kk[4];
  int ki[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int j = 256 * w + lane + 64 * e;
    const KeyIdx v = j < total ? a.ws.cand[((size_t)f * C + j / a.k) * SMP_MAXK + j % a.k] : KeyIdx{-1.f, NO_IDX};
    kk[e] = v.key;
    ki[e] = v.idx;
  }
  int supp = 0;
  if (w == 0)
    for (int u = lane; u < C; u += 64) supp += a.ws.csupp[(size_t)f * C + u];
  if (waves > 1) {
    wave_topk(kk, ki, a.k, list[w]);
    __syncthreads();
    if (w > 0) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = lane + 64 * e;
      const bool on = j < waves * a.k;
      kk[e] = on ? list[j / a.k][j % a.k].key : -1.f;
      ki[e] = on ? list[j / a.k][j % a.k].idx : NO_IDX;
    }
  }
  const int take = min(a.k, wave_sum(supp));
  wave_topk(kk, ki, a.k, best);  // one wave: its lanes run in step, lane 0's writes are in order
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (lane < a.k) {
    const int tok = lane < take && best[lane].idx != NO_IDX ? best[lane].idx : -1;
    a.out_tok[f * a.k + lane] = tok;
    a.out_lp[f * a.k + lane] = tok >= 0 ? logf(q[tok]) : 0.f;
  }
}

// ------------------------------------------------------------- categorical draws
// One draw per row: argmax_y p(y) / E(y), E from the DRAW stream with counter (y / 4, row).
__global__ __launch_bounds__(SMP_THREADS) void draw_chunk_kernel(const float* __restrict__ P, int64_t ldp, int V,
                                                                 Rng rng, SmpWs ws) {
  __shared__ KeyIdx red[16];
  const int row = blockIdx.y, c = blockIdx.x, t = threadIdx.x;
  const int i = c * SMP_CHUNK + t * 4;
  float v[4];
  load4_f32(P + (size_t)row * ldp, i, V, v);
  const U4 r = rng_block(rng, (uint32_t)(i >> 2), (uint32_t)row, TAG_DRAW);
  float best = -1.f;
  int bi = NO_IDX;
  uint32_t on = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) on |= (uint32_t)(i + e < V && v[e] > 0.f) << e;
  for_active(on, [&](int e) {
    const float key = get4(v, e) / exp1_from_bits(u4_get(r, e));
    if (better(key, i + e, best, bi)) {
      best = key;
      bi = i + e;
    }
  });
  KeyIdx w = wave_argmax(best, bi);
  if ((t & 63) == 0) red[t >> 6] = w;
  __syncthreads();
  if (t >= 64) return;
  w = argmax16(red);
  if (t == 0) ws.arg[(size_t)row * ws.C + c] = w;
}

__device__ __forceinline__ KeyIdx merge_chunks(const KeyIdx* part, int C) {
  KeyIdx b{-1.f, NO_IDX};
  for (int c = 0; c < C; ++c)
    if (better(part[c].key, part[c].idx, b.key, b.idx)) b = part[c];
  return b;
}

__global__ void draw_merge_kernel(int rows, SmpWs ws, int* __restrict__ out_tok) {
  const int row = blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= rows) return;
  const KeyIdx b = merge_chunks(ws.arg + (size_t)row * ws.C, ws.C);
  out_tok[row] = b.idx == NO_IDX ? 0 : b.idx;
}

// ----------------------------------------------------------- speculative acceptance
// Verify row r holds node cur = r - 1 (root: r = 0). State j of a node = after its first j
// children (rank order, q0(x) > 0) were rejected:
//   q_0 = q0, q_j(y) = q0(y) [y not rejected] / zq[j]  (zq[j] = sum q0 - sum of rejected q0),
//   p_0 = p,  p_j = (p_{j-1} - q_{j-1})+ / zr[j] when zr[j] = sum (p_{j-1} - q_{j-1})+ > 0,
//             p_j = p_{j-1} otherwise,
// and bonus[j] = the categorical draw from p_j (one shared Exp(1) vector per round: only one
// state's draw is ever used, and which one is decided by the acceptance uniforms alone).
// The first launch over all rows and chunks produces the partials of bonus[0] and of state 1 (its
// residual p - q0 needs no sums), pass j >= 2 those of zr[j] and bonus[j]; partials are combined by whoever
// needs them (the next pass, the walk), always by the same wave reduction (combine_states), so every
// reader sees the same values. The passes are bound by their chains of dependent loads (tree -> tokens ->
// q0), not by bytes: the first one stores each row's child list for the others, loads the rows of P and Q
// beside that chain, and the walk resolves every node at once, one wave each. us for 16 rows of 128256,
// 3 children, before / after: pass 0 13.4 and pass 1 12.0 / first pass 11.4, pass j 12.0 / 8.4, walk
// 8.4 / 6.6.
struct AcceptArgs {
  SsdTree tree;
  const float* P;
  int64_t ldp;
  const float* Q;
  int64_t ldq;
  int V;
  int rows;      // verify rows in P and in the workspace
  int max_kids;  // children considered per node (the launch runs this many rejection passes)
  Rng rng;
  SmpWs ws;
};

constexpr int SMP_MAXNODES = 63;  // verify nodes (rows = nodes + 1 <= 64)

__device__ __forceinline__ int verify_nodes(const SsdTree& t) { return min(t.vmeta[0], SMP_MAXNODES); }

__device__ __forceinline__ const float* q_row(const AcceptArgs& a, int cur) {
  return a.Q + (size_t)(cur < 0 ? 0 : 1 + a.tree.vorig[cur]) * a.ldq;
}

// Children of cur in rank order (ranks are distinct among siblings: they are draw order),
// skipping those with q0(x) <= 0 (verify.py:77-78), built by a whole workgroup of at least 64
// threads (tree nodes staged in LDS; each child finds its position by counting siblings of lower
// rank). Result in `k` (shared), valid after return.
__device__ __forceinline__ void node_kids_block(const AcceptArgs& a, int cur, NodeKids& k, int* sh_par,
                                                int* sh_rank, int* sh_pos) {
  const int vn = verify_nodes(a.tree);
  const int t = threadIdx.x;
  if (t < vn) {
    sh_par[t] = a.tree.vparents[t];
    sh_rank[t] = a.tree.vranks[t];
  }
  if (t < SMP_MAXK) sh_pos[t] = -1;
  __syncthreads();
  if (t < vn && sh_par[t] == cur) {
    int pos = 0;
    for (int o = 0; o < vn; ++o) pos += sh_par[o] == cur && sh_rank[o] < sh_rank[t];
    if (pos < SMP_MAXK) sh_pos[pos] = t;
  }
  __syncthreads();
  if (t < 64) {  // wave 0: lane i takes rank position i (positions are dense from 0), loads in parallel
    const float* q0 = q_row(a, cur);
    int pos = t < a.max_kids && t < SMP_MAXK ? sh_pos[t] : -1;
    // the list ends at the first empty position, as a rank-order scan would stop there
    const uint64_t filled = __ballot(pos >= 0);
    if (t >= __ffsll((unsigned long long)~filled) - 1) pos = -1;
    const int x = pos >= 0 ? a.tree.vtokens[pos] : 0;
    const bool keep = pos >= 0 && q0[x] > 0.f;
    const uint64_t m = __ballot(keep);
    if (keep) {
      const int slot = __popcll(m & ((1ull << t) - 1));  // kept children of lower rank
      k.kid[slot] = pos;
      k.tok[slot] = x;
    }
    if (t == 0) k.n = __popcll(m);
  }
  __syncthreads();
}

struct StateScalars {
  double s0;
  int supp;
  float zr[SMP_MAXK + 1];  // zr[j] for j >= 1 (0 when the residual had no mass)
  float zq[SMP_MAXK + 1];  // zq[0] = 1
};

// Combine the chunk partials of row r: q0's mass and support, and states 1..upto. Called by a
// whole wave: lane l sums chunks l, l + 64, ..., then the wave reduces; every lane returns the
// same values, and every reader (the passes and the walk) uses this code, so all see the same.
__device__ __forceinline__ void combine_states(const AcceptArgs& a, int r, const float* q0, const NodeKids& k,
                                               int upto, StateScalars& s) {
  const int C = a.ws.C, lane = threadIdx.x & 63;
  double s0 = 0.0;
  int supp = 0;
  for (int c = lane; c < C; c += 64) {
    s0 += a.ws.s0[(size_t)r * C + c];
    supp += a.ws.supp[(size_t)r * C + c];
  }
  double z[SMP_MAXK + 1];
#pragma unroll
  for (int j = 1; j <= SMP_MAXK; ++j) {
    z[j] = 0.0;
    if (j <= upto)
      for (int c = lane; c < C; c += 64) z[j] += a.ws.zr[((size_t)r * (SMP_MAXK + 1) + j) * C + c];
  }
  s0 = wave_sum(s0);
  s.s0 = s0;
  s.supp = wave_sum(supp);
  s.zr[0] = 0.f;
  s.zq[0] = 1.f;
  double zq = s0;
#pragma unroll
  for (int j = 1; j <= SMP_MAXK; ++j) {
    if (j <= upto) {  // uniform
      const double zj = wave_sum(z[j]);
      s.zr[j] = zj > 0.0 ? (float)zj : 0.f;
      zq -= (double)q0[k.tok[j - 1]];
      s.zq[j] = (float)zq;
    }
  }
}

// p_j(y) for the state scalars, evaluated at one column. `rej` holds the rejected tokens
// x_1..x_j (only the first j entries are read); the passes and the walk share this code.
__device__ __forceinline__ float chain_p(float p0, float q0, int y, int j, const float* zr, const float* zq,
                                         const int* rej) {
  float pv = p0;
  for (int i = 1; i <= j; ++i) {
    float qv = q0;  // q_{i-1}(y)
    if (i - 1 > 0) {
      bool r = false;
      for (int u = 0; u < i - 1; ++u) r |= rej[u] == y;
      qv = r ? 0.f : q0 / zq[i - 1];
    }
    if (zr[i] > 0.f) pv = fmaxf(pv - qv, 0.f) / zr[i];
  }
  return pv;
}

// Pass 0 and 1: the draws from p_0 and p_1 per chunk, the mass of p_1's residual, q0's mass and support.
// One more workgroup per row (chunk index C) stores the row's child list.
__global__ __launch_bounds__(SMP_THREADS) void state01_kernel(AcceptArgs a) {
  __shared__ KeyIdx red0[16], red1[16];
  __shared__ double red_s[16], red_z[16];
  __shared__ int red_i[16];
  __shared__ int sh_par[64], sh_rank[64], sh_pos[SMP_MAXK];
  __shared__ NodeKids kids;
  const int r = blockIdx.y, c = blockIdx.x, t = threadIdx.x;
  const int cur = r - 1;
  const int i = c * SMP_CHUNK + t * 4;
  float p[4], q[4] = {0.f, 0.f, 0.f, 0.f};
  if (c < a.ws.C) load4_f32(a.P + (size_t)r * a.ldp, i, a.V, p);
  const int vn = verify_nodes(a.tree);
  if (r > vn) return;
  if (c == a.ws.C) {
    node_kids_block(a, cur, kids, sh_par, sh_rank, sh_pos);
    if (t < (int)(sizeof(NodeKids) / 4)) ((int*)&a.ws.kids[r])[t] = ((const int*)&kids)[t];
    return;
  }
  // a row without children in the tree has no draft row (its node may never have proposed)
  if (__syncthreads_or(t < vn && a.max_kids > 0 && a.tree.vparents[t] == cur)) load4_f32(q_row(a, cur), i, a.V, q);
  const U4 rb = rng_block(a.rng, (uint32_t)(i >> 2), 0u, TAG_BONUS);
  float best0 = -1.f, best1 = -1.f;
  int bi0 = NO_IDX, bi1 = NO_IDX, supp = 0;
  double s0 = 0.0, zs = 0.0;
  uint32_t on = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    s0 += (double)q[e];
    supp += q[e] > 0.f;
    if (i + e < a.V) zs += (double)fmaxf(p[e] - q[e], 0.f);  // (p_0 - q_0)+
    on |= (uint32_t)(i + e < a.V && p[e] > 0.f) << e;
  }
  for_active(on, [&](int e) {
    const float pe = get4(p, e), res = fmaxf(pe - get4(q, e), 0.f);
    const float ex = exp1_from_bits(u4_get(rb, e));
    const float k0 = pe / ex, k1 = res / ex;
    if (better(k0, i + e, best0, bi0)) {
      best0 = k0;
      bi0 = i + e;
    }
    if (res > 0.f && better(k1, i + e, best1, bi1)) {
      best1 = k1;
      bi1 = i + e;
    }
  });
  KeyIdx w0 = wave_argmax(best0, bi0), w1 = wave_argmax(best1, bi1);
  s0 = wave_sum(s0);
  zs = wave_sum(zs);
  supp = wave_sum(supp);
  if ((t & 63) == 0) {
    red0[t >> 6] = w0;
    red1[t >> 6] = w1;
    red_s[t >> 6] = s0;
    red_z[t >> 6] = zs;
    red_i[t >> 6] = supp;
  }
  __syncthreads();
  if (t >= 64) return;
  w0 = argmax16(red0);
  w1 = argmax16(red1);
  if (t == 0) {
    const int C = a.ws.C;
    a.ws.bon[((size_t)r * (SMP_MAXK + 1) + 0) * C + c] = w0;
    // of a row without children, state 1 and q0's sums are not read
    a.ws.bon[((size_t)r * (SMP_MAXK + 1) + 1) * C + c] = w1;
    a.ws.zr[((size_t)r * (SMP_MAXK + 1) + 1) * C + c] = sum16(red_z);
    a.ws.s0[(size_t)r * C + c] = sum16(red_s);
    a.ws.supp[(size_t)r * C + c] = sum16(red_i);
  }
}

// Pass j >= 2: residual of state j-1 -> chunk partials of zr[j] and of the draw from p_j.
__global__ __launch_bounds__(SMP_THREADS) void statej_kernel(AcceptArgs a, int j) {
  __shared__ KeyIdx red[16];
  __shared__ double red_d[16];
  __shared__ NodeKids kids;
  __shared__ StateScalars st;
  const int r = blockIdx.y, c = blockIdx.x, t = threadIdx.x;
  if (r > verify_nodes(a.tree)) return;
  const int n = a.ws.kids[r].n;
  const float* q0 = q_row(a, r - 1);
  if (n < j) return;  // uniform: this node has fewer children
  const int i = c * SMP_CHUNK + t * 4;
  float p[4], q[4];
  load4_f32(a.P + (size_t)r * a.ldp, i, a.V, p);
  load4_f32(q0, i, a.V, q);
  if (t < (int)(sizeof(NodeKids) / 4)) ((int*)&kids)[t] = ((const int*)&a.ws.kids[r])[t];
  const U4 rb = rng_block(a.rng, (uint32_t)(i >> 2), 0u, TAG_BONUS);
  __syncthreads();
  if (t < 64) combine_states(a, r, q0, kids, j - 1, st);  // wave 0; its lanes store the same values
  __syncthreads();
  double zs = 0.0;
  float best = -1.f;
  int bi = NO_IDX;
  // p_0(y) = 0 leaves no residual in any state as long as the draft mass left is positive (rounding can
  // leave it at or below 0 once what remains is under 1e-16 of it)
  const bool all = !(st.zq[j - 1] > 0.f);
  uint32_t on = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) on |= (uint32_t)(i + e < a.V && (p[e] > 0.f || all)) << e;
  for_active(on, [&](int e) {
    const int y = i + e;
    const float qe = get4(q, e);
    const float pprev = chain_p(get4(p, e), qe, y, j - 1, st.zr, st.zq, kids.tok);
    bool rj = false;
    for (int u = 0; u < j - 1; ++u) rj |= kids.tok[u] == y;
    const float qprev = rj ? 0.f : qe / st.zq[j - 1];
    const float res = fmaxf(pprev - qprev, 0.f);
    zs += (double)res;
    if (res > 0.f) {
      const float key = res / exp1_from_bits(u4_get(rb, e));
      if (better(key, y, best, bi)) {
        best = key;
        bi = y;
      }
    }
  });
  zs = wave_sum(zs);
  KeyIdx w = wave_argmax(best, bi);
  if ((t & 63) == 0) {
    red_d[t >> 6] = zs;
    red[t >> 6] = w;
  }
  __syncthreads();
  if (t >= 64) return;
  w = argmax16(red);
  if (t == 0) {
    const int C = a.ws.C;
    a.ws.zr[((size_t)r * (SMP_MAXK + 1) + j) * C + c] = sum16(red_d);
    a.ws.bon[((size_t)r * (SMP_MAXK + 1) + j) * C + c] = w;
  }
}

// The walk of sample_verify over the state scalars, then the same bookkeeping as the greedy
// walk: result = [n_new, tokens...], compaction sources, next root token. What happens at a node --
// which child is accepted, or which bonus token is drawn -- depends on that node's row alone, so wave w
// resolves rows w, w + 16, ... (all lanes with the same values; the state sums and the bonus merge are
// wave-wide operations), and one thread then follows the path.
__global__ __launch_bounds__(SMP_THREADS) void sample_walk_kernel(AcceptArgs a, int committed, int* result,
                                                                 int* keep_src, int* n_keep, int* root_token) {
  __shared__ int next[SMP_MAXNODES + 1], drawn[SMP_MAXNODES + 1], tok_sh[SMP_MAXNODES + 1];
  __shared__ NodeKids kids_sh[16];
  __shared__ StateScalars st_sh[16];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int C = a.ws.C, n_rows = min(verify_nodes(a.tree) + 1, a.rows);
  // every node's token: a row's accepted child may lie beyond the launch's rows
  if (threadIdx.x < verify_nodes(a.tree)) tok_sh[threadIdx.x] = a.tree.vtokens[threadIdx.x];
  NodeKids& kids = kids_sh[wv];  // this wave's own, read back by the lanes that wrote them or in step with them
  StateScalars& s = st_sh[wv];
  for (int r = wv; r < n_rows; r += 16) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane < (int)(sizeof(NodeKids) / 4)) ((int*)&kids)[lane] = ((const int*)&a.ws.kids[r])[lane];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int kn = kids.n;
    const float* q0 = q_row(a, r - 1);
    const float* p = a.P + (size_t)r * a.ldp;
    if (kn > 0) combine_states(a, r, q0, kids, kn, s);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // lane i: child i's p and q0
    const int x_l = lane < kn ? kids.tok[lane] : 0;
    const float p_l = lane < kn ? p[x_l] : 0.f, q_l = lane < kn ? q0[x_l] : 0.f;
    int chosen = -1, j = 0;
    for (int i = 0; i < kn; ++i) {  // j == i: the children before i were rejected
      const int x = __shfl(x_l, i);
      const float q0x = __shfl(q_l, i);
      const float pj = chain_p(__shfl(p_l, i), q0x, x, j, s.zr, s.zq, kids.tok);
      const float qj = j == 0 ? q0x : q0x / s.zq[j];
      const double u = uniform_from_bits(rng_block(a.rng, (uint32_t)j, (uint32_t)r, TAG_ACCEPT).x);
      if (u < (double)fminf(1.f, pj / qj)) {
        chosen = kids.kid[i];
        break;
      }
      ++j;
      if (j >= s.supp) break;  // no draft mass left
    }
    KeyIdx b{-1.f, NO_IDX};
    if (chosen < 0) {
      int jj = j;
      while (jj > 0 && !(s.zr[jj] > 0.f)) --jj;  // p_j == p_{j-1} when the residual had no mass
      // the categorical draw from p_jj: the best of the chunks' records (a strict order on
      // (key, column), so any merge order gives the same record)
      const KeyIdx* part = a.ws.bon + ((size_t)r * (SMP_MAXK + 1) + jj) * C;
      for (int c = lane; c < C; c += 64)
        if (better(part[c].key, part[c].idx, b.key, b.idx)) b = part[c];
      b = wave_argmax(b.key, b.idx);
    }
    if (lane == 0) {
      next[r] = chosen;
      drawn[r] = b.idx == NO_IDX ? 0 : b.idx;
    }
  }
  __syncthreads();
  if (threadIdx.x) return;
  int cur = -1, n_acc = 0, bonus = 0;
  for (int step = 0; step <= SMP_MAXDEPTH; ++step) {
    const int r = cur + 1;
    if (r >= n_rows) break;  // a tree larger than the launch's rows (the engine never makes one)
    if (next[r] < 0) {
      bonus = drawn[r];
      break;
    }
    cur = next[r];
    result[1 + n_acc] = tok_sh[cur];
    keep_src[1 + n_acc] = committed + 1 + cur;
    ++n_acc;
  }
  result[1 + n_acc] = bonus;
  result[0] = n_acc + 1;
  keep_src[0] = committed;
  *n_keep = n_acc + 1;
  *root_token = bonus;
}

// ------------------------------------------------------ batched acceptance trials
// Many independent rounds of proposal + acceptance over one fixed set of per-node distributions
// (row 0 the root, row 1 + v node v; P = warped target, Q = warped draft of the node's
// children), one wave per trial, trial t drawing with round counter counter0 + t. The tree is
// unpruned with branch[d] children per node at level d, numbered level by level (level L node with
// in-level index f has children start[L + 1] + f * branch[L + 1] + i, i = draw order). Each trial
// draws only the children on its walk; every draw and decision uses the engine's streams,
// counters and formulas (gumbel_chunk / state01 / statej / sample_walk above): Gumbel keys
// q / Exp(1) from the PROPOSE stream at (column / 4, f | level << 16), acceptance uniforms at
// (rejections, row), residual states through chain_p, the bonus race on the unnormalised
// residual at (column / 4, 0). Sums run over each row's support list (columns where P or Q is
// nonzero; every other column contributes nothing) in double, in lane-strided order. Only the
// sums' rounding order differs from the per-round kernels, so a trial reproduces the engine's
// round with the same counter decision for decision.
constexpr int TRIAL_MAXD = 8;

struct TrialArgs {
  const float* P;
  int64_t ldp;
  const float* Q;
  int64_t ldq;
  const int* cols;  // support columns of row r: cols[off[r] .. off[r + 1]), ascending
  const int* off;
  int depth;
  int branch[TRIAL_MAXD];
  int start[TRIAL_MAXD + 1];
  uint64_t seed, counter0;
  int trials;
  int* out_tok;  // [trials][depth + 1]: accepted tokens, then the bonus
  int* out_n;    // [trials]
};


// q_{j-1}(y) as statej_kernel computes it: rejected tokens have no draft mass left.
__device__ __forceinline__ float trial_qprev(float q0, int y, int j, const float* zq, const int* rej) {
  if (j - 1 <= 0) return q0;
  bool r = false;
  for (int u = 0; u < j - 1; ++u) r |= rej[u] == y;
  return r ? 0.f : q0 / zq[j - 1];
}

__global__ __launch_bounds__(256) void accept_trials_kernel(TrialArgs a) {
  const int lane = threadIdx.x & 63;
  const int trial = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (trial >= a.trials) return;  // whole wave
  const uint64_t ctr = a.counter0 + (uint64_t)trial;
  const Rng rng{(uint32_t)a.seed, (uint32_t)(a.seed >> 32), (uint32_t)ctr, (uint32_t)((ctr >> 32) << 8)};
  int cur = -1, lv = 0, f = 0, n_out = 0, bonus = 0;
  for (;;) {
    const int r = cur + 1;
    const float* p = a.P + (size_t)r * a.ldp;
    const float* q = a.Q + (size_t)r * a.ldq;
    const int* cs = a.cols + a.off[r];
    const int ns = a.off[r + 1] - a.off[r];
    int rej[SMP_MAXK];
    float zr[SMP_MAXK + 1], zq[SMP_MAXK + 1];
    zr[0] = 0.f;
    zq[0] = 1.f;
    int j = 0, chosen = -1;
    if (lv < a.depth) {
      const int k = a.branch[lv];
      // q0's mass and support count, then min(k, support) children by Gumbel top-k
      double s0 = 0.0;
      int supp = 0;
      for (int e = lane; e < ns; e += 64) {
        const float qv = q[cs[e]];
        s0 += (double)qv;
        supp += qv > 0.f;
      }
      s0 = wave_sum(s0);
      supp = wave_sum(supp);
      int take = min(k, supp);
      int tok[SMP_MAXK];
      for (int c = 0; c < take; ++c) {
        float bk = -1.f;
        int bi = NO_IDX;
        for (int e = lane; e < ns; e += 64) {
          const int y = cs[e];
          const float qv = q[y];
          if (!(qv > 0.f)) continue;
          bool taken = false;
          for (int u = 0; u < c; ++u) taken |= tok[u] == y;
          if (taken) continue;
          const U4 rb = rng_block(rng, (uint32_t)(y >> 2), (uint32_t)f | ((uint32_t)lv << 16), TAG_PROPOSE);
          const float key = qv / exp1_from_bits(u4_get(rb, y & 3));
          if (better(key, y, bk, bi)) {
            bk = key;
            bi = y;
          }
        }
        const KeyIdx w = wave_argmax(bk, bi);
        if (w.idx == NO_IDX) {  // no candidate left (cannot happen below the support count)
          take = c;
          break;
        }
        tok[c] = w.idx;
      }
      // the walk over the children in draw order (sample_walk_kernel)
      double zqd = s0;
      for (int i = 0; i < take; ++i) {
        const int x = tok[i];
        const float q0x = q[x];
        const float pj = chain_p(p[x], q0x, x, j, zr, zq, rej);
        const float qj = j == 0 ? q0x : q0x / zq[j];
        const double u = uniform_from_bits(rng_block(rng, (uint32_t)j, (uint32_t)r, TAG_ACCEPT).x);
        if (u < (double)fminf(1.f, pj / qj)) {
          chosen = i;
          break;
        }
        rej[j] = x;
        ++j;
        zqd -= (double)q0x;
        zq[j] = (float)zqd;
        // residual mass of state j (statej_kernel with its first j children rejected)
        double z = 0.0;
        for (int e = lane; e < ns; e += 64) {
          const int y = cs[e];
          const float pprev = chain_p(p[y], q[y], y, j - 1, zr, zq, rej);
          z += (double)fmaxf(pprev - trial_qprev(q[y], y, j, zq, rej), 0.f);
        }
        z = wave_sum(z);
        zr[j] = z > 0.0 ? (float)z : 0.f;
        if (j >= supp) break;  // no draft mass left
      }
      if (chosen >= 0) {
        const int fc = f * k + chosen;  // in-level index of the accepted child
        if (lane == 0) a.out_tok[(size_t)trial * (a.depth + 1) + n_out] = tok[chosen];
        ++n_out;
        cur = a.start[lv] + fc;
        f = fc;
        ++lv;
        continue;
      }
    }
    // bonus: the categorical draw from the last state with residual mass (state 0 at a leaf)
    int jj = j;
    while (jj > 0 && !(zr[jj] > 0.f)) --jj;
    float bk = -1.f;
    int bi = NO_IDX;
    for (int e = lane; e < ns; e += 64) {
      const int y = cs[e];
      float w;
      if (jj == 0) {
        w = p[y];
      } else {
        const float pprev = chain_p(p[y], q[y], y, jj - 1, zr, zq, rej);
        w = fmaxf(pprev - trial_qprev(q[y], y, jj, zq, rej), 0.f);
      }
      if (!(w > 0.f)) continue;
      const float key = w / exp1_from_bits(u4_get(rng_block(rng, (uint32_t)(y >> 2), 0u, TAG_BONUS), y & 3));
      if (better(key, y, bk, bi)) {
        bk = key;
        bi = y;
      }
    }
    const KeyIdx b = wave_argmax(bk, bi);
    bonus = b.idx == NO_IDX ? 0 : b.idx;
    break;
  }
  if (lane == 0) {
    a.out_tok[(size_t)trial * (a.depth + 1) + n_out] = bonus;
    a.out_n[trial] = n_out + 1;
  }
}

// ------------------------------------------------- top-64 draws (batched generation)
// sample_next of ssd/data/generate_selfdistill.py:50-60: the 64 largest logits of a row, the
// temperature + nucleus warp of those 64 alone, one categorical draw among them.
// Candidates are 64-bit records key << 32 | ~column (key = the bf16 logit's monotone key), so
// a larger record is a larger logit or, among equal logits, a lower column; 0 marks no entry.
constexpr int T64 = 64;
constexpr int T64_MAXC = 64;  // chunks per row (rows up to 262144 columns)

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int o) {
  const uint32_t lo = __shfl_xor((uint32_t)v, o), hi = __shfl_xor((uint32_t)(v >> 32), o);
  return ((uint64_t)hi << 32) | lo;
}

// Chunk pass: the chunk's min(64, columns) best records, sorted best first, into
// parts[row][chunk][64] (0-padded). The 64th-best key is found by two 256-bin count histograms
// (key high byte, then low byte inside the cut bin); the records above it are collected in any
// order, its ties by column rank (a block scan of per-thread tie counts: thread order is column
// order), then one wave sorts the 64 (bitonic network over the lanes).
__global__ __launch_bounds__(SMP_THREADS) void top64_chunk_kernel(const bf16_t* __restrict__ logits, int64_t ld,
                                                                  int n, int C, uint64_t* __restrict__ parts) {
  __shared__ uint32_t hist[256];
  __shared__ uint32_t red[16];
  __shared__ uint64_t list[T64];
  __shared__ uint32_t cut_sh, above_sh, cnt_sh;
  const int row = blockIdx.y, c = blockIdx.x, t = threadIdx.x;
  const int i = c * SMP_CHUNK + t * 4;
  uint32_t h[4], k[4];
  load4_bf16(logits + (size_t)row * ld, i, n, h);
#pragma unroll
  for (int e = 0; e < 4; ++e) k[e] = bf_key(h[e]);
  const uint32_t want = (uint32_t)min(T64, n - c * SMP_CHUNK);
  if (t < 256) hist[t] = 0;
  if (t == 0) cnt_sh = 0;
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (i + e < n) atomicAdd(&hist[k[e] >> 8], 1u);
  __syncthreads();
  // bins from the largest key down: the bin holding the want-th record
  uint32_t hv = t < 256 ? hist[255 - t] : 0u;
  uint32_t incl = block_scan(hv, red);
  if (t < 256 && hv > 0 && incl - hv < want && incl >= want) {
    cut_sh = 255u - (uint32_t)t;
    above_sh = incl - hv;
  }
  __syncthreads();
  const uint32_t cb = cut_sh, above1 = above_sh;
  if (t < 256) hist[t] = 0;
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (i + e < n && (k[e] >> 8) == cb) atomicAdd(&hist[k[e] & 255u], 1u);
  __syncthreads();
  hv = t < 256 ? hist[255 - t] : 0u;
  incl = above1 + block_scan(hv, red);
  __syncthreads();
  if (t < 256 && hv > 0 && incl - hv < want && incl >= want) {
    cut_sh = (cb << 8) | (255u - (uint32_t)t);
    above_sh = incl - hv;
  }
  __syncthreads();
  const uint32_t ck = cut_sh, above = above_sh, ties_keep = want - above;
  uint32_t nt = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) nt += (i + e < n && k[e] == ck) ? 1u : 0u;
  uint32_t rank = block_scan(nt, red) - nt;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (i + e >= n) continue;
    const uint64_t rec = ((uint64_t)k[e] << 32) | (uint32_t)~(uint32_t)(i + e);
    if (k[e] > ck) {
      list[atomicAdd(&cnt_sh, 1u)] = rec;  // exactly `above` of these
    } else if (k[e] == ck) {
      if (rank < ties_keep) list[above + rank] = rec;
      ++rank;
    }
  }
  __syncthreads();
  if (t < T64) {
    uint64_t x = (uint32_t)t < want ? list[t] : 0ull;
#pragma unroll
    for (int size = 2; size <= T64; size <<= 1) {
#pragma unroll
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        const uint64_t y = shfl_xor_u64(x, stride);
        const bool desc = (t & size) == 0, lo = (t & stride) == 0;
        x = (lo == desc) ? (x > y ? x : y) : (x < y ? x : y);
      }
    }
    parts[((size_t)row * C + c) * T64 + t] = x;
  }
}

// Merge + warp + draw, one wave per row: the 64 best of the chunk lists (lane c walks list c;
// each round takes the wave's largest head), then in rank order p = softmax(v / T), the
// nucleus cut of warp_probs (an entry is dropped when the sequential fp32 cumulative mass before
// it exceeds top_p; none with top_p >= 1) and a Gumbel-max draw over the kept ranks, Exp(1) of
// rank j from the draw stream (counter (j / 4, row), tag TAG_TOP64).
__global__ __launch_bounds__(64) void top64_draw_kernel(const uint64_t* __restrict__ parts, int C, float temp,
                                                        float top_p, Rng rng, int* __restrict__ out_tok) {
  __shared__ uint64_t L[T64_MAXC * T64];
  const int row = blockIdx.x, lane = threadIdx.x;
  const uint64_t* P = parts + (size_t)row * C * T64;
  for (int j = lane; j < C * T64; j += 64) L[j] = P[j];
  __syncthreads();
  int head = 0;
  uint64_t cur = lane < C ? L[lane * T64] : 0ull, mine = 0ull;
  for (int r = 0; r < T64; ++r) {
    uint64_t best = cur;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint64_t y = shfl_xor_u64(best, o);
      best = y > best ? y : best;
    }
    if (r == lane) mine = best;
    if (best != 0ull && cur == best) {  // records are distinct: exactly one lane advances
      ++head;
      cur = head < T64 ? L[lane * T64 + head] : 0ull;
    }
  }
  const bool has = mine != 0ull;
  const float x = has ? bf2f((bf16_t)key_bf((uint32_t)(mine >> 32))) / temp : -INFINITY;
  const float M = __shfl(x, 0);  // rank 0 holds the largest logit
  const float e = has ? expf(x - M) : 0.f;
  float S = e;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) S += __shfl_xor(S, o);
  const float p = e / S;
  float acc = 0.f, cum = 0.f;
  for (int j = 0; j < 64; ++j) {  // torch.cumsum order: rank 0 first
    acc += __shfl(p, j);
    if (j == lane) cum = acc;
  }
  const bool keep = has && p > 0.f && (top_p >= 1.f || !(cum - p > top_p));
  const U4 rb = rng_block(rng, (uint32_t)(lane >> 2), (uint32_t)row, TAG_TOP64);
  const float key = keep ? p / exp1_from_bits(u4_get(rb, lane & 3)) : -1.f;
  const KeyIdx w = wave_argmax(key, lane);
  const int col = (int)~(uint32_t)mine;
  const int pick = __shfl(col, w.idx == NO_IDX ? 0 : w.idx);
  if (lane == 0) out_tok[row] = pick;
}

}  // namespace ssd

using namespace ssd;

SSD_API int ssd_sample_limits(int32_t* out2) {
  if (!out2) return set_error(SSD_EINVAL, "sample_limits: null");
  out2[0] = SMP_MAXK;
  out2[1] = SMP_CHUNK * SMP_MAXC;
  return SSD_OK;
}

SSD_API int64_t ssd_sample_ws_bytes(int rows, int n) {
  if (rows < 0 || n <= 0 || chunks_of(n) > SMP_MAXC) return -1;
  return smp_layout(rows, chunks_of(n), nullptr, nullptr);
}

static int carve(void* ws, int64_t ws_bytes, int rows, int n, SmpWs* out, const char* what) {
  const int64_t need = ssd_sample_ws_bytes(rows, n);
  if (need < 0) return set_error(SSD_ERANGE, "%s: %d columns > %d", what, n, SMP_CHUNK * SMP_MAXC);
  if (!ws || ws_bytes < need)
    return set_error(SSD_EINVAL, "%s: workspace %lld < %lld bytes", what, (long long)ws_bytes, (long long)need);
  smp_layout(rows, chunks_of(n), (char*)ws, out);
  return SSD_OK;
}

SSD_API int ssd_warp_probs_bf16(const uint16_t* logits, int64_t ld, int rows, int n, const int32_t* vocab_ids,
                                const int32_t* vocab_inv, int V, float temperature, float top_p,
                                const int32_t* tree_meta, int level, float* probs, int64_t ldp, void* ws,
                                int64_t ws_bytes, hipStream_t stream) {
  if (!logits || !probs || (vocab_ids && !vocab_inv)) return set_error(SSD_EINVAL, "warp_probs: null pointer");
  if (rows < 0 || n <= 0 || V <= 0 || (!vocab_ids && n != V) || n > V)
    return set_error(SSD_EINVAL, "warp_probs: bad shape rows=%d n=%d V=%d", rows, n, V);
  if (ld % 4 || ld < (n + 3) / 4 * 4 || ldp % 4 || ldp < V)
    return set_error(SSD_EINVAL, "warp_probs: ld %lld / ldp %lld must be multiples of 4 covering the row",
                     (long long)ld, (long long)ldp);
  if (!(temperature > 0.f)) return set_error(SSD_EINVAL, "warp_probs: temperature must be > 0");
  if (tree_meta && (level < 0 || level >= SMP_MAXDEPTH)) return set_error(SSD_ERANGE, "warp_probs: level %d", level);
  if (rows > 65535) return set_error(SSD_ERANGE, "warp_probs: %d rows", rows);
  if (rows == 0) return SSD_OK;
  SmpWs w;
  if (int rc = carve(ws, ws_bytes, rows, V, &w, "warp_probs")) return rc;
  const int C = chunks_of(n), CV = chunks_of(V);
  w.C = C;  // stats / histograms are per logit chunk (the layout was sized for V >= n chunks)
  const double tp = top_p < 0.f ? 0.0 : (double)top_p;
  WarpArgs a{logits, ld, rows, n, vocab_ids, vocab_inv, V, temperature, top_p,
             (uint64_t)fmin(tp * 0x1p52, 0x1p63), tree_meta, level, probs, ldp, w};
  SSD_LAUNCH(warp_stats_kernel, dim3(C, rows), dim3(SMP_THREADS), 0, stream, a);
  if (top_p < 1.f) {
    SSD_LAUNCH(warp_coarse_kernel, dim3(C, rows), dim3(SMP_THREADS), 0, stream, a);
    SSD_LAUNCH(warp_fine_kernel, dim3(C, rows), dim3(SMP_THREADS), 0, stream, a);
  }
  SSD_LAUNCH(warp_final_kernel, dim3(vocab_ids ? max(C, CV) : C, rows), dim3(SMP_THREADS), 0, stream, a);
  return check_launch("warp_probs");
}

SSD_API int ssd_gumbel_topk(const float* probs, int64_t ldp, int rows, int V, int k, const int32_t* tree_meta,
                            int level, uint64_t seed, uint64_t counter, int32_t* out_tok, float* out_lp, void* ws,
                            int64_t ws_bytes, hipStream_t stream) {
  if (!probs || !out_tok || !out_lp) return set_error(SSD_EINVAL, "gumbel_topk: null pointer");
  if (rows < 0 || V <= 0 || ldp % 4 || ldp < V) return set_error(SSD_EINVAL, "gumbel_topk: bad shape");
  if (k < 1 || k > SMP_MAXK) return set_error(SSD_ERANGE, "gumbel_topk: k=%d not in [1, %d]", k, SMP_MAXK);
  if (tree_meta && (level < 0 || level >= SMP_MAXDEPTH)) return set_error(SSD_ERANGE, "gumbel_topk: level %d", level);
  if (rows > 65535) return set_error(SSD_ERANGE, "gumbel_topk: %d rows", rows);
  if (rows == 0) return SSD_OK;
  SmpWs w;
  if (int rc = carve(ws, ws_bytes, rows, V, &w, "gumbel_topk")) return rc;
  TopkArgs a{probs, ldp, rows, V, k, tree_meta, level, make_rng(seed, counter), out_tok, out_lp, w};
  SSD_LAUNCH(gumbel_chunk_kernel, dim3(w.C, rows), dim3(SMP_THREADS), 0, stream, a);
  SSD_LAUNCH(gumbel_merge_kernel, dim3(rows), dim3(64 * ((w.C * k + 255) / 256)), 0, stream, a);
  return check_launch("gumbel_topk");
}

SSD_API int ssd_sample_rows(const float* probs, int64_t ldp, int rows, int V, uint64_t seed, uint64_t counter,
                            int32_t* out_tok, void* ws, int64_t ws_bytes, hipStream_t stream) {
  if (!probs || !out_tok) return set_error(SSD_EINVAL, "sample_rows: null pointer");
  if (rows < 0 || V <= 0 || ldp % 4 || ldp < V) return set_error(SSD_EINVAL, "sample_rows: bad shape");
  if (rows > 65535) return set_error(SSD_ERANGE, "sample_rows: %d rows", rows);
  if (rows == 0) return SSD_OK;
  SmpWs w;
  if (int rc = carve(ws, ws_bytes, rows, V, &w, "sample_rows")) return rc;
  SSD_LAUNCH(draw_chunk_kernel, dim3(w.C, rows), dim3(SMP_THREADS), 0, stream, probs, ldp, V,
                     make_rng(seed, counter), w);
  SSD_LAUNCH(draw_merge_kernel, dim3((rows + 63) / 64), dim3(64), 0, stream, rows, w, out_tok);
  return check_launch("sample_rows");
}

SSD_API int64_t ssd_sample_top64_ws_bytes(int rows, int V) {
  if (rows < 0 || V < T64 || chunks_of(V) > T64_MAXC) return -1;
  return (int64_t)rows * chunks_of(V) * T64 * (int64_t)sizeof(uint64_t);
}

SSD_API int ssd_sample_top64_bf16(const uint16_t* logits, int64_t ld, int rows, int V, float temperature, float top_p,
                                  uint64_t seed, uint64_t counter, int32_t* out_tok, void* ws, int64_t ws_bytes,
                                  hipStream_t stream) {
  if (!logits || !out_tok) return set_error(SSD_EINVAL, "sample_top64: null pointer");
  if (rows < 0 || V < T64 || chunks_of(V) > T64_MAXC)
    return set_error(SSD_ERANGE, "sample_top64: V=%d outside [%d, %d]", V, T64, SMP_CHUNK * T64_MAXC);
  if (ld % 4 || ld < (V + 3) / 4 * 4)
    return set_error(SSD_EINVAL, "sample_top64: ld %lld must be a multiple of 4 covering the row", (long long)ld);
  if (!(temperature > 0.f) || !(top_p > 0.f))
    return set_error(SSD_EINVAL, "sample_top64: temperature and top_p must be > 0");
  if (rows > 65535) return set_error(SSD_ERANGE, "sample_top64: %d rows", rows);
  if (rows == 0) return SSD_OK;
  const int64_t need = ssd_sample_top64_ws_bytes(rows, V);
  if (!ws || ws_bytes < need || ((uintptr_t)ws & 7))
    return set_error(SSD_EINVAL, "sample_top64: workspace %lld < %lld bytes or misaligned", (long long)ws_bytes,
                     (long long)need);
  const int C = chunks_of(V);
  SSD_LAUNCH(top64_chunk_kernel, dim3(C, rows), dim3(SMP_THREADS), 0, stream, (const bf16_t*)logits, ld, V, C,
             (uint64_t*)ws);
  SSD_LAUNCH(top64_draw_kernel, dim3(rows), dim3(64), 0, stream, (const uint64_t*)ws, C, temperature, top_p,
             make_rng(seed, counter), out_tok);
  return check_launch("sample_top64");
}

SSD_API int ssd_accept_sample(const SsdTree* tree, const float* P, int64_t ldp, const float* Q, int64_t ldq, int V,
                              int rows, int max_kids, uint64_t seed, uint64_t counter, void* ws, int64_t ws_bytes,
                              int committed, int32_t* result, int32_t* keep_src, int32_t* n_keep,
                              int32_t* root_token, hipStream_t stream) {
  if (!tree || !P || !Q || !result || !keep_src || !n_keep || !root_token)
    return set_error(SSD_EINVAL, "accept_sample: null pointer");
  if (V <= 0 || ldp % 4 || ldq % 4 || ldp < V || ldq < V || rows < 1 || rows > 64)
    return set_error(SSD_EINVAL, "accept_sample: bad shape (rows %d must be in [1, 64])", rows);
  if (max_kids < 0 || max_kids > SMP_MAXK)
    return set_error(SSD_ERANGE, "accept_sample: max_kids %d not in [0, %d]", max_kids, SMP_MAXK);
  SmpWs w;
  if (int rc = carve(ws, ws_bytes, rows, V, &w, "accept_sample")) return rc;
  AcceptArgs a{*tree, P, ldp, Q, ldq, V, rows, max_kids, make_rng(seed, counter), w};
  SSD_LAUNCH(state01_kernel, dim3(w.C + 1, rows), dim3(SMP_THREADS), 0, stream, a);
  for (int j = 2; j <= max_kids; ++j)
    SSD_LAUNCH(statej_kernel, dim3(w.C, rows), dim3(SMP_THREADS), 0, stream, a, j);
  SSD_LAUNCH(sample_walk_kernel, dim3(1), dim3(SMP_THREADS), 0, stream, a, committed, result, keep_src, n_keep,
                     root_token);
  return check_launch("accept_sample");
}

// Batched acceptance trials (accept_trials_kernel): trials independent rounds over fixed per-node
// distributions P/Q ([rows][ld] fp32, rows >= 1 + nodes of the unpruned tree given by branch[0 ..
// depth)), support lists cols/col_off (CSR over rows: ascending columns where P or Q > 0).
SSD_API int ssd_accept_sample_trials(const float* P, int64_t ldp, const float* Q, int64_t ldq, int rows,
                                     const int32_t* cols, const int32_t* col_off, int depth, const int32_t* branch,
                                     uint64_t seed, uint64_t counter0, int trials, int32_t* out_tokens,
                                     int32_t* out_n, hipStream_t stream) {
  if (!P || !Q || !cols || !col_off || !branch || !out_tokens || !out_n)
    return set_error(SSD_EINVAL, "accept_trials: null pointer");
  if (depth < 1 || depth > TRIAL_MAXD) return set_error(SSD_ERANGE, "accept_trials: depth %d not in [1, %d]", depth, TRIAL_MAXD);
  if (trials < 0 || ldp % 4 || ldq % 4 || rows < 1) return set_error(SSD_EINVAL, "accept_trials: bad shape");
  TrialArgs a{};
  a.P = P; a.ldp = ldp; a.Q = Q; a.ldq = ldq; a.cols = cols; a.off = col_off; a.depth = depth;
  int64_t level = 1, nodes = 0;
  for (int d = 0; d < depth; ++d) {
    if (branch[d] < 1 || branch[d] > SMP_MAXK)
      return set_error(SSD_ERANGE, "accept_trials: branch[%d]=%d not in [1, %d]", d, branch[d], SMP_MAXK);
    a.branch[d] = branch[d];
    a.start[d] = (int)nodes;
    level *= branch[d];
    nodes += level;
    if (nodes > (1 << 20)) return set_error(SSD_ERANGE, "accept_trials: tree too large");
  }
  a.start[depth] = (int)nodes;
  if (rows < 1 + nodes) return set_error(SSD_EINVAL, "accept_trials: %d rows for a tree of %lld nodes", rows, (long long)nodes);
  a.seed = seed; a.counter0 = counter0; a.trials = trials; a.out_tok = out_tokens; a.out_n = out_n;
  if (trials == 0) return SSD_OK;
  SSD_LAUNCH(accept_trials_kernel, dim3((trials + 3) / 4), dim3(256), 0, stream, a);
  return check_launch("accept_trials");
}

