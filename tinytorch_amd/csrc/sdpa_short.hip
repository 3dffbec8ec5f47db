// Attention, forward and backward, of short sequences: calls of a few row tiles and a few hundred keys, whose time is not work but
// the chain of one wavefront.  Every element type, head_dim up to 128 (16-byte chunks), either causal alignment, per-batch key
// counts, grouped heads; no attnMask, no pages (reference src/Function/FuncNNLayer.h:237-265; it has no backward, :267).
//
// The kernels for long sequences give a wavefront 32 x 32 or 64 x 32 scores at a time, bring K and V through LDS and leave most of the
// chip idle when there are few row tiles.  Here a workgroup owns 16 query rows (backward, dk/dv: 16 keys), its eight wavefronts take
// units of 16 keys (rows) in turn, and a unit's operands come straight from global memory into registers, all of them requested
// at once:
//   scores      S^T[16 keys][16 rows] = K . Q^T on 16 x 16 matrix instructions: lane 16g + i supplies row i of either side and the
//               16-byte chunks g, g + 4, ... of it (which elements a step contracts does not matter as long as both sides agree).
//   P, dS       lane 16g + i holds keys 4g .. 4g+3 of row i in its four registers: the B operand of one 16 x 16 x 16 step in 16 bits
//               (rounded as in the other kernels), register r that of v_mfma_f32_16x16x4_f32 step r in fp32.
//   P.V, dS.K   lane 16g + i loads elements 64h + 4i .. +3 of key 4g + r's row, one vector; their elements e are the A operand of
//               accumulator 4h + e, whose row i is head_dim element 64h + 4i + e.  A lane then holds elements 64h + 16g .. +15 of its
//               row in 16 registers.
// No LDS but for adding the wavefronts' results up, no barrier but for that one.
//
// What bounds it: a launch (4.4 us as the caller sees it), one round trip of a wavefront's loads, a unit's matrix instructions (fp32,
// head_dim 64: 512 cycles a product) and the join; with many workgroups the loads, for every 16 rows read all of K and V.  Hence few
// registers, so that several workgroups share a CU, rather than the next unit's operands ahead (4 x 16 heads x 200 rows, head_dim 64,
// bf16, forward 12.9 us with them, 8.4 so).  Forward / backward, causal, us, the other kernels -> here:
//   4 heads x 128, head_dim 64:     fp32 7.2 / 20.5 -> 5.7 / 15.9     bf16 6.6 / 17.4 -> 4.5 / 9.1
//   4 x 200, 128:                   fp32 16.8 / 50.2 -> 10.2 / 36     bf16 13.8 / 33.5 -> 6.3 / 18.9
//   8 heads on 2 x 320, 64:         fp32 13.2 / 47.9 -> 8.5 / 30.7    bf16 8.6 / 26.9 -> 5.8 / 20.5
//   2 x 16 heads on 4 x 200, 128:   fp32 17.4 / 67.3 -> 15.1 / 61.9   bf16 14.2 / 38.5 -> 8.3 / 34.5
// (4 x 16 x 320, 128, bf16 12.6 / 37.5 -> 19.5 / 85: the other kernels' calls; the host's estimates keep them there.)

#include <type_traits>

#include "sdpa_common.h"

namespace ttsdpa {

namespace {

constexpr int U = 16;     // rows (keys) of a workgroup, keys (rows) of a unit
constexpr int NWAVE = 8;

template <typename T>
struct Elem {  // fp16 / bf16
  typedef T chunk __attribute__((ext_vector_type(8)));
  static constexpr int E = 8;  // elements of a 16-byte chunk
  static __device__ __forceinline__ f32x4 mma(chunk x, chunk y, f32x4 c) {
    if constexpr (std::is_same<T, __bf16>::value) return BF16::mfma16(x, y, c);
    else return F16::mfma16(x, y, c);
  }
  typedef T vec4 __attribute__((ext_vector_type(4)));
  // c += x^T . w over the unit's 16 rows: x[r], this lane's elements e of row 4g + r; w, the weights of those rows for its column
  static __device__ __forceinline__ f32x4 mma_rows(vec4 x, f32x4 w, f32x4 c) {
    const vec4 y = __builtin_convertvector(w, vec4);
    if constexpr (std::is_same<T, __bf16>::value) {
      typedef short s16x4 __attribute__((ext_vector_type(4)));
      return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, x), __builtin_bit_cast(s16x4, y), c, 0, 0, 0);
    } else {
      return __builtin_amdgcn_mfma_f32_16x16x16f16(x, y, c, 0, 0, 0);
    }
  }
  static __device__ __forceinline__ float dot(chunk x, chunk y, float s) {
#pragma unroll
    for (int e = 0; e < 8; e++) s = fmaf((float)x[e], (float)y[e], s);
    return s;
  }
};
template <>
struct Elem<float> {
  typedef f32x4 chunk;
  static constexpr int E = 4;
  static __device__ __forceinline__ f32x4 mma(chunk x, chunk y, f32x4 c) {
#pragma unroll
    for (int e = 0; e < 4; e++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], c, 0, 0, 0);
    return c;
  }
  static __device__ __forceinline__ f32x4 mma_rows(f32x4 x, f32x4 w, f32x4 c) {
#pragma unroll
    for (int r = 0; r < 4; r++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[r], w[r], c, 0, 0, 0);
    return c;
  }
  static __device__ __forceinline__ float dot(chunk x, chunk y, float s) {
#pragma unroll
    for (int e = 0; e < 4; e++) s = fmaf(x[e], y[e], s);
    return s;
  }
};

// A lane's chunks of one row of W elements, of which the tensor has `have` (whole chunks; the rest reads as zeros).
template <typename T, int W>
struct Frag {
  typedef typename Elem<T>::chunk chunk;
  static constexpr int E = Elem<T>::E, N = W / (4 * E);
  chunk c[N];
  __device__ __forceinline__ void load(const T* row, int g, int have) {
#pragma unroll
    for (int s = 0; s < N; s++) {
      const int at = 4 * E * s + E * g;
      chunk t = {};
      if (at < have) t = *(const chunk*)(row + at);
      c[s] = t;
    }
  }
};
// X . Y^T of two fragments, on two accumulators in turn
template <typename T, int W>
__device__ __forceinline__ f32x4 product(const Frag<T, W>& x, const Frag<T, W>& y) {
  f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int i = 0; i < Frag<T, W>::N; i++) s[i & 1] = Elem<T>::mma(x.c[i], y.c[i], s[i & 1]);
  return s[0] + s[1];
}

// Rows 4g .. 4g+3 of a unit, this lane's elements 64h + 4i .. +3 of each; rows from `limit` on are zeros (their weight is 0, but
// 0 times an infinity is not).
template <typename T, int W>
struct Rows {
  typedef T vec4 __attribute__((ext_vector_type(4)));
  vec4 v[W / 64 * 4];
  __device__ __forceinline__ void load(const T* base, long long stride, int row0, int limit, int i, int have) {
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int h = 0; h < W / 64; h++) {
        vec4 t = {};
        if (row0 + r < limit && 64 * h + 4 * i < have) t = *(const vec4*)(base + (row0 + r) * stride + 64 * h + 4 * i);
        v[4 * h + r] = t;
      }
  }
};
// acc += rows^T . w, w: the weights of rows 4g .. 4g+3 for this lane's column
template <typename T, int W>
__device__ __forceinline__ void accumulate(f32x4 (&acc)[W / 16], const Rows<T, W>& x, f32x4 w) {
  typedef T vec4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int h = 0; h < W / 64; h++)
#pragma unroll
    for (int e = 0; e < 4; e++) acc[4 * h + e] = Elem<T>::mma_rows(vec4{x.v[4 * h][e], x.v[4 * h + 1][e], x.v[4 * h + 2][e], x.v[4 * h + 3][e]}, w, acc[4 * h + e]);
}
// What a lane's accumulators hold of elements 64h + 16g + 4r .. +3
template <int N>
__device__ __forceinline__ f32x4 piece_of(const f32x4 (&acc)[N], int h, int r) {
  return f32x4{acc[4 * h][r], acc[4 * h + 1][r], acc[4 * h + 2][r], acc[4 * h + 3][r]};
}
template <typename T>
__device__ __forceinline__ void store4(T* p, f32x4 x) {
  typedef T vec4 __attribute__((ext_vector_type(4)));
  *(vec4*)p = __builtin_convertvector(x, vec4);
}

// Softmax state of this lane's row over the units its wavefront has taken: scores of keys 4g .. 4g+3 -> weights relative to the
// maximum so far; acc is brought to it.
template <int N>
__device__ __forceinline__ f32x4 weigh(f32x4 s, float c, float& m, float& l, f32x4 (&acc)[N]) {
  float top = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
  top = fmaxf(top, __shfl_xor(top, 16));
  top = fmaxf(top, __shfl_xor(top, 32));
  const float m_new = fmaxf(m, top), alpha = fast_exp2((m - m_new) * c);
  m = m_new;
  f32x4 p;
#pragma unroll
  for (int r = 0; r < 4; r++) p[r] = fast_exp2((s[r] - m) * c);
  l = fmaf(l, alpha, (p[0] + p[1]) + (p[2] + p[3]));
#pragma unroll
  for (int n = 0; n < N; n++) acc[n] *= alpha;
  return p;
}

// The wavefronts' (maximum, sum, accumulators) of 16 rows, brought together in wavefront order: this lane's piece (h, r) of its row's
// accumulators, relative to m_all, with the row's sum l_all.  lds: 4 KiB x W / 64 a wavefront, then 128 bytes each.
template <int W>
__device__ __forceinline__ f32x4 join_rows(char* lds, int n, int wave, int lane, float c, float m, float l, const f32x4 (&acc)[W / 16],
                                           float* m_all, float* l_all, int* h, int* r) {
  constexpr int SLOTS = W / 16;  // (h, r)
  f32x4* part = (f32x4*)lds;
  float* ml = (float*)(part + NWAVE * SLOTS * 64);
  const int i = lane & 15;
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (wave < n) {
#pragma unroll
    for (int k = 0; k < SLOTS; k++) part[(wave * SLOTS + k) * 64 + lane] = piece_of(acc, k >> 2, k & 3);
    if (lane < 32) ml[wave * 32 + lane] = lane < 16 ? m : l;
  }
  __syncthreads();
  *h = wave >> 2, *r = wave & 3;
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
  if (wave >= SLOTS) return x;
  // (all reads at once; wavefronts without units: the first one's numbers, as zeros)
  float mw[NWAVE], lw[NWAVE];
  f32x4 y[NWAVE];
#pragma unroll
  for (int w = 0; w < NWAVE; w++) {
    const int at = w < n ? w : 0;
    mw[w] = ml[at * 32 + i], lw[w] = ml[at * 32 + 16 + i], y[w] = part[(at * SLOTS + wave) * 64 + lane];
  }
  float most = mw[0], sum = 0.f;
#pragma unroll
  for (int w = 1; w < NWAVE; w++) most = fmaxf(most, mw[w]);
#pragma unroll
  for (int w = 0; w < NWAVE; w++) {
    if (w >= n) lw[w] = 0.f, y[w] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float f = fast_exp2((mw[w] - most) * c);
    sum = fmaf(f, lw[w], sum);
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = fmaf(f, y[w][e], x[e]);
  }
  *m_all = most, *l_all = sum;
  return x;
}
template <int W>
constexpr int kJoinBytes = NWAVE * (W / 16 * 1024 + 128);

// Scores of keys key0 .. key0+3 that a row whose last visible key (under a causal mask) is `last` does not see.
template <bool CAUSAL>
__device__ __forceinline__ void hide_keys(f32x4& s, int key0, int S, int last) {
#pragma unroll
  for (int r = 0; r < 4; r++)
    if (key0 + r >= S || (CAUSAL && key0 + r > last)) s[r] = -INFINITY;
}

// Rows q0 .. q0+15: units of keys they see.
__device__ __forceinline__ int units_of_rows(const KArgs& a, int q0, int S, int coff, bool causal) {
  int last = S - 1;
  if (causal) {
    const int v = (q0 + U < a.L ? q0 + U : a.L) - 1 + coff;
    last = v < last ? v : last;
  }
  return last / U + 1;
}

// ---- forward --------------------------------------------------------------------------------------------------------
template <typename T, int W, bool CAUSAL>
__global__ __launch_bounds__(64 * NWAVE, 1) void short_forward_kernel(KArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[kJoinBytes<W>];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int ntile = (a.L + U - 1) / U;
  int pair, in;
  map_workgroup(blockIdx.x, a.B * a.Hq, ntile, &pair, &in);
  const int h = pair % a.Hq, b = pair / a.Hq, hk = h / a.G;
  const int q0 = (CAUSAL ? ntile - 1 - in : in) * U, row = q0 + i;
  const T* kp = (const T*)a.k + b * a.ks[0] + hk * a.ks[1];
  const T* vp = (const T*)a.v + b * a.vs[0] + hk * a.vs[1];
  T* op = (T*)a.out + b * a.os[0] + h * a.os[1] + row * a.os[2];

  Frag<T, W> q;
  q.load((const T*)a.q + b * a.qs[0] + h * a.qs[1] + (row < a.L ? row : a.L - 1) * a.qs[2], g, a.D);
  const int S = keys_of_batch(a, b);
  if (S == 0) {  // no keys: zeros
    if (wave == 0 && row < a.L)
      for (int d = 4 * g; d < a.D; d += 16) store4(op + d, f32x4{0.f, 0.f, 0.f, 0.f});
    return;
  }
  const int coff = CAUSAL ? causal_offset(a, S) : 0, nunit = units_of_rows(a, q0, S, coff, CAUSAL);
  const float c = a.scale * kLog2e;
  float m = -FLT_MAX, l = 0.f;
  f32x4 acc[W / 16] = {};
  for (int u = wave; u < nunit; u += NWAVE) {
    const int k0 = u * U;
    Frag<T, W> k;
    Rows<T, W> v;
    k.load(kp + (k0 + i < S ? k0 + i : S - 1) * a.ks[2], g, a.D);
    v.load(vp, a.vs[2], k0 + 4 * g, S, i, a.D);
    f32x4 s = product(k, q);
    hide_keys<CAUSAL>(s, k0 + 4 * g, S, row + coff);
    accumulate<T, W>(acc, v, weigh(s, c, m, l, acc));
  }
  float m_all, l_all;
  int ph, pr;
  const f32x4 x = join_rows<W>(lds, nunit < NWAVE ? nunit : NWAVE, wave, lane, c, m, l, acc, &m_all, &l_all, &ph, &pr);
  const int d = 64 * ph + 16 * g + 4 * pr;
  if (wave < W / 16 && row < a.L && d < a.D) {
    const float inv = 1.f / l_all;
    store4(op + d, x * inv);
  }
}

// ---- backward -------------------------------------------------------------------------------------------------------
// dout . out of this lane's row, whose chunks the four lanes of a row hold between them
template <typename T, int W>
__device__ __forceinline__ float row_delta(const Frag<T, W>& o, const Frag<T, W>& go) {
  float delta = 0.f;
#pragma unroll
  for (int n = 0; n < Frag<T, W>::N; n++) delta = Elem<T>::dot(o.c[n], go.c[n], delta);
  delta += __shfl_xor(delta, 16);
  return delta + __shfl_xor(delta, 32);
}

// dq of 16 rows; STATS: and their statistics for the dk / dv workgroups of a second launch.
template <typename T, int W, bool CAUSAL, bool STATS>
__device__ __forceinline__ void dq_rows(const BwdArgs& a, int block, char* lds) {
  const KArgs& f = a.f;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int ntile = (f.L + U - 1) / U;
  int pair, in;
  map_workgroup(block, f.B * f.Hq, ntile, &pair, &in);
  const int h = pair % f.Hq, b = pair / f.Hq, hk = h / f.G;
  const int q0 = (CAUSAL ? ntile - 1 - in : in) * U, row = q0 + i, rowc = row < f.L ? row : f.L - 1;
  const T* kp = (const T*)f.k + b * f.ks[0] + hk * f.ks[1];
  const T* vp = (const T*)f.v + b * f.vs[0] + hk * f.vs[1];
  T* dqp = (T*)a.dq + b * a.dqs[0] + h * a.dqs[1] + row * a.dqs[2];

  const int S = keys_of_batch(f, b);
  if (S == 0) {  // no keys: the output did not depend on q
    if (wave == 0 && row < f.L)
      for (int d = 4 * g; d < f.D; d += 16) store4(dqp + d, f32x4{0.f, 0.f, 0.f, 0.f});
    return;
  }
  const int coff = CAUSAL ? causal_offset(f, S) : 0, nunit = units_of_rows(f, q0, S, coff, CAUSAL);
  const float c = f.scale * kLog2e;
  Frag<T, W> q, go, o;
  q.load((const T*)f.q + b * f.qs[0] + h * f.qs[1] + rowc * f.qs[2], g, f.D);
  go.load((const T*)a.dout + b * a.dos[0] + h * a.dos[1] + rowc * a.dos[2], g, f.D);
  o.load((const T*)f.out + b * f.os[0] + h * f.os[1] + rowc * f.os[2], g, f.D);
  float m = -FLT_MAX, l = 0.f, delta = 0.f;
  f32x4 acc[W / 16] = {};
  for (int u = wave; u < nunit; u += NWAVE) {
    const int k0 = u * U, keyc = k0 + i < S ? k0 + i : S - 1;
    Frag<T, W> k, v;
    Rows<T, W> kr;
    k.load(kp + keyc * f.ks[2], g, f.D);
    v.load(vp + keyc * f.vs[2], g, f.D);
    kr.load(kp, f.ks[2], k0 + 4 * g, S, i, f.D);
    if (u == wave) delta = row_delta(o, go);  // (here, behind the loads of the first unit)
    f32x4 s = product(k, q);
    const f32x4 dp = product(v, go);
    hide_keys<CAUSAL>(s, k0 + 4 * g, S, row + coff);
    f32x4 p = weigh(s, c, m, l, acc);
#pragma unroll
    for (int r = 0; r < 4; r++) p[r] *= dp[r] - delta;
    accumulate<T, W>(acc, kr, p);
  }
  float m_all, l_all;
  int ph, pr;
  const f32x4 x = join_rows<W>(lds, nunit < NWAVE ? nunit : NWAVE, wave, lane, c, m, l, acc, &m_all, &l_all, &ph, &pr);
  if (wave >= W / 16 || row >= f.L) return;
  if (STATS && wave == 0 && g == 0)
    *(float2*)(a.stats + 2 * (((long long)b * f.Hq + h) * f.L + row)) = make_float2(l_all == 0.f ? 1e30f : m_all * c + __log2f(l_all), delta);
  const int d = 64 * ph + 16 * g + 4 * pr;
  // (a row without weight, all its scores -infinity: no gradient)
  if (d < f.D) store4(dqp + d, l_all == 0.f ? f32x4{0.f, 0.f, 0.f, 0.f} : x * (f.scale / l_all));
}

// dk and dv of 16 keys.  STATS: the rows' statistics are in a.stats; else they are formed here, a score product more for every key
// that a unit's rows see.
template <typename T, int W, bool CAUSAL, bool STATS>
__device__ __forceinline__ void dkv_keys(const BwdArgs& a, int block, char* lds) {
  constexpr int SLOTS = W / 16;
  const KArgs& f = a.f;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int nblk = (f.S + U - 1) / U;
  int wg, split;  // the units are divided among a.dkv_splits workgroups, which leave partial sums
  split_of_workgroup(block, a.dkv_splits, f.B * f.Hkv, &wg, &split);
  int pair, kb;  // the first keys are seen by every row: the longest
  map_workgroup(wg, f.B * f.Hkv, nblk, &pair, &kb);
  const int hk = pair % f.Hkv, b = pair / f.Hkv;
  const int k0 = kb * U, key = k0 + i;
  const int S = keys_of_batch(f, b);
  const T* kp = (const T*)f.k + b * f.ks[0] + hk * f.ks[1];
  T* dkp = (T*)a.dk + b * a.dks[0] + hk * a.dks[1] + key * a.dks[2];
  T* dvp = (T*)a.dv + b * a.dvs[0] + hk * a.dvs[1] + key * a.dvs[2];
  const int coff = CAUSAL ? causal_offset(f, S) : 0;
  const int it0 = CAUSAL && k0 > coff ? (k0 - coff) / U : 0, ntq = (f.L + U - 1) / U;
  const int all = k0 < S && it0 < ntq ? f.G * (ntq - it0) : 0;
  const int nunit = split < all ? (all - split + a.dkv_splits - 1) / a.dkv_splits : 0;  // units split, split + dkv_splits, ...
  const float c = f.scale * kLog2e;

  Frag<T, W> k, v;
  if (nunit > 0) {
    const int keyc = key < S ? key : S - 1;
    k.load(kp + keyc * f.ks[2], g, f.D);
    v.load((const T*)f.v + b * f.vs[0] + hk * f.vs[1] + keyc * f.vs[2], g, f.D);
  }
  f32x4 dk[W / 16] = {}, dv[W / 16] = {};
  for (int u = wave; u < nunit; u += NWAVE) {
    // (the longest streams first: the wavefronts without a second unit are those with the most keys to go over)
    const int at = split + u * a.dkv_splits;
    const int h = hk * f.G + at % f.G, i0 = (ntq - 1 - at / f.G) * U;
    const int rowc = i0 + i < f.L ? i0 + i : f.L - 1;
    const T* qb = (const T*)f.q + b * f.qs[0] + h * f.qs[1];
    const T* gb = (const T*)a.dout + b * a.dos[0] + h * a.dos[1];
    Frag<T, W> q, go;
    Rows<T, W> qr, gr;
    q.load(qb + rowc * f.qs[2], g, f.D);
    go.load(gb + rowc * a.dos[2], g, f.D);
    f32x4 lse, delta;
    if constexpr (STATS) {
      const float* st = a.stats + 2 * ((long long)b * f.Hq + h) * f.L;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int at = i0 + 4 * g + r;
        const float2 t = *(const float2*)(st + 2 * (at < f.L ? at : f.L - 1));
        lse[r] = t.x, delta[r] = t.y;
      }
    }
    // (fp32 at head_dim 128: in the registers of q and dout, when those are done with)
    constexpr bool LATE = W > 64 && sizeof(T) == 4;
    if constexpr (!LATE) {
      gr.load(gb, a.dos[2], i0 + 4 * g, f.L, i, f.D);
      qr.load(qb, f.qs[2], i0 + 4 * g, f.L, i, f.D);
    }
    if constexpr (!STATS) {
      Frag<T, W> o;
      o.load((const T*)f.out + b * f.os[0] + h * f.os[1] + rowc * f.os[2], g, f.D);
      // this lane's row is i0 + i here, its keys 4g .. 4g+3 of each unit
      float m = -FLT_MAX, l = 0.f;
      const int n = units_of_rows(f, i0, S, coff, CAUSAL);
      auto fetch = [&](Frag<T, W>& x, int j) __attribute__((always_inline)) {
        const int kc = j * U + i < S ? j * U + i : S - 1;
        x.load(kp + kc * f.ks[2], g, f.D);
      };
      auto add = [&](const Frag<T, W>& x, int j) __attribute__((always_inline)) {
        f32x4 s = product(x, q);
        hide_keys<CAUSAL>(s, j * U + 4 * g, S, i0 + i + coff);
        const float m_new = fmaxf(m, fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])));
        l *= fast_exp2((m - m_new) * c);
        m = m_new;
#pragma unroll
        for (int r = 0; r < 4; r++) l += fast_exp2((s[r] - m) * c);
      };
      Frag<T, W> x, y;  // the next unit's keys are on their way while one's are worked on
      fetch(x, 0);
      for (int j = 0; j < n; j += 2) {
        if (j + 1 < n) fetch(y, j + 1);
        add(x, j);
        if (j + 1 >= n) break;
        if (j + 2 < n) fetch(x, j + 2);
        add(y, j + 1);
      }
      float most = fmaxf(m, __shfl_xor(m, 16));
      most = fmaxf(most, __shfl_xor(most, 32));
      l *= fast_exp2((m - most) * c);
      l += __shfl_xor(l, 16);
      l += __shfl_xor(l, 32);
      const float row_lse = l == 0.f ? 1e30f : most * c + __log2f(l), own = row_delta(o, go);
#pragma unroll
      for (int r = 0; r < 4; r++) lse[r] = __shfl(row_lse, 4 * g + r), delta[r] = __shfl(own, 4 * g + r);
    }
    const f32x4 s = product(q, k), dp = product(go, v);
    f32x4 p, ds;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int at = i0 + 4 * g + r;
      const bool hidden = at >= f.L || (CAUSAL && key > at + coff);
      p[r] = hidden ? 0.f : fast_exp2(fmaf(s[r], c, -lse[r]));
      ds[r] = hidden ? 0.f : p[r] * (dp[r] - delta[r]);
    }
    if constexpr (LATE) gr.load(gb, a.dos[2], i0 + 4 * g, f.L, i, f.D);
    accumulate<T, W>(dv, gr, p);
    if constexpr (LATE) qr.load(qb, f.qs[2], i0 + 4 * g, f.L, i, f.D);
    accumulate<T, W>(dk, qr, ds);
  }
  // the wavefronts' sums, added in wavefront order
  f32x4* part = (f32x4*)lds;
  const int n = nunit < NWAVE ? nunit : NWAVE;
  if (wave < n) {
#pragma unroll
    for (int j = 0; j < SLOTS; j++) {
      part[(wave * 2 * SLOTS + j) * 64 + lane] = piece_of(dk, j >> 2, j & 3);
      part[(wave * 2 * SLOTS + SLOTS + j) * 64 + lane] = piece_of(dv, j >> 2, j & 3);
    }
  }
  __syncthreads();
  if (key >= f.S) return;
#pragma unroll
  for (int j0 = 0; j0 < 2 * SLOTS; j0 += NWAVE) {
    const int j = j0 + wave;
    f32x4 x = {0.f, 0.f, 0.f, 0.f}, y[NWAVE];
#pragma unroll
    for (int w = 0; w < NWAVE; w++) y[w] = part[((w < n ? w : 0) * 2 * SLOTS + j) * 64 + lane];
#pragma unroll
    for (int w = 0; w < NWAVE; w++) x += w < n ? y[w] : f32x4{0.f, 0.f, 0.f, 0.f};
    if (key >= S) x = f32x4{0.f, 0.f, 0.f, 0.f};  // at or beyond the batch entry's key count
    const int slot = j % SLOTS, d = 64 * (slot >> 2) + 16 * g + 4 * (slot & 3);
    if (d >= f.D) continue;
    if (j < SLOTS) x *= f.scale;
    if (a.dkv_splits > 1) {  // dense [split][dk | dv][B][Hkv][S][D]
      const long long plane = (long long)f.B * f.Hkv * f.S * f.D;
      *(f32x4*)(a.partial + (2 * split + (j < SLOTS ? 0 : 1)) * plane + (((long long)b * f.Hkv + hk) * f.S + key) * f.D + d) = x;
    } else {
      store4((j < SLOTS ? dkp : dvp) + d, x);
    }
  }
}
template <int W>
constexpr int kDkvBytes = NWAVE * 2 * (W / 16) * 1024;

template <typename T, int W, bool CAUSAL>
__global__ __launch_bounds__(64 * NWAVE, 1) void short_dq_kernel(BwdArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[kJoinBytes<W>];
  dq_rows<T, W, CAUSAL, true>(a, blockIdx.x, lds);
}
template <typename T, int W, bool CAUSAL>
__global__ __launch_bounds__(64 * NWAVE, 1) void short_dkv_kernel(BwdArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[kDkvBytes<W>];
  dkv_keys<T, W, CAUSAL, true>(a, blockIdx.x, lds);
}
// Both in one launch: the workgroups of the keys, which take longer, first.
template <typename T, int W, bool CAUSAL>
__global__ __launch_bounds__(64 * NWAVE, 1) void short_backward_kernel(BwdArgs a, int of_keys) {
  __shared__ __attribute__((aligned(16))) char lds[kDkvBytes<W>];
  static_assert(kDkvBytes<W> >= kJoinBytes<W>, "");
  if ((int)blockIdx.x < of_keys) dkv_keys<T, W, CAUSAL, false>(a, blockIdx.x, lds);
  else dq_rows<T, W, CAUSAL, false>(a, blockIdx.x - of_keys, lds);
}

template <typename T, int W, bool CAUSAL>
int launch_forward_k(const KArgs& a, hipStream_t stream) {
  const long long n = (long long)a.B * a.Hq * ((a.L + U - 1) / U);
  hipLaunchKernelGGL((short_forward_kernel<T, W, CAUSAL>), dim3((unsigned)n), dim3(64 * NWAVE), 0, stream, a);
  return (int)hipGetLastError();
}

template <typename T, int W, bool CAUSAL>
int launch_backward_k(const BwdArgs& a, bool joint, hipStream_t stream) {
  const KArgs& f = a.f;
  const long long of_rows = (long long)f.B * f.Hq * ((f.L + U - 1) / U);
  const long long of_keys = (long long)f.B * f.Hkv * ((f.S + U - 1) / U) * a.dkv_splits;
  if (joint) {
    if constexpr (W > 64 && sizeof(T) == 4)
      return (int)hipErrorInvalidValue;  // (the registers of both roles do not fit; the caller keeps to this)
    else
      hipLaunchKernelGGL((short_backward_kernel<T, W, CAUSAL>), dim3((unsigned)(of_keys + of_rows)), dim3(64 * NWAVE), 0, stream, a, (int)of_keys);
  } else {
    hipLaunchKernelGGL((short_dq_kernel<T, W, CAUSAL>), dim3((unsigned)of_rows), dim3(64 * NWAVE), 0, stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    hipLaunchKernelGGL((short_dkv_kernel<T, W, CAUSAL>), dim3((unsigned)of_keys), dim3(64 * NWAVE), 0, stream, a);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || a.dkv_splits == 1) return (int)e;
  return launch_backward_dkv_sum<T>(a, stream);
}

// the callers keep to this: rows of whole 16-byte chunks, no mask, no pages
bool takes(const KArgs& a, int dtype) {
  return a.D >= 4 && a.D <= 128 && a.D % (dtype == 0 ? 4 : 8) == 0 && a.mask_kind == 0 && !a.block_table && a.L >= 1 && a.S >= 1;
}

template <typename T>
int launch_forward_t(const KArgs& a, hipStream_t stream) {
  if (a.D <= 64) return a.causal ? launch_forward_k<T, 64, true>(a, stream) : launch_forward_k<T, 64, false>(a, stream);
  return a.causal ? launch_forward_k<T, 128, true>(a, stream) : launch_forward_k<T, 128, false>(a, stream);
}
template <typename T>
int launch_backward_t(const BwdArgs& a, bool joint, hipStream_t stream) {
  if (a.f.D <= 64) return a.f.causal ? launch_backward_k<T, 64, true>(a, joint, stream) : launch_backward_k<T, 64, false>(a, joint, stream);
  return a.f.causal ? launch_backward_k<T, 128, true>(a, joint, stream) : launch_backward_k<T, 128, false>(a, joint, stream);
}

}  // namespace

int launch_short_forward(const KArgs& a, int dtype, hipStream_t stream) {
  if (!takes(a, dtype) || a.pack_L) return (int)hipErrorInvalidValue;
  return dtype == 0 ? launch_forward_t<float>(a, stream) : dtype == 1 ? launch_forward_t<_Float16>(a, stream) : launch_forward_t<__bf16>(a, stream);
}

int launch_short_backward(const BwdArgs& a, int dtype, bool joint, hipStream_t stream) {
  if (!takes(a.f, dtype)) return (int)hipErrorInvalidValue;
  return dtype == 0   ? launch_backward_t<float>(a, joint, stream)
         : dtype == 1 ? launch_backward_t<_Float16>(a, joint, stream)
                      : launch_backward_t<__bf16>(a, joint, stream);
}

}  // namespace ttsdpa
