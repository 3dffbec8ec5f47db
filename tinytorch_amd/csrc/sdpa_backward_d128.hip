// Attention backward for fp16 / bf16, head_dim 128, without an attnMask, on gfx950 matrix cores: dq and the row statistics
// (sdpa_backward_mfma.hip has the mathematics and the other half).
//
// A workgroup owns 128 query rows of one (batch, query head), a wavefront 32 of them (Q and dout in registers); keys stream in tiles
// of 32.  Per tile a wavefront forms S^T = K.Q^T and dP^T = V.dout^T, turns them into P and dS on the vector ALU and accumulates dq^T +=
// K^T.dS^T: 24 matrix instructions (768 cycles) and 88 vector ones, 16 of them exponentials (about 550 cycles of issue, beside 16 for every
// matrix instruction).  In the compiler's order the three followed each other, the wavefronts of a SIMD hardly overlapping: 3250 cycles
// a tile of two wavefronts, the matrix pipe 44 % busy at 1.99 GHz.  Here a step is a stream of hand-ordered instructions
// (gen_backward128_steps.py) over three tiles: scores and dP of tile i+1 and dq of tile i-1 on the matrix pipe, the vector work of
// tile i between them.  2 x 32 heads (8) x 4096 x 4096, causal: 420 -> 378 us, the matrix pipe 58 % busy and the clock down at 1.69 GHz: as
// in the forward kernel, power is what bounds it now.
//
// K and V come by direct global->LDS loads, four stages each (K of tiles i-1, i, i+1 and, on its way, i+2): a tile is eight groups of
// four 256-byte rows, 1040 bytes apart, chunk c of 16 bytes of row i of a group at slot c ^ 4i, so that one copy serves the
// row-major reads and the transposed ones without bank conflicts and both take four address registers.

#include "backward128_steps.inc"  // hand-ordered instruction streams (gen_backward128_steps.py)
#include "sdpa_common.h"

namespace ttsdpa {

namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x32 __attribute__((ext_vector_type(32)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) void lds_void;

constexpr int D = 128, KSTEPS = D / 16, DBLK = D / 32;
constexpr int BM = 128;                 // query rows of a workgroup
constexpr int BN = 32;                  // keys of a tile
constexpr int ROW_BYTES = 2 * D;
constexpr int GROUP_BYTES = 4 * ROW_BYTES + 16;
constexpr int TILE_BYTES = 8 * GROUP_BYTES;
constexpr int STAGES = 4;
constexpr int DQ_LDS = 2 * STAGES * TILE_BYTES;
constexpr float kSumLimit = 256.f;      // a lane's 16 probabilities of a tile may sum to this much before the maximum is raised

// The lane's byte offsets of row-major operands (row lane%32, k-step ks: r[ks / 2] + 32 (ks % 2)) and transposed ones (rows 16t .. of
// block db, half ld: tr[db] + (4t + 2ld) GROUP_BYTES) in a tile.
__device__ __forceinline__ void operand_offsets(int lane, u32x4& r, u32x4& tr) {
  const int lq = lane & 31, lh = lane >> 5, s = lane & 15, dhalf = (lane >> 4) & 1;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    r[i] = (unsigned)((lq >> 2) * GROUP_BYTES + (lq & 3) * ROW_BYTES + 16 * lh + 64 * (i ^ (lq & 3)));
    tr[i] = (unsigned)(lh * GROUP_BYTES + (s >> 2) * ROW_BYTES + 64 * (i ^ (s >> 2)) + 32 * dhalf + 16 * ((s & 3) >> 1) + 8 * (s & 1));
  }
}

template <typename TR, bool CAUSAL>
__global__ __launch_bounds__(256, 2) void backward_dq128_kernel(BwdArgs a) {
  typedef typename TR::elem T;
  typedef typename TR::vec8 vec8;
  constexpr bool kIsBf16 = __is_same(T, __bf16);
  const KArgs& f = a.f;

  extern __shared__ __attribute__((aligned(16))) char smem[];
  const unsigned smem_addr = (unsigned)(unsigned long)(lds_void*)smem;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane & 31, lh = lane >> 5;

  const int ntile = (f.L + BM - 1) / BM;
  int pair, in, piece;  // piece: this workgroup's share of the row block's key range (dq_splits > 1)
  {
    int n;
    split_of_workgroup(blockIdx.x, a.dq_splits, f.B * f.Hq, &n, &piece);
    map_workgroup(n, f.B * f.Hq, ntile, &pair, &in);
  }
  const int h = pair % f.Hq, b = pair / f.Hq;
  const int hk = h / f.G;
  const int rt = CAUSAL ? ntile - 1 - in : in;  // longest rows first
  const int q0 = rt * BM, qw0 = q0 + wave * 32;

  const int S = keys_of_batch(f, b);
  if (S == 0) {  // no keys (an empty cache entry): the output did not depend on q
    if (a.dq_splits > 1) return;  // the merge kernel writes the zeros
    const int qi = qw0 + lq;
    if (qi < f.L) {
      T* dqp = (T*)a.dq + b * a.dqs[0] + h * a.dqs[1] + qi * a.dqs[2];
      typename TR::vec4 zero;
#pragma unroll
      for (int i = 0; i < 4; i++) zero[i] = (T)0.f;
      for (int d = 4 * lh; d < D; d += 8) *(typename TR::vec4*)(dqp + d) = zero;
    }
    return;
  }
  const int coff = CAUSAL ? causal_offset(f, S) : 0;
  int ntiles_kv = (S + BN - 1) / BN;
  if (CAUSAL) {
    const int last = (q0 + BM - 1 < f.L - 1 ? q0 + BM - 1 : f.L - 1) + coff;  // last key any row of the workgroup sees
    const int lastkv = last < S - 1 ? last : S - 1;
    ntiles_kv = lastkv / BN + 1;
  }
  // this workgroup's tiles: all of them, or piece `piece` of dq_splits nearly equal ones (possibly none)
  const int t0 = (int)((long long)ntiles_kv * piece / a.dq_splits), t1 = (int)((long long)ntiles_kv * (piece + 1) / a.dq_splits), nt = t1 - t0;
  auto first_key = [&](int i) __attribute__((always_inline)) { return (t0 + i) * BN; };
  // ... of which the wavefront's rows see `mine`; steps 1 .. nfast (an even number) take the stream: their tiles hide nothing
  int seen = t1, clear = S / BN;
  if (CAUSAL) {
    const int last = (qw0 + 31 + coff) / BN + 1, whole = (qw0 + coff + 1) / BN;
    seen = last < seen ? last : seen;
    clear = whole < clear ? whole : clear;
  }
  const int mine = qw0 < f.L && seen > t0 ? seen - t0 : 0;
  int nfast = clear - t0 - 1;
  nfast = mine - 1 < nfast ? mine - 1 : nfast;
  nfast = __builtin_amdgcn_readfirstlane(nfast > 0 ? nfast & ~1 : 0);

  // ---- tiles: wavefront w brings rows 8w .. 8w+7 (two groups) of K and of V --------------------------------------------------------
  auto dma16 = [&](const char* sbase, unsigned voff, unsigned lds_addr) __attribute__((always_inline)) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_addr) : "memory", "m0");
  };
  const T* kp = (const T*)f.k + b * f.ks[0] + hk * f.ks[1];
  const T* vp = (const T*)f.v + b * f.vs[0] + hk * f.vs[1];
  const unsigned chunk = (unsigned)((lane & 15) ^ (4 * (lane >> 4)));
  const unsigned koff = ((unsigned)(lane >> 4) * (unsigned)f.ks[2] + 8u * chunk) * 2u, voff = ((unsigned)(lane >> 4) * (unsigned)f.vs[2] + 8u * chunk) * 2u;
  auto dma_tile = [&](int i) __attribute__((always_inline)) {
    const int kv0 = first_key(i);
    const unsigned at = smem_addr + (i & 3) * TILE_BYTES + 2 * wave * GROUP_BYTES;
    if (__builtin_expect(kv0 + BN <= S, 1)) {
#pragma unroll
      for (int g = 0; g < 2; g++) {
        const int row = kv0 + 8 * wave + 4 * g;
        dma16((const char*)(kp + (long long)row * f.ks[2]), koff, at + g * GROUP_BYTES);
        dma16((const char*)(vp + (long long)row * f.vs[2]), voff, at + STAGES * TILE_BYTES + g * GROUP_BYTES);
      }
    } else {  // rows past the end re-read the last key (hidden below)
#pragma unroll
      for (int g = 0; g < 2; g++) {
        int row = 8 * wave + 4 * g + (lane >> 4);
        asm volatile("" : "+v"(row));  // keeps this rarely taken path's address arithmetic inside the branch
        const int rowc = kv0 + row < S ? row : S - 1 - kv0;
        const unsigned ch = (unsigned)((lane & 15) ^ (4 * (lane >> 4)));
        dma16((const char*)(kp + (long long)kv0 * f.ks[2]), ((unsigned)rowc * (unsigned)f.ks[2] + 8u * ch) * 2u, at + g * GROUP_BYTES);
        dma16((const char*)(vp + (long long)kv0 * f.vs[2]), ((unsigned)rowc * (unsigned)f.vs[2] + 8u * ch) * 2u, at + STAGES * TILE_BYTES + g * GROUP_BYTES);
      }
    }
  };
  if (nt > 0) dma_tile(0);
  if (nt > 1) dma_tile(1);
  if (nt > 2) dma_tile(2);

  // ---- this lane's query row: q and dout as B operands, delta = dout . out ---------------------------------------------------------
  u32x32 qv, gv;  // k-step ks in elements 4ks .. 4ks+3
  float delta;
  {
    int row = qw0 + lq;
    row = row < f.L ? row : f.L - 1;
    const T* qr = (const T*)f.q + b * f.qs[0] + h * f.qs[1] + row * f.qs[2] + 8 * lh;
    const T* gr = (const T*)a.dout + b * a.dos[0] + h * a.dos[1] + row * a.dos[2] + 8 * lh;
    const T* orow = (const T*)f.out + b * f.os[0] + h * f.os[1] + row * f.os[2] + 8 * lh;
    float part = 0.f;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) {
      const u32x4 q4 = *(const u32x4*)(qr + 16 * ks), g4 = *(const u32x4*)(gr + 16 * ks);
      const vec8 o = *(const vec8*)(orow + 16 * ks), g = __builtin_bit_cast(vec8, g4);
#pragma unroll
      for (int i = 0; i < 4; i++) qv[4 * ks + i] = q4[i], gv[4 * ks + i] = g4[i];
#pragma unroll
      for (int i = 0; i < 8; i++) part = fmaf((float)o[i], (float)g[i], part);
    }
    delta = part + __shfl_xor(part, 32);
  }
  auto operand_of = [&](const u32x32& v, int ks) __attribute__((always_inline)) {
    u32x4 w;
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = v[4 * ks + i];
    return __builtin_bit_cast(vec8, w);
  };

  f32x16 dqacc[DBLK];
#pragma unroll
  for (int i = 0; i < DBLK; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) dqacc[i][r] = 0.f;
  const float c = f.scale * kLog2e;
  const float c_s = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, c)));
  float m_use = -1e30f, mc = m_use * c, l_run = 0.f;
  u32x4 row_addr, tr_addr;
  operand_offsets(lane, row_addr, tr_addr);

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  // State between steps: scores s and dP d of a tile (even tiles in sX, dX, odd ones in sY, dY); dS, in pairs of 16 bits, takes the first
  // eight registers of d.
  f32x16 sX, sY, dX, dY;
  auto product = [&](f32x16& acc, const char* tile, const u32x32& own) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) acc = TR::mfma32(*(const vec8*)(tile + row_addr[ks >> 1] + 32 * (ks & 1)), operand_of(own, ks), acc);
  };
  auto k_tile = [&](int i) __attribute__((always_inline)) { return smem + (i & 3) * TILE_BYTES; };
  auto v_tile = [&](int i) __attribute__((always_inline)) { return smem + (STAGES + (i & 3)) * TILE_BYTES; };
  auto row_max = [&](const f32x16& s) __attribute__((always_inline)) {
    float m = s[0];
#pragma unroll
    for (int r = 1; r < 16; r++) m = fmaxf(m, s[r]);
    return fmaxf(m, __shfl_xor(m, 32));  // the other 16 keys of this query sit in lane l^32
  };
  // the maximum raised to that of the scores, sum and accumulators brought to it
  auto raise = [&](const f32x16& s) __attribute__((always_inline)) {
    const float m_new = fmaxf(m_use, row_max(s));
    const float alpha = fast_exp2((m_use - m_new) * c);
    m_use = m_new;
    mc = m_new * c;
    l_run *= alpha;
#pragma unroll
    for (int i = 0; i < DBLK; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) dqacc[i][r] *= alpha;
  };
  auto weigh = [&](const f32x16& s, f32x16& d) __attribute__((always_inline)) {  // P from s, dS into d; the lane's sum of P
    float psum = 0.f;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      f32x8 x;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const float p = fast_exp2(fmaf(s[8 * t + i], c, -mc));
        psum += p;
        x[i] = p * (d[8 * t + i] - delta);
      }
      const u32x4 w = __builtin_bit_cast(u32x4, __builtin_convertvector(x, vec8));
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const unsigned one = w[i];
        d[4 * t + i] = __builtin_bit_cast(float, one);
      }
    }
    return psum;
  };
  auto hide = [&](f32x16& s, int kv0) __attribute__((always_inline)) {
    if ((CAUSAL && kv0 + BN - 1 > qw0 + coff) || kv0 + BN > S) {
      const int qi = qw0 + lq + coff;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int key = kv0 + 8 * (r >> 2) + 4 * lh + (r & 3);
        if (key >= S || (CAUSAL && key > qi)) s[r] = -INFINITY;
      }
    }
  };
  // General form of step i: dq of tile i-1, scores and dP of tile i+1, dS of tile i, as far as they are the wavefront's.
  auto slow_step = [&](int i, f32x16& s_cur, f32x16& d_cur, f32x16& s_new, f32x16& d_new) __attribute__((always_inline)) {
    if (i - 1 < mine) {
#pragma unroll
      for (int t = 0; t < 2; t++) {
        u32x4 w;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float one = d_new[4 * t + e];
          w[e] = __builtin_bit_cast(unsigned, one);
        }
#pragma unroll
        for (int db = 0; db < DBLK; db++) {
          const char* at = k_tile(i - 1) + tr_addr[db] + 4 * t * GROUP_BYTES;
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at);
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 2 * GROUP_BYTES));
          dqacc[db] = TR::mfma32(__builtin_bit_cast(vec8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7)), __builtin_bit_cast(vec8, w), dqacc[db]);
        }
      }
    }
    if (i + 1 < mine) product(s_new, k_tile(i + 1), qv), product(d_new, v_tile(i + 1), gv);
    if (i < mine) {
      hide(s_cur, first_key(i));
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(row_max(s_cur) > m_use + 8.f / c) != 0, 0)) raise(s_cur);
      l_run += weigh(s_cur, d_cur);
    }
  };
  auto step_dma = [&](int i) __attribute__((always_inline)) {
    if (i + 2 < nt) dma_tile(i + 2);
  };
  // what step i sent for is in place for the next one
  auto sync = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  u32x32 ring;
#pragma unroll
  for (int i = 0; i < 32; i++) ring[i] = 0u;
#pragma unroll
  for (int r = 0; r < 16; r++) sX[r] = 0.f, sY[r] = 0.f, dX[r] = 0.f, dY[r] = 0.f;
  if (mine > 0) {
    product(sX, k_tile(0), qv), product(dX, v_tile(0), gv);
    if (mine > 1) product(sY, k_tile(1), qv), product(dY, v_tile(1), gv);
    hide(sX, first_key(0));
    raise(sX);
    l_run = weigh(sX, dX);
  }
  int i = 1;
  if (nfast > 0) {
    float psum;
    // A lane's probabilities left the range the maximum allows (or are not numbers): dP anew, the maximum raised.
    // (the ring's requests for the next step are dropped and sent for again: the path needs its registers)
#define TT_DQ_SETTLE(S, D_, PREFETCH)                                                                                     \
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(psum <= kSumLimit)) != 0, 0)) {                                   \
      asm volatile("s_waitcnt lgkmcnt(0)" ::"{v[224:255]}"(ring) : "memory");                                            \
      product(D_, v_tile(i), gv);                                                                                        \
      raise(S);                                                                                                          \
      psum = weigh(S, D_);                                                                                               \
      asm volatile(PREFETCH : "={v[224:255]}"(ring) : "{v[88:91]}"(row_addr), "{v[92:95]}"(tr_addr) : "memory");          \
    }                                                                                                                    \
    l_run += psum;
#define TT_DQ_RUN(TXT)                                                                                                    \
  asm volatile(TXT                                                                                                       \
               : [o0] "+v"(dqacc[0]), [o1] "+v"(dqacc[1]), [o2] "+v"(dqacc[2]), [o3] "+v"(dqacc[3]), [ps] "=&v"(psum),      \
                 "+{v[160:175]}"(sX), "+{v[176:191]}"(sY), "+{v[192:207]}"(dX), "+{v[208:223]}"(dY), "+{v[224:255]}"(ring)  \
               : [c] "s"(c_s), [mc] "v"(mc), [dl] "v"(delta), "{v[96:127]}"(qv), "{v[128:159]}"(gv), "{v[88:91]}"(row_addr), "{v[92:95]}"(tr_addr) \
               : "v82", "v83", "v84", "v85", "v86", "v87", "memory")
#define TT_DQ_STEP(U, NEXT, S_CUR, D_CUR)                                                                                       \
    if (U % 2 == 0 && i > nfast) break;                                                                                  \
    step_dma(i);                                                                                                         \
    if constexpr (kIsBf16) TT_DQ_RUN(TT_B128_DQ_BF16_U##U);                                                              \
    else TT_DQ_RUN(TT_B128_DQ_F16_U##U);                                                                                 \
    TT_DQ_SETTLE(S_CUR, D_CUR, TT_B128_DQ_PREFETCH_U##NEXT)                                                               \
    sync();                                                                                                              \
    i++;
    asm volatile(TT_B128_DQ_PREFETCH_U0 : "+{v[224:255]}"(ring) : "{v[88:91]}"(row_addr), "{v[92:95]}"(tr_addr) : "memory");
    for (;;) {
      TT_DQ_STEP(0, 1, sY, dY)
      TT_DQ_STEP(1, 2, sX, dX)
      TT_DQ_STEP(2, 3, sY, dY)
      TT_DQ_STEP(3, 0, sX, dX)
    }
#undef TT_DQ_STEP
#undef TT_DQ_SETTLE
#undef TT_DQ_RUN
    // the ring's last requests land, and the last matrix instructions end, before the compiler's code goes on with the registers
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 15" : "+{v[224:255]}"(ring), "+{v[160:175]}"(sX), "+{v[176:191]}"(sY), "+{v[192:207]}"(dX), "+{v[208:223]}"(dY) : : "memory");
  }
  // (at an odd step; the last one is that behind the last tile)
  for (; i <= nt; i += 2) {
    step_dma(i);
    slow_step(i, sY, dY, sX, dX);
    sync();
    step_dma(i + 1);
    slow_step(i + 1, sX, dX, sY, dY);
    sync();
  }

  const float l_tot = l_run + __shfl_xor(l_run, 32);
  int ln;  // the lane number anew (as asm: the compiler would otherwise keep the values derived from it alive through the loop)
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
  const int half = ln >> 5, qi = qw0 + (ln & 31);
  if (qi >= f.L) return;
  const long long row_id = ((long long)b * f.Hq + h) * f.L + qi;
  if (a.dq_splits > 1) {
    store_dq_partial<D>(a, piece, row_id, half, dqacc, m_use * c, l_tot, delta);
    return;
  }
  if (half == 0) *(float2*)(a.stats + 2 * row_id) = make_float2(m_use * c + __log2f(l_tot), delta);
  const float w = f.scale / l_tot;
  T* dqp = (T*)a.dq + b * a.dqs[0] + h * a.dqs[1] + qi * a.dqs[2] + 4 * half;
#pragma unroll
  for (int db = 0; db < DBLK; db++)
#pragma unroll
    for (int rg = 0; rg < 4; rg++) {
      f32x4 x;
#pragma unroll
      for (int e = 0; e < 4; e++) x[e] = dqacc[db][4 * rg + e] * w;
      *(typename TR::vec4*)(dqp + 32 * db + 8 * rg) = __builtin_convertvector(x, typename TR::vec4);
    }
}

template <typename TR, bool CAUSAL>
int launch_dq(const BwdArgs& a, hipStream_t stream) {
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  const hipError_t granted = grant_dynamic_lds((const void*)backward_dq128_kernel<TR, CAUSAL>, DQ_LDS, state, done);
  if (granted != hipSuccess) return (int)granted;
  const long long grid = (long long)a.f.B * a.f.Hq * ((a.f.L + BM - 1) / BM) * a.dq_splits;
  hipLaunchKernelGGL((backward_dq128_kernel<TR, CAUSAL>), dim3((unsigned)grid), dim3(256), DQ_LDS, stream, a);
  return (int)hipGetLastError();
}

}  // namespace

int launch_backward_dq_d128(const BwdArgs& a, bool bf16, hipStream_t stream) {
  if (bf16) return a.f.causal ? launch_dq<BF16, true>(a, stream) : launch_dq<BF16, false>(a, stream);
  return a.f.causal ? launch_dq<F16, true>(a, stream) : launch_dq<F16, false>(a, stream);
}

}  // namespace ttsdpa
