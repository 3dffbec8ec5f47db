// Attention backward for fp16 / bf16, head_dim 128, without an attnMask, on gfx950 matrix cores (sdpa_backward_mfma.hip has
// the mathematics).
//
// dq and the row statistics: a workgroup owns 128 query rows of one (batch, query head), a wavefront 32 of them (Q and dout in registers); keys stream in tiles
// of 32.  Per tile a wavefront forms S^T = K.Q^T and dP^T = V.dout^T, turns them into P and dS on the vector ALU and accumulates dq^T +=
// K^T.dS^T: 24 matrix instructions (768 cycles) and 88 vector ones, 16 of them exponentials (about 550 cycles of issue, beside 16 for every
// matrix instruction).  In the compiler's order the three followed each other, the wavefronts of a SIMD hardly overlapping: 3250 cycles
// a tile of two wavefronts, the matrix pipe 44 % busy at 1.99 GHz.  Here a step is a stream of hand-ordered instructions
// (gen_backward128_steps.py) over three tiles: scores and dP of tile i+1 and dq of tile i-1 on the matrix pipe, the vector work of
// tile i between them.  2 x 32 heads (8) x 4096 x 4096, causal: 420 -> 378 us, the matrix pipe 58 % busy and the clock down at 1.69 GHz.
// Two things bound both kernels: the clock, which falls with the power of the operands' bits (on zeros dq takes 262 us of 370, dk/dv 361 of
// 480), and the instructions that a step still has beside its matrix ones: a compiler-made wait taken out of the loops gave 4.6 % (below).
//
// K and V come by direct global->LDS loads, four stages each (K of tiles i-1, i, i+1 and, on its way, i+2): a tile is eight groups of
// four 256-byte rows, 1040 bytes apart, chunk c of 16 bytes of row i of a group at slot c ^ 4i, so that one copy serves the
// row-major reads and the transposed ones without bank conflicts and both take four address registers.

// dk and dv: a workgroup owns 128 keys.  A tile of 32 query rows costs a wavefront 32 matrix instructions (1024 cycles), 80 vector ones
// and 44 KB of LDS operands, a SIMD's two wavefronts the LDS's whole 2050 cycles; here everything of a tile is one stream, a step, with its
// operands requested into the register ring 6 ahead (the next tile's first before the step ends) and all that is not a matrix
// instruction spread between those.  Same call: 620 -> 566 us in the first launches, the matrix pipe 55 % busy at 1.73 GHz
// (45 % at 1.87 in the compiler's order), 545 -> 520 among others once the chip is warm.  V's row addresses in four registers of
// their own instead of eight additions a step: forward and backward of this call 1160 -> 1152 us.  Without the compiler's wait for K in the loop (below)
// -> 1089 (1139 with both as before, on that box).

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
  // The lanes' offsets are formed for each tile from the lane number anew (a dozen instructions), but for bf16 under a causal mask.  Kept, they were
  // spilled, and a reload's wait in front of each request was one for the tiles in flight.  Forward and backward, f16, 2 x 32 heads (8) x 4096 causal
  // 1165 -> 1151 us, 4 x 8 x 1545 144.0 -> 141.4, 1 x 32 (4) x 2111 229.6 -> 225.8; 2 x 32 (8) x 2000 without a mask 626 -> 619.  bf16 without a mask, twelve
  // calls of 512 to 4096 rows, 1.7 % (1 x 32 (8) x 700 80.0 -> 77.3, 4 x 32 (8) x 1024 310.8 -> 304.9, 2 x 32 (8) x 4096 2052 -> 2040; 1 x 28 (4) x 1311 161.3 ->
  // 162.9, 2 x 7 (1) x 3000 333.0 -> 337.1).  bf16 causal spills nothing and keeps them: formed anew, 2 x 16 (8) x 1023 94.4 -> 95.9.
  constexpr bool kLaneKept = kIsBf16 && CAUSAL;
  auto lane_now = [&]() __attribute__((always_inline)) {
    int ln = lane;
    if constexpr (!kLaneKept) asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
    return ln;
  };
  const unsigned chunk = (unsigned)((lane & 15) ^ (4 * (lane >> 4)));
  const unsigned koff_kept = ((unsigned)(lane >> 4) * (unsigned)f.ks[2] + 8u * chunk) * 2u, voff_kept = ((unsigned)(lane >> 4) * (unsigned)f.vs[2] + 8u * chunk) * 2u;
  auto dma_tile = [&](int i) __attribute__((always_inline)) {
    const int kv0 = first_key(i);
    const unsigned at = smem_addr + (i & 3) * TILE_BYTES + 2 * wave * GROUP_BYTES;
    if (__builtin_expect(kv0 + BN <= S, 1)) {
      unsigned koff = koff_kept, voff = voff_kept;
      if constexpr (!kLaneKept) {
        const int ln = lane_now();
        const unsigned ch = (unsigned)((ln & 15) ^ (4 * (ln >> 4)));
        koff = ((unsigned)(ln >> 4) * (unsigned)f.ks[2] + 8u * ch) * 2u, voff = ((unsigned)(ln >> 4) * (unsigned)f.vs[2] + 8u * ch) * 2u;
      }
#pragma unroll
      for (int g = 0; g < 2; g++) {
        const int row = kv0 + 8 * wave + 4 * g;
        dma16((const char*)(kp + (long long)row * f.ks[2]), koff, at + g * GROUP_BYTES);
        dma16((const char*)(vp + (long long)row * f.vs[2]), voff, at + STAGES * TILE_BYTES + g * GROUP_BYTES);
      }
    } else {  // rows past the end re-read the last key (hidden below)
#pragma unroll
      for (int g = 0; g < 2; g++) {
        const int ln = lane_now();
        int row = 8 * wave + 4 * g + (ln >> 4);
        asm volatile("" : "+v"(row));  // keeps this rarely taken path's address arithmetic inside the branch
        const int rowc = kv0 + row < S ? row : S - 1 - kv0;
        const unsigned ch = (unsigned)((ln & 15) ^ (4 * (ln >> 4)));
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

  // (with the operands named the compiler's own wait for their loads lies here and not in the loop, where it would be one for the tile
  // just asked for)
  asm volatile("s_waitcnt vmcnt(0)" : "+v"(qv), "+v"(gv) : : "memory");
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
      const int ln = lane_now(), lh = ln >> 5, qi = qw0 + (ln & 31) + coff;
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
    store_dq_partial<D>(a, piece, row_id, half, dqacc, m_use * c, l_tot, -delta);
    return;
  }
  if (half == 0) *(float2*)(a.stats + 2 * row_id) = make_float2(m_use * c + __log2f(l_tot), -delta);  // -delta: see the dk/dv kernel
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

// ---- dk, dv ----------------------------------------------------------------------------------------------------------------
// A workgroup owns 128 keys of a (batch, KV head), a wavefront 32 of them (K in registers, V in LDS): the 32-row tiles of the query
// heads that see them stream past.  Eight wavefronts in two groups of four: both groups own the same keys and take alternate tiles, each
// with its own ring of three stages, and the second's gradients join the first's at the end — under a causal mask the first key block
// sees every row of every head of its group, the longest workgroup of the launch.
constexpr int KV_STAGES = 3, KV_STAGE_BYTES = 2 * TILE_BYTES + 256;  // Q, dout, lse and delta of 32 rows
constexpr int V_BYTES = 4 * TILE_BYTES;
constexpr int KV_LDS = V_BYTES + 2 * KV_STAGES * KV_STAGE_BYTES;
static_assert(KV_LDS >= 2 * 128 * 64 * 4, "the sum of one gradient needs 64 KiB");

__device__ __forceinline__ int ceil_div(int a, int b) { return a > 0 ? (a + b - 1) / b : 0; }

template <typename TR, bool CAUSAL>
__global__ __launch_bounds__(512, 2) void backward_dkv128_kernel(BwdArgs a) {
  typedef typename TR::elem T;
  typedef typename TR::vec8 vec8;
  typedef __attribute__((address_space(3))) vec8 lds_vec8;
  typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
  constexpr bool kIsBf16 = __is_same(T, __bf16);
  const KArgs& f = a.f;

  extern __shared__ __attribute__((aligned(16))) char smem[];
  const unsigned smem_addr = (unsigned)(unsigned long)(lds_void*)smem;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2, gw = wave & 3;  // group, wavefront of it
  const int lq = lane & 31, lh = lane >> 5;

  const int nkb = (f.S + BM - 1) / BM;
  const int nsplit = a.dkv_splits;
  int wg, split;  // this workgroup takes entries split, split + nsplit, ... of key-block workgroup wg
  split_of_workgroup(blockIdx.x, nsplit, f.B * f.Hkv, &wg, &split);
  int pair, kb;
  map_workgroup(wg, f.B * f.Hkv, nkb, &pair, &kb);
  const int hk = pair % f.Hkv, b = pair / f.Hkv;
  const int k0 = kb * BM, kw0 = k0 + gw * 32;
  const int S = keys_of_batch(f, b);  // rows of dk / dv from here to f.S are written as zeros
  if (k0 >= S) {
    if (grp == 0) zero_key_rows<TR, D>(a, split, b, hk, kw0 + lq, lh);
    return;
  }
  const int coff = CAUSAL ? causal_offset(f, S) : 0;

  // (asm: the compiler would make every LDS read wait for all loads that store there)
  auto dma16 = [&](const char* sbase, unsigned voff, unsigned lds_addr) __attribute__((always_inline)) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_addr) : "memory", "m0");
  };
  auto dma4 = [&](const char* sbase, unsigned voff, unsigned lds_addr) __attribute__((always_inline)) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_addr) : "memory", "m0");
  };

  // ---- V into LDS (wavefront w brings rows 16w .. 16w+15), this wavefront's K into registers -------------------------------------------
  {
    const char* vb = (const char*)((const T*)f.v + b * f.vs[0] + hk * f.vs[1] + (long long)k0 * f.vs[2]);
    const unsigned ch = (unsigned)((lane & 15) ^ (4 * (lane >> 4)));
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int row = 16 * wave + 4 * g + (lane >> 4);
      const int rowc = k0 + row < S ? row : S - 1 - k0;  // rows past the end re-read the last key (never stored)
      dma16(vb, ((unsigned)rowc * (unsigned)f.vs[2] + 8u * ch) * 2u, smem_addr + (4 * wave + g) * GROUP_BYTES);
    }
  }
  u32x32 kv;  // k-step ks in elements 4ks .. 4ks+3
  {
    int row = kw0 + lq;
    row = row < S ? row : S - 1;
    const T* kr = (const T*)f.k + b * f.ks[0] + hk * f.ks[1] + row * f.ks[2] + 8 * lh;
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) {
      const u32x4 k4 = *(const u32x4*)(kr + 16 * ks);
#pragma unroll
      for (int i = 0; i < 4; i++) kv[4 * ks + i] = k4[i];
    }
  }

  // Query tiles it0 .. ntq-1 of each of the G heads see keys of this workgroup.  They are taken from the last tile down (or
  // up: dkv_walks_up), the heads of a tile one after the other: every key block of a (batch, KV head) then starts at the same tile and
  // walks in step with the others (one further down the causal triangle just stops earlier), so the tile one workgroup
  // fetches from HBM is in the XCD's L2 for the others.  This workgroup's entries are split, split + nsplit, ... of that
  // list; entry idx of ITS list belongs to group idx % 2.
  const int ntq = (f.L + 31) / 32;
  int it0 = 0;
  if (CAUSAL) it0 = (k0 - coff > 0 ? k0 - coff : 0) / 32;
  const int nt = ntq > it0 ? ntq - it0 : 0;
  const int total = split < f.G * nt ? (f.G * nt - split + nsplit - 1) / nsplit : 0;
  const int niter = (total + 1) / 2;  // iterations of either group (the second may have one entry less)
  const bool walk_up = dkv_walks_up(a, CAUSAL, wg);
  // wavefront gw of a group brings rows 8gw .. 8gw+7 (two groups of four) of the Q tile and of the dout tile into the group's ring, and
  // the statistics (all four the same): lse of the 32 rows, then -delta, where the sums of dP - delta start
  const unsigned ring_addr = smem_addr + V_BYTES + grp * KV_STAGES * KV_STAGE_BYTES;
  const unsigned chunk = (unsigned)((lane & 15) ^ (4 * (lane >> 4)));
  const u32x2 offs = {((unsigned)(lane >> 4) * (unsigned)f.qs[2] + 8u * chunk) * 2u, ((unsigned)(lane >> 4) * (unsigned)a.dos[2] + 8u * chunk) * 2u};
  // what the next request is for: entry, head of the group, first row, and where this wavefront's part begins
  int next = grp, next_head = (split + nsplit * grp) % f.G, next_row = 32 * (walk_up ? it0 + (split + nsplit * grp) / f.G : ntq - 1 - (split + nsplit * grp) / f.G);
  const int dir = walk_up ? 32 : -32, step_head = 2 * nsplit % f.G, step_row = 2 * nsplit / f.G * dir;
  const long long head0 = (long long)b * f.Hq + hk * f.G + next_head;
  const char* q_next = (const char*)((const T*)f.q + b * f.qs[0] + (hk * f.G + next_head) * f.qs[1] + (long long)(next_row + 8 * gw) * f.qs[2]);
  const char* g_next = (const char*)((const T*)a.dout + b * a.dos[0] + (hk * f.G + next_head) * a.dos[1] + (long long)(next_row + 8 * gw) * a.dos[2]);
  const char* s_next = (const char*)(a.stats + 2 * (head0 * f.L + next_row));
  const long long q_step = 2 * (step_head * f.qs[1] + step_row * f.qs[2]), q_wrap = 2 * (dir * f.qs[2] - f.G * f.qs[1]);
  const long long g_step = 2 * (step_head * a.dos[1] + step_row * a.dos[2]), g_wrap = 2 * (dir * a.dos[2] - f.G * a.dos[1]);
  const long long s_step = 8 * ((long long)step_head * f.L + step_row), s_wrap = 8 * (dir - (long long)f.G * f.L);
  auto dma_next = [&](int stage) __attribute__((always_inline)) {
    const bool more = next < total;
    if (more) {
      const unsigned at = ring_addr + stage * KV_STAGE_BYTES, mine = at + 2 * gw * GROUP_BYTES;
      int ln;  // the lane number anew: nothing derived from it lives through the loop
      asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
      if (__builtin_expect(next_row + 32 <= f.L, 1)) {
        dma16(q_next, offs[0], mine);
        dma16(g_next, offs[1], mine + TILE_BYTES);
        dma16(q_next + 8 * f.qs[2], offs[0], mine + GROUP_BYTES);
        dma16(g_next + 8 * a.dos[2], offs[1], mine + TILE_BYTES + GROUP_BYTES);
        dma4(s_next, (unsigned)(2 * (ln & 31) + (ln >> 5)) * 4u, at + 2 * TILE_BYTES);
      } else {  // rows past the end re-read the last row (weight forced to 0)
        const unsigned ch = (unsigned)((ln & 15) ^ (4 * (ln >> 4)));
        const char *qb = q_next - 16 * gw * f.qs[2], *gb = g_next - 16 * gw * a.dos[2];
#pragma unroll
        for (int g = 0; g < 2; g++) {
          const int row = 8 * gw + 4 * g + (ln >> 4), rowc = next_row + row < f.L ? row : f.L - 1 - next_row;
          dma16(qb, ((unsigned)rowc * (unsigned)f.qs[2] + 8u * ch) * 2u, mine + g * GROUP_BYTES);
          dma16(gb, ((unsigned)rowc * (unsigned)a.dos[2] + 8u * ch) * 2u, mine + TILE_BYTES + g * GROUP_BYTES);
        }
        const int row = ln & 31, rowc = next_row + row < f.L ? row : f.L - 1 - next_row;
        dma4(s_next, (unsigned)(2 * rowc + (ln >> 5)) * 4u, at + 2 * TILE_BYTES);
      }
    }
    const bool wrap = next_head + step_head >= f.G;
    next += 2;
    next_head += step_head - (wrap ? f.G : 0), next_row += step_row + (wrap ? dir : 0);
    q_next += q_step + (wrap ? q_wrap : 0), g_next += g_step + (wrap ? g_wrap : 0), s_next += s_step + (wrap ? s_wrap : 0);
    return more;
  };
  int row_now = next_row;  // first rows of the tiles of this iteration and the next
  dma_next(0);
  int row_next = next_row;
  dma_next(1);

  // Iterations j0 .. j1-1 take the stream: tiles that hide nothing from the wavefront's keys.
  int j0 = niter, j1 = niter;
  if (kw0 + 32 <= S) {
    int lo = it0, hi = f.L / 32;  // first such tile and the one behind the last
    if (CAUSAL) {
      const int first = ceil_div(kw0 + 31 - coff, 32);
      lo = first > lo ? first : lo;
    }
    lo = lo < hi ? lo : hi;
    const int e0 = f.G * (walk_up ? lo - it0 : ntq - hi), e1 = f.G * (walk_up ? hi - it0 : ntq - lo);
    j0 = ceil_div(ceil_div(e0 - split, nsplit) - grp, 2);
    j1 = ceil_div(ceil_div(e1 - split, nsplit) - grp, 2);
    j0 = __builtin_amdgcn_readfirstlane(j0 < niter ? j0 : niter), j1 = __builtin_amdgcn_readfirstlane(j1 < niter ? j1 : niter);
  }

  f32x16 dkacc[DBLK], dvacc[DBLK];
#pragma unroll
  for (int i = 0; i < DBLK; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) dkacc[i][r] = 0.f, dvacc[i][r] = 0.f;
  const float c = f.scale * kLog2e;
  const float c_s = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, c)));
  u32x4 row_addr, tr_addr;
  operand_offsets(lane, row_addr, tr_addr);
#pragma unroll
  for (int i = 0; i < 4; i++) row_addr[i] += ring_addr, tr_addr[i] += ring_addr;
  const unsigned v_from_ring = (unsigned)__builtin_amdgcn_readfirstlane((int)(smem_addr + gw * TILE_BYTES - ring_addr));

  asm volatile("s_waitcnt vmcnt(0)" : "+v"(kv) : : "memory");  // (named for the reason given in the dq kernel)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  // every wavefront is through with its reads, and the next tile is in place (what was asked for last may still be on its way)
  auto sync = [&](bool more) __attribute__((always_inline)) {
    if (more) asm volatile("s_waitcnt vmcnt(5) lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // General form of iteration j.  The operand addresses are the ring's current stage's.
  auto slow_step = [&](int j, int stage) __attribute__((always_inline)) {
    const int i0 = row_now;
    row_now = row_next, row_next = next_row;
    const bool more = dma_next(stage == 0 ? 2 : stage - 1);
    const unsigned at_stage = stage * KV_STAGE_BYTES;
    const int idx = 2 * j + grp;
    if (idx < total) {
      int ln;
      asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
      const int lh = ln >> 5;
      const unsigned st = ring_addr + at_stage + 2 * TILE_BYTES + 16 * lh;
      f32x16 s, d;
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        const f32x4 minus_delta = *(lds_f32x4*)(st + 128 + 32 * rg);
#pragma unroll
        for (int e = 0; e < 4; e++) s[4 * rg + e] = 0.f, d[4 * rg + e] = minus_delta[e];
      }
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ks++) {
        u32x4 w;
#pragma unroll
        for (int i = 0; i < 4; i++) w[i] = kv[4 * ks + i];
        s = TR::mfma32(*(lds_vec8*)(row_addr[ks >> 1] + 32 * (ks & 1)), __builtin_bit_cast(vec8, w), s);
      }
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ks++)
        d = TR::mfma32(*(lds_vec8*)(row_addr[ks >> 1] + TILE_BYTES + 32 * (ks & 1)), *(lds_vec8*)(row_addr[ks >> 1] + (v_from_ring - at_stage) + 32 * (ks & 1)), d);
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        const f32x4 lse = *(lds_f32x4*)(st + 32 * rg);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int r = 4 * rg + e;
          s[r] = fast_exp2(fmaf(s[r], c, -lse[e]));
          d[r] *= s[r];
        }
      }
      // (a wavefront whose keys no row of the tile sees runs it with every weight 0)
      if ((CAUSAL && kw0 + 31 > i0 + coff) || kw0 + 32 > S || i0 + 32 > f.L) {
        const int key = kw0 + (ln & 31);
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const int qrow = i0 + 8 * (r >> 2) + 4 * lh + (r & 3);
          const bool hidden = (key >= S) | (qrow >= f.L) | (CAUSAL && key > qrow + coff);
          s[r] = hidden ? 0.f : s[r], d[r] = hidden ? 0.f : d[r];
        }
      }
#pragma unroll
      for (int t = 0; t < 2; t++) {
        f32x8 x, y;
#pragma unroll
        for (int i = 0; i < 8; i++) x[i] = s[8 * t + i], y[i] = d[8 * t + i];
        const vec8 p = __builtin_convertvector(x, vec8), ds = __builtin_convertvector(y, vec8);
#pragma unroll
        for (int db = 0; db < DBLK; db++) {
          const unsigned at = tr_addr[db] + 4 * t * GROUP_BYTES;
          const s16x4 glo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + TILE_BYTES));
          const s16x4 ghi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + TILE_BYTES + 2 * GROUP_BYTES));
          const s16x4 qlo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at);
          const s16x4 qhi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 2 * GROUP_BYTES));
          dvacc[db] = TR::mfma32(__builtin_bit_cast(vec8, (s16x8)__builtin_shufflevector(glo, ghi, 0, 1, 2, 3, 4, 5, 6, 7)), p, dvacc[db]);
          dkacc[db] = TR::mfma32(__builtin_bit_cast(vec8, (s16x8)__builtin_shufflevector(qlo, qhi, 0, 1, 2, 3, 4, 5, 6, 7)), ds, dkacc[db]);
        }
      }
    }
    const unsigned advance = stage == 2 ? 0u - 2 * KV_STAGE_BYTES : KV_STAGE_BYTES;
#pragma unroll
    for (int i = 0; i < 4; i++) row_addr[i] += advance, tr_addr[i] += advance;
    sync(more);
  };

  int j = 0, stage = 0;
#pragma nounroll
  for (int turn = 0; turn < 2; turn++) {
    for (const int end = turn == 0 ? j0 : niter; j < end; j++) {
      slow_step(j, stage);
      stage = stage == 2 ? 0 : stage + 1;
    }
    if (j >= j1) continue;
    u32x32 ring;
    f32x16 tmp[3];
#pragma unroll
    for (int i = 0; i < 32; i++) ring[i] = 0u;
    u32x4 v_addr;
#pragma unroll
    for (int i = 0; i < 4; i++) v_addr[i] = row_addr[i] + (v_from_ring - stage * KV_STAGE_BYTES);
    asm volatile(TT_B128_DKV_PREFETCH : "+{v[224:255]}"(ring) : "{v[140:143]}"(row_addr) : "memory");
#define TT_DKV_RUN(TXT)                                                                                                        \
  asm volatile(TXT                                                                                                            \
               : [o0] "+{v[0:15]}"(dkacc[0]), [o1] "+{v[16:31]}"(dkacc[1]), [o2] "+{v[32:47]}"(dkacc[2]), [o3] "+{v[48:63]}"(dkacc[3]), [o4] "+{v[64:79]}"(dvacc[0]),       \
                 [o5] "+{v[80:95]}"(dvacc[1]), [o6] "+{v[96:111]}"(dvacc[2]), [o7] "+{v[112:127]}"(dvacc[3]), "+{v[224:255]}"(ring), "=&{v[144:159]}"(tmp[0]), \
                 "=&{v[160:175]}"(tmp[1]), "=&{v[176:191]}"(tmp[2]), "+{v[140:143]}"(row_addr), "+{v[136:139]}"(tr_addr)       \
               : [c] "s"(c_s), [st] "s"(ring_addr + at_stage), [adv] "s"(advance),           \
                 [more] "s"(more), "{v[192:223]}"(kv), "{v[128:131]}"(v_addr), "{v[132:133]}"(offs)                                                    \
               : "memory", "scc")
    do {
      row_now = row_next, row_next = next_row;
      const int more = __builtin_amdgcn_readfirstlane((int)dma_next(stage == 0 ? 2 : stage - 1));
      const unsigned at_stage = stage * KV_STAGE_BYTES, advance = stage == 2 ? 0u - 2 * KV_STAGE_BYTES : KV_STAGE_BYTES;
      if constexpr (kIsBf16) TT_DKV_RUN(TT_B128_DKV_BF16);
      else TT_DKV_RUN(TT_B128_DKV_F16);
      stage = stage == 2 ? 0 : stage + 1;
    } while (++j < j1);
#undef TT_DKV_RUN
    // the ring's last requests land, and the last matrix instructions end, before the compiler's code goes on with the registers
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 15" : "+{v[224:255]}"(ring), "+v"(dkacc[0]), "+v"(dkacc[1]), "+v"(dkacc[2]), "+v"(dkacc[3]),
                 "+v"(dvacc[0]), "+v"(dvacc[1]), "+v"(dvacc[2]), "+v"(dvacc[3]) : : "memory");
  }

  // ---- the second group's gradients join the first's, one (64 KiB of fp32) at a time -------------------------------------------------
  int ln;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
  float* red = (float*)smem;
  const int slot = gw * 64 + ln;
#pragma unroll
  for (int which = 0; which < 2; which++) {
    f32x16* acc = which == 0 ? dkacc : dvacc;
    if (grp == 1) {
#pragma unroll
      for (int db = 0; db < DBLK; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) red[(db * 16 + r) * 256 + slot] = acc[db][r];
    }
    __syncthreads();
    if (grp == 0) {
#pragma unroll
      for (int db = 0; db < DBLK; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[db][r] += red[(db * 16 + r) * 256 + slot];
    }
    __syncthreads();
  }
  if (grp == 0) store_key_grads<TR, D>(a, split, b, hk, kw0 + (ln & 31), ln >> 5, dkacc, dvacc, f.scale);
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

template <typename TR, bool CAUSAL>
int launch_dkv(const BwdArgs& args, hipStream_t stream) {
  BwdArgs a = args;
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  const hipError_t granted = grant_dynamic_lds((const void*)backward_dkv128_kernel<TR, CAUSAL>, KV_LDS, state, done);
  if (granted != hipSuccess) return (int)granted;
  static int round_cache[kMaxDevices];
  a.dkv_round = CAUSAL ? dkv_round_of((const void*)backward_dkv128_kernel<TR, CAUSAL>, 512, KV_LDS, round_cache) : 0;
  const long long grid = (long long)a.f.B * a.f.Hkv * ((a.f.S + BM - 1) / BM) * a.dkv_splits;
  hipLaunchKernelGGL((backward_dkv128_kernel<TR, CAUSAL>), dim3((unsigned)grid), dim3(512), KV_LDS, stream, a);
  return (int)hipGetLastError();
}

}  // namespace

int launch_backward_dq_d128(const BwdArgs& a, bool bf16, hipStream_t stream) {
  if (bf16) return a.f.causal ? launch_dq<BF16, true>(a, stream) : launch_dq<BF16, false>(a, stream);
  return a.f.causal ? launch_dq<F16, true>(a, stream) : launch_dq<F16, false>(a, stream);
}

int launch_backward_dkv_d128(const BwdArgs& a, bool bf16, hipStream_t stream) {
  if (bf16) return a.f.causal ? launch_dkv<BF16, true>(a, stream) : launch_dkv<BF16, false>(a, stream);
  return a.f.causal ? launch_dkv<F16, true>(a, stream) : launch_dkv<F16, false>(a, stream);
}

}  // namespace ttsdpa
