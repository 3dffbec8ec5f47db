// Flash-attention forward for fp16 / bf16, head_dim 128 and 64, for calls whose 256-row tiles would not fill the chip evenly: the
// pipelined prefill kernel (sdpa_prefill_d128.hip, sdpa_prefill_d64.hip) with 128 rows to a workgroup and a row's keys dealt out to
// two groups of four wavefronts.
//
// What it is for.  The pipelined kernels' workgroup of 256 rows walks its keys tile by tile, 1.4 us each, one workgroup to a CU: a
// launch lasts as long as its longest workgroup.  Under a causal mask that is twice the average, and with fewer row tiles than CUs the
// rest of the chip is idle (us on that kernel and here, head_dim 128, causal: 16 heads x 1327 rows 34.4 and 22.9, 16 x 756 24.3 and
// 16.5, 32 x 1539 41 and 33; 6 x 32 x 326 on 3781 keys of a paged cache 162 and 126; head_dim 64, 32 x 727 18.1 and 12.8).  Here wavefront w of a group owns rows 32 w .. 32 w + 31 of the workgroup's 128, and of a row's keys, in
// halves of 32, group 0 takes the even ones and group 1 the odd ones: twice the workgroups, each half as long, and no records in memory:
// the two groups' accumulators come together in LDS.  The matrix work and the LDS bytes per key and row are the same; what it costs is
// twice the tile loads (each half serves four wavefronts instead of eight, from the XCD's L2), a barrier per 32 keys of a group instead
// of per 64, and the exchange at the end.
//
// LDS.  Each group has a ring of four halves for K and one for V.  Half n (of the group's own: the keys 64 n + 32 group ..) sits in
// place n % 4.  Step n forms the scores of half n+2, takes the exponentials of half n+1 and accumulates P.V of half n, as in the
// pipelined kernels, and its last LDS requests are for the operands of step n+1 (K of n+3, V of n+1).  K is therefore requested five
// halves ahead and V three, in the place of the half that step n-1 was the last to read, and everything sent for in step n-1 is in
// place when step n+1 starts: a load has a whole step (0.7 us at head_dim 128) to arrive, as in the pipelined kernels.
// The streams are theirs with rings of two tiles (TT_P128_DSTEP_.., gen_prefill128_steps.py).

#include "sdpa_common.h"
#include "prefill128_steps.inc"  // hand-ordered instruction streams of the steady state (gen_prefill128_steps.py)
#include "prefill64_steps.inc"

namespace ttsdpa {

namespace {

constexpr int NW = 8;           // wavefronts per workgroup
constexpr int GW = NW / 2;      // ... of a group
constexpr int WM = 32;          // query rows per wavefront
constexpr int BM = GW * WM;     // query rows per workgroup
constexpr int RING = 4;         // halves of K (of V) that a group has in LDS
constexpr float kSumLimit = 1024.f;  // a lane's 16 probabilities of a half may sum to this much before the maximum is raised

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) void lds_void;

template <int D>
struct Sizes {
  static constexpr int ROW = 2 * D;                 // bytes of a K or V row
  static constexpr int HALF = 32 * ROW;             // ... of a half
  static constexpr int GROUP = RING * HALF;         // ... of a group's ring
  static constexpr int STAGES = 2 * 2 * GROUP;      // ... of K, both groups, then V
  static constexpr int OUT = WM * D;                // output staging of a wavefront: half of the columns of its rows
  static constexpr int LDS = STAGES + NW * OUT;
  static constexpr int LOADS = D / 64;              // load instructions of a wavefront for a half: 512 / D rows each
  static constexpr int EXCHANGE = GW * 2 * (D / 16) * 1024;  // what the groups hand each other: half of their accumulators
  static_assert(EXCHANGE + GW * 2 * 512 <= STAGES, "the exchange takes the place of the stages");
};

template <int D>
__device__ __forceinline__ int swz(int row) {
  return D == 128 ? ((row & 3) << 2) | ((row >> 2) & 3) : (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}

// PAGED, SPLIT: as in sdpa_prefill_d128.hip; the first key of a split is a multiple of 256.
template <typename TR, int D, bool CAUSAL, bool PAGED, bool SPLIT>
__global__ __launch_bounds__(NW * 64, 2) void prefill_dealt_kernel(KArgs a) {
  typedef typename TR::elem T;
  typedef typename TR::vec8 vec8;
  typedef Sizes<D> Z;
  constexpr int KST = D / 16, NDB = D / 32, LPR = D / 8;  // k-steps of a score product; head_dim blocks; lanes of a row's load
  typedef uint32_t u32xq __attribute__((ext_vector_type(4 * KST)));
  typedef uint32_t u32xa __attribute__((ext_vector_type(KST)));
  typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
  typedef uint32_t u32x32 __attribute__((ext_vector_type(32)));

  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2, gw = wave & 3;  // the group, the wavefront's place in it
  const int lq = lane & 31;
  const int lh = lane >> 5;

  // ---- workgroup -> (batch, kv head, query head in group, row tile): as in sdpa_prefill_d128.hip, single row tiles ----------
  const int ntile = (a.L + BM - 1) / BM;
  const int npair = a.B * a.Hkv;
  int pair, in, split = 0;
  if (SPLIT) {
    if (!find_piece(a, BM, CAUSAL, &pair, &in, &split)) return;
  } else {
    const int n = blockIdx.x;
    const int gq = pair_classes(npair);
    const int xcd = n & 7, slot = n >> 3;
    const int cls = xcd % gq, sub = xcd / gq;
    const long long item = (long long)slot * (8 / gq) + sub;  // work item of the class
    const int ppc = npair / gq;
    if (item >= (long long)ppc * a.G * ntile) return;  // the grid is rounded up to a multiple of 8
    if (CAUSAL) {  // longest row tiles first across all the pairs of the class
      pair = cls + gq * (int)(item % ppc);
      in = (int)(item / ppc);
    } else {
      pair = cls + gq * (int)(item / (a.G * ntile));
      in = (int)(item % (a.G * ntile));
    }
  }
  const int b = pair / a.Hkv, hk = pair % a.Hkv;
  const int h = hk * a.G + in % a.G;
  const int q0 = (CAUSAL ? ntile - 1 - in / a.G : in / a.G) * BM;
  const int n0 = SPLIT ? split * (a.kv_chunk / 64) : 0;  // the groups' first half (a multiple of the ring's length)

  const T* qp = (const T*)a.q + b * a.qs[0] + h * a.qs[1];
  const int* table = PAGED ? a.block_table + (long long)b * a.bt_stride : nullptr;
  const T* kp = (const T*)a.k + (PAGED ? 0 : b * a.ks[0]) + hk * a.ks[1];
  const T* vp = (const T*)a.v + (PAGED ? 0 : b * a.vs[0]) + hk * a.vs[1];
  const int S = keys_of_batch(a, b);
  // Wavefronts w and w+4 share a SIMD: under a causal mask the second group takes its rows in reverse, so that every SIMD has a long
  // and a short one.
  const int rowgroup = (CAUSAL && grp) ? GW - 1 - gw : gw;
  const int qw0 = q0 + rowgroup * WM;

  if (SPLIT && n0 * 64 >= S) return;  // beyond the keys (none at all: the merge kernel writes zeros)
  if (S == 0) {  // no keys for this batch entry: zeros, the reference's empty contraction (kept out of the main loop)
    T* obase = (T*)a.out + b * a.os[0] + h * a.os[1];
    vec8 zero;
#pragma unroll
    for (int i = 0; i < 8; i++) zero[i] = (T)0.f;
    for (int row = q0 + tid / LPR; row < q0 + BM && row < a.L; row += NW * 64 / LPR) *(vec8*)(obase + row * a.os[2] + 8 * (tid % LPR)) = zero;
    return;
  }

  // Query row i sees keys up to i + coff (coff = 0: the reference's top-left aligned mask); qc0 is this wavefront's first row in key
  // coordinates.
  const int coff = CAUSAL ? causal_offset(a, S) : 0;
  const int qc0 = qw0 + coff;
  // Halves of the workgroup's row tile (both groups'), and how many of them are this group's; the wavefront's own, under a causal mask
  // those that start at or before its last row.  Counts are from the first key on, also in a split.
  int halves = (S + 31) / 32;
  if (CAUSAL) {
    const int last = (q0 + BM < a.L ? q0 + BM : a.L) - 1 + coff;
    halves = last / 32 + 1 < halves ? last / 32 + 1 : halves;
  }
  if (SPLIT) {
    const int end = 2 * n0 + a.kv_chunk / 32;
    halves = end < halves ? end : halves;
  }
  if (SPLIT && 2 * n0 >= halves) return;  // a row tile that ends before this split
  const int steps = (halves + 1) / 2, loaded = (halves + 1 - grp) / 2;
  const int seen = CAUSAL ? (qc0 + WM - 1) / 32 + 1 : halves;  // (beyond the workgroup's halves where keys or split end earlier)
  const int my_halves = ((seen < halves ? seen : halves) + 1 - grp) / 2;

  // ---- global -> LDS: a group's wavefront moves rows 8 gw .. 8 gw + 7 of a half, 512 / D rows (1 KiB) per instruction; the 16-byte
  // chunk c of row r sits at chunk slot c ^ swz(r), so a lane fetches the chunk that belongs in its slot --------------------------
  unsigned ld_koff[Z::LOADS], ld_voff[Z::LOADS];
#pragma unroll
  for (int i = 0; i < Z::LOADS; i++) {
    const int row = 8 * gw + 4 * i + lane / LPR;
    const int chunk = (lane % LPR) ^ swz<D>(row);
    ld_koff[i] = ((unsigned)row * (unsigned)a.ks[2] + 8u * chunk) * 2u;  // the host checks that 64 rows fit 32 bits
    ld_voff[i] = ((unsigned)row * (unsigned)a.vs[2] + 8u * chunk) * 2u;
  }
  // asm, with wait states for a scalar base that a vector instruction restored: as in sdpa_prefill_d128.hip
  auto dma_issue = [&](const char* sbase, unsigned voff, unsigned lds_addr) __attribute__((always_inline)) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_addr) : "memory", "m0");
  };
  const unsigned ring_addr = (unsigned)(unsigned long)(lds_void*)smem + grp * Z::GROUP;  // the group's K ring; its V ring STAGES / 2 on
  // Paged cache: a window of 64 entries of the table in a register, the next one in another (sdpa_prefill_d128.hip)
  unsigned ptab[2] = {0u, 0u};
  const int last_entry = PAGED ? (S - 1) >> a.page_shift : 0;
  auto entry_off = [&](int w) __attribute__((always_inline)) {
    const int e = 64 * w + lane;
    return 4u * (unsigned)(e < last_entry ? e : last_entry);
  };
  auto first_key = [&](int n) __attribute__((always_inline)) { return 32 * (2 * n + grp); };
  auto dma_half = [&](const T* base, long long rstride, long long pstride, const unsigned (&off)[Z::LOADS], int kv0, unsigned addr) __attribute__((always_inline)) {
    long long toff = (long long)kv0 * rstride;
    if (PAGED) {
      const int e = kv0 >> a.page_shift;
      const int p0 = __builtin_amdgcn_readlane(ptab[0], e & 63), p1 = __builtin_amdgcn_readlane(ptab[1], e & 63);
      toff = (long long)((e & 64) ? p1 : p0) * pstride + (long long)(kv0 & ((1 << a.page_shift) - 1)) * rstride;
    }
    const char* src = (const char*)(base + toff);
    if (__builtin_expect(kv0 + 32 <= S, 1)) {
#pragma unroll
      for (int i = 0; i < Z::LOADS; i++) dma_issue(src, off[i], addr + (8 * gw + 4 * i) * Z::ROW);
    } else {  // ragged last half: rows past the end re-read the last valid row (their scores are masked)
#pragma unroll
      for (int i = 0; i < Z::LOADS; i++) {
        int row = 8 * gw + 4 * i + lane / LPR;
        asm volatile("" : "+v"(row));  // keeps this rarely taken path's address arithmetic inside the branch
        const int chunk = (lane % LPR) ^ swz<D>(row);
        const int rowc = row < S - kv0 ? row : S - 1 - kv0;
        dma_issue(src, ((unsigned)rowc * (unsigned)rstride + 8u * chunk) * 2u, addr + (8 * gw + 4 * i) * Z::ROW);
      }
    }
  };
  auto dma_k = [&](int n) __attribute__((always_inline)) { dma_half(kp, a.ks[2], a.ks[0], ld_koff, first_key(n), ring_addr + (n & 3) * Z::HALF); };
  auto dma_v = [&](int n) __attribute__((always_inline)) {
    dma_half(vp, a.vs[2], a.vs[0], ld_voff, first_key(n), ring_addr + Z::STAGES / 2 + (n & 3) * Z::HALF);
  };
  // Wait until at most this wavefront's newest `keep` halves are still in flight (loads complete in issue order), then meet the other
  // wavefronts: what was sent for before those is visible to all.
  auto dma_wait_and_sync = [&](int keep) __attribute__((always_inline)) {
    if (__builtin_expect(keep >= 2, 1)) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * Z::LOADS) : "memory");
    else if (keep == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(Z::LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // bare barrier: the loads above carry the ordering; __syncthreads() would also drain the LDS operand prefetch
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // ---- LDS operand addresses (bytes), loop-invariant: as in sdpa_prefill_d128.hip, in the group's rings -----------------------------
  u32xa k_addr;
  {
    const unsigned base = (unsigned)(grp * Z::GROUP + lq * Z::ROW + 16 * (lh ^ swz<D>(lq)));
#pragma unroll
    for (int ks = 0; ks < KST; ks++) k_addr[ks] = base ^ (unsigned)(32 * ks);
  }
  u32xa v_addr;  // index 2 * db + ld; the V region's base folded in
  {
    const int s = lane & 15, dhalf = (lane >> 4) & 1;
#pragma unroll
    for (int ld = 0; ld < 2; ld++) {
      const int row = 8 * ld + 4 * lh + (s >> 2);
#pragma unroll
      for (int db = 0; db < NDB; db++) {
        const int chunk = 4 * db + 2 * dhalf + ((s & 3) >> 1);
        v_addr[2 * db + ld] = (unsigned)(Z::STAGES / 2 + grp * Z::GROUP + row * Z::ROW + 16 * (chunk ^ swz<D>(row)) + 8 * (s & 1));
      }
    }
  }

  // ---- first loads: K of halves 0 .. 3, V of 0 .. 2 ----------------------------------------------------------------------------------
  if (PAGED) {  // the table's windows of the first entry and behind it (s_nop: the base as in dma_issue)
    const int w = (n0 * 64) >> a.page_shift >> 6;
    asm volatile("s_nop 4\n\tglobal_load_dword %0, %2, %4\n\tglobal_load_dword %1, %3, %4\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(ptab[0]), "=&v"(ptab[1])
                 : "v"(entry_off(w + (w & 1))), "v"(entry_off(w + ((w & 1) ^ 1))), "s"(table)
                 : "memory");
  }
  if (n0 < loaded) dma_k(n0), dma_v(n0);
  if (n0 + 1 < loaded) dma_k(n0 + 1), dma_v(n0 + 1);
  if (n0 + 2 < loaded) dma_k(n0 + 2), dma_v(n0 + 2);
  if (n0 + 3 < loaded) dma_k(n0 + 3);
  // Q into its registers, and everything sent for so far in place: one statement (sdpa_prefill_d128.hip)
  u32xq qv;
  {
    const int first = qw0 < a.L ? qw0 : a.L - 1;  // rows past the end re-read the last row (never stored)
    int row = qw0 + lq;
    row = row < a.L ? row : a.L - 1;
    const char* qbase = (const char*)(qp + (long long)first * a.qs[2]);
    const unsigned qoff = ((unsigned)(row - first) * (unsigned)a.qs[2] + 8u * lh) * 2u;  // the host checks that 32 rows fit 32 bits
    if constexpr (D == 128)
      asm volatile(
          "s_nop 4\n\t"
          "global_load_dwordx4 v[120:123], %1, %2\n\t"
          "global_load_dwordx4 v[124:127], %1, %2 offset:32\n\t"
          "global_load_dwordx4 v[128:131], %1, %2 offset:64\n\t"
          "global_load_dwordx4 v[132:135], %1, %2 offset:96\n\t"
          "global_load_dwordx4 v[136:139], %1, %2 offset:128\n\t"
          "global_load_dwordx4 v[140:143], %1, %2 offset:160\n\t"
          "global_load_dwordx4 v[144:147], %1, %2 offset:192\n\t"
          "global_load_dwordx4 v[148:151], %1, %2 offset:224\n\t"
          "s_waitcnt vmcnt(0)"
          : "={v[120:151]}"(qv)
          : "v"(qoff), "s"(qbase)
          : "memory");
    else
      asm volatile(
          "s_nop 4\n\t"
          "global_load_dwordx4 v[120:123], %1, %2\n\t"
          "global_load_dwordx4 v[124:127], %1, %2 offset:32\n\t"
          "global_load_dwordx4 v[128:131], %1, %2 offset:64\n\t"
          "global_load_dwordx4 v[132:135], %1, %2 offset:96\n\t"
          "s_waitcnt vmcnt(0)"
          : "={v[120:135]}"(qv)
          : "v"(qoff), "s"(qbase)
          : "memory");
  }

  // Steps in the fast form.  Its exponentials are those of half n+1, which has to be whole and either the wavefront's or hidden by the
  // causal predicate altogether (what a place holds beyond the loaded halves is hidden with it), its P.V that of half n, the wavefront's;
  // scores beyond the wavefront's halves are formed and not used.  From step nfast on the streams apply the predicate.
  int nfast_all, nfast;
  {
    const int whole = S >= 96 + 32 * grp ? (S - 96 - 32 * grp) / 64 + 1 : 0;
    int own = my_halves;
    if (!CAUSAL || (seen + 1 - grp) / 2 > my_halves) own--;  // half n+1 beyond the last one is not hidden by the diagonal
    nfast_all = whole < own ? whole : own;
    nfast = nfast_all;
    if (CAUSAL) {
      const int clear = qc0 >= 31 + 32 * grp ? (qc0 - 31 - 32 * grp) / 64 : 0;
      nfast = clear < nfast ? clear : nfast;
      nfast = __builtin_amdgcn_readfirstlane(nfast);  // scalar registers: operands of the step statements derive from them
    }
    nfast_all = __builtin_amdgcn_readfirstlane(nfast_all) & ~1;  // two at a time
  }

  auto q_of = [&](int ks) __attribute__((always_inline)) {
    u32x4 w;
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = qv[4 * ks + i];
    return __builtin_bit_cast(vec8, w);
  };
  f32x16 oacc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; db++)
#pragma unroll
    for (int r = 0; r < 16; r++) oacc[db][r] = 0.f;
  const float c = a.scale * kLog2e;
  const float c_s = CAUSAL ? __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, c))) : 0.f;
  float m_use = -1e30f;  // maximum the exponentials are taken against (raw scores)
  float mc = m_use * c;
  float l_run = 0.f;

  auto k_half = [&](int n) __attribute__((always_inline)) { return smem + (n & 3) * Z::HALF; };  // k_addr and v_addr hold the rings' bases
  auto qk_half = [&](f32x16& s, const char* kh) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KST; ks++) s = TR::mfma32(*(const vec8*)(kh + k_addr[ks]), q_of(ks), s);
  };
  auto mask_half = [&](f32x16& s, int kv0) __attribute__((always_inline)) {
    const int qi = qc0 + lq;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int key = kv0 + 8 * (r >> 2) + 4 * lh + (r & 3);
      if (key >= S || (CAUSAL && key > qi)) s[r] = -INFINITY;
    }
  };
  auto row_max = [&](const f32x16& s) __attribute__((always_inline)) {
    float m = s[0];
#pragma unroll
    for (int r = 1; r < 16; r++) m = fmaxf(m, s[r]);
    unsigned lo = __builtin_bit_cast(unsigned, m), hi = lo;  // the other 16 keys of this query sit in lane l^32
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(lo), "+v"(hi));
    return fmaxf(__builtin_bit_cast(float, lo), __builtin_bit_cast(float, hi));
  };
  auto exp_half = [&](const f32x16& s, vec8 (&pb)[2]) __attribute__((always_inline)) {
    float psum = 0.f;
#pragma unroll
    for (int t = 0; t < 2; t++) {
      f32x8 x;
#pragma unroll
      for (int i = 0; i < 8; i++) {
        x[i] = fast_exp2(fmaf(s[8 * t + i], c, -mc));
        psum += x[i];
      }
      pb[t] = __builtin_convertvector(x, vec8);
    }
    return psum;
  };
  // The lazily raised maximum, as in sdpa_prefill_d128.hip.
  const int rl = CAUSAL ? qc0 + lq - 4 * lh : 0;  // the causal predicate's lane operand: key k of a score is visible iff k - 4*(lane/32) <= rl
  auto settle_half = [&](f32x16& s, vec8 (&pb)[2], float psum, int masked_kv0 = -1) __attribute__((always_inline)) {
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(psum <= kSumLimit)) != 0, 0)) {
      if (CAUSAL && masked_kv0 >= 0) {
#pragma unroll
        for (int r = 0; r < 16; r++)
          if (masked_kv0 + 8 * (r >> 2) + (r & 3) > rl) s[r] = -INFINITY;  // the streams' predicate
      }
      const float m_new = fmaxf(m_use, row_max(s));
      const float alpha = fast_exp2((m_use - m_new) * c);
      m_use = m_new;
      mc = m_new * c;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[db][r] *= alpha;
      psum = exp_half(s, pb);
    }
    l_run += psum;
  };
  auto pv_half = [&](const vec8 (&pb)[2], const char* vh) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int db = 0; db < NDB; db++) {
        s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vh + v_addr[2 * db] + 16 * t * Z::ROW));
        s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(vh + v_addr[2 * db + 1] + 16 * t * Z::ROW));
        vec8 va = __builtin_bit_cast(vec8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        oacc[db] = TR::mfma32(va, pb[t], oacc[db]);
      }
  };
  // General form of a step (any half may be masked or missing); the compiler orders it.
  auto slow_step = [&](int n, const vec8 (&p_cur)[2], f32x16& s_nxt, f32x16& s_new, vec8 (&p_nxt)[2]) __attribute__((always_inline)) {
    if (n + 2 < my_halves) qk_half(s_new, k_half(n + 2));
    if (n < my_halves) pv_half(p_cur, k_half(n));
    if (n + 1 < my_halves) {
      const int kv0 = first_key(n + 1);
      if ((CAUSAL && kv0 + 31 > qc0) || kv0 + 32 > S) mask_half(s_nxt, kv0);
      settle_half(s_nxt, p_nxt, exp_half(s_nxt, p_nxt));
    }
  };

  // ---- fast form of a step: one statement of hand-ordered instructions; registers as in the pipelined kernels ------------------------
  u32x32 ring;
#pragma unroll
  for (int i = 0; i < 32; i++) ring[i] = 0u;
#define TT_DEALT_STEP_128(TXT)                                                                                         \
  asm volatile(TXT                                                                                                     \
               : [o0] "+v"(oacc[0]), [o1] "+v"(oacc[1]), [o2] "+v"(oacc[2 % NDB]), [o3] "+v"(oacc[3 % NDB]), [ps] "=&v"(psum_step),  \
                 "+{v[160:175]}"(sB), "+{v[176:191]}"(sC), "+{v[192:199]}"(pAv), "+{v[200:207]}"(pBv),                   \
                 "+{v[208:239]}"(ring)                                                                                 \
               : [c] "s"(c_s), [mc] "v"(mc), [rl] "v"(rl), [mk] "s"(mk), [kvs] "s"(kvs), "{v[120:151]}"(qv), "{v[152:159]}"(v_addr), "{v[248:255]}"(k_addr) \
               : "v240", "v241", "v242", "v243", "v244", "v245", "vcc", "scc", "m0", "memory")
#define TT_DEALT_PSTEP_128(TXT)                                                                                        \
  asm volatile(TXT                                                                                                     \
               : [o0] "+v"(oacc[0]), [o1] "+v"(oacc[1]), [o2] "+v"(oacc[2 % NDB]), [o3] "+v"(oacc[3 % NDB]), [ps] "=&v"(psum_step),  \
                 "+{v[160:175]}"(sB), "+{v[176:191]}"(sC), "+{v[192:199]}"(pAv), "+{v[200:207]}"(pBv),                   \
                 "+{v[208:239]}"(ring)                                                                                 \
               : [c] "v"(c), [mc] "v"(mc), "{v[120:151]}"(qv), "{v[152:159]}"(v_addr), "{v[248:255]}"(k_addr)            \
               : "v240", "v241", "v242", "v243", "v244", "v245", "memory")
#define TT_DEALT_STEP_64(TXT)                                                                                          \
  asm volatile(TXT                                                                                                     \
               : [o0] "+v"(oacc[0]), [o1] "+v"(oacc[1]), [ps] "=&v"(psum_step),                                          \
                 "+{v[160:175]}"(sB), "+{v[176:191]}"(sC), "+{v[192:199]}"(pAv), "+{v[200:207]}"(pBv),                   \
                 "+{v[208:239]}"(ring)                                                                                 \
               : [c] "s"(c_s), [mc] "v"(mc), [rl] "v"(rl), [mk] "s"(mk), [kvs] "s"(kvs), "{v[120:135]}"(qv), "{v[152:155]}"(v_addr), "{v[248:251]}"(k_addr) \
               : "v240", "v241", "v242", "v243", "v244", "v245", "vcc", "scc", "m0", "memory")
#define TT_DEALT_PSTEP_64(TXT)                                                                                         \
  asm volatile(TXT                                                                                                     \
               : [o0] "+v"(oacc[0]), [o1] "+v"(oacc[1]), [ps] "=&v"(psum_step),                                          \
                 "+{v[160:175]}"(sB), "+{v[176:191]}"(sC), "+{v[192:199]}"(pAv), "+{v[200:207]}"(pBv),                   \
                 "+{v[208:239]}"(ring)                                                                                 \
               : [c] "v"(c), [mc] "v"(mc), "{v[120:135]}"(qv), "{v[152:155]}"(v_addr), "{v[248:251]}"(k_addr)            \
               : "v240", "v241", "v242", "v243", "v244", "v245", "memory")
#define TT_DEALT_STREAM(N)                                                                                             \
  if constexpr (D == 128 && CAUSAL && kIsBf16) TT_DEALT_STEP_128(TT_P128_DSTEP_BF16_N##N);                             \
  else if constexpr (D == 128 && CAUSAL) TT_DEALT_STEP_128(TT_P128_DSTEP_F16_N##N);                                    \
  else if constexpr (D == 128 && kIsBf16) TT_DEALT_PSTEP_128(TT_P128_DPSTEP_BF16_N##N);                                \
  else if constexpr (D == 128) TT_DEALT_PSTEP_128(TT_P128_DPSTEP_F16_N##N);                                            \
  else if constexpr (CAUSAL && kIsBf16) TT_DEALT_STEP_64(TT_P64_DSTEP_BF16_N##N);                                      \
  else if constexpr (CAUSAL) TT_DEALT_STEP_64(TT_P64_DSTEP_F16_N##N);                                                  \
  else if constexpr (kIsBf16) TT_DEALT_PSTEP_64(TT_P64_DPSTEP_BF16_N##N);                                              \
  else TT_DEALT_PSTEP_64(TT_P64_DPSTEP_F16_N##N)
  constexpr bool kIsBf16 = __is_same(T, __bf16);

  f32x16 sB, sC;
  vec8 pA[2], pB[2];
  u32x8 pAv, pBv;  // P of a half as two MFMA B operands (k-steps of 16 keys), 4 registers each
  float psum_step;
  auto p_load = [&](const u32x8& pv, vec8 (&p)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; t++) {
      u32x4 w;
#pragma unroll
      for (int i = 0; i < 4; i++) w[i] = pv[4 * t + i];
      p[t] = __builtin_bit_cast(vec8, w);
    }
  };
  auto p_store = [&](u32x8& pv, const vec8 (&p)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const u32x4 w = __builtin_bit_cast(u32x4, p[t]);
#pragma unroll
      for (int i = 0; i < 4; i++) pv[4 * t + i] = w[i];
    }
  };

  // every wavefront's waits for the first halves (with Q) are behind it: they are visible to all
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  {  // P(0) and the scores of half 1 (a group without a half: every key hidden, zeros)
    const int kb = first_key(n0);
    qk_half(sC, k_half(n0));
    if (n0 + 1 < my_halves) qk_half(sB, k_half(n0 + 1));
    if ((CAUSAL && kb + 31 > qc0) || kb + 32 > S) mask_half(sC, kb);
    m_use = fmaxf(m_use, row_max(sC));
    mc = m_use * c;
    l_run = exp_half(sC, pA);
  }
  // every wavefront has read K(0) and K(1): their places are free
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if (n0 + 4 < loaded) dma_k(n0 + 4);

  auto step_dma = [&](int n) __attribute__((always_inline)) {
    int keep = 0;
    if (__builtin_expect(n + 3 < loaded, 1)) {
      if (__builtin_expect(n + 5 < loaded, 1)) {
        if (PAGED) {  // half way through a window (no stream is in the one before it any more): the one behind it
          const int kv0 = 64 * (n + 5), e = kv0 >> a.page_shift, w = (e >> 6) + 1;
          if (__builtin_expect((e & 63) == 32 && (kv0 & ((1 << a.page_shift) - 1)) == 0 && 64 * w <= last_entry, 0)) {
            unsigned next;
            asm volatile("s_nop 4\n\tglobal_load_dword %0, %1, %2\n\ts_waitcnt vmcnt(0)" : "=v"(next) : "v"(entry_off(w)), "s"(table) : "memory");
            if (w & 1) ptab[1] = next;
            else ptab[0] = next;
          }
        }
        dma_k(n + 5);
        keep = 2;
      } else {
        keep = 1;
      }
      dma_v(n + 3);
    }
    return keep;
  };
  // The fast form's requests where both halves are whole: through two running pointers (the general form multiplies the half's number
  // out and has the ragged and paged cases); N = n % 4 makes the places constants.
  const char* kfast = (const char*)(kp + (long long)first_key(n0 + 5) * a.ks[2]);
  const char* vfast = (const char*)(vp + (long long)first_key(n0 + 3) * a.vs[2]);
  const long long kfast_step = (long long)128 * a.ks[2], vfast_step = (long long)128 * a.vs[2];  // bytes of 64 keys
  const int straight = PAGED ? 0 : (first_key(loaded) - 32 <= S ? loaded : loaded - 1);  // halves of the group that are whole
  auto step_dma_fast = [&](int n, int N) __attribute__((always_inline)) {
    int keep = 2;
    if (__builtin_expect(n + 5 < straight, 1)) {
#pragma unroll
      for (int i = 0; i < Z::LOADS; i++) dma_issue(kfast, ld_koff[i], ring_addr + ((N + 1) & 3) * Z::HALF + (8 * gw + 4 * i) * Z::ROW);
#pragma unroll
      for (int i = 0; i < Z::LOADS; i++)
        dma_issue(vfast, ld_voff[i], ring_addr + Z::STAGES / 2 + ((N + 3) & 3) * Z::HALF + (8 * gw + 4 * i) * Z::ROW);
    } else {
      keep = step_dma(n);
    }
    kfast += kfast_step;
    vfast += vfast_step;
    return keep;
  };
  int n = n0;
  if (nfast_all > n0) {
    auto settle_fast = [&](f32x16& s, u32x8& pv, int masked_kv0) __attribute__((always_inline)) {
      vec8 p[2];
      p_load(pv, p);
      settle_half(s, p, psum_step, masked_kv0);
      p_store(pv, p);
    };
    p_store(pAv, pA);
    p_store(pBv, pB);
    if constexpr (D == 128) asm volatile(TT_P128_PREFETCH : "+{v[208:239]}"(ring) : "{v[152:159]}"(v_addr), "{v[248:255]}"(k_addr) : "memory");
    else asm volatile(TT_P64_PREFETCH : "+{v[208:239]}"(ring) : "{v[152:155]}"(v_addr), "{v[248:251]}"(k_addr) : "memory");
    // Four steps per trip so that a half's place is a constant of its statement; the trip may end after any of them.
#define TT_DEALT_HALF(N, S_NXT, P_NXT)                                                                   \
    if (N % 2 == 0 && __builtin_expect(n >= nfast_all, 0)) break;                                         \
    {                                                                                                    \
      const int keep = PAGED ? step_dma(n) : step_dma_fast(n, N);                                        \
      /* mk = 1: the exponentials take the causal predicate; kvs = first key of the half whose they are; kvm = kvs then, else -1 \
         (scalar instructions, as in sdpa_prefill_d128.hip) */                                            \
      int mk = 0, kvs = first_key(n + 1), kvm = -1;                                                      \
      if constexpr (CAUSAL)                                                                              \
        asm("s_cmp_ge_i32 %2, %3\n\ts_cselect_b32 %0, 1, 0\n\ts_cselect_b32 %1, %4, -1"                   \
            : "=&s"(mk), "=&s"(kvm) : "s"(n), "s"(nfast), "s"(kvs) : "scc");                              \
      TT_DEALT_STREAM(N);                                                                                \
      settle_fast(S_NXT, P_NXT, kvm);                                                                    \
      dma_wait_and_sync(keep);                                                                           \
      n++;                                                                                               \
    }
    for (;;) {
      TT_DEALT_HALF(0, sB, pBv)
      TT_DEALT_HALF(1, sC, pAv)
      TT_DEALT_HALF(2, sB, pBv)
      TT_DEALT_HALF(3, sC, pAv)
    }
#undef TT_DEALT_HALF
    // the ring's last requests belong to a step that takes the general form: let them land before the registers are reused
    asm volatile("s_waitcnt lgkmcnt(0)" : "+{v[208:239]}"(ring) : : "memory");
    p_load(pAv, pA);
    p_load(pBv, pB);
  }
  for (; n < steps; n += 2) {
    int keep = step_dma(n);
    slow_step(n, pA, sB, sC, pB);
    dma_wait_and_sync(keep);
    keep = step_dma(n + 1);
    slow_step(n + 1, pB, sC, sB, pA);
    dma_wait_and_sync(keep);
  }

  // ---- the groups come together: each hands the other half of its columns' accumulators (head_dim blocks) and keeps the others --------
  int ln;  // the lane number anew (as asm: the compiler would otherwise keep the values derived from it alive through the whole kernel)
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(ln));
  const float l_own = l_run + __shfl_xor(l_run, 32);
  char* xch = smem + rowgroup * (Z::EXCHANGE / GW);
  f32x2* stat = (f32x2*)(smem + Z::EXCHANGE) + rowgroup * 128;
  auto hand = [&](auto other) __attribute__((always_inline)) {
    constexpr int O = decltype(other)::value;
#pragma unroll
    for (int db = 0; db < NDB / 2; db++)
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        const f32x16& x = oacc[O * (NDB / 2) + db];
        *(f32x4*)(xch + (O * (D / 16) + 4 * db + rg) * 1024 + 16 * ln) = (f32x4){x[4 * rg], x[4 * rg + 1], x[4 * rg + 2], x[4 * rg + 3]};
      }
  };
  if (grp) hand(std::integral_constant<int, 0>{});
  else hand(std::integral_constant<int, 1>{});
  stat[64 * grp + ln] = (f32x2){m_use, l_own};
  __syncthreads();
  const f32x2 st = stat[64 * (grp ^ 1) + ln];
  const float m_all = fmaxf(m_use, st[0]);
  const float w_own = fast_exp2((m_use - m_all) * c), w_oth = fast_exp2((st[0] - m_all) * c);
  const float l0 = grp ? w_oth * st[1] : w_own * l_own, l1 = grp ? w_own * l_own : w_oth * st[1];
  const float l_all = l0 + l1;  // (the same in both groups)
  f32x4 y[NDB / 2][4];
  auto take = [&](auto own) __attribute__((always_inline)) {
    constexpr int O = decltype(own)::value;
#pragma unroll
    for (int db = 0; db < NDB / 2; db++)
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        const f32x16& x = oacc[O * (NDB / 2) + db];
        const f32x4 z = *(const f32x4*)(xch + (O * (D / 16) + 4 * db + rg) * 1024 + 16 * ln);
#pragma unroll
        for (int i = 0; i < 4; i++) y[db][rg][i] = fmaf(w_oth, z[i], w_own * x[4 * rg + i]);
      }
  };
  if (grp) take(std::integral_constant<int, 1>{});
  else take(std::integral_constant<int, 0>{});

  if (SPLIT && last_key_of_rows(a, q0, BM, S) >= a.kv_chunk) {  // a record instead of the output (store_split_record)
    if (qw0 >= a.L) return;
    float* rec = a.ws + ((((long long)b * a.Hq + h) * a.kv_splits + split) * ((a.L + 31) / 32) + qw0 / 32) * (32 * (D + 2));
#pragma unroll
    for (int db = 0; db < NDB / 2; db++)
#pragma unroll
      for (int rg = 0; rg < 4; rg++) *(f32x4*)(rec + 256 * (4 * (grp * (NDB / 2) + db) + rg) + 4 * ln) = y[db][rg];
    if (grp == 0) rec[32 * D + ln] = ln < 32 ? m_all : l_all;
    return;
  }

  // ---- normalise, transpose through LDS, store: a wavefront the 32 rows' pieces of D / 2 columns, chunk c of row r at slot
  // c ^ r % (D / 16) ----------------------------------------------------------------------------------------------------------------------
  {
    constexpr int CH = D / 16;  // 16-byte chunks of such a piece
    const float inv = 1.f / l_all;
    char* tbuf = smem + Z::STAGES + wave * Z::OUT;
    T* obase = (T*)a.out + b * a.os[0] + h * a.os[1] + grp * (D / 2);
    const int rr = ln & 31, lho = ln >> 5;
#pragma unroll
    for (int db = 0; db < NDB / 2; db++)
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        f32x4 x;
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = y[db][rg][i] * inv;
        *(typename TR::vec4*)(tbuf + rr * D + (((4 * db + rg) ^ (rr & (CH - 1))) << 4) + 8 * lho) = __builtin_convertvector(x, typename TR::vec4);
      }
    // the reads below fetch what other lanes of the wavefront wrote: keep the compiler from relating them to this lane's
    // own accesses.  The LDS runs a wavefront's instructions in order; nothing else is needed.
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < CH / 2; i++) {
      const int row = 64 / CH * i + ln / CH, cc = ln & (CH - 1);
      const vec8 v = *(const vec8*)(tbuf + row * D + ((cc ^ (row & (CH - 1))) << 4));
      const int qi = qw0 + row;
      if (qi < a.L) __builtin_nontemporal_store(v, (vec8*)(obase + qi * a.os[2] + 8 * cc));  // written once, not read here
    }
  }
}

template <typename TR, int D, bool CAUSAL, bool PAGED, bool SPLIT>
int launch_v(const KArgs& a, dim3 grid, hipStream_t stream) {
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  const hipError_t granted = grant_dynamic_lds((const void*)prefill_dealt_kernel<TR, D, CAUSAL, PAGED, SPLIT>, Sizes<D>::LDS, state, done);
  if (granted != hipSuccess) return (int)granted;
  hipLaunchKernelGGL((prefill_dealt_kernel<TR, D, CAUSAL, PAGED, SPLIT>), grid, dim3(NW * 64), Sizes<D>::LDS, stream, a);
  return (int)hipGetLastError();
}

template <typename TR, int D, bool CAUSAL>
int launch_k(const KArgs& a, dim3 grid, hipStream_t stream) {
  if constexpr (D == 128)  // (paged caches of head_dim 64 are the 4-wavefront kernel's)
    if (a.block_table) return a.kv_splits > 1 ? launch_v<TR, D, CAUSAL, true, true>(a, grid, stream) : launch_v<TR, D, CAUSAL, true, false>(a, grid, stream);
  return a.kv_splits > 1 ? launch_v<TR, D, CAUSAL, false, true>(a, grid, stream) : launch_v<TR, D, CAUSAL, false, false>(a, grid, stream);
}

template <int D>
int launch_d(const KArgs& a, int dtype, dim3 grid, hipStream_t stream) {
  if (dtype == 1) return a.causal ? launch_k<F16, D, true>(a, grid, stream) : launch_k<F16, D, false>(a, grid, stream);
  return a.causal ? launch_k<BF16, D, true>(a, grid, stream) : launch_k<BF16, D, false>(a, grid, stream);
}

}  // namespace

int launch_prefill_dealt(const KArgs& a, int dtype, hipStream_t stream) {
  if (a.mask_kind != 0 || !(a.D == 128 || (a.D == 64 && !a.block_table))) return (int)hipErrorInvalidValue;  // (the host sends none of these here)
  long long nwg;
  if (a.kv_splits > 1) {
    nwg = split_grid(a, BM);
  } else {  // the kernel's XCD-aware numbering addresses workgroups in groups of 8: rounded up, the extras return
    const int gq = pair_classes(a.B * a.Hkv);
    const long long per_class = (long long)(a.B * a.Hkv / gq) * a.G * ((a.L + BM - 1) / BM);
    nwg = (per_class + 8 / gq - 1) / (8 / gq) * 8;
  }
  const dim3 grid((unsigned)nwg);
  const int rc = a.D == 128 ? launch_d<128>(a, dtype, grid, stream) : launch_d<64>(a, dtype, grid, stream);
  if (rc != 0 || a.kv_splits <= 1) return rc;
  return launch_split_merge(a, dtype, a.D, BM, stream);
}

}  // namespace ttsdpa
