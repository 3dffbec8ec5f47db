// Split-KV attention for decode: a few query rows per KV head against a long, contiguous KV cache (head_dim 128 or 64).  Memory-bound: every K and V byte is read exactly once with 16-byte loads, whatever the number of
// query heads sharing the KV head, instead of the reference's GEMM -> scale -> softmax -> GEMM chain over a
// materialised score tensor (reference src/Function/FuncNNLayer.h:237-265).
//
// Work split.  Grid = splits x Hkv x B workgroups of 4 wavefronts, or of 8 up to 8 rows (plan_decode).  A split is a contiguous range of keys; its
// wavefronts take 32-key blocks round-robin.  All query rows that read this KV head — the L * (Hq/Hkv) rows
// (l, g), at most 16 — are handled together, so the cache is streamed once for the whole group.
//
// Per 32-key block and wavefront:
//   scores  v_mfma_f32_16x16x32: A = the query rows (16 x 32 slice of head_dim, zero rows where unused), B = K^T taken
//           straight from global memory: lane l supplies key l%16 and the 8 head_dim elements of group l/16, i.e. one
//           16-byte load; head_dim/32 MFMAs cover the head (fp32: 4 elements per load, four v_mfma_f32_16x16x4 each).  Query row x sits at MFMA row 4*(x%4) + x/4, so the
//           result lane (key l%16, group l/16) holds rows l/16, l/16+4, ... in registers 0, 1, ...
//   softmax running max per row (reduced over the 16 key lanes with DPP row rotations), exp2 with scale*log2e folded
//   P.V     on the vector ALUs: with C 16-byte chunks per row, lane l owns the elements of chunk l%C of keys
//           l/C, l/C + 64/C, ... (one 16-byte load per key, a wavefront load instruction covers 64/C whole V rows =
//           1 KiB contiguous); the probabilities
//           travel from the score lanes to the value lanes through a per-wavefront LDS patch.
// Each wavefront ends with (max, sum, acc) per row; the workgroup merges its four or eight, then either writes the final
// output (splits == 1) or a partial (max, sum, acc) record that merge_kernel combines by log-sum-exp.

#include "sdpa_common.h"

namespace ttsdpa {

namespace {

constexpr int KB = 32;       // keys per wavefront block

// What the kernel needs to know about the element type: 16 bytes of it as an MFMA operand, and as floats.
template <typename TR>
struct Dec {
  typedef typename TR::elem elem;
  typedef typename TR::vec8 chunk;
  static __device__ __forceinline__ f32x4 mma(chunk q, chunk k, f32x4 c) { return TR::mfma16(q, k, c); }
  static __device__ __forceinline__ void floats(u32x4 v, float (&f)[8]) {
#pragma unroll
    for (int w = 0; w < 4; w++) f[2 * w] = TR::lo(v[w]), f[2 * w + 1] = TR::hi(v[w]);
  }
};
struct F32 {};
template <>
struct Dec<F32> {
  typedef float elem;
  typedef f32x4 chunk;
  // four v_mfma_f32_16x16x4, instruction e contracting the lanes' e-th elements: the same head_dim elements on both sides
  static __device__ __forceinline__ f32x4 mma(chunk q, chunk k, f32x4 c) {
#pragma unroll
    for (int e = 0; e < 4; e++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(q[e], k[e], c, 0, 0, 0);
    return c;
  }
  static __device__ __forceinline__ void floats(u32x4 v, float (&f)[4]) {
    const f32x4 x = __builtin_bit_cast(f32x4, v);
#pragma unroll
    for (int w = 0; w < 4; w++) f[w] = x[w];
  }
};

// max over the 16 lanes of a DPP row (lanes 16*i .. 16*i+15), result in every lane of the row
__device__ __forceinline__ float row16_max(float x) {
  x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x128, 0xf, 0xf, false)));  // row_ror:8
  x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x124, 0xf, 0xf, false)));  // row_ror:4
  x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x122, 0xf, 0xf, false)));  // row_ror:2
  x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x121, 0xf, 0xf, false)));  // row_ror:1
  return x;
}
__device__ __forceinline__ float row16_sum(float x) {
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x128, 0xf, 0xf, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x124, 0xf, 0xf, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x122, 0xf, 0xf, false));
  x += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0x121, 0xf, 0xf, false));
  return x;
}

// Sums of N values of a lane over the lanes of its chunk (lane % CH), neighbouring phases first: a swap of two registers' rows of 16 lanes (of
// their halves) and one addition fold two values into one register, so that four (CH = 32: two) values end in one, each in its own rows:
// value phase_value + 4 i (2 i) in element i.  (As 2 shuffles through LDS for each value, 64 a wavefront, this took 0.7 us.  Folding the
// halves first, which saves the narrow rows three additions in four, adds in another order: results of 16 bits then differ in their last place.)
__device__ __forceinline__ float fold16(float a, float b) {
  const auto t = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, a), __builtin_bit_cast(int, b), false, false);
  const int lo = t[0], hi = t[1];
  return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
__device__ __forceinline__ float fold32(float a, float b) {
  const auto t = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, a), __builtin_bit_cast(int, b), false, false);
  const int lo = t[0], hi = t[1];
  return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
template <int CH>
__device__ __forceinline__ int phase_value(int lane) {
  return CH < 32 ? lane >> 4 : lane >> 5;
}
template <int CH, int N>
__device__ __forceinline__ void add_phases(float* x) {
  static_assert(CH == 8 || CH == 16 || CH == 32, "");
  if constexpr (CH == 8) {
#pragma unroll
    for (int i = 0; i < N; i++) x[i] += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x[i]), 0x128, 0xf, 0xf, true));  // row_ror:8
  }
  if constexpr (CH == 32) {
#pragma unroll
    for (int i = 0; i < N / 2; i++) x[i] = fold32(x[2 * i], x[2 * i + 1]);
  } else {
#pragma unroll
    for (int i = 0; i < N / 4; i++) x[i] = fold32(fold16(x[4 * i], x[4 * i + 1]), fold16(x[4 * i + 2], x[4 * i + 3]));
  }
}

// Make this wavefront's LDS writes visible to its own later reads and keep the compiler from reordering across.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// R = registers of query rows per score lane: rows handled = up to 4*R.
// PAGED: K/V are page pools addressed through a block table (a variant of its own, so that the contiguous kernel
// carries none of the lookups).
// PAD: the tensors' head_dim a.D is a multiple of 8 below DD.  The 16-byte chunks of a row beyond it read as zeros (q, k)
// or are left out of the output (v: the lanes of those chunks fetch the row's first chunk instead, so that the loads stay
// unconditional); the split records keep the pitch DD + 2.
template <typename TR, int R, int DD, bool PAGED, bool PAD, int NWAVE>
__global__ __launch_bounds__(64 * NWAVE, 2) void decode_kernel(KArgs a, int splits, int chunk, float* __restrict__ ws) {
  typedef typename Dec<TR>::elem T;
  typedef typename Dec<TR>::chunk chunk_t;
  constexpr int E = 16 / sizeof(T);  // elements of a 16-byte chunk
  constexpr int NR = 4 * R;          // row slots
  constexpr int KS = DD / (4 * E);   // chunks of a key per score lane
  constexpr int CH = DD / E;         // 16-byte chunks of a V row = value lanes per key
  constexpr int PH = 64 / CH;  // keys a wavefront V load covers (key phases)

  // per-wavefront patch: probabilities [KB keys][NR rows] + rescale factors [NR]; reused for the final merge
  __shared__ __attribute__((aligned(16))) float Pl[NWAVE][KB * NR + NR];
  __shared__ __attribute__((aligned(16))) float Om[NWAVE][NR][DD + 2];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;  // (forcing it scalar measured slower, also for the page lookups)
  const int l16 = lane & 15;  // score lanes: key within a 16-key group
  const int lg = lane >> 4;   // score lanes: row group
  const int vc = lane % CH;   // value lanes: 16-byte chunk of the row
  const int vph = lane / CH;  // value lanes: key phase

  // Workgroup i runs on XCD i % 8: the splits of neighbouring pairs begin at different XCDs, so that sequences too short for
  // all of theirs do not leave the same XCDs idle.
  int n = blockIdx.x / splits;
  const int split = (int)((blockIdx.x + n) % splits);
  const int hk = n % a.Hkv;
  const int b = n / a.Hkv;
  const int rows = a.L * a.G;  // query rows sharing this KV head, row x = (l, g) = (x / G, x % G)
  int S = a.S;                 // keys of this batch entry: the whole cache, or its filled prefix
  if (a.kv_len) {
    int len = a.kv_len[b];
    S = len < 0 ? 0 : (len < S ? len : S);
    // a sequence's own keys over all of its splits (24 sequences of 1000 .. 3000 keys, 4 KV heads: with the longest one's
    // chunk 32.3 us, the short ones' work on the first splits' XCDs; 25.8 so)
    const int own = (S + splits * NWAVE * KB - 1) / (splits * NWAVE * KB) * (NWAVE * KB);
    chunk = own < chunk ? own : chunk;
  }

  const T* kp = (const T*)a.k + b * a.ks[0] + hk * a.ks[1];
  const T* vp = (const T*)a.v + b * a.vs[0] + hk * a.vs[1];

  // ---- query rows as MFMA A operands: lane l supplies MFMA row l%16, head_dim 4*E*ks + E*(l/16) .. +E-1 -----------
  chunk_t qa[KS];
  {
    int mrow = l16;                       // MFMA row
    int x = (mrow & 3) * 4 + (mrow >> 2); // query row stored there: row x sits at 4*(x%4) + x/4
    bool used = (mrow & 3) < R && x < rows;
    int xl = used ? x / a.G : 0, xg = used ? x % a.G : 0;
    const T* qr = (const T*)a.q + b * a.qs[0] + (hk * a.G + xg) * a.qs[1] + xl * a.qs[2] + E * lg;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      const bool there = used && (!PAD || 4 * E * ks + E * lg < a.D);
      const chunk_t t = *(const chunk_t*)(there ? qr + 4 * E * ks : qr - E * lg);
#pragma unroll
      for (int i = 0; i < E; i++) qa[ks][i] = there ? t[i] : (T)0.f;
    }
  }

  // lane-local state: score lanes track rows lg + 4r; value lanes accumulate all rows for their 8 dims
  float m_run[R], l_run[R];
#pragma unroll
  for (int r = 0; r < R; r++) m_run[r] = -1e30f, l_run[r] = 0.f;
  float acc[NR][E];
#pragma unroll
  for (int x = 0; x < NR; x++)
#pragma unroll
    for (int i = 0; i < E; i++) acc[x][i] = 0.f;
  const float c = a.scale * kLog2e;

  const int s_begin = split * chunk;
  const int s_end = s_begin + chunk < S ? s_begin + chunk : S;
  float* pl = Pl[wave];
  // First hidden key per row of this score lane: the end of the split, or under a (bottom-right aligned) causal mask
  // the key after the row's own position S - L + l.
  int klim[R], klim_min = s_end;
#pragma unroll
  for (int r = 0; r < R; r++) {
    klim[r] = s_end;
    if (a.causal) {
      int own = causal_offset(a, S) + (lg + 4 * r) / a.G + 1;
      klim[r] = own < s_end ? own : s_end;
    }
    klim_min = klim[r] < klim_min ? klim[r] : klim_min;
  }

  // Paged cache: the 32 keys of a block lie in one page (pages hold a power of two >= 32 rows and blocks start at
  // multiples of 32); its number is read one block ahead.
  const int* table = PAGED ? a.block_table + (long long)b * a.bt_stride : nullptr;
  int page_next = 0;
  if (PAGED && s_begin + wave * KB < s_end) page_next = table[(s_begin + wave * KB) >> a.page_shift];

  for (int k0 = s_begin + wave * KB; k0 < s_end; k0 += NWAVE * KB) {
    const T* kpb = kp;
    const T* vpb = vp;
    int key0 = 0;  // first key of the memory region kpb / vpb point to
    if (PAGED) {
      kpb = (const T*)a.k + (long long)page_next * a.ks[0] + hk * a.ks[1];
      vpb = (const T*)a.v + (long long)page_next * a.vs[0] + hk * a.vs[1];
      key0 = (k0 >> a.page_shift) << a.page_shift;
      if (k0 + NWAVE * KB < s_end) page_next = table[(k0 + NWAVE * KB) >> a.page_shift];
    }
    // ---- issue all loads of the block: K for the score MFMAs, V for the accumulation ----------------------------------
    u32x4 kreg[2][KS];
#pragma unroll
    for (int gi = 0; gi < 2; gi++) {
      int key = k0 + 16 * gi + l16;
      key = (key < S ? key : S - 1) - key0;
      const T* kr = kpb + key * a.ks[2] + E * lg;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        if (!PAD) {
          kreg[gi][ks] = __builtin_nontemporal_load((const u32x4*)(kr + 4 * E * ks));  // read once: keep it out of the caches
        } else {
          const bool there = 4 * E * ks + E * lg < a.D;
          const u32x4 t = __builtin_nontemporal_load((const u32x4*)(there ? kr + 4 * E * ks : kr - E * lg));
          kreg[gi][ks] = there ? t : u32x4{0u, 0u, 0u, 0u};
        }
      }
    }
    u32x4 vreg[KB / PH];
#pragma unroll
    for (int i = 0; i < KB / PH; i++) {
      int key = k0 + PH * i + vph;
      key = (key < S ? key : S - 1) - key0;
      vreg[i] = __builtin_nontemporal_load((const u32x4*)(vpb + key * a.vs[2] + (PAD && E * vc >= a.D ? 0 : E * vc)));
    }

    // ---- scores --------------------------------------------------------------------------------------------------------
    f32x4 sc[2];
#pragma unroll
    for (int gi = 0; gi < 2; gi++) {
      sc[gi] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ks++)
        sc[gi] = Dec<TR>::mma(qa[ks], __builtin_bit_cast(chunk_t, kreg[gi][ks]), sc[gi]);
      if (k0 + 16 * gi + l16 >= klim_min) {
#pragma unroll
        for (int r = 0; r < 4; r++)
          if (r >= R || k0 + 16 * gi + l16 >= klim[r < R ? r : 0]) sc[gi][r] = -INFINITY;
      }
    }

    // ---- running softmax per row (register r of score-lane group lg is row lg + 4r) -----------------------------------
#pragma unroll
    for (int r = 0; r < R; r++) {
      float mloc = row16_max(fmaxf(sc[0][r], sc[1][r]));
      float m_new = fmaxf(m_run[r], mloc);
      float alpha = fast_exp2((m_run[r] - m_new) * c);
      float mc = m_new * c;
      m_run[r] = m_new;
      float p0 = fast_exp2(fmaf(sc[0][r], c, -mc));
      float p1 = fast_exp2(fmaf(sc[1][r], c, -mc));
      l_run[r] = l_run[r] * alpha + p0 + p1;
      pl[(l16)*NR + 4 * r + lg] = p0;
      pl[(16 + l16) * NR + 4 * r + lg] = p1;
      if (l16 == 0) pl[KB * NR + 4 * r + lg] = alpha;
    }
    wave_lds_sync();

    // ---- rescale and accumulate P.V -------------------------------------------------------------------------------------
#pragma unroll
    for (int r = 0; r < R; r++) {
      f32x4 al = *(const f32x4*)(pl + KB * NR + 4 * r);
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < E; i++) acc[4 * r + j][i] *= al[j];
    }
#pragma unroll
    for (int i = 0; i < KB / PH; i++) {
      float vf[E];
      Dec<TR>::floats(vreg[i], vf);
#pragma unroll
      for (int r = 0; r < R; r++) {
        f32x4 p = *(const f32x4*)(pl + (PH * i + vph) * NR + 4 * r);
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int e = 0; e < E; e++) acc[4 * r + j][e] = fmaf(p[j], vf[e], acc[4 * r + j][e]);
      }
    }
    wave_lds_sync();
  }

  // ---- wavefront totals: sums over the 16 key lanes; accumulators over the key phases ------------------------------------
#pragma unroll
  for (int r = 0; r < R; r++) l_run[r] = row16_sum(l_run[r]);
  add_phases<CH, NR * E>(&acc[0][0]);
  if (CH > 8 || (lane & 8) == 0) {
#pragma unroll
    for (int i = 0; i < NR * E / (CH < 32 ? 4 : 2); i++) {
      const int v = phase_value<CH>(lane) + (CH < 32 ? 4 : 2) * i;  // of the lane's chunk
      Om[wave][v / E][E * vc + v % E] = (&acc[0][0])[i];
    }
  }
  if (l16 == 0) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      Om[wave][4 * r + lg][DD] = m_run[r];
      Om[wave][4 * r + lg][DD + 1] = l_run[r];
    }
  }
  __syncthreads();

  // ---- merge the wavefronts; thread t handles (row slot, dim) pairs ------------------------------------------------------
  for (int e = tid; e < NR * DD; e += 64 * NWAVE) {
    int x = e / DD, d = e % DD;  // row slot x holds query row x (slot index == query row index)
    if (x >= rows) continue;
    float mx = Om[0][x][DD];
#pragma unroll
    for (int w = 1; w < NWAVE; w++) mx = fmaxf(mx, Om[w][x][DD]);
    float lsum = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < NWAVE; w++) {
      float f = fast_exp2((Om[w][x][DD] - mx) * c);
      lsum += f * Om[w][x][DD + 1];
      o += f * Om[w][x][d];
    }
    if (splits == 1) {
      int xl = x / a.G, xg = x % a.G;
      T* op = (T*)a.out + b * a.os[0] + (hk * a.G + xg) * a.os[1] + xl * a.os[2];
      if (!PAD || d < a.D) store_from_float(op + d, S > 0 ? o / lsum : 0.f);  // no keys at all: zeros, as the reference's empty contraction
    } else {
      float* rec = ws + ((long long)blockIdx.x * rows + x) * (DD + 2);
      rec[d] = o;
      if (d == 0) {
        rec[DD] = mx;
        rec[DD + 1] = lsum;
      }
    }
  }
}

// Combine the per-split records of one query row: one workgroup of head_dim threads per (batch, kv head, row).  The first
// wavefront turns the (max, sum) pairs of the up to 64 splits into weights (one split per lane, wave reductions);
// then thread d accumulates head_dim element d over the splits with independent, coalesced loads.
constexpr int kMaxSplits = 64;
template <typename T, int DD>
__global__ __launch_bounds__(DD) void merge_kernel(KArgs a, int splits, const float* __restrict__ ws) {
  __shared__ float weight[kMaxSplits];
  __shared__ float total;
  const int rows = a.L * a.G;
  const int pair = blockIdx.x / rows, x = blockIdx.x % rows;  // pair = b * Hkv + hk
  const int hk = pair % a.Hkv, b = pair / a.Hkv;
  const float c = a.scale * kLog2e;
  const float* rec0 = ws + ((long long)pair * splits * rows + x) * (DD + 2);
  const long long step = (long long)rows * (DD + 2);
  const int t = threadIdx.x;
  if (t < 64) {
    const bool have = t < splits;
    const float m = have ? rec0[t * step + DD] : -1e30f;
    const float l = have ? rec0[t * step + DD + 1] : 0.f;
    float mx = m;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    const float f = have ? fast_exp2((m - mx) * c) : 0.f;
    float lsum = f * l;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) lsum += __shfl_xor(lsum, off);
    weight[t] = f;
    if (t == 0) total = lsum;
  }
  __syncthreads();
  float o = 0.f;
#pragma unroll 8
  for (int s = 0; s < splits; s++) o = fmaf(weight[s], rec0[s * step + t], o);
  const int xl = x / a.G, xg = x % a.G;
  T* op = (T*)a.out + b * a.os[0] + (hk * a.G + xg) * a.os[1] + xl * a.os[2];
  const bool empty = a.kv_len && a.kv_len[b] <= 0;  // (as the decode kernel has it)
  if (t < a.D) store_from_float(op + t, empty ? 0.f : o / total);  // (a.D < DD: the decode kernel's zero-column variant)
}

template <typename TR, int R, int DD, bool PAD, int NWAVE>
void launch_decode_w(const KArgs& a, const DecodePlan& pl, float* ws, hipStream_t stream) {
  const dim3 grid((unsigned)((long long)a.B * a.Hkv * pl.splits)), block(64 * NWAVE);
  if (a.block_table) hipLaunchKernelGGL((decode_kernel<TR, R, DD, true, PAD, NWAVE>), grid, block, 0, stream, a, pl.splits, pl.chunk, ws);
  else hipLaunchKernelGGL((decode_kernel<TR, R, DD, false, PAD, NWAVE>), grid, block, 0, stream, a, pl.splits, pl.chunk, ws);
}
template <typename TR, int R, int DD, bool PAD>
void launch_decode_r(const KArgs& a, const DecodePlan& pl, float* ws, hipStream_t stream) {
  if constexpr (R <= 2)
    if (pl.waves == 8) return launch_decode_w<TR, R, DD, PAD, 8>(a, pl, ws, stream);
  launch_decode_w<TR, R, DD, PAD, 4>(a, pl, ws, stream);
}
template <typename TR, int DD, bool PAD>
int launch_decode_t(const KArgs& a, const DecodePlan& pl, float* ws, hipStream_t stream) {
  typedef typename Dec<TR>::elem T;
  switch ((pl.rows + 3) / 4) {
    case 1: launch_decode_r<TR, 1, DD, PAD>(a, pl, ws, stream); break;
    case 2: launch_decode_r<TR, 2, DD, PAD>(a, pl, ws, stream); break;
    case 3: launch_decode_r<TR, 3, DD, PAD>(a, pl, ws, stream); break;
    default: launch_decode_r<TR, 4, DD, PAD>(a, pl, ws, stream); break;
  }
  int rc = (int)hipGetLastError();
  if (rc != 0 || pl.splits == 1) return rc;
  hipLaunchKernelGGL((merge_kernel<T, DD>), dim3((unsigned)((long long)a.B * a.Hkv * pl.rows)), dim3(DD), 0, stream, a, pl.splits, ws);
  return (int)hipGetLastError();
}

}  // namespace

DecodePlan plan_decode(const KArgs& a, bool f32) {
  DecodePlan p;
  p.rows = a.L * a.G;
  const int round = 4 * KB;
  p.waves = 4;
  long long pairs = (long long)a.B * a.Hkv;
  // two blocks of keys per wavefront at least, or one where that leaves most of the CUs idle (1 sequence of 1500 keys, 8 KV heads
  // 11.2 -> 9.5 us, 2 of 324, one KV head 12.2 -> 10.3; not for a single chunk: the merge costs more)
  int max_splits = (a.S + 2 * round - 1) / (2 * round);
  if (pairs * max_splits < 128 && a.S > 2 * round) max_splits = (a.S + round - 1) / round;
  if (max_splits < 1) max_splits = 1;
  if (max_splits > kMaxSplits) max_splits = kMaxSplits;
  // Two workgroups per CU or a few more: the count, up to four per CU, that fills its last round best (a CU takes in its
  // workgroups' keys at a rate of its own, so 2.25 per CU cost as much as 3: 24 sequences of 3000 keys on 4 KV heads, 96
  // pairs, 37.7 us in 6 splits of the keys and 31 in 8), the smaller of two that are equally good.  Few pairs: as many as may be,
  // without a look at counts beyond that (one pair: 524 of them, 1.5 us of host time in each of a call's three plans).
  const long long first = (500 + pairs - 1) / pairs;
  int splits = first < max_splits ? 1 : max_splits;
  double best = 0;
  for (long long s = first; first < max_splits && s <= max_splits && (s == 1 || s * pairs <= 4 * 256); s++) {
    const long long wgs = s * pairs, rounds = (wgs + 255) / 256;
    const double fill = (double)wgs / (double)(rounds * 256) - 0.01 * rounds;
    if (s > 1 && fill <= best) continue;
    best = fill, splits = (int)s;
  }
  int chunk = (a.S + splits - 1) / splits;
  chunk = (chunk + round - 1) / round * round;
  if (chunk < round) chunk = round;
  splits = (a.S + chunk - 1) / chunk;
  if (splits < 1) splits = 1;
  // A workgroup of four or eight wavefronts for all of a sequence's keys, in one launch, where that is shorter than the split and its
  // merge: us for a turn of the wavefronts (32 keys each), the merge's launch, a CU's further workgroups (four wavefronts of them: each, and
  // for a turn), and twice the wavefronts, by head_dim, element type and rows; fitted to 400 calls of 1 to 1500 (sequence, KV head)
  // pairs on 128 to 4096 keys (9 to 15 % off; a turn is the vector ALUs' P.V for the most part: requesting the next turn's keys ahead gave
  // nothing).  24 x 8 pairs on up to 1024 keys 13.3 -> 9.5 us, 12 x 8 on 178 of 1024 9.6 -> 6.4; 12 x 1 on 1024 stay split, 8.2 and 14.2.  Not
  // beyond the keys it was fitted on, where memory's rate is all that counts: 64 x 8 on 8192 316 us with four wavefronts and 323 with eight.
  // A cache is taken to be full: by nine tenths of its keys, a last turn was missed (fp32, 21 x 2 on 284, head_dim 80, 13.7 us divided, 16.3).
  static constexpr double fit[2][2][2][5] = {{{{1.2, 3.6, 0.40, 0, 0.8}, {1.25, 3.0, 1.5, 0, 0.4}}, {{1.95, 3.6, 0, 0.80, 1.35}, {2.5, 4.8, 2.2, 0, 1.8}}},
                                             {{{2.0, 3.7, 0, 0.68, 1.15}, {2.15, 3.5, 1.5, 0.62, 1.2}}, {{3.8, 4.3, 1.3, 0.86, 2.6}, {4.7, 4.5, 0.93, 1.55, 2.6}}}};
  // Sequences of unlike lengths: the longest one's chain lasts while the others' workgroups have ended, and a wavefront more does not shorten
  // it (a CU takes in 35 KB of K and V a us).  Up to 256 KB of K the merge makes up for it in most batches (780 drawn ones of a third to all keys 0.99 to
  // 2.2x, with a single long sequence among short ones of 60 keys 0.79 to 2.2x); beyond that their keys stay divided.
  // bf16, head_dim 128, us divided and in one launch, lengths spread evenly / one long among short ones: 32 x 8 on 1024 21.8 and 20.9 / 17.1
  // and 17.6, on 2048 35.7 and 37.2 / 27.1 and 32.7, on 4096 64.2 and 70.7 / 46.1 and 62.3; fp32 on 1024 34.7 and 36.5 / 26.1 and 31.5.
  // Eight wavefronts only while a CU has one workgroup (up to head_dim 64: less than two): 64 x 8 on 1024 51.0 us with four, 54.5 with eight, a
  // tenth full 12.2 and 13.0; 70 x 4 on 1206, head_dim 80, 35.8 divided and 41.7; 79 x 8, head_dim 64, on 1097 40.1 and 42.2.
  const bool unlike = a.kv_len && a.B > 1;
  if (p.rows <= 8 && a.S <= 4096 && (!unlike || (long long)a.S * a.D * (f32 ? 4 : 2) <= 256 << 10)) {
    const double* f = fit[a.D > 64][f32][p.rows > 4];
    const double keys = a.S, fixed = 2.5 + 1e-7 * pairs * keys * a.D * (f32 ? 8 : 4);  // (0.1 us for a MB)
    auto us = [&](int waves, int n) {
      const double further = (double)((pairs * n + 255) / 256 - 1) * waves / 4, turns = ceil(ceil(keys / n) / (KB * waves));
      return fixed + f[0] * turns + (n > 1 ? f[1] : 0) + (f[2] + f[3] * turns) * further + (waves > 4 ? f[4] : 0);
    };
    const double split = us(4, splits), four = us(4, 1), eight = pairs <= (a.D > 64 ? 256 : 511) ? us(8, 1) : four;
    if ((four < eight ? four : eight) < 0.95 * split) splits = 1, chunk = (a.S + round - 1) / round * round, p.waves = eight < four ? 8 : 4;
  }
  p.splits = splits;
  p.chunk = chunk;
  p.ws_bytes = splits > 1 ? (size_t)pairs * splits * p.rows * ((a.D <= 64 ? 64 : 128) + 2) * sizeof(float) : 0;  // the kernel's head_dim: 64 or 128
  return p;
}

namespace {

// head_dim 64 and 128; any other whole number of 16-byte chunks up to 128: the kernel of the next size up, the missing
// columns as zeros
template <typename TR>
int launch_decode_d(const KArgs& a, const DecodePlan& pl, float* ws, hipStream_t stream) {
  constexpr int E = 16 / (int)sizeof(typename Dec<TR>::elem);
  if (a.D % E != 0 || a.D < E || a.D > 128) return (int)hipErrorInvalidValue;  // (the callers keep to this)
  if (a.D == 64) return launch_decode_t<TR, 64, false>(a, pl, ws, stream);
  if (a.D == 128) return launch_decode_t<TR, 128, false>(a, pl, ws, stream);
  return a.D < 64 ? launch_decode_t<TR, 64, true>(a, pl, ws, stream) : launch_decode_t<TR, 128, true>(a, pl, ws, stream);
}

}  // namespace

int launch_decode(const KArgs& a, int dtype, void* workspace, hipStream_t stream) {
  const DecodePlan pl = plan_decode(a, dtype == 0);
  switch (dtype) {
    case 0: return launch_decode_d<F32>(a, pl, (float*)workspace, stream);
    case 1: return launch_decode_d<F16>(a, pl, (float*)workspace, stream);
    default: return launch_decode_d<BF16>(a, pl, (float*)workspace, stream);
  }
}

}  // namespace ttsdpa
