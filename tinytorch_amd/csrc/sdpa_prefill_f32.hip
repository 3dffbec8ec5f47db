// Flash-attention forward for fp32 tensors on the gfx950 matrix cores (v_mfma_f32_32x32x2_f32, full fp32 products
// and sums): fp32 is the reference's default dtype, and its fp32 path is what the 1e-4 parity bar is stated against.
// Replaces the same device chain as the 16-bit kernels (reference src/Function/FuncNNLayer.h:237-265): the score
// matrix never leaves registers.  head_dim 64 or 128; attnMask and per-batch key counts are applied in the kernel.
//
// A workgroup of 4 wavefronts owns 128 query rows of one (batch, query head), 32 rows per wavefront; keys/values come
// in tiles of 32, staged global -> registers -> LDS, double-buffered.
// Per wavefront and tile, with v_mfma_f32_32x32x2 (A: 32 rows x 2, B: 2 x 32 cols, lane l supplies row/col l%32 and
// contraction element l/32; C: lane l holds column l%32 and rows 8*(r/4) + 4*(l/32) + r%4):
//   S^T[32 keys x 32 queries] = K . Q^T   MFMA ks contracts head_dim elements ks (lanes 0-31) and ks + D/2 (lanes 32-63),
//                                         so a lane's Q operands are one contiguous half of its query row (registers)
//                                         and K comes from LDS rows padded by one float (conflict-free columns);
//                                         two accumulators take alternate ks so the chain never waits on itself
//   P^T = exp2((S^T - m) * scale*log2e)   a query is one lane column; its other 16 keys sit in lane l^32
//   O^T[D x 32 queries] += V^T . P^T      MFMA t contracts the two keys that the lane halves hold in accumulator
//                                         register t, so P^T feeds the pipe straight from those registers and
//                                         V^T[d][key] is a plain row-major LDS read along d
// With few row tiles a CU's time is one wavefront's chain of 64-cycle matrix instructions (2.7 us a tile at head_dim 64, 4.6 at
// 128): KEYS gives a workgroup 32 query rows and each of its wavefronts every fourth key tile, staged in a part of LDS of its
// own, and adds the four partial results up through LDS.  Four times as many workgroups, each a quarter as long: 4
// heads x 128 rows, head_dim 64, causal 14.8 -> 7.3 us, 4 x 8 heads x 300 rows, head_dim 128 49.6 -> 23.1.
// The running maximum is raised only when exceeded by 2^8 in the exponent.  Causal masking as in the 16-bit kernels
// (top-left aligned, reference src/Operation/OpTransformCpu.h:202-209): tiles above the diagonal are skipped.

#include "sdpa_common.h"

namespace ttsdpa {

namespace {

constexpr int BM = 128;  // query rows per workgroup
constexpr int BN = 32;   // keys per tile
constexpr float kLazyExp = 8.f;

template <int D>
struct F32Lds {
  static constexpr int K_PITCH = D + 1;   // floats; a column of 32 keys falls into 32 different banks
  static constexpr int V_PITCH = D + 32;  // floats; rows stay 16-byte aligned, the two lane halves use disjoint banks
  static constexpr int STAGE = BN * (K_PITCH + V_PITCH);
};

// MASK: 0 none; 1 a Bool attnMask, 2 an additive one (variants of their own: the mask addressing costs registers the unmasked ones keep).
// With a Bool mask, mostly a batch padded to one length, a tile whose keys are hidden from all of the wavefront's rows is left out:
// its weights are 0 (a tile whose V holds infinities or NaN is taken, 0 times those counts).  A tile is 2.7 us of matrix
// instructions: 30 x 16 heads x 300 rows, head_dim 64, lengths 75 to 300 154 -> 110 us; 4 x 8 x 1001 100 -> 90, its longest
// entry's tiles in a row.
// SPLIT: whether the keys are divided among workgroups: 0 no, 1 yes, 2 told at run time.  Without a mask variants of their own: as a
// run-time branch it made launches without divided keys slower (64 heads x 2527 rows, head_dim 64, causal 489 us, 484 so).  With a
// mask the unsplit variant takes more registers than the one that asks (head_dim below 64, Bool: a wavefront a SIMD less).
// PAD: the tensors' head_dim a.D is a multiple of 4 below D; the 16-byte chunks of a row beyond it are taken as zeros (Q
// and K: nothing added to a score; V: output columns that are not stored).  The reference takes any head size
// (src/Function/FuncNNLayer.h:231-236).
template <int D, bool CAUSAL, int MASK, bool PAD, bool KEYS, int SPLIT>
__global__ __launch_bounds__(256, (KEYS ? 1 : 2)) void prefill_f32_kernel(KArgs a) {
  typedef F32Lds<D> Lds;
  constexpr int K_PITCH = Lds::K_PITCH, V_PITCH = Lds::V_PITCH;
  constexpr bool MASKED = MASK != 0;
  if (MASK != 0) __builtin_assume(a.mask_kind == MASK);
  constexpr int KSTEPS = D / 2;   // MFMAs along head_dim for S^T
  constexpr int DBLK = D / 32;    // 32-row blocks of O^T
  constexpr int ROWS = KEYS ? 32 : BM;                // query rows of the workgroup
  constexpr int STAGERS = KEYS ? 64 : 256;            // threads that bring a tile
  constexpr int NLD = BN * D / 4 / STAGERS;           // 16-byte chunks per thread per tile, for K and for V
  constexpr int STEP = KEYS ? 4 : 1;                  // a wavefront's (workgroup's) tiles: every STEP-th

  extern __shared__ __attribute__((aligned(16))) float smem_f32[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float* smem = smem_f32 + (KEYS ? wave * Lds::STAGE : 0);
  const int lq = lane & 31;
  const int lh = lane >> 5;

  // ---- workgroup -> (batch, kv head, query head in group, row tile); workgroup n runs on XCD n % 8 -------------
  const int ntile = (a.L + ROWS - 1) / ROWS;
  const int inner = a.G * ntile;
  const int npair = a.B * a.Hkv;
  int pair, in;
  static_assert(!(KEYS && SPLIT), "keys are divided among workgroups or among wavefronts");
  const bool divided = SPLIT == 1 || (SPLIT == 2 && a.kv_splits > 1);
  int split = 0;  // key range of this workgroup (the only one unless the keys are divided)
  if (divided) {
    if (!find_piece(a, ROWS, CAUSAL, &pair, &in, &split)) return;
  } else {
    const int n = blockIdx.x;
    if ((npair & 7) == 0) {
      int xcd = n & 7, slot = n >> 3;
      pair = (slot / inner) * 8 + xcd;
      in = slot % inner;
    } else {
      pair = n / inner;
      in = n % inner;
    }
  }
  const int b = pair / a.Hkv, hk = pair % a.Hkv;
  const int g = in % a.G;
  const int rt = CAUSAL ? ntile - 1 - in / a.G : in / a.G;  // longest rows first
  const int h = hk * a.G + g;
  const int q0 = rt * ROWS;
  const int qw0 = KEYS ? q0 : q0 + wave * 32;

  const float* qp = (const float*)a.q + b * a.qs[0] + h * a.qs[1];
  const int* table = a.block_table ? a.block_table + (long long)b * a.bt_stride : nullptr;  // paged cache
  const float* kp = (const float*)a.k + (table ? 0 : b * a.ks[0]) + hk * a.ks[1];
  const float* vp = (const float*)a.v + (table ? 0 : b * a.vs[0]) + hk * a.vs[1];

  // ---- Q: this lane's half of its query row, the B operands of the S^T MFMAs ---------------------------------------
  float qreg[KSTEPS];
  {
    int row = qw0 + lq;
    row = row < a.L ? row : a.L - 1;
    const float* qr = qp + row * a.qs[2] + lh * (D / 2);
#pragma unroll
    for (int i = 0; i < KSTEPS / 4; i++) {
      f32x4 t = {0.f, 0.f, 0.f, 0.f};
      if (!PAD || lh * (D / 2) + 4 * i < a.D) t = *(const f32x4*)(qr + 4 * i);
#pragma unroll
      for (int e = 0; e < 4; e++) qreg[4 * i + e] = t[e];
    }
  }

  f32x16 oacc[DBLK];
#pragma unroll
  for (int i = 0; i < DBLK; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) oacc[i][r] = 0.f;
  const float c = MASKED ? scores_unit(a) : a.scale * kLog2e;
  const float lazy = kLazyExp / c;
  float m_use = MASKED ? -FLT_MAX : -1e30f;
  float mc = m_use * c;
  float l_run = 0.f;

  int S = a.S;  // keys of this batch entry: all of them, or the filled prefix of a cache / the unpadded length
  if (a.kv_len) {
    int len = __builtin_amdgcn_readfirstlane(a.kv_len[b]);
    S = len < 0 ? 0 : (len < S ? len : S);
  }
  if (S == 0 && !divided) {  // no keys: zeros, the reference's empty contraction
    const int qi = qw0 + lq;
    if (qi < a.L) {
      float* op = (float*)a.out + b * a.os[0] + h * a.os[1] + qi * a.os[2];
      for (int d = 4 * lh; d < (PAD ? a.D : D); d += 8) *(f32x4*)(op + d) = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    return;
  }
  const int coff = CAUSAL ? causal_offset(a, S) : 0;  // query position i sees keys up to i + coff
  // Query position of a row under the causal mask: the row itself, or with packed heads row % pack_L — then positions
  // are not monotone in the row, and the tile-level tests below use the range of all positions.
  const int pos_lo = a.pack_L ? 0 : qw0, pos_hi = a.pack_L ? a.pack_L - 1 : qw0 + 31;
  const int ntiles_kv = (last_key_of_rows(a, q0, ROWS, S) + BN) / BN;
  // tiles jt0 .. jt1-1 are this workgroup's: all of them, or those of its split (kv_chunk is a multiple of the tile)
  int jt0 = 0, jt1 = ntiles_kv;
  if (divided) {
    jt0 = split * (a.kv_chunk / BN);
    const int end = jt0 + a.kv_chunk / BN;
    jt1 = end < jt1 ? end : jt1;
    if (jt0 >= jt1) return;  // beyond the keys
  }
  const bool wave_live = qw0 < a.L;  // a wavefront without query rows only helps to stage the tiles

  // ---- global -> register -> LDS staging: thread t moves 16-byte chunks t, t+256, ... of a tile ----------------------
  f32x4 kst[NLD], vst[NLD];
  int lrow[NLD], lcol[NLD], gcol[NLD];
  bool cval[NLD];  // PAD: the chunk lies inside the tensors' rows; the others are loaded from the row's first chunk instead
                   // (the loads stay unconditional) and reach LDS as zeros
#pragma unroll
  for (int i = 0; i < NLD; i++) {
    int cidx = (KEYS ? lane : tid) + STAGERS * i;
    lrow[i] = cidx / (D / 4);
    lcol[i] = cidx % (D / 4);
    cval[i] = !PAD || 4 * lcol[i] < a.D;
    gcol[i] = cval[i] ? lcol[i] : 0;
  }
  auto load_tile = [&](int kv0) {
    const float* ktile = kp + kv_tile_offset(a, table, kv0, a.ks[2], a.ks[0]);
    const float* vtile = vp + kv_tile_offset(a, table, kv0, a.vs[2], a.vs[0]);
#pragma unroll
    for (int i = 0; i < NLD; i++) {
      int row = lrow[i];
      row = kv0 + row < S ? row : S - 1 - kv0;  // rows past the end re-read the last valid row (masked later)
      kst[i] = *(const f32x4*)(ktile + row * a.ks[2] + 4 * gcol[i]);
      vst[i] = *(const f32x4*)(vtile + row * a.vs[2] + 4 * gcol[i]);
    }
  };
  auto store_tile = [&](int stage) {
    float* Ks = smem + stage * Lds::STAGE;
    float* Vs = Ks + BN * K_PITCH;
#pragma unroll
    for (int i = 0; i < NLD; i++) {
#pragma unroll
      for (int e = 0; e < 4; e++) Ks[lrow[i] * K_PITCH + 4 * lcol[i] + e] = cval[i] ? kst[i][e] : 0.f;  // rows are not 16-byte aligned
      *(f32x4*)(Vs + lrow[i] * V_PITCH + 4 * lcol[i]) = cval[i] ? vst[i] : (f32x4){0.f, 0.f, 0.f, 0.f};
    }
  };

  const int k_lane = lq * K_PITCH + lh * (D / 2);  // floats
  const int v_lane = 4 * lh * V_PITCH + lq;        // floats; + (8*(t/4) + t%4) * V_PITCH + 32*db

  long long mrow = 0;
  if (MASKED) {
    const int qi = qw0 + lq;
    mrow = b * a.ms[0] + h * a.ms[1] + (qi < a.L ? qi : a.L - 1) * a.ms[2];
  }

  if (KEYS) jt0 += wave;
  MaskBlock<float> next_mask = {};  // MASK 1: a tile's mask is requested a tile ahead
  if (MASK == 1 && jt0 < jt1) next_mask = load_attn_mask<float, true>(a, mrow, jt0 * BN, lh, S);
  if (KEYS) {
    if (jt0 < jt1) load_tile(jt0 * BN);
  } else {
    if (jt0 < jt1) {
      load_tile(jt0 * BN);
      store_tile(0);
      if (jt0 + 1 < jt1) load_tile((jt0 + 1) * BN);
    }
    __syncthreads();
  }

  for (int jt = jt0; jt < jt1; jt += STEP) {
    const int kv0 = jt * BN;
    const int cur = KEYS ? 0 : (jt - jt0) & 1;
    if (KEYS) {  // the wavefront's own stage: its LDS reads and writes stay in order, no other wavefront sees them
      __builtin_amdgcn_wave_barrier();
      store_tile(0);
      __builtin_amdgcn_wave_barrier();
      if (jt + STEP < jt1) load_tile(kv0 + STEP * BN);
    } else if (jt + 1 < jt1) {
      store_tile(cur ^ 1);  // stage cur^1 was last read before the barrier that ended the previous iteration
      if (jt + 2 < jt1) load_tile(kv0 + 2 * BN);
    }

    bool live = wave_live && (!CAUSAL || kv0 <= pos_hi + coff);  // else: the whole tile is above this wavefront's diagonal
    MaskBlock<float> mask = next_mask;
    if (MASK == 1) {
      if (jt + STEP < jt1) next_mask = load_attn_mask<float, true>(a, mrow, kv0 + STEP * BN, lh, S);
      if (live && !mask_sees_any<float>(mask)) {  // taken only for infinities and NaN in V
        const float* Vs = smem + cur * Lds::STAGE + BN * K_PITCH;
        uint32_t odd = 0;  // the exponent's lowest bit added: a carry into the sign's place where it is all ones
#pragma unroll
        for (int i = 0; i < BN * D / 64; i++) {
          const float v = Vs[(64 * i + lane) / D * V_PITCH + (64 * i + lane) % D];
          odd |= (__builtin_bit_cast(uint32_t, v) & 0x7fffffffu) + 0x00800000u;
        }
        live = __builtin_amdgcn_ballot_w64((odd >> 31) != 0) != 0;
      }
    }
    if (live) {
      const float* Ks = smem + cur * Lds::STAGE;
      const float* Vs = Ks + BN * K_PITCH;

      if (MASK == 2) mask = load_attn_mask<float>(a, mrow, kv0, lh, S);  // requested here, used behind the score products

      // ---- S^T = K . Q^T, two accumulators over alternate k-steps ----------------------------------------------------
      f32x16 s0, s1;
#pragma unroll
      for (int r = 0; r < 16; r++) s0[r] = 0.f, s1[r] = 0.f;
      const float* krow = Ks + k_lane;
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ks += 2) {
        s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(krow[ks], qreg[ks], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_32x32x2f32(krow[ks + 1], qreg[ks + 1], s1, 0, 0, 0);
      }
      f32x16 s;
#pragma unroll
      for (int r = 0; r < 16; r++) s[r] = s0[r] + s1[r];

      if (MASK == 1 ? !mask_sees_all<float>(mask) : MASKED) apply_attn_mask<float, MASK == 1>(a, s, mask, kv0, lh, S);

      // ---- mask the diagonal / ragged tile -----------------------------------------------------------------------------
      if ((CAUSAL && kv0 + BN - 1 > pos_lo + coff) || (kv0 + BN > S)) {
        const int qi = (a.pack_L ? (qw0 + lq) % a.pack_L : qw0 + lq) + coff;
#pragma unroll
        for (int r = 0; r < 16; r++) {
          int key = kv0 + 8 * (r >> 2) + 4 * lh + (r & 3);
          bool hidden = key >= S || (CAUSAL && key > qi);
          if (hidden) s[r] = -INFINITY;
        }
      }

      // ---- online softmax with a lazily raised maximum -----------------------------------------------------------------
      float mloc = s[0];
#pragma unroll
      for (int r = 1; r < 16; r++) mloc = fmaxf(mloc, s[r]);
      mloc = fmaxf(mloc, __shfl_xor(mloc, 32));
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(mloc > m_use + lazy) != 0, 0)) {
        const float m_new = fmaxf(m_use, mloc);
        const float alpha = fast_exp2((m_use - m_new) * c);
        m_use = m_new;
        mc = m_new * c;
        l_run *= alpha;
#pragma unroll
        for (int i = 0; i < DBLK; i++)
#pragma unroll
          for (int r = 0; r < 16; r++) oacc[i][r] *= alpha;
      }
      float psum = 0.f;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        s[r] = fast_exp2(MASKED ? (s[r] - m_use) * c : fmaf(s[r], c, -mc));
        psum += s[r];
      }
      l_run += psum;

      // ---- O^T += V^T . P^T: MFMA t contracts the keys held in accumulator register t of the two lane halves -------------
      const float* vl = Vs + v_lane;
#pragma unroll
      for (int t = 0; t < 16; t++) {
#pragma unroll
        for (int db = 0; db < DBLK; db++) {
          float va = vl[(8 * (t >> 2) + (t & 3)) * V_PITCH + 32 * db];
          oacc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(va, s[t], oacc[db], 0, 0, 0);
        }
      }
    }
    if (!KEYS) __syncthreads();
  }

  // ---- normalise and store ----------------------------------------------------------------------------------------------
  float l_tot = l_run + __shfl_xor(l_run, 32);
  const int qi = qw0 + lq;
  if constexpr (KEYS) {  // the four wavefronts' results to their common maximum, added in wavefront order
    float* ml = smem_f32 + 4 * D * 32;  // [wavefront][maximum, sum][32 rows], behind the accumulators
    static_assert(4 * D * 32 + 4 * 64 <= 4 * Lds::STAGE, "");
    __syncthreads();
    ml[wave * 64 + lane] = lh ? l_tot : m_use;
    __syncthreads();
    float m_all = ml[lq];
#pragma unroll
    for (int w = 1; w < 4; w++) m_all = fmaxf(m_all, ml[w * 64 + lq]);
    float l_all = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) l_all = fmaf(fast_exp2((ml[w * 64 + lq] - m_all) * c), ml[w * 64 + 32 + lq], l_all);
    const float f = fast_exp2((m_use - m_all) * c);
    float* mine = smem_f32 + wave * D * 32 + lane;
#pragma unroll
    for (int db = 0; db < DBLK; db++)
#pragma unroll
      for (int r = 0; r < 16; r++) mine[(16 * db + r) * 64] = oacc[db][r] * f;
    __syncthreads();
    const float inv = 1.f / l_all;
    if (qi < a.L) {
      float* op = (float*)a.out + b * a.os[0] + h * a.os[1] + qi * a.os[2];
#pragma unroll
      for (int db = 0; db < DBLK; db++) {
        const int d = 32 * db + 8 * wave + 4 * lh;
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const float* at = smem_f32 + (16 * db + 4 * wave + e) * 64 + lane;
          x[e] = (((at[0] + at[D * 32]) + at[2 * D * 32]) + at[3 * D * 32]) * inv;
        }
        if (!PAD || d < a.D) *(f32x4*)(op + d) = x;
      }
    }
    return;
  }
  if (divided && ntiles_kv * BN > a.kv_chunk) {  // a partial result (else the row tile's keys end in the first split: the output itself)
    store_split_record<D>(a, (long long)b * a.Hq + h, split, qw0, lane, oacc, m_use, l_tot);
    return;
  }
  const float inv = 1.f / l_tot;
  if (qi < a.L) {
    float* op = (float*)a.out + b * a.os[0] + h * a.os[1] + qi * a.os[2];
#pragma unroll
    for (int db = 0; db < DBLK; db++)
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        f32x4 x;
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = oacc[db][4 * rg + i] * inv;
        if (!PAD || 32 * db + 8 * rg + 4 * lh < a.D) *(f32x4*)(op + 32 * db + 8 * rg + 4 * lh) = x;
      }
  }
}

template <int D, bool CAUSAL, int MASK, bool PAD, bool KEYS, int SPLIT>
int launch_f32_v(const KArgs& a, hipStream_t stream) {
  constexpr int lds = (KEYS ? 4 : 2) * F32Lds<D>::STAGE * 4, rows = KEYS ? 32 : BM;
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  const hipError_t granted = grant_dynamic_lds((const void*)prefill_f32_kernel<D, CAUSAL, MASK, PAD, KEYS, SPLIT>, lds, state, done);
  if (granted != hipSuccess) return (int)granted;
  const long long nwg = a.kv_splits > 1 ? split_grid(a, rows) : (long long)a.B * a.Hq * ((a.L + rows - 1) / rows);
  if (nwg > 0x7fffffffLL) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL((prefill_f32_kernel<D, CAUSAL, MASK, PAD, KEYS, SPLIT>), dim3((unsigned)nwg), dim3(256), lds, stream, a);
  return (int)hipGetLastError();
}

// Key tiles walked by one wavefront, times the rounds of the CUs: in workgroups of 128 rows, or of 32 with the tiles dealt out to
// the wavefronts (one such workgroup per CU; half a tile's time to add the results up).
bool keys_among_wavefronts(const KArgs& a, double* tiles_walked = nullptr) {
  if (a.kv_splits > 1) return false;
  const long long heads = (long long)a.B * a.Hq, wide = heads * ((a.L + BM - 1) / BM), narrow = heads * ((a.L + 31) / 32);
  const long long tiles = ((a.causal && !a.pack_L && !a.kv_len && a.L < a.S ? a.L : a.S) + BN - 1) / BN;
  // under a causal mask a launch of several rounds has a little more than half of the tiles to take
  auto rounds = [&](long long wgs) {
    const double r = (double)wgs * (a.causal ? 0.6 : 1.0) / 256;
    return r > 1 ? r : 1.0;
  };
  // several rounds of the narrow ones: nothing overlaps a workgroup's loads, where two of the wide ones share a CU (4 x 8 heads x
  // 778 rows, head_dim 80: 196 us dealt out, 125 whole)
  const double whole = (double)tiles * rounds(wide), narrow_rounds = narrow <= 512 ? (double)((narrow + 255) / 256) : rounds(narrow);
  const double dealt = (double)((tiles + 3) / 4) * (narrow_rounds > 1 ? 1.4 * narrow_rounds : 1.0) + 0.5;
  // (head_dim 128: a dealt tile's loads overlap only its wavefront's own work, 6.2 us a tile instead of 4.6: 3 x 8 heads x 200 rows on
  // 2000 keys 96 us dealt out, 71 in splits)
  if (tiles_walked) *tiles_walked = dealt < 0.9 * whole ? dealt * (a.D > 64 ? 1.35 : 1.0) : whole;
  return dealt < 0.9 * whole;
}

template <int D, bool CAUSAL, int MASK, bool PAD>
int launch_f32_k(const KArgs& a, hipStream_t stream) {
  if (a.kv_splits <= 1 && keys_among_wavefronts(a)) return launch_f32_v<D, CAUSAL, MASK, PAD, true, 0>(a, stream);
  if constexpr (MASK != 0) {
    return launch_f32_v<D, CAUSAL, MASK, PAD, false, 2>(a, stream);
  } else {
    return a.kv_splits > 1 ? launch_f32_v<D, CAUSAL, MASK, PAD, false, 1>(a, stream) : launch_f32_v<D, CAUSAL, MASK, PAD, false, 0>(a, stream);
  }
}

template <int D, bool PAD>
int launch_f32_d(const KArgs& a, hipStream_t stream) {
  // the callers keep to this (rows are read in 16-byte chunks)
  if (PAD && (a.D % 4 != 0 || a.D >= D || a.D < 4)) return (int)hipErrorInvalidValue;
  // (exclusive with causal: validated by the caller, as the reference asserts)
  if (a.mask_kind != 0) return a.mask_kind == 1 ? launch_f32_k<D, false, 1, PAD>(a, stream) : launch_f32_k<D, false, 2, PAD>(a, stream);
  return a.causal ? launch_f32_k<D, true, 0, PAD>(a, stream) : launch_f32_k<D, false, 0, PAD>(a, stream);
}

}  // namespace

double prefill_f32_tiles(const KArgs& a, bool* dealt) {
  double tiles = 0;
  const bool among = keys_among_wavefronts(a, &tiles);
  if (dealt) *dealt = among;
  return tiles;
}

int launch_prefill_f32(const KArgs& a, hipStream_t stream) {
  if (a.D == 128) return launch_f32_d<128, false>(a, stream);
  if (a.D == 64) return launch_f32_d<64, false>(a, stream);
  // any other multiple of 4 up to 128: the kernel of the next size up, the missing columns as zeros
  return a.D < 64 ? launch_f32_d<64, true>(a, stream) : launch_f32_d<128, true>(a, stream);
}

}  // namespace ttsdpa
