// Attention of short sequences and many heads with an attnMask, 16-bit tensors: a batch of sentences padded to one length.  Up to 256
// keys and rows, head_dim up to 64; no pages (reference src/Function/FuncNNLayer.h:237-265).
//
// A workgroup brings all of a head's K and V into LDS at once, and a wavefront takes 16 R rows against all keys: their scores (up to
// 64 registers for 16 rows) stay in place, so that the maximum is known before the first exponential and there is one barrier in all.
//   scores   S^T[16 keys][16 rows] = K . Q^T by 16 x 16 x 32 matrix instructions: lane 16g + i holds keys 4g .. 4g+3 of row i.
//   P.V      a pair of 16-key units is one 16 x 16 x 32 step: lane 16g + i's eight probabilities are those of keys 4g .. 4g+3 of
//            either unit, and V^T comes by transposing LDS reads in the same order.  A lane ends with elements 16n + 4g .. +3 of row i.
// Rows in LDS are of 16-byte chunks, chunk c of row r in place c ^ swz(r), so that neither read has bank conflicts.
//
// KEYS, a Bool mask without a row index: hidden keys' K rows are zeros in LDS and the score products start from -inf there, 0
// elsewhere; what lies behind the last visible key is left out, unless V has an infinity or NaN somewhere (0 times those counts).
// Other masks: a lane's four keys of every unit are requested before the scores.  FULLP: probabilities with all their fp32 bits, as in
// prefill_kernel; an operand of V is read once for all parts, and infinities in it meet the first part only.
//
// What bounds it (16 x 12 heads x 197 rows, fp16, lengths 49 to 197, core cycles of a workgroup): 6300 until K and V are in LDS, 2800 for
// the scores, 4000 for the exponentials, their parts and P.V on each of a SIMD's two wavefronts, whose vector and matrix work hardly
// overlap, 1200 for the rows' way out; a launch is 4.4 us of the 12.0 that the caller sees (prefill_kernel: 13.0).  What was slower:
// 13 wavefronts of 16 rows, 128 registers each (12.2), no requests ahead with 16 rows (12.8), operands ahead with 32 (spills, 16.1).

#include <type_traits>

#include "sdpa_common.h"

namespace ttsdpa {

namespace {

constexpr int U = 16;            // keys of a unit
constexpr int kMostPairs = 8;    // pairs of units
constexpr int kMostWaves = 8;
constexpr int W = 64, ROWB = 2 * W, CH = W / 8;

__device__ __forceinline__ int swz(int row) { return (row & 6) | ((row >> 3) & 1); }  // by the row's place among 16

typedef short s16x4 __attribute__((ext_vector_type(4)));

template <typename TR, bool KEYS, bool FULLP, int R>
__global__ __launch_bounds__(64 * kMostWaves) void heads_kernel(KArgs a, int units) {
  typedef typename TR::elem T;
  typedef typename TR::vec8 vec8;
  typedef typename TR::vec4 vec4;
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  constexpr int KS = W / 32, NDB = W / 16, BATCH = 4, ROWS = 16 * R;
  constexpr int NB = R == 1 ? 2 : 1;  // a pair's operands are requested while the pair before is computed, where registers allow
  constexpr bool FLAGS = KEYS || FULLP;
  constexpr bool SHIFT = FULLP && __is_same(T, _Float16);
  constexpr uint32_t kExp = __is_same(T, _Float16) ? 0x7c00u : 0x7f80u;  // a value's exponent: all ones in infinities and NaN

  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, nthr = blockDim.x, nwave = nthr >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, g = lane >> 4;

  const int nrow = (a.L + ROWS - 1) / ROWS, nblk = (nrow + units - 1) / units;
  int pair, in;
  map_workgroup(blockIdx.x, a.B * a.Hq, nblk, &pair, &in);
  const int h = pair % a.Hq, b = pair / a.Hq, hk = h / a.G;
  const int first = in * units, end = first + units < nrow ? first + units : nrow;  // wavefronts' units of rows
  const T* qp = (const T*)a.q + b * a.qs[0] + h * a.qs[1];
  const T* kp = (const T*)a.k + b * a.ks[0] + hk * a.ks[1];
  const T* vp = (const T*)a.v + b * a.vs[0] + hk * a.vs[1];
  T* op = (T*)a.out + b * a.os[0] + h * a.os[1];
  const int S = keys_of_batch(a, b);

  vec8 q[R][KS];
  auto load_q = [&](int ru) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < R; x++) {
      const int row = ru * ROWS + 16 * x + i;
      const T* qr = qp + (row < a.L ? row : a.L - 1) * a.qs[2];
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        vec8 t = {};
        if (32 * ks + 8 * g < a.D) t = *(const vec8*)(qr + 32 * ks + 8 * g);
        q[x][ks] = t;
      }
    }
  };
  load_q(first + wave < end ? first + wave : first);

  if (S == 0) {  // no keys: zeros
    for (int row = first * ROWS + wave * 16 + i; row < end * ROWS && row < a.L; row += 16 * nwave)
      for (int d = 4 * g; d < a.D; d += 16) *(vec4*)(op + row * a.os[2] + d) = vec4{};
    return;
  }

  uint32_t seen = 0;  // KEYS: bytes of keys 4 lane .. +3, zeros beyond the last one
  if (KEYS) {
    const uint8_t* mp = (const uint8_t*)a.mask + b * a.ms[0] + h * a.ms[1];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int key = 4 * lane + e;
      const uint8_t x = mp[(key < S ? key : S - 1) * a.ms[3]];
      if (key < S && x != 0) seen |= 1u << (8 * e);
    }
  }

  const int npair_all = (S + 31) / 32;
  char* ks0 = smem;
  char* vs0 = smem + npair_all * 32 * ROWB;
  float* bias = (float*)(smem + (a.S + 31) / 32 * 32 * 2 * ROWB);
  int* flags = (int*)(bias + 256);
  uint32_t odd = 0;
  for (int base = 0; base < npair_all * 32 * CH; base += nthr * BATCH) {
    u32x4 kx[BATCH], vx[BATCH];
#pragma unroll
    for (int j = 0; j < BATCH; j++) {
      const int idx = base + j * nthr + tid, row = idx / CH, col = idx % CH;
      kx[j] = u32x4{0u, 0u, 0u, 0u}, vx[j] = kx[j];
      if (row < S && 8 * col < a.D) {
        kx[j] = *(const u32x4*)(kp + row * a.ks[2] + 8 * col);
        vx[j] = *(const u32x4*)(vp + row * a.vs[2] + 8 * col);
      }
    }
#pragma unroll
    for (int j = 0; j < BATCH; j++) {
      const int idx = base + j * nthr + tid, row = idx / CH, col = idx % CH;
      if (KEYS) {
        const uint32_t w = (uint32_t)__shfl((int)seen, (row >> 2) & 63);
        if (((w >> (8 * (row & 3))) & 1u) == 0) kx[j] = u32x4{0u, 0u, 0u, 0u};
      }
      if (FLAGS) {  // the exponent's lowest bit added: a carry into the sign's place where it is all ones
#pragma unroll
        for (int w = 0; w < 4; w++) odd |= ((vx[j][w] & 0x7fff7fffu) + (kExp & (0u - kExp)) * 0x10001u) & 0x80008000u;
      }
      if (row < npair_all * 32) {
        const int at = row * ROWB + 16 * (col ^ swz(row));
        *(u32x4*)(ks0 + at) = kx[j];
        *(u32x4*)(vs0 + at) = vx[j];
      }
    }
  }
  if (FLAGS) {
    const bool any = __builtin_amdgcn_ballot_w64(odd != 0) != 0;
    if (lane == 0) flags[wave] = any;
  }
  int npair = npair_all;  // pairs of units that are taken: up to the last visible key
  if (KEYS) {
    const unsigned long long vis = __builtin_amdgcn_ballot_w64(seen != 0);
    npair = vis == 0 ? 1 : (63 - __builtin_clzll(vis)) / 8 + 1;
    if (wave == 0) {
      f32x4 x;
#pragma unroll
      for (int e = 0; e < 4; e++) x[e] = (seen >> (8 * e)) & 1u ? 0.f : -INFINITY;
      *(f32x4*)(bias + 4 * lane) = x;
    }
  }
  __syncthreads();
  bool whole = false;  // V has infinities or NaN
  if (FLAGS) {
    whole = __builtin_amdgcn_ballot_w64(lane < nwave && flags[lane & 15] != 0) != 0;
    if (whole) npair = npair_all;
  }

  const float c = scores_unit(a);
  const int vrow = 4 * g + (i >> 2);
  const char* klane[KS];
  const char* vlane[NDB];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) klane[ks] = ks0 + i * ROWB + 16 * ((4 * ks + g) ^ swz(i));
#pragma unroll
  for (int n = 0; n < NDB; n++) vlane[n] = vs0 + vrow * ROWB + 16 * ((2 * n + ((i & 3) >> 1)) ^ swz(vrow)) + 8 * (i & 1);

  for (int ru = first + wave; ru < end; ru += nwave) {
    const int q0 = ru * ROWS;

    // ---- without KEYS: the mask's keys 4g .. 4g+3 of every unit, all requested ahead of the scores ------------------------
    typedef uint32_t loose32 __attribute__((aligned(1)));
    typedef unsigned long long loose64 __attribute__((aligned(2)));
    unsigned long long mk[R][KEYS ? 1 : 2 * kMostPairs];
    int room = S - 4 - 4 * g;  // where the last group of four keys starts, from the lane's own first one
    asm volatile("" : "+v"(room));  // (else what follows from it is kept in registers over the rows' loop)
    if constexpr (!KEYS) {
#pragma unroll
      for (int x = 0; x < R; x++) {
        const int row = q0 + 16 * x + i;
        const long long mrow = b * a.ms[0] + h * a.ms[1] + (row < a.L ? row : a.L - 1) * a.ms[2] + 4 * g;
#pragma unroll
        for (int u = 0; u < 2 * kMostPairs; u++) {
          mk[x][u] = 0;
          if (u >= 2 * npair) continue;
          const int past = U * u > room ? U * u - room : 0;  // a group that runs past the last key: read from key S - 4 on, and shifted
          if (a.mask_kind == 1) mk[x][u] = *(const loose32*)((const uint8_t*)a.mask + mrow + (U * u - past)) >> (8 * (past & 3));
          else mk[x][u] = *(const loose64*)((const uint16_t*)a.mask + mrow + (U * u - past)) >> (16 * (past & 3));
        }
      }
    }

    // ---- scores ---------------------------------------------------------------------------------------------------------
    f32x4 s[R][2 * kMostPairs];
    float m[R];
#pragma unroll
    for (int x = 0; x < R; x++) m[x] = -FLT_MAX;
    vec8 kb[NB][2][KS];
    f32x4 c0[NB][2];
    auto load_k = [&](int buf, int t) __attribute__((always_inline)) {
#pragma unroll
      for (int y = 0; y < 2; y++) {
        c0[buf][y] = KEYS ? *(const f32x4*)(bias + U * (2 * t + y) + 4 * g) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ks++) kb[buf][y][ks] = *(const vec8*)(klane[ks] + U * (2 * t + y) * ROWB);
      }
    };
    if (NB == 2) load_k(0, 0);
#pragma unroll
    for (int t = 0; t < kMostPairs; t++) {
      if (t >= npair) continue;
      if (NB == 1) load_k(0, t);
      else if (t + 1 < kMostPairs) load_k((t + 1) & 1, t + 1 < npair_all ? t + 1 : t);
#pragma unroll
      for (int y = 0; y < 2; y++)
#pragma unroll
        for (int x = 0; x < R; x++) {
          const int u = 2 * t + y;
          f32x4 z = c0[t & (NB - 1)][y];
#pragma unroll
          for (int ks = 0; ks < KS; ks++) z = TR::mfma16(kb[t & (NB - 1)][y][ks], q[x][ks], z);
          if constexpr (!KEYS) {
            if (a.mask_kind == 1) {
#pragma unroll
              for (int r = 0; r < 4; r++)
                if (((mk[x][u] >> (8 * r)) & 0xffu) == 0) z[r] = -INFINITY;
            } else {
              const vec4 bv = __builtin_bit_cast(vec4, mk[x][u]);
#pragma unroll
              for (int r = 0; r < 4; r++) z[r] = fmaf(z[r], a.scale, (float)bv[r]);
            }
            if (U * u + U > S) {
#pragma unroll
              for (int r = 0; r < 4; r++)
                if (U * u + r - 4 >= room) z[r] = -INFINITY;
            }
          }
          s[x][u] = z;
          m[x] = fmaxf(m[x], fmaxf(fmaxf(z[0], z[1]), fmaxf(z[2], z[3])));
        }
    }
    vec8 vb[NB][NDB];
    auto load_v = [&](int buf, int t) __attribute__((always_inline)) {
#pragma unroll
      for (int n = 0; n < NDB; n++) {
        const char* va = vlane[n] + 2 * U * t * ROWB;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)va);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(va + U * ROWB));
        vb[buf][n] = __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
    if (NB == 2) load_v(0, 0);
    float l[R];
#pragma unroll
    for (int x = 0; x < R; x++) {
      m[x] = fmaxf(m[x], __shfl_xor(m[x], 16));
      m[x] = fmaxf(m[x], __shfl_xor(m[x], 32));
      l[x] = 0.f;
    }
    if (NB == 2 && ru + nwave < end) load_q(ru + nwave);

    // ---- P.V ------------------------------------------------------------------------------------------------------------
    constexpr int NP = FULLP ? TR::kParts : 1;
    f32x4 acc[R][NDB];
#pragma unroll
    for (int x = 0; x < R; x++)
#pragma unroll
      for (int n = 0; n < NDB; n++) acc[x][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto take = [&](auto clean) __attribute__((always_inline)) {  // clean: infinities and NaN in V meet the first part only
#pragma unroll
      for (int t = 0; t < kMostPairs; t++) {
        if (t >= npair) continue;
        if (NB == 1) load_v(0, t);
        else if (t + 1 < kMostPairs) load_v((t + 1) & 1, t + 1 < npair_all ? t + 1 : t);
        vec8 pb[R][NP];
#pragma unroll
        for (int x = 0; x < R; x++) {
          f32x8 p;
#pragma unroll
          for (int e = 0; e < 8; e++) {
            const float d = s[x][2 * t + (e >> 2)][e & 3] - m[x];
            p[e] = fast_exp2(SHIFT ? fmaf(d, c, 10.f) : d * c);
            l[x] += p[e];
          }
#pragma unroll
          for (int k = 0; k < NP; k++) pb[x][k] = FULLP ? TR::take_part(p) : __builtin_convertvector(p, vec8);
        }
#pragma unroll
        for (int n = 0; n < NDB; n++) {
          vec8 v = vb[t & (NB - 1)][n];
#pragma unroll
          for (int x = 0; x < R; x++) acc[x][n] = TR::mfma16(v, pb[x][0], acc[x][n]);
          if constexpr (FULLP) {
            if constexpr (decltype(clean)::value) {
              u32x4 w = __builtin_bit_cast(u32x4, v);
#pragma unroll
              for (int j = 0; j < 4; j++) {
                if ((w[j] & kExp) == kExp) w[j] &= 0xffff0000u;
                if ((w[j] & (kExp << 16)) == kExp << 16) w[j] &= 0xffffu;
              }
              v = __builtin_bit_cast(vec8, w);
            }
#pragma unroll
            for (int k = 1; k < NP; k++)
#pragma unroll
              for (int x = 0; x < R; x++) acc[x][n] = TR::mfma16(v, pb[x][k], acc[x][n]);
          }
        }
      }
    };
    if (FULLP && whole) take(std::integral_constant<bool, true>{});
    else take(std::integral_constant<bool, false>{});
#pragma unroll
    for (int x = 0; x < R; x++) {
      const int row = q0 + 16 * x + i;
      l[x] += __shfl_xor(l[x], 16);
      l[x] += __shfl_xor(l[x], 32);
      const float inv = 1.f / l[x];
      if (row < a.L) {
#pragma unroll
        for (int n = 0; n < NDB; n++)
          if (16 * n + 4 * g < a.D) *(vec4*)(op + row * a.os[2] + 16 * n + 4 * g) = __builtin_convertvector(acc[x][n] * inv, vec4);
      }
    }
    if (NB == 1 && ru + nwave < end) load_q(ru + nwave);
  }
}

bool keys_only_mask(const KArgs& a) { return a.mask_kind == 1 && a.ms[2] == 0; }

// Workgroups of a launch with 16 R rows a wavefront: a head's rows in as many as they need, or as there are CUs for, of two row units
// at least; four wavefronts at least (they bring K and V).
struct HeadsShape {
  int units, waves;  // row units of a workgroup
  long long wgs;
  HeadsShape(const KArgs& a, int R) {
    const int nrow = (a.L + 16 * R - 1) / (16 * R);
    const long long heads = (long long)a.B * a.Hq, room = heads >= 256 ? 1 : 256 / heads;
    int blocks = (nrow + kMostWaves - 1) / kMostWaves;
    if (blocks < room) blocks = (int)(room < (nrow + 1) / 2 ? room : (nrow + 1) / 2);
    units = (nrow + blocks - 1) / blocks;
    wgs = heads * ((nrow + units - 1) / units);
    waves = units < 4 ? 4 : units < kMostWaves ? units : kMostWaves;
  }
};

template <typename TR, bool KEYS, bool FULLP, int R>
int launch_k(const KArgs& a, hipStream_t stream) {
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  constexpr int kFixed = 256 * 4 + 64, kMostBytes = 256 * 2 * ROWB + kFixed;
  hipError_t e = grant_dynamic_lds((const void*)heads_kernel<TR, KEYS, FULLP, R>, kMostBytes, state, done);
  if (e != hipSuccess) return (int)e;
  const HeadsShape n(a, R);
  const int lds = (a.S + 31) / 32 * 32 * 2 * ROWB + kFixed;
  hipLaunchKernelGGL((heads_kernel<TR, KEYS, FULLP, R>), dim3((unsigned)n.wgs), dim3(64 * n.waves), lds, stream, a, n.units);
  return (int)hipGetLastError();
}

template <typename TR>
int launch_t(const KArgs& a, int rows, hipStream_t stream) {
  if (!keys_only_mask(a)) return a.full_p ? launch_k<TR, false, true, 1>(a, stream) : launch_k<TR, false, false, 1>(a, stream);
  if (rows == 16) return a.full_p ? launch_k<TR, true, true, 1>(a, stream) : launch_k<TR, true, false, 1>(a, stream);
  return a.full_p ? launch_k<TR, true, true, 2>(a, stream) : launch_k<TR, true, false, 2>(a, stream);
}

}  // namespace

// Rows of a wavefront of the kernel for a call, 0: another kernel is the shorter way (or the only one).  a.full_p as the call has it.
// 16 rows where the workgroups run side by side, at most two rounds of them of the shortest heads; 32, with half the LDS reads for
// each product but nothing requested ahead, where more are needed and the mask is the keys' alone.  Against the other kernel, us, key
// padding / additive [H, L, L]:
//   8 heads x 94       7.0 ->  5.3              16 x 49 (bf16)          6.7 -> 5.7
//   64 x 247 (bf16)   12.2 ->  8.3              64 x 217 (bf16)        15.8 -> 10.5
//   128 x 136          8.4 ->  6.5              128 x 93 (bf16)        10.2 -> 6.8
//   192 x 197         13.0 -> 12.0 (32 rows)    256 x 189              16.8 -> 16.8 (there; 19.6 here)
//   256 x 137         11.7 ->  9.1 (32 rows)    384 x 104 (bf16)       10.1 -> 10.1 (there; 13.3 here)
//   768 x 174         32.4 -> 26.9 (32 rows)    768 x 47 (bf16)        12.7 -> 10.6
// head_dim 32 and below has tiles of its own in the other kernel.  Its time over this one's there, geometric means of 3800 calls: keys 1.05
// to 1.2, but 0.82 with two rounds of workgroups at 32, or where it reads the mask four keys at a time; Bool rows 0.95 to 0.98 up to 64 rows (0.7 with two rounds), 1.02 to 1.07 beyond;
// additive ones 1.06 to 1.4, but where it reads their keys four at a time 0.9 to 0.95 with more than 96 rows and 1024 units of 16 in all.  At 40
// to 64 the same are 1.1 to 1.5 throughout, Bool rows up to 32 1.00 to 1.2.
int heads_rows(const KArgs& a, int dtype) {
  if (dtype == 0 || a.D < 8 || a.D > W || a.D % 8 != 0 || a.S < 1 || a.S > 32 * kMostPairs || a.L < 16 || a.L > 256 || a.block_table ||
      a.pack_L || a.causal || a.mask_kind == 0)
    return 0;
  const bool keys_only = keys_only_mask(a);
  if (!keys_only && (a.ms[3] != 1 || a.S < 4 || a.kv_len)) return 0;  // (it reads such masks four keys at a time)
  const HeadsShape n(a, 1);
  const long long side = 256ll * (kMostWaves / n.waves);
  const bool narrow = a.D <= 32;
  bool best = n.wgs <= (n.waves <= 4 ? 2 : 1) * side;
  if (keys_only) best = best && !(narrow && n.wgs >= 512 && (a.D == 32 || !a.full_p));
  else if (a.mask_kind == 1) best = best && (!narrow || a.L > 64);
  else if (narrow && !a.full_p) best = best && (a.L <= 96 || n.wgs * n.units < 1024);
  if (best) return 16;
  return keys_only && !narrow ? 32 : 0;
}

int launch_heads(const KArgs& a, int dtype, hipStream_t stream) {
  const int rows = heads_rows(a, dtype);
  if (rows == 0) return (int)hipErrorInvalidValue;
  return dtype == 1 ? launch_t<F16>(a, rows, stream) : launch_t<BF16>(a, rows, stream);
}

}  // namespace ttsdpa
