// Products whose wavefronts divide the contraction among themselves, for gfx950: few rows of x against a large weight
// (a decode step's projections), small layers, and operands of any alignment and size (reference: op::matmul,
// src/Operation/OpLinalg.cpp:52-276; device GEMM src/Operation/OpLinalgCuda.cuh:239-293).
//
//   out[m][n] = bias[n] + sum_k x(m,k) w(n,k)     x(m,k) = XT ? x[k*ldx + m] : x[m*ldx + k], w(n,k) likewise
//
// What bounds these shapes is latency and the bytes in flight, not the matrix pipe: a workgroup owns a small tile of the
// output (16*MB rows of x by 16*NB of w) and its W wavefronts take the 128-byte pieces (units) of the contraction in turn,
// each with a ring of P units of its own in registers; no barrier until the partial sums meet in LDS at the end.
//   operands     a step of a unit is the 16 bytes that a lane supplies to v_mfma_f32_16x16x32 (16-bit: row l%16, k = 8(l/16)
//                .. +7) or to four v_mfma_f32_16x16x4 (fp32: k = 4(l/16) + e in instruction e, the same pairing on both
//                sides)
//   loads        into registers, at any alignment, eight lanes to the 128 bytes of a row; then through a piece of LDS of the
//                wavefront's own into operand order.  (Straight into operand order saves the LDS, but there 16 neighbouring
//                lanes belong to 16 rows: a CU took in 16 bytes per clock, 24 x 2048 x 5632 ran 13 us instead of 7.4.)
//   k-major      an operand stored [K, rows]: 16-bit loads 16 bytes along the rows and reads LDS transposed
//                (ds_read_b64_tr_b16); fp32 loads its elements straight into operand order (64 contiguous bytes per k)
//   edges        rows past the end re-read the last one (k-major: the last tile is moved back to end with the matrix).

#include "../../include/ttsdpa.h"
#include "linear_args.h"

namespace ttsdpa {
namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// 16 bytes at any element's address (rows may begin anywhere)
typedef uint32_t loose16 __attribute__((ext_vector_type(4), aligned(2)));

template <typename TR>
struct Step {
  typedef typename TR::elem elem;
  typedef typename TR::vec8 frag;
  static constexpr int KV = 8;  // consecutive k of a lane
  static __device__ __forceinline__ f32x4 mma(frag a, frag b, f32x4 c) { return TR::mfma16(a, b, c); }
};
struct F32 {};
template <>
struct Step<F32> {
  typedef float elem;
  typedef f32x4 frag;
  static constexpr int KV = 4;
  static __device__ __forceinline__ f32x4 mma(frag a, frag b, f32x4 c) {
#pragma unroll
    for (int e = 0; e < 4; e++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
    return c;
  }
};

// One operand of a tile: R blocks of 16 rows from `row0` on.  A unit of the contraction is 128 bytes of a row: 64 k of a
// 16-bit type, 32 of fp32, two steps of 16 bytes per lane of an operand register.
template <typename TR, bool KMAJOR, int R>
struct Operand {
  typedef Step<TR> S;
  typedef typename S::elem T;
  typedef typename S::frag frag;
  static constexpr int KV = S::KV, KU = 8 * KV;             // k of a unit
  static constexpr bool DIRECT = KMAJOR && KV == 4;         // fp32, k-major: no LDS
  static constexpr int PITCH = 32 * R + 16;                 // 16-bit, k-major: bytes of a k-row in LDS (4 rows in different banks)
  static constexpr int LDS = DIRECT ? 0 : KMAJOR ? KU * PITCH : 16 * R * 128;
  static constexpr int NL = 2 * R;                        // 16-byte registers of a unit
  static constexpr int CPR = KMAJOR ? 2 * R : 8, RPI = 64 / CPR;  // 16-byte chunks of a row as loaded, rows of one load instruction

  const char* base;  // of the first row at k = 0
  unsigned off[NL];  // bytes from base (+ the unit's advance) of what this lane loads
  long long ld;      // bytes
  int lane;

  // `rows`: rows of the tile, at most 16 * R; those beyond re-read its last one
  __device__ __forceinline__ void init(const void* p, long long row0, int rows, long long ld_elems, int lane_) {
    lane = lane_;
    ld = ld_elems * (long long)sizeof(T);
    base = (const char*)p + (KMAJOR ? row0 * (long long)sizeof(T) : row0 * ld);
#pragma unroll
    for (int i = 0; i < NL; i++) {
      if constexpr (DIRECT) {  // register i: block i / 2, step i % 2, k = 16 (i % 2) + 4 (lane / 16) + element
        off[i] = (unsigned)((16 * (i & 1) + 4 * (lane >> 4)) * ld + (16 * (i >> 1) + (lane & 15)) * (long long)sizeof(T));
      } else {
        const int r = RPI * i + lane / CPR;
        off[i] = (unsigned)((KMAJOR || r < rows ? r : rows - 1) * ld + 16 * (lane % CPR));
      }
    }
  }

  // k0: the unit's first k
  __device__ __forceinline__ void load(u32x4 (&v)[NL], long long k0) const {
    const char* at = base + k0 * (KMAJOR ? ld : (long long)sizeof(T));
#pragma unroll
    for (int i = 0; i < NL; i++) {
      if constexpr (DIRECT) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[i][e] = *(const uint32_t*)(at + e * ld + off[i]);
      } else {
        v[i] = *(const loose16*)(at + off[i]);
      }
    }
  }

  // k of the first element that this lane loaded into register i, from the unit's first
  __device__ __forceinline__ int k_of(int i) const {
    return DIRECT ? 16 * (i & 1) + 4 * (lane >> 4) : KMAJOR ? RPI * i + lane / CPR : KV * (lane % CPR);
  }

  // zeros for the first `skip` k of the unit (the last unit of a contraction that is no whole number of units begins
  // before the one in front of it ends)
  __device__ __forceinline__ void clear(u32x4 (&v)[NL], int skip) const {
#pragma unroll
    for (int i = 0; i < NL; i++) {
      const int gone = skip - k_of(i);
      if constexpr (KMAJOR && !DIRECT) {
        if (gone > 0) v[i] = u32x4{0u, 0u, 0u, 0u};
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if constexpr (KV == 4) v[i][e] = e < gone ? 0u : v[i][e];
          else v[i][e] = 2 * e + 1 < gone ? 0u : 2 * e < gone ? v[i][e] & 0xffff0000u : v[i][e];
        }
      }
    }
  }

  // a contraction of K < KU elements, then zeros
  __device__ __forceinline__ void load_short(u32x4 (&v)[NL], int K) const {
#pragma unroll
    for (int i = 0; i < NL; i++) {
      v[i] = u32x4{0u, 0u, 0u, 0u};
      const int left = K - k_of(i);
      if constexpr (KMAJOR && !DIRECT) {
        if (left > 0) v[i] = *(const loose16*)(base + off[i]);
      } else {
#pragma unroll
        for (int e = 0; e < KV; e++)
          if (e < left) {
            const char* p = base + off[i] + (DIRECT ? e * ld : e * (long long)sizeof(T));
            if constexpr (KV == 4) v[i][e] = *(const uint32_t*)p;
            else v[i][e >> 1] |= (uint32_t)*(const uint16_t*)p << (16 * (e & 1));
          }
      }
    }
  }

  // what was loaded, into the wavefront's piece of LDS (its LDS instructions run in order: no waits between the two)
  __device__ __forceinline__ void stage(const u32x4 (&v)[NL], char* lds) const {
    if constexpr (!DIRECT)
#pragma unroll
      for (int i = 0; i < NL; i++) {
        const int r = RPI * i + lane / CPR, c = lane % CPR;
        if constexpr (KMAJOR) *(u32x4*)(lds + r * PITCH + 16 * c) = v[i];
        else *(u32x4*)(lds + r * 128 + 16 * (c ^ ((r >> 1) & 7))) = v[i];  // 16 rows of a chunk fall into different banks
      }
  }

  // operand registers of step s (0 or 1) of the unit
  __device__ __forceinline__ void frags(frag (&f)[R], const u32x4 (&v)[NL], const char* lds, int s) const {
    const int r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int b = 0; b < R; b++) {
      if constexpr (DIRECT) {
        f[b] = __builtin_bit_cast(frag, v[2 * b + s]);
      } else if constexpr (KMAJOR) {
        const char* from = lds + (32 * s + 8 * q + (r >> 2)) * PITCH + 8 * (r & 3) + 32 * b;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)from);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(from + 4 * PITCH));
        f[b] = __builtin_bit_cast(frag, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      } else {
        f[b] = *(const frag*)(lds + (16 * b + r) * 128 + 16 * ((4 * s + q) ^ ((r >> 1) & 7)));
      }
    }
  }
};

template <typename TR, bool XT, bool WT, int MB, int NB, int W>
struct StreamLds {
  static constexpr int STAGE = Operand<TR, XT, MB>::LDS + Operand<TR, WT, NB>::LDS;  // per wavefront
  static constexpr int PITCH = 16 * NB + 4;                                            // floats of a row of partial sums
  static constexpr int SUMS = 16 * MB * PITCH * 4;                                     // per wavefront
  static constexpr int BYTES = W * (STAGE > SUMS ? STAGE : SUMS);
};

// One tile of the product: workgroup `block` of those of entry `entry`.  ROWSUM: the workgroups of the first column of tiles
// also write a.rowsum[m] = sum_k x(m,k) (a product with ones that rides along in the matrix pipe).
//
// GROUP: a.tile_waves of the workgroup's wavefronts share a tile, the others have tiles of their own (waves_of_call).
template <typename TR, bool XT, bool WT, int MB, int NB, int W, int P, bool ROWSUM, bool GROUP = false>
__device__ __forceinline__ void stream_tile(const LinArgs& a, char* smem, int block, int entry) {
  typedef Operand<TR, XT, MB> OX;
  typedef Operand<TR, WT, NB> OW;
  typedef StreamLds<TR, XT, WT, MB, NB, W> Lds;
  typedef typename Step<TR>::elem T;
  typedef typename Step<TR>::frag frag;
  constexpr int TM = 16 * MB, TN = 16 * NB, KU = OX::KU;
  const int lane = threadIdx.x & 63;
  const int wg_wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = GROUP ? a.tile_waves : W;  // wavefronts of a tile
  const int wave = GROUP ? wg_wave & (G - 1) : wg_wave, first_wave = wg_wave - wave, per_block = GROUP ? W / G : 1;  // tiles of a workgroup

  // workgroup -> tile: an XCD (workgroup i runs on XCD i % 8) takes a contiguous band of tiles, rows of x fastest, so that
  // the workgroups that read a piece of w run side by side
  const int tiles_m = (int)((a.M + TM - 1) / TM), tiles_n = (int)((a.N + TN - 1) / TN);
  const int blocks = GROUP ? (tiles_m * tiles_n + per_block - 1) / per_block : tiles_m * tiles_n;
  const int band = (blocks + 7) / 8;
  const int split = block / (8 * band);  // range of the contraction
  block -= split * 8 * band;
  block = (block & 7) * band + (block >> 3);
  if (block >= blocks) return;
  int tile = GROUP ? block * per_block + first_wave / G : block;
  const bool idle = GROUP && tile >= tiles_m * tiles_n;  // (the last workgroup's)
  if (idle) tile = 0;
  long long m0 = (long long)(tile % tiles_m) * TM, n0 = (long long)(tile / tiles_m) * TN;
  if (XT && m0 > a.M - TM) m0 = a.M - TM;  // k-major operands have at least a tile of rows (the host sees to it)
  if (WT && n0 > a.N - TN) n0 = a.N - TN;

  OX ox;
  OW ow;
  ox.init((const T*)a.x + (long long)entry * a.bsx, m0, a.M - m0 < TM ? (int)(a.M - m0) : TM, a.ldx, lane);
  ow.init((const T*)a.w + (long long)entry * a.bsw, n0, a.N - n0 < TN ? (int)(a.N - n0) : TN, a.ldw, lane);
  char* stage = smem + wg_wave * Lds::STAGE;

  f32x4 acc[NB][MB];
#pragma unroll
  for (int i = 0; i < NB; i++)
#pragma unroll
    for (int j = 0; j < MB; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  f32x4 rowsum[ROWSUM ? MB : 1];
  frag ones;
  bool sums_rows = false;
  if constexpr (ROWSUM) {
    sums_rows = a.rowsum && tile < tiles_m && !idle;
#pragma unroll
    for (int j = 0; j < MB; j++) rowsum[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < Step<TR>::KV; e++) ones[e] = (T)1.f;
  }

  u32x4 xv[P][OX::NL], wv[P][OW::NL];
  auto use = [&](int p) __attribute__((always_inline)) {
    ow.stage(wv[p], stage + OX::LDS);
    ox.stage(xv[p], stage);
#pragma unroll
    for (int s = 0; s < 2; s++) {
      frag xf[MB], wf[NB];
      ow.frags(wf, wv[p], stage + OX::LDS, s);
      ox.frags(xf, xv[p], stage, s);
#pragma unroll
      for (int i = 0; i < NB; i++)
#pragma unroll
        for (int j = 0; j < MB; j++) acc[i][j] = Step<TR>::mma(wf[i], xf[j], acc[i][j]);
      if constexpr (ROWSUM)
        if (sums_rows)
#pragma unroll
          for (int j = 0; j < MB; j++) rowsum[j] = Step<TR>::mma(ones, xf[j], rowsum[j]);
    }
  };

  // unit i of the contraction belongs to wavefront i % G of the tile's; a last, incomplete one is read as the KU elements in front of
  // the end, those of the unit before it as zeros
  const int K = (int)a.K, all_units = (K + KU - 1) / KU;
  const int per_split = (all_units + a.splits - 1) / a.splits;
  const int u0 = split * per_split;  // the split's units: u0 .. u0 + units - 1
  const int units = all_units - u0 < per_split ? all_units - u0 : per_split;
  const int n = units > wave && !idle ? (units - wave + G - 1) / G : 0;
  const bool overlaps = K % KU != 0 && n > 0 && u0 + (n - 1) * G + wave == all_units - 1;  // this wavefront's last unit is that one
  auto first_k = [&](int j) __attribute__((always_inline)) {
    const int k = (u0 + (j < n ? j : n - 1) * G + wave) * KU;  // requests past the end repeat the last unit (never used)
    return (long long)(k < K - KU ? k : K - KU);
  };
  if (K < KU) {
    if (n > 0) {
      ow.load_short(wv[0], K);
      ox.load_short(xv[0], K);
      use(0);
    }
  } else if (n > 0) {
#pragma unroll
    for (int p = 0; p < P; p++) {
      if (GROUP && p > 0 && n == 1) break;  // a short contraction: nothing to repeat
      ow.load(wv[p], first_k(p));
      ox.load(xv[p], first_k(p));
    }
    int j0 = 0;
    for (; j0 + P < n; j0 += P)
#pragma unroll
      for (int p = 0; p < P; p++) {
        use(p);
        ow.load(wv[p], first_k(j0 + P + p));
        ox.load(xv[p], first_k(j0 + P + p));
      }
#pragma unroll
    for (int p = 0; p < P; p++)
      if (j0 + p < n) {
        if (overlaps && j0 + p == n - 1) {
          ow.clear(wv[p], KU - K % KU);
          ox.clear(xv[p], KU - K % KU);
        }
        use(p);
      }
  }

  // partial sums: a lane holds rows m = 16j + l%16, columns n = 16i + 4(l/16) .. +3
  __syncthreads();  // (the staging pieces of other wavefronts lie where the sums go)
  float* sums = (float*)smem + wg_wave * (Lds::SUMS / 4);
#pragma unroll
  for (int i = 0; i < NB; i++)
#pragma unroll
    for (int j = 0; j < MB; j++) *(f32x4*)(sums + (16 * j + (lane & 15)) * Lds::PITCH + 16 * i + 4 * (lane >> 4)) = acc[i][j];
  if constexpr (ROWSUM)
    if (sums_rows && lane < 16)  // (every row of the product with ones is the same)
#pragma unroll
      for (int j = 0; j < MB; j++) ((float*)(smem + Lds::BYTES))[wg_wave * TM + 16 * j + lane] = rowsum[j][0];
  __syncthreads();
  if (idle) return;
  const int thread = threadIdx.x - 64 * first_wave;  // of the tile's
  const float* const tile_sums = (const float*)smem + first_wave * (Lds::SUMS / 4);
  float* part = a.part ? a.part + split * (a.M * a.N + a.M) : nullptr;  // this split's sums: of the product, then of x's rows
  if constexpr (ROWSUM)
    if (sums_rows && thread < TM && m0 + thread < a.M) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < (GROUP ? G : W); w++) v += ((const float*)(smem + Lds::BYTES))[(first_wave + w) * TM + thread];
      if (part) part[a.M * a.N + m0 + thread] = v;
      else store_from_float((T*)a.rowsum + m0 + thread, v);
    }
  const bool whole = (a.ldo & 3) == 0 && ((uintptr_t)a.out & (4 * sizeof(T) - 1)) == 0 && (a.bso & 3) == 0 && (n0 & 3) == 0;
  for (int g = thread; g < TM * (TN / 4); g += 64 * G) {
    const int r = g / (TN / 4), c = 4 * (g % (TN / 4));
    const long long m = m0 + r, col = n0 + c;
    if (m >= a.M || col >= a.N) continue;
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
    const float* from = tile_sums + r * Lds::PITCH + c;
    if constexpr (!GROUP) {
#pragma unroll
      for (int w = 0; w < W; w++) v += *(const f32x4*)(from + w * (Lds::SUMS / 4));
    } else {
      for (int w = 0; w < G; w++) v += *(const f32x4*)(from + w * (Lds::SUMS / 4));
    }
    const int have = a.N - col < 4 ? (int)(a.N - col) : 4;
    if (part) {
      float* dst = part + m * a.N + col;
      if (have == 4 && ((a.N | n0) & 3) == 0) *(f32x4*)dst = v;
      else
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (e < have) dst[e] = v[e];
      continue;
    }
    if (a.bias)
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (e < have) v[e] += load_as_float((const T*)a.bias + col + e);
    T* dst = (T*)a.out + (long long)entry * a.bso + m * a.ldo + col;
    if (whole && have == 4) {
      typedef T out4 __attribute__((ext_vector_type(4)));
      *(out4*)dst = __builtin_convertvector(v, out4);
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (e < have) store_from_float(dst + e, v[e]);
    }
  }
}

// out = bias + the sum of the splits' partial products, and the same of the row sums.  An index into a split has 32 bits (plan_tiles; divided
// tiles are few).
template <typename T>
__global__ __launch_bounds__(256) void linear_merge_kernel(LinArgs a) {
  typedef float loose4 __attribute__((ext_vector_type(4), aligned(4)));  // (a split begins at any element)
  typedef T out4 __attribute__((ext_vector_type(4)));
  const long long total = a.M * a.N + a.M;
  const long long per = a.rowsum ? total : a.M * a.N;
  const bool fours = ((a.N | a.ldo) & 3) == 0;
  const bool whole = ((uintptr_t)a.out & (4 * sizeof(T) - 1)) == 0;
  for (long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4; i < per; i += (long long)gridDim.x * 1024) {
    if (i + 4 <= a.M * a.N && fours) {
      f32x4 v = *(const loose4*)(a.part + i);
#pragma unroll 4
      for (int s = 1; s < a.splits; s++) v += (f32x4)*(const loose4*)(a.part + s * total + i);
      const uint32_t m = (uint32_t)i / (uint32_t)a.N, n = (uint32_t)i - m * (uint32_t)a.N;
      if (a.bias)
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] += load_as_float((const T*)a.bias + n + e);
      T* dst = (T*)a.out + (long long)m * a.ldo + n;
      if (whole) *(out4*)dst = __builtin_convertvector(v, out4);
      else
#pragma unroll
        for (int e = 0; e < 4; e++) store_from_float(dst + e, v[e]);
    } else {
      for (long long k = i; k < i + 4 && k < per; k++) {
        float v = 0.f;
#pragma unroll 4
        for (int s = 0; s < a.splits; s++) v += a.part[s * total + k];
        if (k >= a.M * a.N) store_from_float((T*)a.rowsum + (k - a.M * a.N), v);
        else store_from_float((T*)a.out + k / a.N * a.ldo + k % a.N, v + (a.bias ? load_as_float((const T*)a.bias + k % a.N) : 0.f));
      }
    }
  }
}

template <typename T>
int launch_merge(const LinArgs& a, hipStream_t stream) {
  const long long groups = (a.M * a.N + a.M + 1023) / 1024;
  const dim3 grid((unsigned)(groups < 2048 ? groups : 2048));
  if (a.M * a.N + a.M >= 0x7fffffffLL) return TTSDPA_ERR_SHAPE;  // (the plans keep to this)
  hipLaunchKernelGGL((linear_merge_kernel<T>), grid, dim3(256), 0, stream, a);
  return (int)hipGetLastError();
}

}  // namespace

int launch_linear_merge(const LinArgs& a, int dtype, hipStream_t stream) {
  return dtype == 0 ? launch_merge<float>(a, stream) : dtype == 1 ? launch_merge<_Float16>(a, stream) : launch_merge<__bf16>(a, stream);
}

namespace {

// Wavefronts and units in flight of each by the tile's size in blocks of 16: eight with a ring of as many units as their registers
// hold; on the largest tile four, which have twice the registers (eight measure the same, and spill).
template <int R>
struct Shape {
  static constexpr int W = R == 4 ? 4 : 8, P = 4 / R;
};

template <typename TR, bool XT, bool WT, int R, bool GROUP>
__global__ __launch_bounds__(64 * Shape<R>::W, Shape<R>::W / 4) void linear_stream_kernel(LinArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  stream_tile<TR, XT, WT, R, R, Shape<R>::W, Shape<R>::P, XT && WT, GROUP>(a, smem, blockIdx.x, blockIdx.y);  // row sums: a weight's gradient
}

// Few rows of x (one tile of them) against a weight that 32 x 32 tiles cut into more pieces than there are CUs, up to twice as many: tiles
// of as many of its rows as make one round; and rows that leave much of a square tile idle (few_rows_tile).
template <typename TR, bool WT, int MB, int NB, int P>
__global__ __launch_bounds__(512, 2) void linear_rows_kernel(LinArgs a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  stream_tile<TR, false, WT, MB, NB, 8, P, false>(a, smem, blockIdx.x, blockIdx.y);
}

// Both products of a linear layer's backward in one launch, the first `split` workgroups those of the weight's gradient
// (grad^T . x, with grad's column sums: the bias's gradient), the others those of the input's (grad . w).
template <typename TR, int RW, int RI, bool GROUP>
__global__ __launch_bounds__(64 * Shape<RW>::W, Shape<RW>::W / 4) void linear_stream_pair_kernel(LinArgs gw, LinArgs gi, int split) {
  static_assert(Shape<RW>::W == Shape<RI>::W, "one workgroup size");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  if ((int)blockIdx.x < split) stream_tile<TR, true, true, RW, RW, Shape<RW>::W, Shape<RW>::P, true, GROUP>(gw, smem, blockIdx.x, 0);
  else stream_tile<TR, false, true, RI, RI, Shape<RI>::W, Shape<RI>::P, false>(gi, smem, blockIdx.x - split, 0);
}

template <int R>
int tiles_of_block(const LinArgs& a) {
  return a.tile_waves ? Shape<R>::W / a.tile_waves : 1;
}

template <int R>
long long blocks_of(const LinArgs& a) {
  const long long tiles = ((a.M + 16 * R - 1) / (16 * R)) * ((a.N + 16 * R - 1) / (16 * R)), per_block = tiles_of_block<R>(a);
  return ((tiles + per_block - 1) / per_block + 7) / 8 * 8 * a.splits;
}

template <typename TR, bool XT, bool WT, int R, bool GROUP = false>
int launch_kernel(const LinArgs& a, hipStream_t stream, unsigned entries) {
  if constexpr (XT && WT && !GROUP)
    if (tiles_of_block<R>(a) > 1) return launch_kernel<TR, XT, WT, R, true>(a, stream, entries);
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  constexpr int lds = StreamLds<TR, XT, WT, R, R, Shape<R>::W>::BYTES + (XT && WT ? Shape<R>::W * 16 * R * 4 : 0);
  const hipError_t granted = grant_dynamic_lds((const void*)linear_stream_kernel<TR, XT, WT, R, GROUP>, lds, state, done);
  if (granted != hipSuccess) return (int)granted;
  const long long blocks = blocks_of<R>(a);
  if (blocks > 0x3fffffffLL) return TTSDPA_ERR_SHAPE;
  hipLaunchKernelGGL((linear_stream_kernel<TR, XT, WT, R, GROUP>), dim3((unsigned)blocks, entries), dim3(64 * Shape<R>::W), lds, stream, a);
  return (int)hipGetLastError();
}

template <typename TR, bool WT, int MB, int NB, int P>
int launch_rows_kernel(const LinArgs& a, hipStream_t stream) {
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  constexpr int lds = StreamLds<TR, false, WT, MB, NB, 8>::BYTES;
  const hipError_t granted = grant_dynamic_lds((const void*)linear_rows_kernel<TR, WT, MB, NB, P>, lds, state, done);
  if (granted != hipSuccess) return (int)granted;
  const long long tiles = ((a.M + 16 * MB - 1) / (16 * MB)) * ((a.N + 16 * NB - 1) / (16 * NB));
  hipLaunchKernelGGL((linear_rows_kernel<TR, WT, MB, NB, P>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(512), lds, stream, a);
  return (int)hipGetLastError();
}

template <typename TR, int RW, int RI, bool GROUP = false>
int launch_pair_kernel(const LinArgs& gw, const LinArgs& gi, hipStream_t stream) {
  if constexpr (!GROUP)
    if (tiles_of_block<RW>(gw) > 1) return launch_pair_kernel<TR, RW, RI, true>(gw, gi, stream);
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  constexpr int W = Shape<RW>::W;
  constexpr int lds_w = StreamLds<TR, true, true, RW, RW, W>::BYTES + W * 16 * RW * 4, lds_i = StreamLds<TR, false, true, RI, RI, W>::BYTES;
  constexpr int lds = lds_w > lds_i ? lds_w : lds_i;
  const hipError_t granted = grant_dynamic_lds((const void*)linear_stream_pair_kernel<TR, RW, RI, GROUP>, lds, state, done);
  if (granted != hipSuccess) return (int)granted;
  const long long split = blocks_of<RW>(gw), all = split + blocks_of<RI>(gi);
  if (all > 0x3fffffffLL) return TTSDPA_ERR_SHAPE;
  hipLaunchKernelGGL((linear_stream_pair_kernel<TR, RW, RI, GROUP>), dim3((unsigned)all), dim3(64 * W), lds, stream, gw, gi, (int)split);
  return (int)hipGetLastError();
}

}  // namespace

namespace {

constexpr int wavefronts(int R) { return R == 4 ? Shape<4>::W : Shape<1>::W; }  // of a workgroup

// Wavefronts that a tile has work for where both operands are k-major (a weight's gradient) and a short contraction has fewer units
// than a workgroup wavefronts; 0: for all.
int waves_of_tile(const LinArgs& a, int esz, int R) {
  if (!a.xt || !a.wt) return 0;
  int G = 1;
  while (G < wavefronts(R) && (long long)G * (128 / esz) < a.K) G *= 2;
  return G < wavefronts(R) ? G : 0;
}

double tiles_of(const LinArgs& a, int R) { return (double)((a.M + 16 * R - 1) / (16 * R)) * (double)((a.N + 16 * R - 1) / (16 * R)); }

// Wavefronts that share a tile of a call (others, RI: tiles and size of another product in the launch).  A workgroup takes as many tiles
// as leave none of its wavefronts idle; backward of a layer, us, a tile to a workgroup -> so: fp32 19 x 2048 x 2048 54 -> 20; 16-bit 62 x
// 1024 x 1024 13.5 -> 6.0.  But where all tiles run side by side there is nothing to gain, and those of a workgroup wait for each other:
// 16-bit layers of up to 256 tiles 4.2 us a tile to a workgroup, 4.5 in groups; fp32 24 x 512 x 320 5.4 and 7.7, whose 32 x 32 tiles
// share a CU in pairs, where one unit is all their work or the other product's tiles are of that size too (20 x 40 x 3328, 312 tiles, 5.5 and
// 7.3; 72 x 576 x 320, 280 tiles of three units and 16-row ones, 6.8 and 6.1).
int waves_of_call(const LinArgs& a, int esz, int R, int S, double entries, double others, int RI) {
  const int W = wavefronts(R), G = S > 1 ? 0 : waves_of_tile(a, esz, R);
  if (G == 0) return W;
  const double tiles = 8 * ceil(tiles_of(a, R) / 8) * entries;
  const bool pairs = esz == 4 && R == 2 && (RI == 2 || (G == 1 && tiles <= 256));
  return tiles + 8 * ceil(others / 8) <= (pairs ? 512 : 256) ? W : G;
}

double rounds_of(const LinArgs& a, long long tm, long long tn, double entries) {
  const double tiles = (double)((a.M + tm - 1) / tm) * (double)((a.N + tn - 1) / tn) * entries;
  return tiles > 256 ? tiles / 256 : 1;
}

// Microseconds of a product on tiles of 16*R rows of x by 16*R of w, its contraction divided among S workgroups per tile, from
// measurements (MI355X, 16-bit unless said): 3 us of launch, latency and the meeting of the partial sums (2 more on the
// largest tile: a wavefront's sums are 16 KB); then, for each round of the 256 CUs, half a microsecond and the operands of
// a tile at the 65 GB/s that a CU takes in (it measured 60-75 over all shapes that the L2s hold or that are read once: when
// both operands are larger, all tiles together take theirs in at 8 TB/s, 1636 x 3775 x 2025 100 us, with k-major operands at
// 10, 205 x 4096 x 25472 160; 16-bit k-major operands come in pieces of
// 32*R bytes, which costs 2.6, 1.6 and 1.1 times that), or the tile's products where those take longer (fp32: 0.45 TFLOP/s
// of a CU's 0.61 on the largest tile while a CU has one, 0.36 with more, 0.3 on the others).  With S > 1 another launch and the partial products written and
// read.
//   measured / this: 1000^3 on 16, 32, 64: 25 / 26, 12 / 13, 9.5 / 9.4; 24 x 2048 x 5632: 7.4 / 9, 10.5 / 13, 19 / 21;
//   64 x 4096 x 4096: 17 / 20, 11 / 12, 21 / 22; fp32 1000^3: 42 / 43, 30 / 32, 25 / 24; both k-major, 500 x 500 x 8192:
//   88 / 90, 29 / 29, 40 / 40
// whole: fp32's largest tiles are bound by the matrix cores, so that the 8 of 264 that make a second round take as long as it (62 x 16896
// x 3072, 138 us; 130 x 3072 x 8448 182, divided among more 95).  A call's own plan goes by this; which way a product runs goes by the other, for the tiled kernels, which
// would then be taken for more calls, add up the contraction in fewer and longer chains.
// Several tiles to a workgroup (a weight's gradient of few rows), 16-bit: by its wavefronts with work, 1024 of which run at once; tiles of
// 16, 32 and 64 rows take 0.9, 1.9 and 7.7 us for each 1024 more: in 32 x 32 tiles 20 x 2048 x 2048 9.8 us, 120 x 2048 x 1024
// 6.9, 250 x 2048 x 1024 12.9, 24 x 11264 x 2048 42.  fp32, whose products bound it, takes what the rounds say but for single units on the largest
// tiles: 20 x 9000 x 3000 66 us in 32 x 32 ones, 98 in 64 x 64.
double stream_us(const LinArgs& a, int esz, int R, int S, double entries, bool whole = false) {
  if (esz == 4 && R == 4 && S == 1 && waves_of_tile(a, esz, R) == 1) return 5 + 3 * rounds_of(a, 64, 64, entries);
  if (const int G = esz == 2 && S == 1 ? waves_of_tile(a, esz, R) : 0) {
    const double tiles = tiles_of(a, R) * entries, waves = tiles * G / 1024;
    return 3 + (waves <= 1 && R < 4 ? 0.5 : waves * (R == 1 ? 0.9 : R == 2 ? 1.9 : 7.7));
  }
  const double tm = 16 * R, tn = 16 * R;
  const double tiles = tiles_of(a, R) * entries * S;
  // (16-bit x . w^T, 64 rows: a second round lasts as long as the first, however few its tiles: 720 x 1536 x 1536, 288 tiles, 18.2 us, on the
  // tiled kernel 14.8; k-major operands bound such calls otherwise.  The shares of such calls are counted so too, lest two of them look
  // shorter: 54 x 18688 x 3072, 292 tiles, 32.7, in two shares 35.2)
  const bool whole_rounds = R == 4 && (whole || (esz == 2 && !a.xt && !a.wt && (tiles < 512 || (tiles > 256 * S && tiles < 512 * S))));
  const double rounds = tiles <= 256 ? 1 : whole_rounds ? ceil(tiles / 256) : tiles / 256;
  const double narrow = esz == 4 ? 1 : R == 1 ? 2.6 : R == 2 ? 1.6 : 1.1;
  const double k = (double)a.K / S;
  const double bytes = ((a.M < tm ? a.M : tm) * (a.xt ? narrow : 1) + (a.N < tn ? a.N : tn) * (a.wt ? narrow : 1)) * k * esz;
  const double rate = esz == 2 ? 4e6 : R < 4 ? 0.3e6 : rounds > 1.5 ? 0.36e6 : 0.45e6, flops = 2 * tm * tn * k;
  const double per = bytes / 65e3 > flops / rate ? bytes / 65e3 : flops / rate;
  const double few = (double)(a.M < a.N ? a.M : a.N) * a.K * esz, all = (double)(a.M + a.N) * a.K * esz;
  // (one round of tiles on rows of whole lines: they go along the contraction together, and the L2s hold what they are at: 539 x 1600 x 2432
  // 14.1 us, 22.5 by the rate; rows across lines up to 1.4 times that)
  const bool together = esz == 2 && S == 1 && !a.xt && !a.wt && tiles <= 256 && (a.ldx | a.ldw) % 64 == 0;
  const double missed = few > 2e6 && all > 8e6 && !together ? tiles * bytes / (esz == 2 && (a.xt || a.wt) ? 10e6 : 8e6) : 0;
  // 16-bit: the next tile's first loads and the last one's output do not overlap (tiles of 64 rows: 72 of k into 960 x 7552, 7 rounds
  // 38 us, 752 into 1906 x 2088, 3.9: 32; of 32: 327 into 310 x 4245, 5.2: 17.6, 262 k-major into 2545 x 866, 8.8: 27)
  // (two workgroups of 32 rows share a CU: two rounds are one)
  const double turns = esz == 4 || R == 1 ? 0 : R == 4 ? 3 * (rounds - 1) : rounds > 2 ? 0.75 * (rounds - 1) : 0;
  const double work = rounds * (0.5 + per) + turns;
  return (R == 4 ? 5 : 3) + (work > missed ? work : missed) + (S > 1 ? 3 + S * 8.0 * a.M * a.N / 4e6 : 0);
}

// The cheapest tile (rows in blocks of 16: 1, 2 or 4, as far as a k-major operand has them; R = 0: none) and, when the caller
// has scratch for partial products, division of the contraction (no less than 512 of it per workgroup).
StreamPlan plan_tiles(const LinArgs& a, int esz, double entries, bool may_split, int least = 1, int most = 4, bool whole = false, int chains = 0) {
  StreamPlan best{0, 1, 0};
  for (int R = least; R <= most; R *= 2) {
    if ((a.xt && a.M < 16 * R) || (a.wt && a.N < 16 * R)) break;
    // half of a 64 square tile idle: its few workgroups stream a weight slower than the estimate, which has every round full (12 x
    // 5120 x 34944: 87 us in 64-row tiles, 69 in 32-row ones; 12 x 4096 x 28672 54 and 45)
    if (R == 4 && R > least && (a.M <= 32 || a.N <= 32)) break;
    for (int S = 1; S <= 32 && (S == 1 || (may_split && a.K >= 512 * S && a.M * a.N + a.M < 0x7fffffffLL)); S *= 2) {
      if (wavefronts(R) * S < chains) continue;
      const double t = stream_us(a, esz, R, S, entries, whole);
      if (!best.R || t < best.us) best = {R, S, t};
    }
  }
  return best;
}

// The tile for up to 32 rows of x where 32 x 32 ones would be taken, 16-bit x . w^T.  Those of one to two rounds of the 256 CUs last as
// long as two.  A tile's eight wavefronts take its units of 64 of K in turn, with four on their way in 16-row tiles: those go by
// whole rings (K 1536, 2048, 3584, 4096, 6144, 8192, or a few units more), while a ring of one or two at the end costs what the smaller tile
// gained.  Times of 32 x 32 tiles over those of others, weights from memory, geometric means of 6500 products by K and tiles:
//   257 to 384 tiles    up to 16 rows, whole rings    K < 2560  16 x 64 1.14 to 1.24, 32 x 48 1.02 to 1.18    beyond  16 x 16 1.11 to 1.23
//                       others                        32 x 48 1.07 to 1.31 (16 x 16 1.0 to 1.17, K 1024 0.9)
//   385 to 512          up to 16 rows, whole rings    K < 2560  16 x 64 1.05 to 1.14    beyond  up to 8  16 x 16 1.01 to 1.12, more  16 x 64 1.02 to 1.10
//                       others                        16 x 16 0.82 to 0.98, 16 x 64 0.95 to 1.08, 32 x 48 0.75
//   more, 200 MB        up to 8 rows, whole rings     16 x 16 1.00 to 1.08 (28672 x 4096 1.06, 32000 x 4096 1.14)
//                       others                        16 x 16 K 1024 0.75 to 0.85, 2560 0.91, 3072 0.97, 5120 0.98
//   24 rows x 8704, K 1024, 2048, 4096    8.4, 14.2, 23.5 us -> 7.1, 11.6, 18.6 (32 x 48)
// k-major w (a layer's input gradient), us, rows x columns x contraction: up to 16 rows in 16 x 32 tiles, 16 x 8192 x 2048 12.6 -> 11.0 (5 x 7839 x 731
// 6.4 -> 7.2, hence the least contraction; 5850 products by units of a wavefront: 3 and 4 1.10, 8, 12 and 16 1.03 to 1.04, other odd ones 1.02, 6
// 0.98, 10 and 14 1.00); 32 x 64 ones where 32 x 32 make one to two rounds, 30 x 11264 x 4096 38 -> 28, 8 x 10880 x 5760 40
// -> 30; 33 to 48 rows in 48 x 64 tiles of eight wavefronts instead of 64 x 64 of four, 42 x 11200 x 4096 28 -> 23, 37 x 17280 x 5120 58 -> 54.
enum class Tile { Square, Square16, Rows32x48, Rows16x64, Rows16x32, Rows32x64, Rows48x64 };
Tile few_rows_tile(const LinArgs& a, int R) {
  if (a.wt && !a.xt) {
    if (R == 4) return a.M > 32 && a.M <= 48 ? Tile::Rows48x64 : Tile::Square;
    const long long pieces = (a.N + 31) / 32;
    if (a.M > 32 || pieces > 512) return Tile::Square;
    if (pieces > 256) return Tile::Rows32x64;
    const int each = (int)((a.K + 511) / 512);  // units of a wavefront: rings of four
    return a.M <= 16 && a.K >= 1200 && (each & 3) != 2 ? Tile::Rows16x32 : Tile::Square;
  }
  if (a.xt || a.M > 32 || R != 2) return Tile::Square;
  const long long tiles = (a.N + 31) / 32;
  const int units = (int)((a.K + 63) / 64), rest = units & 31;  // beyond whole rings of all wavefronts
  const bool whole_rings = rest == 0 || rest >= 22 || (rest <= 4 && units > 64);
  if (tiles > 512) return a.M <= 8 && whole_rings && a.K > 1400 && a.N * a.K > 100000000ll ? Tile::Square16 : Tile::Square;
  if (tiles <= 256) return Tile::Square;
  if (a.M <= 16 && a.K >= 1536) {
    if (a.K < 2560 && (whole_rings || tiles > 384)) return Tile::Rows16x64;
    if (whole_rings) return tiles > 384 && a.M > 8 ? Tile::Rows16x64 : Tile::Square16;
  }
  return tiles <= 384 ? Tile::Rows32x48 : Tile::Square;  // (a round of 32 x 48)
}

// The tile of a call
Tile tile_of_call(const LinArgs& a, int dtype, unsigned entries, const StreamPlan& p) {
  return dtype != 0 && entries == 1 && p.S == 1 && p.R >= 2 ? few_rows_tile(a, p.R) : Tile::Square;
}

template <typename TR>
int launch_rows_type(const LinArgs& a, Tile tile, hipStream_t stream) {
  switch (tile) {
    case Tile::Rows32x48: return launch_rows_kernel<TR, false, 2, 3, 2>(a, stream);
    case Tile::Rows16x64: return launch_rows_kernel<TR, false, 1, 4, 4>(a, stream);
    case Tile::Rows16x32: return launch_rows_kernel<TR, true, 1, 2, 4>(a, stream);
    case Tile::Rows32x64: return launch_rows_kernel<TR, true, 2, 4, 2>(a, stream);
    default: return launch_rows_kernel<TR, true, 3, 4, 1>(a, stream);
  }
}

size_t part_bytes(const LinArgs& a, int S) { return S > 1 ? (size_t)S * (size_t)(a.M * a.N + a.M) * sizeof(float) : 0; }

template <typename TR, bool XT, bool WT>
int launch_rows(const LinArgs& a, int R, hipStream_t stream, unsigned entries) {
  if (R == 1) return launch_kernel<TR, XT, WT, 1>(a, stream, entries);
  if (R == 2) return launch_kernel<TR, XT, WT, 2>(a, stream, entries);
  return launch_kernel<TR, XT, WT, 4>(a, stream, entries);
}

template <typename TR>
int launch_type(const LinArgs& a, int R, hipStream_t stream, unsigned entries) {
  if (a.xt) return a.wt ? launch_rows<TR, true, true>(a, R, stream, entries) : launch_rows<TR, true, false>(a, R, stream, entries);
  return a.wt ? launch_rows<TR, false, true>(a, R, stream, entries) : launch_rows<TR, false, false>(a, R, stream, entries);
}

template <typename TR>
int launch_pair_type(const LinArgs& gw, const LinArgs& gi, int RW, int RI, hipStream_t stream) {
  if (RW == 4) return launch_pair_kernel<TR, 4, 4>(gw, gi, stream);
  if (RW == 2) return RI == 2 ? launch_pair_kernel<TR, 2, 2>(gw, gi, stream) : launch_pair_kernel<TR, 2, 1>(gw, gi, stream);
  return RI == 2 ? launch_pair_kernel<TR, 1, 2>(gw, gi, stream) : launch_pair_kernel<TR, 1, 1>(gw, gi, stream);
}

// Tiles of the two products of a layer's backward: one workgroup size, so both of 64 rows or both of fewer.
PairPlan plan_pair(const LinArgs& gw, const LinArgs& gi, int esz) {
  PairPlan few{plan_tiles(gw, esz, 1, true, 1, 2), plan_tiles(gi, esz, 1, false, 1, 2)};
  // one round of the CUs with both, if that only takes larger tiles of the other (16-bit; 60 x 777 x 1001 10.8 -> 6.1, 60 x 512 x 1024 6.5 -> 5.0)
  if (const int G = esz == 2 && few.gw.S == 1 && few.gw.R == 2 && few.gi.R == 1 && gi.N >= 32 ? waves_of_tile(gw, esz, 2) : 0) {
    const double blocks = floor(tiles_of(gw, 2) * G / wavefronts(2));
    if (blocks + tiles_of(gi, 1) > 256 && blocks + tiles_of(gi, 2) <= 256) few.gi = {2, 1, stream_us(gi, esz, 2, 1, 1)};
  }
  // and a round with a tile of the weight's gradient to a workgroup, if larger ones of it make that (97 x 320 x 232 5.0 -> 4.2)
  if (esz == 2 && few.gw.S == 1 && few.gw.R == 1 && gw.M >= 32 && gw.N >= 32 && waves_of_tile(gw, esz, 1) > 0) {
    const double of_i = tiles_of(gi, few.gi.R);
    if (tiles_of(gw, 1) + of_i > 256 && tiles_of(gw, 2) + of_i <= 240) few.gw.R = 2;
  }
  const PairPlan many{plan_tiles(gw, esz, 1, true, 4, 4), plan_tiles(gi, esz, 1, false, 4, 4)};
  return many.gw.R && many.gi.R && many.gw.us + many.gi.us < few.gw.us + few.gi.us ? many : few;
}

}  // namespace

bool stream_takes(const LinArgs& a, int dtype) {
  // a tile's rows and a unit's k-rows are addressed with 32-bit byte offsets; a k-major operand has a tile's rows at least
  const long long ld_max = 1ll << 24;
  return a.K >= 1 && a.K <= 0x3fffffffLL && a.ldx < ld_max && a.ldw < ld_max && (!a.xt || a.M >= 16) && (!a.wt || a.N >= 16);
}

StreamPlan plan_stream(const LinArgs& a, int dtype, unsigned entries, bool may_split) {
  return plan_tiles(a, dtype == 0 ? 4 : 2, entries, may_split);
}

// fp32: by whole rounds, which count on the largest tiles, with as many chains of sums (wavefronts and shares) as the other estimate's
// plan has.
StreamPlan plan_stream_call(const LinArgs& a, int dtype, unsigned entries, bool may_split, const StreamPlan& p) {
  if (dtype != 0 || p.R != 4) return p;
  const StreamPlan q = plan_tiles(a, 4, entries, may_split, 1, 4, true, wavefronts(p.R) * p.S);
  return q.us < 0.9 * stream_us(a, 4, p.R, p.S, entries, true) ? q : p;
}

size_t stream_part_bytes(const LinArgs& a, const StreamPlan& call) { return part_bytes(a, call.S); }

StreamTiles stream_tiles(const LinArgs& a, int dtype, unsigned entries, const StreamPlan& call, const LinArgs* other, int RI) {
  switch (tile_of_call(a, dtype, entries, call)) {
    case Tile::Square16: return {16, 16, 1};
    case Tile::Rows32x48: return {32, 48, 1};
    case Tile::Rows16x64: return {16, 64, 1};
    case Tile::Rows16x32: return {16, 32, 1};
    case Tile::Rows32x64: return {32, 64, 1};
    case Tile::Rows48x64: return {48, 64, 1};
    default: break;
  }
  return {16 * call.R, 16 * call.R, wavefronts(call.R) / waves_of_call(a, dtype == 0 ? 4 : 2, call.R, call.S, entries, other ? tiles_of(*other, RI) : 0, RI)};
}

int launch_stream(const LinArgs& args, int dtype, hipStream_t stream, const StreamPlan& chosen, unsigned entries, void* scratch, size_t scratch_bytes) {
  LinArgs a = args;
  StreamPlan p = plan_stream_call(a, dtype, entries, entries == 1 && scratch, chosen);
  if (part_bytes(a, p.S) > scratch_bytes) p = plan_stream_call(a, dtype, entries, false, plan_stream(a, dtype, entries, false));
  a.splits = p.S;
  a.part = p.S > 1 ? (float*)scratch : nullptr;
  a.tile_waves = waves_of_call(a, dtype == 0 ? 4 : 2, p.R, p.S, entries, 0, 0);
  int rc;
  const Tile tile = tile_of_call(a, dtype, entries, p);
  if (tile == Tile::Square16) p.R = 1;
  else if (tile != Tile::Square) return dtype == 1 ? launch_rows_type<F16>(a, tile, stream) : launch_rows_type<BF16>(a, tile, stream);
  switch (dtype) {
    case 0: rc = launch_type<F32>(a, p.R, stream, entries); break;
    case 1: rc = launch_type<F16>(a, p.R, stream, entries); break;
    default: rc = launch_type<BF16>(a, p.R, stream, entries);
  }
  return rc != 0 || p.S == 1 ? rc : launch_linear_merge(a, dtype, stream);
}

PairPlan plan_stream_pair(const LinArgs& gw, const LinArgs& gi, int dtype) { return plan_pair(gw, gi, dtype == 0 ? 4 : 2); }

int launch_stream_pair(const LinArgs& gw_, const LinArgs& gi, int dtype, hipStream_t stream, const PairPlan& p, void* scratch) {
  LinArgs gw = gw_;
  gw.splits = p.gw.S;
  gw.part = p.gw.S > 1 ? (float*)scratch : nullptr;
  gw.tile_waves = waves_of_call(gw, dtype == 0 ? 4 : 2, p.gw.R, p.gw.S, 1, tiles_of(gi, p.gi.R), p.gi.R);
  int rc;
  switch (dtype) {
    case 0: rc = launch_pair_type<F32>(gw, gi, p.gw.R, p.gi.R, stream); break;
    case 1: rc = launch_pair_type<F16>(gw, gi, p.gw.R, p.gi.R, stream); break;
    default: rc = launch_pair_type<BF16>(gw, gi, p.gw.R, p.gi.R, stream);
  }
  return rc != 0 || p.gw.S == 1 ? rc : launch_linear_merge(gw, dtype, stream);
}

}  // namespace ttsdpa
