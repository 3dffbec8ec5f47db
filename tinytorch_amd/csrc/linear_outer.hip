// The weight's gradient of a layer with few rows, for gfx950: out[m][n] = sum_k x[k*ldx + m] w[k*ldw + n] (x: the incoming gradient, w: the
// layer's input) over a contraction of at most a few units of rows, with x's column sums (the bias's gradient) on the way; any
// alignment (reference: FuncLinear::backward, src/Function/FuncNNLayer.h:20-33).
//
// What bounds it is writing the result.  A workgroup of four wavefronts owns 128 x 128 of it: a unit of either operand's rows (64, fp32 32)
// goes through registers into LDS, the next unit's is requested meanwhile, a wavefront computes 64 x 64.  The last tiles are moved
// back to end with the matrix, rows past the contraction's end are zeros.
//   16-bit   operands by transposing LDS reads (rows 8 (l/16) + (l%16)/4 and those + 4, in both); the result leaves through LDS as the
//            tile's 256 bytes of a row.  Few registers and 34 KB, so that four (two units and more: three) workgroups share a CU
//            and some write while others load.
//   fp32     lane l reads four neighbouring elements of row 4 (l/16) + e, one vector: the operands of four blocks of
//            v_mfma_f32_16x16x4 step e.  w's groups of four are dealt out so that the four lanes of a row store 64 bytes side by
//            side.  One unit only: longer contractions are the streaming kernel's, which adds them up in several chains.
// The other ways were the streaming kernel's small tiles or copies in the tiled kernels' layout, their 128 x 128 tiles and launches for the
// bias.  A layer's backward, us, before -> so (16-bit): 16 x 4096 x 4096 31 -> 21 (this kernel 9.1, 33 MB), 24 x 11264 x 2048 40 -> 27 (10.6, 46 MB),
// 42 x 4096 x 11200 62 -> 45, 129 x 2048 x 2048 28 -> 17, 100 x 1000 x 4000 26 -> 15, 256 x 2048 x 8192 54 -> 46; fp32 24 x 3072 x 3072 54 -> 38.

#include <type_traits>

#include "../../include/ttsdpa.h"
#include "linear_args.h"

namespace ttsdpa {
namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef uint32_t loose16 __attribute__((ext_vector_type(4), aligned(2)));  // 16 bytes at any element's address

struct F32 {
  typedef float elem;
};

constexpr int kTile = 128, kThreads = 256;

template <typename TR>
struct Outer {
  typedef typename TR::elem T;
  static constexpr bool FP32 = sizeof(T) == 4;
  static constexpr int KU = FP32 ? 32 : 64;                      // rows of a unit
  static constexpr int CPR = kTile * (int)sizeof(T) / 16;          // 16-byte chunks of a row of the tile
  static constexpr int RPI = kThreads / CPR, NL = KU / RPI;      // rows of one load of the workgroup, loads of a unit
  static constexpr int PITCH = kTile * (int)sizeof(T) + 16, HALF = KU * PITCH;
};

// ONE: the contraction is one unit, so that no loads are in flight while it is computed.
template <typename TR, bool ONE>
__global__ __launch_bounds__(kThreads, ONE ? 4 : 3) void linear_outer_kernel(LinArgs a) {
  typedef Outer<TR> O;
  typedef typename O::T T;
  constexpr bool FP32 = O::FP32;
  static_assert(ONE || !FP32, "fp32: one unit");
  constexpr int KU = O::KU, PITCH = O::PITCH, NL = O::NL;
  __shared__ __attribute__((aligned(16))) char smem[2 * O::HALF];
  static_assert(FP32 || 2 * O::HALF >= kTile * PITCH, "the result fits where the operands lie");
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;

  // an XCD (workgroup i runs on XCD i % 8) takes a contiguous band of tiles, those of a row of tiles side by side
  const int tiles_m = (int)((a.M + kTile - 1) / kTile), tiles_n = (int)((a.N + kTile - 1) / kTile);
  const int band = (tiles_m * tiles_n + 7) / 8;
  const int tile = ((int)blockIdx.x & 7) * band + ((int)blockIdx.x >> 3);
  if (tile >= tiles_m * tiles_n) return;
  long long m0 = (long long)(tile / tiles_n) * kTile, n0 = (long long)(tile % tiles_n) * kTile;
  if (m0 > a.M - kTile) m0 = a.M - kTile;
  if (n0 > a.N - kTile) n0 = a.N - kTile;
  const bool sums_rows = a.rowsum && tile % tiles_n == 0 && wn == 0;

  const int K = (int)a.K, row = tid / O::CPR, chunk = tid % O::CPR;
  const char* xp = (const char*)((const T*)a.x + m0) + 16 * chunk;
  const char* wp = (const char*)((const T*)a.w + n0) + 16 * chunk;
  const long long ldx = a.ldx * (long long)sizeof(T), ldw = a.ldw * (long long)sizeof(T);
  u32x4 xv[NL], wv[NL];
  auto load = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NL; i++) {
      const int k = k0 + O::RPI * i + row, at = k < K ? k : K - 1;
      xv[i] = *(const loose16*)(xp + at * ldx);
      wv[i] = *(const loose16*)(wp + at * ldw);
    }
  };
  auto stage = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NL; i++) {
      const bool past = k0 + O::RPI * i + row >= K;
      char* to = smem + (O::RPI * i + row) * PITCH + 16 * chunk;
      *(u32x4*)to = past ? u32x4{0u, 0u, 0u, 0u} : xv[i];
      *(u32x4*)(to + O::HALF) = past ? u32x4{0u, 0u, 0u, 0u} : wv[i];
    }
  };

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[4][4], rowsum[4];  // acc[i][j]: block i of w's elements, j of x's
#pragma unroll
  for (int j = 0; j < 4; j++) {
    rowsum[j] = zero;
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i][j] = zero;
  }

  load(0);
  for (int k0 = 0; k0 < (ONE ? 1 : K); k0 += KU) {
    if (!ONE && k0 > 0) __syncthreads();
    stage(k0);
    __syncthreads();
    if (!ONE && k0 + KU < K) load(k0 + KU);
    if constexpr (FP32) {
      const char* xf_at = smem + 4 * q * PITCH + 256 * wm + 16 * r;
      const char* wf_at = smem + O::HALF + 4 * q * PITCH + 256 * wn + 16 * (4 * (r & 3) + (r >> 2));
#pragma unroll
      for (int s = 0; s < KU / 16; s++) {
        if (16 * s >= K) break;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const f32x4 xf = *(const f32x4*)(xf_at + (16 * s + e) * PITCH), wf = *(const f32x4*)(wf_at + (16 * s + e) * PITCH);
#pragma unroll
          for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i], xf[j], acc[i][j], 0, 0, 0);
          if (sums_rows)
#pragma unroll
            for (int j = 0; j < 4; j++) rowsum[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(1.f, xf[j], rowsum[j], 0, 0, 0);
        }
      }
    } else {
      typedef typename TR::vec8 frag;
      const char* at = smem + (8 * q + (r >> 2)) * PITCH + 8 * (r & 3);
      auto operand = [&](const char* from) __attribute__((always_inline)) {
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)from);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(from + 4 * PITCH));
        return __builtin_bit_cast(frag, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      };
      frag ones;
#pragma unroll
      for (int e = 0; e < 8; e++) ones[e] = (T)1.f;
#pragma unroll
      for (int s = 0; s < 2; s++) {
        if (s == 1 && K - k0 <= 32) break;
        frag xf[4], wf[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          wf[i] = operand(at + O::HALF + 32 * s * PITCH + 128 * wn + 32 * i);
          xf[i] = operand(at + 32 * s * PITCH + 128 * wm + 32 * i);
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int j = 0; j < 4; j++) acc[i][j] = TR::mfma16(wf[i], xf[j], acc[i][j]);
        if (sums_rows)
#pragma unroll
          for (int j = 0; j < 4; j++) rowsum[j] = TR::mfma16(ones, xf[j], rowsum[j]);
      }
    }
  }

  // every row of the product with ones is the same
  if (sums_rows && lane < 16)
#pragma unroll
    for (int j = 0; j < 4; j++) store_from_float((T*)a.rowsum + m0 + 64 * wm + (FP32 ? 4 * r + j : 16 * j + r), rowsum[j][0]);

  if (a.bias) {
    const T* bias = (const T*)a.bias + n0 + 64 * wn;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float b = load_as_float(bias + (FP32 ? 16 * e + 4 * q + i : 16 * i + 4 * q + e));
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j][e] += b;
      }
  }

  T* out = (T*)a.out + m0 * a.ldo + n0;
  if constexpr (FP32) {
    typedef float loose4 __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int e = 0; e < 4; e++)
        *(loose4*)(out + (64 * wm + 4 * r + j) * a.ldo + 64 * wn + 16 * e + 4 * q) = f32x4{acc[0][j][e], acc[1][j][e], acc[2][j][e], acc[3][j][e]};
  } else {
    typedef T out4 __attribute__((ext_vector_type(4)));
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        *(out4*)(smem + (64 * wm + 16 * j + r) * PITCH + 128 * wn + 32 * i + 8 * q) = __builtin_convertvector(acc[i][j], out4);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTile / O::RPI; i++) {
      const int m = O::RPI * i + row;
      *(loose16*)((char*)(out + m * a.ldo) + 16 * chunk) = *(const u32x4*)(smem + m * PITCH + 16 * chunk);
    }
  }
}

template <typename TR>
int launch(const LinArgs& a, hipStream_t stream) {
  const long long tiles = ((a.M + kTile - 1) / kTile) * ((a.N + kTile - 1) / kTile);
  if (tiles > 0x3fffffffLL) return TTSDPA_ERR_SHAPE;
  const dim3 grid((unsigned)((tiles + 7) / 8 * 8));
  if (Outer<TR>::FP32 || a.K <= Outer<TR>::KU) hipLaunchKernelGGL((linear_outer_kernel<TR, true>), grid, dim3(kThreads), 0, stream, a);
  else hipLaunchKernelGGL((linear_outer_kernel<TR, Outer<TR>::FP32>), grid, dim3(kThreads), 0, stream, a);
  return (int)hipGetLastError();
}

}  // namespace

bool outer_takes(const LinArgs& a, int dtype) {
  return a.xt && a.wt && a.M >= kTile && a.N >= kTile && a.K >= 1 && a.K <= (dtype == TTSDPA_F32 ? 32 : 256);
}

// A launch, the result written at 5.3 TB/s (fp32 4.5), and a tile's further units (fp32: its products) in each round of the CUs.
double outer_cost(const LinArgs& a, int dtype) {
  const double tiles = (double)((a.M + kTile - 1) / kTile) * (double)((a.N + kTile - 1) / kTile), rounds = tiles > 256 ? tiles / 256 : 1;
  if (dtype == TTSDPA_F32) return 5 + (double)a.M * (double)a.N * 4 / 4.5e6 + 2 * rounds;
  return 3 + (double)a.M * (double)a.N * 2 / 5.3e6 + 0.8 * rounds * (double)((a.K - 1) / 64);
}

int launch_outer(const LinArgs& a, int dtype, hipStream_t stream) {
  switch (dtype) {
    case TTSDPA_F32: return launch<F32>(a, stream);
    case TTSDPA_F16: return launch<F16>(a, stream);
    default: return launch<BF16>(a, stream);
  }
}

}  // namespace ttsdpa
