// The linear layer y = x . w^T + bias on gfx950 (reference: op::matmul(input, weight, false, true, bias) behind
// function::linear, src/Function/FuncNNLayer.h:14-19; device GEMM src/Operation/OpLinalgCuda.cuh:239-293).
//
// linear_mfma_kernel (fp16 / bf16 on v_mfma_f32_32x32x16, fp32 on v_mfma_f32_32x32x2 with full fp32 products): a workgroup of 8
// wavefronts owns a 256 x 256 tile of the output and walks K in steps of 128 bytes (64 or 32 elements).  Both operands have K
// contiguous ("NT"), which is the layout v_mfma_f32_32x32x16 wants for both inputs: a lane supplies 8 consecutive k of one row, so
// operand fragments are plain 16-byte LDS reads, no transposes.
//   global -> LDS   global_load_lds_dwordx4, two (or four) stages, of 64 KB for this tile (x tile 256 x 64, w tile 256 x 64); the 16-byte chunks
//                   of a 128-byte LDS row are XOR-swizzled with half the row number so that the 32 rows a fragment read
//                   touches spread over the banks; the loads for tile t+2 are requested while tile t's last k-step
//                   runs, one barrier per tile
//   MFMA            the wavefront's 64 (n) x 128 (m) part is computed transposed, A = w rows, B = x rows, so that an
//                   accumulator register group holds 4 consecutive n of one m: the output is stored as 8-byte pieces
//                   along its contiguous axis without a transpose
//   accumulators    start from the bias (the reference writes the bias into C and accumulates onto it), fp32
// Workgroups are numbered so that the 32 that run together on one XCD (workgroup i runs on XCD i % 8) form a 4 x 8
// block of tiles: they share their x and w panels through that XCD's L2 (tile_of_block).
//
// linear_general_kernel: any element type and shape, fp32 arithmetic on the vector ALUs (64 x 64 tiles); what neither this
// file's matrix-core kernels nor the streaming one (linear_stream.hip) take.

#include <type_traits>
#include "../../include/ttlinear.h"
#include "linear_args.h"

namespace ttsdpa {
namespace {

typedef __attribute__((address_space(3))) void lds_void_t;

typedef uint32_t loose16 __attribute__((ext_vector_type(4), aligned(2)));  // 16 bytes at any element's address

constexpr int ROWB = 128;  // bytes of an LDS row: 64 k of a 16-bit type, 32 k of fp32

// What the kernel needs to know about the element type.  A fragment is the 16 bytes a lane reads per 32 x 32 block and
// k-step: 8 consecutive k (16-bit: one v_mfma_f32_32x32x16) or 4 (fp32: four v_mfma_f32_32x32x2, MFMA e contracting the
// lanes' e-th elements — lanes 0-31 hold k .. k+3, lanes 32-63 k+4 .. k+7, the same pairing for both operands).
template <typename TR>
struct Gemm {
  typedef typename TR::elem elem;
  typedef typename TR::vec8 frag;
  typedef typename TR::vec4 out4;
  static constexpr int KPC = 8;  // elements per 16-byte chunk
  static __device__ __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) { return TR::mfma32(a, b, c); }
  static __device__ __forceinline__ out4 cvt(f32x4 v) { return __builtin_convertvector(v, out4); }
};
// The tile of this workgroup.  Tiles are numbered down strips of four tile rows, column by column, and each XCD takes an
// eighth of that sequence: every XCD has as many tiles, and any 32 in a row are a 4 x 8 block.  (Whole 4 x 8 blocks dealt to
// the XCDs in turn gave one of them twice the work where there were nine: 1501 x 2501 x 1999 fp32, 240 tiles, 260 -> 156 us.)
template <int TM, int TN>
__device__ __forceinline__ bool tile_of_block(const LinArgs& a, int slot, int* tm, int* tn) {
  const int tiles_m = (int)((a.M + TM - 1) / TM), tiles_n = (int)((a.N + TN - 1) / TN);
  const int tiles = tiles_m * tiles_n, per = (tiles + 7) / 8;
  const int at = (int)(blockIdx.x & 7) * per + slot;
  if (slot >= per || at >= tiles) return false;
  const int strip = at / (4 * tiles_n), rest = at - strip * 4 * tiles_n;
  const int high = tiles_m - 4 * strip < 4 ? tiles_m - 4 * strip : 4;
  *tm = 4 * strip + rest % high;
  *tn = rest / high;
  return true;
}

template <int N>
__device__ __forceinline__ void wait_loads() {
  static_assert(N == 0 || N == 4 || N == 8 || N == 12 || N == 16, "add the matching wait");
  if constexpr (N == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if constexpr (N == 4) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
  if constexpr (N == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  if constexpr (N == 12) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
  if constexpr (N == 16) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
}

struct F32 {};
template <>
struct Gemm<F32> {
  typedef float elem;
  typedef f32x4 frag;
  typedef f32x4 out4;
  static constexpr int KPC = 4;
  static __device__ __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) {
#pragma unroll
    for (int e = 0; e < 4; e++) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
    return c;
  }
  static __device__ __forceinline__ out4 cvt(f32x4 v) { return v; }
};

// TM x TN: the workgroup's output tile, 256 x 256 (two stages of 64 KB) or 128 x 128 for problems with too few large
// tiles to fill the chip.
// WN x WM wavefronts share the tile: a wavefront's part is (TN/WN n) x (TM/WM m).
// ST: k-tiles in LDS.  Four (128 KB) where a CU has one 128 x 128 tile anyway: with two, each tile's loads were requested one tile's
// work ahead and their latency was waited for; with several workgroups on a CU one computes while another waits.
template <typename TR, int TM, int TN, int WN, int WM, int ST>
__global__ __launch_bounds__(WN * WM * 64, 1) void linear_mfma_kernel(LinArgs a) {
  constexpr int NW = WN * WM;
  constexpr int XTILE = TM * ROWB;
  constexpr int STAGE = (TM + TN) * ROWB;
  constexpr int XI = TM / NW / 8, WI = TN / NW / 8;  // load instructions per wavefront and tile
  constexpr int NI = TN / WN / 32, MJ = TM / WM / 32;  // 32 x 32 blocks of a wavefront's part
  typedef Gemm<TR> G;
  typedef typename G::elem T;
  typedef typename G::frag vec8;  // the 16-byte operand fragment
  constexpr int BK = (ROWB / 16) * G::KPC;  // k per tile
  constexpr int ESZ = 16 / G::KPC;
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane & 31, lh = lane >> 5;

  int tm, tn, split = 0, slot = blockIdx.x >> 3, step0 = 0, ntk = (int)(a.K / BK);
  if (TM == 128 && TN == 128 && a.part) {  // the contraction is divided: all tiles of the first share of it, of the second, ...
    const int per = (((int)a.M + TM - 1) / TM * (((int)a.N + TN - 1) / TN) + 7) / 8;
    split = slot / per, slot %= per;
    step0 = ntk * split / a.splits;  // (few steps and shares: launch_packed)
    ntk = ntk * (split + 1) / a.splits - step0;
  }
  if (!tile_of_block<TM, TN>(a, slot, &tm, &tn)) return;
  const long long m0 = (long long)tm * TM, n0 = (long long)tn * TN;

  // ---- global -> LDS: wavefront w moves rows (TM/8)w .. of the x tile and (TN/8)w .. of the w tile, 8 rows (1 KB) per instruction
  // lane l fills (row l/8, chunk slot l%8) and therefore fetches chunk (l%8) ^ ((row / 2) % 8) — two rows share 256
  // bytes of LDS, so 16 consecutive rows of one logical chunk land in 16 different bank groups; rows past the end of the
  // matrix re-read its last row (their products land in outputs that are not stored)
  // The byte offset of a lane's chunk is recomputed per request (a handful of vector-ALU operations against the 2048+
  // MFMA cycles of a tile) rather than held in registers for every row group.
  const long long mlim = a.M - 1 - m0, nlim = a.N - 1 - n0;  // last valid row of the tiles
  auto lane_off = [&](int row, long long lim, long long ld) __attribute__((always_inline)) {
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    const long long r = row < lim ? row : lim;
    return (unsigned)((r * ld + G::KPC * chunk) * ESZ);
  };
  const char* xbase = (const char*)((const T*)a.x + (long long)blockIdx.y * a.bsx + m0 * a.ldx) + (long long)step0 * ROWB;
  const char* wbase = (const char*)((const T*)a.w + (long long)blockIdx.y * a.bsw + n0 * a.ldw) + (long long)step0 * ROWB;
  const unsigned smem_addr = (unsigned)(unsigned long)(lds_void_t*)smem;
  // issued as asm so that the compiler does not treat it as an LDS store it must order every later LDS read behind
  // (the lane's full address goes in a register pair: a scalar base operand is not always kept in scalar registers by
  // the compiler once the tile requests are unrolled)
  auto dma_issue = [&](const char* sbase, unsigned voff, unsigned lds_addr) __attribute__((always_inline)) {
    const char* p = sbase + voff;
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(p), "s"(lds_addr) : "memory", "m0");
  };
  auto dma_tile = [&](int t, int stage) __attribute__((always_inline)) {
    const char* xs = xbase + (long long)t * ROWB;
    const char* ws = wbase + (long long)t * ROWB;
    const unsigned dst = smem_addr + stage * STAGE;
#pragma unroll
    for (int i = 0; i < XI; i++) {
      const int row = (TM / NW) * wave + 8 * i + (lane >> 3);
      dma_issue(xs, lane_off(row, mlim, a.ldx), dst + ((TM / NW) * wave + 8 * i) * ROWB);
    }
#pragma unroll
    for (int i = 0; i < WI; i++) {
      const int row = (TN / NW) * wave + 8 * i + (lane >> 3);
      dma_issue(ws, lane_off(row, nlim, a.ldw), dst + XTILE + ((TN / NW) * wave + 8 * i) * ROWB);
    }
  };

  // ---- this wavefront's part: n rows (TN/4)*wn .. of the w tile (A operand), m rows (TM/2)*wm .. of the x tile (B) ---------
  const int wn = wave % WN, wm = wave / WN;
  // fragment (block, ks): row 32*block + lq, chunk 2*ks + lh at row*128 + 16 * (chunk ^ ((row/2) % 8)); (row/2) % 8 == (lq/2) % 8
  const unsigned frag = (unsigned)(lq * ROWB + 16 * (lh ^ ((lq >> 1) & 7)));
  const unsigned wfrag = XTILE + ((TN / WN) * wn) * ROWB + frag;
  const unsigned xfrag = ((TM / WM) * wm) * ROWB + frag;

  f32x16 acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const long long n = n0 + (TN / WN) * wn + 32 * i + 8 * (r >> 2) + 4 * lh + (r & 3);
      const float b = (a.bias && !a.part && n < a.N) ? (float)((const T*)a.bias)[n] : 0.f;
#pragma unroll
      for (int j = 0; j < MJ; j++) acc[i][j][r] = b;
    }

  // Operand fragments are double-buffered in registers: while the MFMAs of k-step ks run, the fragments of ks+1 are
  // on their way from LDS.  The one barrier per tile sits before the MFMAs of a tile's last k-step: by then every
  // wavefront has taken its last fragment of tile t (its stage may be overwritten: tile t+2 is requested) and its own
  // loads of tile t+1 have landed (requested a tile earlier), so right after the barrier the first fragments of tile
  // t+1 are requested and arrive while the last 8 MFMAs of tile t run.
  vec8 fw[2][NI], fx[2][MJ];
  auto load_frag = [&](int buf, const char* st, int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NI; i++) fw[buf][i] = *(const vec8*)(st + ((wfrag + 32 * i * ROWB) ^ (unsigned)(32 * ks)));
#pragma unroll
    for (int j = 0; j < MJ; j++) fx[buf][j] = *(const vec8*)(st + ((xfrag + 32 * j * ROWB) ^ (unsigned)(32 * ks)));
  };
  auto mma = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
      for (int j = 0; j < MJ; j++) acc[i][j] = G::mma(fw[buf][i], fx[buf][j], acc[i][j]);
  };

  // Past the last tile it is requested again, into stages that nothing reads any more: the number of loads in flight behind
  // every wait is the same.
  if (ntk > 0) {
#pragma unroll
    for (int t = 0; t < ST; t++) dma_tile(t < ntk ? t : ntk - 1, t);
    wait_loads<(ST - 1) * (XI + WI)>();  // tile 0's
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    load_frag(0, smem, 0);
  }
  for (int t = 0; t < ntk; t++) {
    const char* st = smem + (t % ST) * STAGE;
    load_frag(1, st, 1);
    mma(0);
    __builtin_amdgcn_sched_barrier(0);
    load_frag(0, st, 2);
    mma(1);
    __builtin_amdgcn_sched_barrier(0);
    load_frag(1, st, 3);
    mma(0);
    __builtin_amdgcn_sched_barrier(0);
    wait_loads<(ST - 2) * (XI + WI)>();  // tile t+1's
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    dma_tile(t + ST < ntk ? t + ST : ntk - 1, t % ST);
    if (t + 1 < ntk) load_frag(0, smem + ((t + 1) % ST) * STAGE, 0);
    mma(1);
    __builtin_amdgcn_sched_barrier(0);
  }
  wait_loads<0>();  // none may write LDS that has passed to another workgroup

  if constexpr (TM == 128 && TN == 128) {
    // The tile leaves through LDS as whole rows, 16 bytes at any alignment a lane (four elements of a row each, as the
    // accumulators lie, took 56 us for a 4095 x 4095 x 64 product's rows of odd length, 25 so): 16-byte chunk c of row r at slot c ^ (r % chunks).
    constexpr int CH = TN * ESZ / 16;  // chunks of a row
    __builtin_amdgcn_s_barrier();      // every wavefront has taken its last operands
    if (a.part) {  // fp32 sums of this share of the contraction, rows of 512 bytes
#pragma unroll
      for (int j = 0; j < MJ; j++) {
        const int row = (TM / WM) * wm + 32 * j + lq;
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
          for (int rg = 0; rg < 4; rg++) {
            const int c = (TN / WN) / 4 * wn + 8 * i + 2 * rg + lh;
            f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = acc[i][j][4 * rg + e];
            *(f32x4*)(smem + row * TN * 4 + 16 * (c ^ (row & 31))) = v;
          }
      }
      __syncthreads();
      float* part = a.part + split * (a.M * a.N + a.M);
#pragma unroll
      for (int it = 0; it < TM * 32 / (NW * 64); it++) {
        const int row = NW * 2 * it + tid / 32, c = tid % 32;
        const u32x4 v = *(const u32x4*)(smem + row * TN * 4 + 16 * (c ^ (row & 31)));
        const long long m = m0 + row, n = n0 + 4 * c;
        if (m >= a.M) continue;
        float* dst = part + m * a.N + n;
        if (n + 4 <= a.N) {
          *(loose16*)dst = v;
        } else {
          const f32x4 o = __builtin_bit_cast(f32x4, v);
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (n + e < a.N) dst[e] = o[e];
        }
      }
      return;
    }
#pragma unroll
    for (int j = 0; j < MJ; j++) {
      const int row = (TM / WM) * wm + 32 * j + lq;
#pragma unroll
      for (int i = 0; i < NI; i++)
#pragma unroll
        for (int rg = 0; rg < 4; rg++) {
          const int col = (TN / WN) * wn + 32 * i + 8 * rg + 4 * lh;
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = acc[i][j][4 * rg + e];
          *(typename G::out4*)(smem + row * TN * ESZ + 16 * ((col / G::KPC) ^ (row & (CH - 1))) + (col % G::KPC) * ESZ) = G::cvt(v);
        }
    }
    __syncthreads();
    constexpr int PER = NW * 64 / CH;  // rows at a time
#pragma unroll
    for (int it = 0; it < TM / PER; it++) {
      const int row = PER * it + tid / CH, c = tid % CH;
      const u32x4 v = *(const u32x4*)(smem + row * TN * ESZ + 16 * (c ^ (row & (CH - 1))));
      const long long m = m0 + row, n = n0 + c * G::KPC;
      if (m >= a.M) continue;
      T* dst = (T*)a.out + (long long)blockIdx.y * a.bso + m * a.ldo + n;
      if (n + G::KPC <= a.N) {
        *(loose16*)dst = v;
      } else {
        const vec8 o = __builtin_bit_cast(vec8, v);
#pragma unroll
        for (int e = 0; e < G::KPC; e++)
          if (n + e < a.N) dst[e] = o[e];
      }
    }
    return;
  }

  // ---- store: register group rg of acc[i][j] is out[m = .. + 32j + lq][n = .. + 32i + 8rg + 4lh .. +3] ----------------------
  const bool whole = ((a.N | a.ldo) & 3) == 0 && ((uintptr_t)a.out & (4 * ESZ - 1)) == 0;
#pragma unroll
  for (int j = 0; j < MJ; j++) {
    const long long m = m0 + (TM / WM) * wm + 32 * j + lq;
    if (m >= a.M) continue;
    T* orow = (T*)a.out + (long long)blockIdx.y * a.bso + m * a.ldo;
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        const long long n = n0 + (TN / WN) * wn + 32 * i + 8 * rg + 4 * lh;
        if (n < a.N) {
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = acc[i][j][4 * rg + e];
          const typename G::out4 o = G::cvt(v);
          if (whole) {
            *(typename G::out4*)(orow + n) = o;
          } else {  // rows that do not begin at, or end with, groups of four
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (n + e < a.N) orow[n + e] = o[e];
          }
        }
      }
  }
}

// ---- 16-bit tensors with an operand stored contraction-major (op::matmul's other transpose flags) -------------------------
// out[m][n] = sum_k x(m,k) w(n,k) + bias[n] with x(m,k) = XT ? x[k*ldx + m] : x[m*ldx + k] and w(n,k) = WT ? w[k*ldw + n] :
// w[n*ldw + k]: the operands of op::matmul(a, b, transA, transB) as they lie in memory (reference
// src/Operation/OpLinalg.cpp:107-150 hands its flags to the GEMM; no transposed copy is made here either).
// Same tiles, workgroup order, stages and pipeline as linear_mfma_kernel.  What differs is the tile of a contraction-major
// operand and how fragments are read:
//  * such a tile is 64 k-rows of its 128 or 256 columns, kept as sub-tiles of 128 columns (64 rows x 256 bytes, the
//    layout of the attention kernels' V tile: 16-byte chunk c of row r at slot c ^ f(r), f(r) = (r%4)*4 + (r/4)%4), and a
//    fragment of it comes through the LDS transpose load: two ds_read_b64_tr_b16 give a lane the k values
//    {4h..4h+3} and {8+4h..8+4h+3} of a 16-k step for its row (h = lane/32);
//  * the contraction index has to be permuted identically on both sides, so a row-major operand's fragment is read in
//    the same order, as two 8-byte pieces (chunks 2ks and 2ks+1 of the k-step, bytes 8h..8h+7 of each).
namespace lint {
__device__ __forceinline__ int swz(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
}  // namespace lint

template <typename TR, int TM, int TN, bool XT, bool WT>
__global__ __launch_bounds__(512, 1) void linear_mfma_t_kernel(LinArgs a) {
  static_assert(XT || WT, "both operands row-major: linear_mfma_kernel");
  constexpr int WN = 4, WM = 2, NW = 8;
  constexpr int XTILE = TM * ROWB, STAGE = (TM + TN) * ROWB;  // bytes: 64 k of 2 bytes per row or column, either layout
  constexpr int XI = TM / NW / 8, WI = TN / NW / 8;           // load instructions per wavefront and tile, either layout
  constexpr int NI = TN / WN / 32, MJ = TM / WM / 32;
  constexpr int BK = 64, SUB = 64 * 256;                      // k per tile; bytes of a 128-column sub-tile
  typedef typename TR::elem T;
  typedef typename TR::vec8 vec8;
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane & 31, lh = lane >> 5;

  int tm, tn;
  if (!tile_of_block<TM, TN>(a, blockIdx.x >> 3, &tm, &tn)) return;
  const long long m0 = (long long)tm * TM, n0 = (long long)tn * TN;

  // ---- global -> LDS -------------------------------------------------------------------------------------------------------
  // row-major operand: wavefront w moves rows (T/8)w .. of the tile, 8 rows (1 KB) per instruction, lane l fills (row l/8,
  // chunk slot l%8) with chunk (l%8) ^ ((row/2) % 8); rows past the end re-read the last row.
  // contraction-major operand: wavefront w moves k-rows 8w .. 8w+7 of every 128-column sub-tile, 4 rows (1 KB) per
  // instruction, lane l fills (row l/16, chunk slot l%16) with chunk (l%16) ^ f(row); columns past the end re-read the
  // last 8 valid ones (their products land in outputs that are not stored).
  const long long mlim = a.M - 1 - m0, nlim = a.N - 1 - n0;
  auto rm_off = [&](int row, long long lim, long long ld) __attribute__((always_inline)) {
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    const long long r = row < lim ? row : lim;
    return (unsigned)((r * ld + 8 * chunk) * 2);
  };
  auto km_off = [&](int row, int sub, long long cols_left, long long ld) __attribute__((always_inline)) {  // cols_left: valid columns from the tile's first
    const int chunk = (lane & 15) ^ lint::swz(row);
    long long col = 128 * sub + 8 * chunk;
    col = col + 8 <= cols_left ? col : cols_left - 8;
    return (unsigned)(((long long)row * ld + col) * 2);
  };
  const T* xb = (const T*)a.x + (long long)blockIdx.y * a.bsx;
  const T* wb = (const T*)a.w + (long long)blockIdx.y * a.bsw;
  const char* xbase = (const char*)(XT ? xb + m0 : xb + m0 * a.ldx);
  const char* wbase = (const char*)(WT ? wb + n0 : wb + n0 * a.ldw);
  const unsigned smem_addr = (unsigned)(unsigned long)(lds_void_t*)smem;
  auto dma_issue = [&](const char* sbase, unsigned voff, unsigned lds_addr) __attribute__((always_inline)) {
    const char* p = sbase + voff;
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(p), "s"(lds_addr) : "memory", "m0");
  };
  auto dma_operand = [&](bool km, const char* base, long long ld, long long lim, int T_, int NINSTR, long long t, unsigned dst) __attribute__((always_inline)) {
    if (km) {
      const char* src = base + t * BK * ld * 2;  // 64 k-rows further
#pragma unroll
      for (int i = 0; i < NINSTR; i++) {
        const int sub = i >> 1, row = 8 * wave + 4 * (i & 1) + (lane >> 4);
        dma_issue(src, km_off(row, sub, lim + 1, ld), dst + sub * SUB + (8 * wave + 4 * (i & 1)) * 256);
      }
    } else {
      const char* src = base + t * ROWB;
#pragma unroll
      for (int i = 0; i < NINSTR; i++) {
        const int row = (T_ / NW) * wave + 8 * i + (lane >> 3);
        dma_issue(src, rm_off(row, lim, ld), dst + ((T_ / NW) * wave + 8 * i) * ROWB);
      }
    }
  };
  auto dma_tile = [&](int t, int stage) __attribute__((always_inline)) {
    const unsigned dst = smem_addr + stage * STAGE;
    dma_operand(XT, xbase, a.ldx, mlim, TM, XI, t, dst);
    dma_operand(WT, wbase, a.ldw, nlim, TN, WI, t, dst + XTILE);
  };

  // ---- fragments ---------------------------------------------------------------------------------------------------------------
  const int wn = wave % WN, wm = wave / WN;
  // row-major: (block, ks, piece p): row 32*block + lq, bytes 8lh .. 8lh+7 of chunk 2ks + p
  const unsigned rm_base = (unsigned)(lq * ROWB + 8 * lh + 16 * ((lq >> 1) & 7));
  // contraction-major: piece ld of k-step ks for the 32 columns 32*db .. of a sub-tile (see sdpa_prefill_d128.hip, V operand)
  unsigned km_base[2];
  {
    const int s = lane & 15, dhalf = (lane >> 4) & 1;
#pragma unroll
    for (int ld = 0; ld < 2; ld++) {
      const int row = 8 * ld + 4 * lh + (s >> 2);
      const int chunk = 2 * dhalf + ((s & 3) >> 1);
      km_base[ld] = (unsigned)(row * 256 + 16 * (chunk ^ lint::swz(row)) + 8 * (s & 1));
    }
  }
  // fragment of the 32 rows / columns starting at `first` of an operand's tile at `region`, k-step ks
  auto frag_of = [&](bool km, const char* region, int first, int ks) __attribute__((always_inline)) {
    if (km) {
      const char* sub = region + (first >> 7) * SUB + 16 * ks * 256;
      const unsigned db = (unsigned)((first & 127) >> 5);
      const lint::s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lint::lds_s16x4*)(sub + (km_base[0] ^ (64u * db))));
      const lint::s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lint::lds_s16x4*)(sub + (km_base[1] ^ (64u * db))));
      return __builtin_bit_cast(vec8, (lint::s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      const char* rows = region + first * ROWB;
      const lint::s16x4 lo = *(const lint::s16x4*)(rows + (rm_base ^ (unsigned)(32 * ks)));
      const lint::s16x4 hi = *(const lint::s16x4*)(rows + (rm_base ^ (unsigned)(32 * ks + 16)));
      return __builtin_bit_cast(vec8, (lint::s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };

  f32x16 acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const long long n = n0 + (TN / WN) * wn + 32 * i + 8 * (r >> 2) + 4 * lh + (r & 3);
      const float b = (a.bias && n < a.N) ? (float)((const T*)a.bias)[n] : 0.f;
#pragma unroll
      for (int j = 0; j < MJ; j++) acc[i][j][r] = b;
    }

  vec8 fw[2][NI], fx[2][MJ];
  auto load_frag = [&](int buf, const char* st, int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NI; i++) fw[buf][i] = frag_of(WT, st + XTILE, (TN / WN) * wn + 32 * i, ks);
#pragma unroll
    for (int j = 0; j < MJ; j++) fx[buf][j] = frag_of(XT, st, (TM / WM) * wm + 32 * j, ks);
  };
  auto mma = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
      for (int j = 0; j < MJ; j++) acc[i][j] = TR::mfma32(fw[buf][i], fx[buf][j], acc[i][j]);
  };

  // the pipeline of linear_mfma_kernel: fragments double-buffered in registers, one barrier per tile before its last k-step
  const int ntk = (int)(a.K / BK);
  if (ntk > 0) {
    dma_tile(0, 0);
    if (ntk > 1) {
      dma_tile(1, 1);
      if constexpr (XI + WI == 8) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      static_assert(XI + WI == 8 || XI + WI == 4, "add the matching wait");
    } else {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    load_frag(0, smem, 0);
  }
  for (int t = 0; t < ntk; t++) {
    const char* st = smem + (t & 1) * STAGE;
    load_frag(1, st, 1);
    mma(0);
    __builtin_amdgcn_sched_barrier(0);
    load_frag(0, st, 2);
    mma(1);
    __builtin_amdgcn_sched_barrier(0);
    load_frag(1, st, 3);
    mma(0);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + 2 < ntk) dma_tile(t + 2, t & 1);
    if (t + 1 < ntk) load_frag(0, smem + ((t + 1) & 1) * STAGE, 0);
    mma(1);
    __builtin_amdgcn_sched_barrier(0);
  }

  // store: register group rg of acc[i][j] is out[m = .. + 32j + lq][n = .. + 32i + 8rg + 4lh .. +3]
#pragma unroll
  for (int j = 0; j < MJ; j++) {
    const long long m = m0 + (TM / WM) * wm + 32 * j + lq;
    if (m >= a.M) continue;
    T* orow = (T*)a.out + (long long)blockIdx.y * a.bso + m * a.ldo;
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        const long long n = n0 + (TN / WN) * wn + 32 * i + 8 * rg + 4 * lh;
        if (n < a.N) {  // N is a multiple of 4 on this route
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; e++) v[e] = acc[i][j][4 * rg + e];
          *(typename TR::vec4*)(orow + n) = __builtin_convertvector(v, typename TR::vec4);
        }
      }
  }
}

// ---- 16-bit tensors, 256 x 256 tiles: four wavefronts with 128 x 128 each and the tile's arithmetic as one hand-ordered stream
// Same tiles, LDS layout and direct loads as linear_mfma_kernel<TR, 256, 256>; what differs is who owns what, the matrix
// instruction and who orders the instructions.  The clock of these kernels is power-managed, so what a tile costs is
// energy rather than issue slots:
//  * a wavefront owns 128 x 128 of the tile (256 accumulator registers, in AGPRs: one wavefront per SIMD), so an operand
//    read from LDS feeds eight matrix instructions — LDS operand traffic is the second consumer after the matrix pipe;
//  * v_mfma_f32_16x16x32 instead of 32x32x16: with random operands the chip sustains 2.10 against 1.84 PFLOP/s of them;
//  * the body of a tile (accumulators from the bias, K loop, conversion into LDS) is a single asm statement
//    (linear256_loop.inc, written by gen_linear256_loop.py): the compiler's version of the loop requested the operands
//    of a k-step in one burst behind the matrix instructions and waited for them before the next, and put the tile
//    loads and the next operands between the barrier and the matrix instructions behind it;
//  * the output leaves through LDS as whole lines: written 8 bytes at a time the tile's stores took 16 % of the kernel
//    (every instruction touched 32 rows, 16 bytes each; the L2 takes a request per piece).
#include "linear256_loop.inc"
#include "linear128_loop.inc"

typedef unsigned u32x8 __attribute__((ext_vector_type(8)));

// The bodies: of a TM x 256 tile.  lds_x, lds_w: where the wavefront's first x and w row of stage 0 goes; left: k-tiles; adv: of
// them, those behind the ones that xp and wp (the next to be loaded) point to.
template <typename TR, int TM>
struct Lin256Body;
template <>
struct Lin256Body<BF16, 256> {
  static __device__ __forceinline__ void run(f32x16 bias_lo, f32x16 bias_hi, u32x8 xoff, u32x8 woff, u32x4 raddr, u32x8 eaddr,
                                             unsigned long long xp, unsigned long long wp, unsigned lds_x, unsigned lds_w, unsigned left, unsigned adv) {
    (void)lds_w;
    const unsigned m0base = lds_x;
#define TT_LIN256_TEXT TT_LIN256_BODY_BF16
#include "linear256_stmt.inc"
#undef TT_LIN256_TEXT
  }
};
template <>
struct Lin256Body<F16, 256> {
  static __device__ __forceinline__ void run(f32x16 bias_lo, f32x16 bias_hi, u32x8 xoff, u32x8 woff, u32x4 raddr, u32x8 eaddr,
                                             unsigned long long xp, unsigned long long wp, unsigned lds_x, unsigned lds_w, unsigned left, unsigned adv) {
    (void)lds_w;
    const unsigned m0base = lds_x;
#define TT_LIN256_TEXT TT_LIN256_BODY_F16
#include "linear256_stmt.inc"
#undef TT_LIN256_TEXT
  }
};
#define TT_LIN128_RUN(TXT)                                                                                              \
  u32x4 raddr_out;                                                                                                      \
  unsigned long long xp_out, wp_out;                                                                                    \
  unsigned left_out, adv_out;                                                                                           \
  const u32x4 xoff4 = {xoff[0], xoff[1], xoff[2], xoff[3]};                                                             \
  asm volatile(TXT                                                                                                      \
               : "={v[56:59]}"(raddr_out), "={s[40:41]}"(xp_out), "={s[42:43]}"(wp_out), "={s45}"(left_out), "={s46}"(adv_out) \
               : "0"(raddr), "1"(xp), "2"(wp), "3"(left), "4"(adv), "{s44}"(lds_x), "{s51}"(lds_w), "{v[60:63]}"(raddr),  \
                 "{v[64:67]}"(xoff4), "{v[72:79]}"(woff), "{v[80:87]}"(eaddr), "{v[96:111]}"(bias_lo), "{v[112:127]}"(bias_hi) \
               : TT_LIN128_CLOBBERS)
template <>
struct Lin256Body<BF16, 128> {
  static __device__ __forceinline__ void run(f32x16 bias_lo, f32x16 bias_hi, u32x8 xoff, u32x8 woff, u32x4 raddr, u32x8 eaddr,
                                             unsigned long long xp, unsigned long long wp, unsigned lds_x, unsigned lds_w, unsigned left, unsigned adv) {
    TT_LIN128_RUN(TT_LIN128_BODY_BF16);
  }
};
template <>
struct Lin256Body<F16, 128> {
  static __device__ __forceinline__ void run(f32x16 bias_lo, f32x16 bias_hi, u32x8 xoff, u32x8 woff, u32x4 raddr, u32x8 eaddr,
                                             unsigned long long xp, unsigned long long wp, unsigned lds_x, unsigned lds_w, unsigned left, unsigned adv) {
    TT_LIN128_RUN(TT_LIN128_BODY_F16);
  }
};

template <int TM>
constexpr int kLin256Lds = (TM == 256 ? 2 : 3) * (TM + 256) * ROWB;

// The tile of TM x 256 outputs from (m0, n0) on.  TM: 256, or 128 where the large tiles leave CUs idle (three stages of half the size
// less: the body's comment).
template <typename TR, int TM>
__device__ __forceinline__ void linear256_tile(const LinArgs& a, long long m0, long long n0) {
  constexpr int TN = 256, ST = TM == 256 ? 2 : 3;  // stages
  constexpr int XI = TM / 32;                       // x load instructions of a wavefront and k-tile (w: 8)
  constexpr int XTILE = TM * ROWB;
  constexpr int STAGE = (TM + TN) * ROWB;
  typedef typename TR::elem T;
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;

  // global -> LDS: wavefront v moves rows 64v .. 64v+63 of both tiles (a quarter of the x tile), 8 rows (1 KB) per instruction; lane l fills
  // (row l/8, chunk slot l%8) and fetches chunk (l%8) ^ ((row/2) % 8); rows past the end re-read the last row
  const long long mlim = a.M - 1 - m0, nlim = a.N - 1 - n0;
  u32x8 xoff, woff;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int row = 64 * wave + 8 * i + (lane >> 3), xrow = TM / 4 * wave + 8 * (i % XI) + (lane >> 3);
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);  // (of xrow too: they differ by a multiple of 16)
    xoff[i] = (unsigned)(((xrow < mlim ? xrow : mlim) * a.ldx + 8 * chunk) * 2);
    woff[i] = (unsigned)(((row < nlim ? row : nlim) * a.ldw + 8 * chunk) * 2);
  }
  // (the 64-bit products are formed on the vector ALUs; the loads want their base in scalar registers)
  auto uniform = [](const void* p) __attribute__((always_inline)) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (const char*)(((unsigned long long)hi << 32) | lo);
  };
  const char* xbase = uniform((const T*)a.x + m0 * a.ldx);
  const char* wbase = uniform((const T*)a.w + n0 * a.ldw);
  const unsigned smem_addr = (unsigned)(unsigned long)(lds_void_t*)smem;
  auto dma_tile = [&](long long t, int stage) __attribute__((always_inline)) {
    const char* xs = xbase + t * ROWB;
    const char* ws = wbase + t * ROWB;
    const unsigned xdst = smem_addr + stage * STAGE + wave * (XI * 1024), wdst = smem_addr + stage * STAGE + XTILE + wave * 8192;
#pragma unroll
    for (int i = 0; i < XI; i++)
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(xoff[i]), "s"(xs), "s"(xdst + 1024 * i) : "memory", "m0");
#pragma unroll
    for (int i = 0; i < 8; i++)
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(woff[i]), "s"(ws), "s"(wdst + 1024 * i) : "memory", "m0");
  };

  // this wavefront's part: n rows 128*wn .. of the w tile (A operand), m rows TM/2*wm .. of the x tile (B operand);
  // operand (block, s): row 16*block + lane%16, chunk 4*s + lane/16 at row*128 + 16 * (chunk ^ ((row/2) % 8))
  const int wn = wave & 1, wm = wave >> 1;
  const unsigned frag = (unsigned)(lr * ROWB + 16 * (lg ^ ((lr >> 1) & 7)));
  u32x4 raddr;
#pragma unroll
  for (int s = 0; s < 2; s++) {
    raddr[2 * s] = smem_addr + ((TM / 2 * wm * ROWB + frag) ^ (unsigned)(64 * s));
    raddr[2 * s + 1] = smem_addr + ((128 * wn * ROWB + frag) ^ (unsigned)(64 * s));
  }
  // block (i, j) leaves the lane with out[m = .. + 16j + lane%16][n = .. + 16i + 4(lane/16) .. +3]: 8 bytes of row 16j + lane%16
  // of the wavefront's quarter of LDS (rows of 256 bytes, the 16-byte chunks of row r at slot c ^ (r % 16))
  u32x8 eaddr;
#pragma unroll
  for (int i = 0; i < 8; i++) eaddr[i] = smem_addr + wave * (TM * 128) + lr * 256 + 16 * ((2 * i + (lg >> 1)) ^ lr) + 8 * (lg & 1);
  // accumulators start from the bias (the reference writes the bias into C and accumulates onto it)
  f32x16 bias_lo, bias_hi;
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const long long n = n0 + 128 * wn + 16 * i + 4 * lg + e;
      const float b = (a.bias && n < a.N) ? (float)((const T*)a.bias)[n] : 0.f;
      if (i < 4) bias_lo[4 * i + e] = b;
      else bias_hi[4 * (i - 4) + e] = b;
    }

  const long long ntk = a.K / 64;  // > 0 on this route
#pragma unroll
  for (int t = 0; t < ST; t++) dma_tile(t < ntk ? t : ntk - 1, t);  // (the last one again where there are fewer)
  if constexpr (ST == 2) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  {
    // the loop's loads: k-tile min(t + ST, ntk - 1) while k-tile t is computed
    const long long first = ntk > ST ? ST : ntk - 1;
    Lin256Body<TR, TM>::run(bias_lo, bias_hi, xoff, woff, raddr, eaddr, (unsigned long long)(xbase + first * ROWB),
                            (unsigned long long)(wbase + first * ROWB), smem_addr + wave * (XI * 1024), smem_addr + XTILE + wave * 8192,
                            (unsigned)ntk, ntk > ST + 1 ? (unsigned)(ntk - ST - 1) : 0u);
  }

  // 16 lanes read a row of the wavefront's quarter back and store its 256 bytes (a wavefront reads only what it wrote)
  const char* mine = smem + wave * (TM * 128);
  const long long nbase = n0 + 128 * wn;
#pragma unroll 8
  for (int it = 0; it < TM / 8; it++) {
    const int row = 4 * it + (lane >> 4);
    const int c = (lane & 15) ^ (row & 15);
    const u32x4 v = *(const u32x4*)(mine + row * 256 + 16 * (lane & 15));
    const long long m = m0 + TM / 2 * wm + row, n = nbase + 8 * c;
    if (m < a.M) {
      T* dst = (T*)a.out + m * a.ldo + n;
      if (n + 8 <= a.N) {
        *(loose16*)dst = v;  // rows of any length and alignment; aligned ones take the same instruction
      } else {
        const typename TR::vec8 o = __builtin_bit_cast(typename TR::vec8, v);
#pragma unroll
        for (int e = 0; e < 8; e++)
          if (n + e < a.N) dst[e] = o[e];
      }
    }
  }
}

template <typename TR, int TM>
__global__ __launch_bounds__(256, 1) void linear256_kernel(LinArgs a) {
  int tm, tn;
  if (!tile_of_block<TM, 256>(a, blockIdx.x >> 3, &tm, &tn)) return;
  linear256_tile<TR, TM>(a, (long long)tm * TM, (long long)tn * 256);
}

// Large tiles in whole rounds of the CUs (an XCD has 32), what is left over in halves: a last round of large tiles that is half full
// or less takes nearly as long as a full one; in halves it is a full one, but of tiles half as long, and a half takes the place of a
// tile as soon as a CU is free.  Forward and both gradients, in us, without and with it: 2048 x 4096 x 9216 518, 459; 5000 x 4096 x
// 3584 475, 417; 8192 x 4096 x 6144 1025, 984 (there the weight's gradient alone is such a product: 384 tiles).
constexpr int kCusOfXcd = 32;

template <typename TR>
__global__ __launch_bounds__(256, 1) void linear256_mixed_kernel(LinArgs a, int whole /* large tiles of an XCD, the first ones */) {
  const int slot = blockIdx.x >> 3;
  int tm, tn;
  if (slot < whole) {
    if (tile_of_block<256, 256>(a, slot, &tm, &tn)) linear256_tile<TR, 256>(a, (long long)tm * 256, (long long)tn * 256);
    return;
  }
  if (!tile_of_block<256, 256>(a, whole + (slot - whole) / 2, &tm, &tn)) return;
  const long long m0 = (long long)tm * 256 + 128 * ((slot - whole) & 1);
  if (m0 < a.M) linear256_tile<TR, 128>(a, m0, (long long)tn * 256);
}

// Any element type and shape: 64 x 64 output tile per workgroup, 4 x 4 outputs per lane, K in steps of 16 through LDS.
template <typename T>
__global__ __launch_bounds__(256) void linear_general_kernel(LinArgs a) {
  __shared__ float Xs[16][64 + 1], Ws[16][64 + 1];
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const long long m0 = (long long)blockIdx.y * 64, n0 = (long long)blockIdx.x * 64;
  const T* x = (const T*)a.x + (long long)blockIdx.z * a.bsx;
  const T* w = (const T*)a.w + (long long)blockIdx.z * a.bsw;
  float acc[4][4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const long long n = n0 + 4 * tx + j;
    const float b = (a.bias && n < a.N) ? load_as_float((const T*)a.bias + n) : 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i][j] = b;
  }
  for (long long k0 = 0; k0 < a.K; k0 += 16) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int e = tid + 256 * i;
      const int row = e >> 4, kk = e & 15;
      const bool kin = k0 + kk < a.K;
      const long long xat = a.xt ? (k0 + kk) * a.ldx + m0 + row : (m0 + row) * a.ldx + k0 + kk;
      const long long wat = a.wt ? (k0 + kk) * a.ldw + n0 + row : (n0 + row) * a.ldw + k0 + kk;
      Xs[kk][row] = (kin && m0 + row < a.M) ? load_as_float(x + xat) : 0.f;
      Ws[kk][row] = (kin && n0 + row < a.N) ? load_as_float(w + wat) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; kk++) {
      float xv[4], wv[4];
#pragma unroll
      for (int i = 0; i < 4; i++) xv[i] = Xs[kk][4 * ty + i], wv[i] = Ws[kk][4 * tx + i];
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = fmaf(xv[i], wv[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const long long m = m0 + 4 * ty + i;
    if (m >= a.M) continue;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const long long n = n0 + 4 * tx + j;
      if (n < a.N) store_from_float((T*)a.out + (long long)blockIdx.z * a.bso + m * a.ldo + n, acc[i][j]);
    }
  }
}

// Operands brought into the layout of the x . w^T kernels: dst dense rows of `ldd` elements (a multiple of a k-tile), the
// elements past the operand's own zeros.  Bound by memory: 16-byte accesses on both sides whatever the source's alignment.
template <typename T>
__global__ __launch_bounds__(256) void pack_rows_kernel(const T* src, T* dst, long long R, long long C, long long ld, long long ldd) {
  constexpr int VEC = 16 / sizeof(T);
  typedef T vecT __attribute__((ext_vector_type(VEC)));
  const long long c = ((long long)blockIdx.x * 64 + (threadIdx.x & 63)) * VEC;
  if (c >= ldd) return;
  const long long r0 = (long long)blockIdx.y * 16 + (threadIdx.x >> 6);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const long long r = r0 + 4 * i;
    if (r >= R) return;
    const T* p = src + r * ld + c;
    vecT v;
    if (c + VEC <= C) {
      v = __builtin_bit_cast(vecT, (u32x4)*(const loose16*)p);
    } else {
#pragma unroll
      for (int e = 0; e < VEC; e++) v[e] = c + e < C ? p[e] : (T)0;
    }
    *(vecT*)(dst + r * ldd + c) = v;
  }
}

// dst[c, r] = src[r, c] for src [R, C] with row stride ld; dst [C, ldd].  A workgroup takes 64 columns of kPackRows rows through
// LDS in 64 x 64 tiles (pitch: two dwords more than the tile's row, so that the eight lanes that read down a column of
// eight rows each fall into different banks).  SUMS: also the fp32 sums of its rows' columns, to part[blockIdx.y][C]
// (colsum_merge_kernel adds them): the bias's gradient costs no reading of its own.  6144 x 4096 bf16: 20 us, 5.0 TB/s.
constexpr int kPackRows = 256;

template <typename T, bool SUMS>
__global__ __launch_bounds__(256) void pack_transposed_kernel(const T* src, T* dst, long long R, long long C, long long ld, long long ldd, float* part) {
  constexpr int VEC = 16 / sizeof(T);
  constexpr int PITCH = 64 + 4 / (int)sizeof(T);
  constexpr int CPR = 64 / VEC;  // 16-byte chunks per tile row
  typedef T vecT __attribute__((ext_vector_type(VEC)));
  __shared__ uint32_t tile_words[64 * PITCH * sizeof(T) / 4];
  T* tile = (T*)tile_words;
  const long long c0 = (long long)blockIdx.x * 64;
  float sums[64 * CPR / 256];
#pragma unroll
  for (int i = 0; i < 64 * CPR / 256; i++) sums[i] = 0.f;
  for (int t = 0; t < kPackRows / 64; t++) {
    const long long r0 = (long long)blockIdx.y * kPackRows + 64 * t;
    if (r0 >= ldd) break;
    if (t) __syncthreads();
#pragma unroll
    for (int i = 0; i < 64 * CPR / 256; i++) {
      const int chunk = threadIdx.x + 256 * i;
      const int row = chunk / CPR, cc = (chunk % CPR) * VEC;
      const long long r = r0 + row, c = c0 + cc;
      const T* p = src + r * ld + c;
      u32x4 v = {0, 0, 0, 0};
      if (r < R) {
        if (c + VEC <= C) {
          v = *(const loose16*)p;
        } else {
          vecT w;
#pragma unroll
          for (int e = 0; e < VEC; e++) w[e] = c + e < C ? p[e] : (T)0;
          v = __builtin_bit_cast(u32x4, w);
        }
      }
#pragma unroll
      for (int e = 0; e < 4; e++) tile_words[(row * PITCH + cc) * (int)sizeof(T) / 4 + e] = v[e];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 64 * CPR / 256; i++) {
      const int chunk = threadIdx.x + 256 * i;
      const int orow = chunk / CPR, oc = (chunk % CPR) * VEC;  // output row = source column; first of VEC source rows
      const long long c = c0 + orow, r = r0 + oc;
      vecT v;
#pragma unroll
      for (int e = 0; e < VEC; e++) v[e] = tile[(oc + e) * PITCH + orow];
      if constexpr (SUMS) {
#pragma unroll
        for (int e = 0; e < VEC; e++) sums[i] += (float)v[e];
      }
      if (c < C && r < ldd) *(vecT*)(dst + c * ldd + r) = v;
    }
  }
  if constexpr (SUMS) {
#pragma unroll
    for (int i = 0; i < 64 * CPR / 256; i++) {
      float v = sums[i];
#pragma unroll
      for (int m = 1; m < CPR; m <<= 1) v += __shfl_xor(v, m);
      const int chunk = threadIdx.x + 256 * i;
      const long long c = c0 + chunk / CPR;
      if (chunk % CPR == 0 && c < C) part[(long long)blockIdx.y * C + c] = v;
    }
  }
}

// A product's operand [rows, K] (kmajor: stored [K, rows]) to rows of kpad elements.
template <typename T>
int launch_pack(const void* src, void* dst, long long rows, long long K, long long ld, long long kpad, bool kmajor, float* part, hipStream_t stream) {
  if (kmajor) {
    const dim3 grid((unsigned)((rows + 63) / 64), (unsigned)((kpad + kPackRows - 1) / kPackRows));
    if (part)
      hipLaunchKernelGGL((pack_transposed_kernel<T, true>), grid, dim3(256), 0, stream, (const T*)src, (T*)dst, K, rows, ld, kpad, part);
    else
      hipLaunchKernelGGL((pack_transposed_kernel<T, false>), grid, dim3(256), 0, stream, (const T*)src, (T*)dst, K, rows, ld, kpad, part);
  } else {
    constexpr int VEC = 16 / (int)sizeof(T);
    const dim3 grid((unsigned)((kpad / VEC + 63) / 64), (unsigned)((rows + 15) / 16));
    hipLaunchKernelGGL((pack_rows_kernel<T>), grid, dim3(256), 0, stream, (const T*)src, (T*)dst, rows, K, ld, kpad);
  }
  return (int)hipGetLastError();
}

// Column sums out[n] = sum_m x[m][n] in fp32 (the bias's gradient; reference op::sumOnDim behind src/Function/FuncNNLayer.h:30).
// Bound by reading x: 1024 lanes take 16 (fp32: 8) columns of 16 bytes side by side and 64 rows at a time, so a column
// block of 1000 rows is some 16 loads in flight per lane and the chip is filled with row ranges (blockIdx.y), whose
// partial sums `part` [ranges][N] colsum_merge_kernel adds.  8192 x 6144 bf16: 16 + 3 us; the cast, the library
// reduction and the cast back that it replaces took 44 + 47 + 5.
template <typename T>
__global__ __launch_bounds__(1024) void colsum_kernel(const T* x, long long M, long long N, long long ld, long long rows, T* out, float* part) {
  constexpr int V = 16 / sizeof(T), LANES = 16;
  __shared__ float sums[64][LANES * V + 1];
  const int c = threadIdx.x % LANES, g = threadIdx.x / LANES;  // 16 bytes of columns, row group
  const long long n0 = (long long)blockIdx.x * (LANES * V), n = n0 + V * c;
  const long long m0 = blockIdx.y * rows, m1 = m0 + rows < M ? m0 + rows : M;
  float acc[V];
#pragma unroll
  for (int e = 0; e < V; e++) acc[e] = 0.f;
  if (n + V <= N) {
    const T* p = x + n;
#pragma unroll 8
    for (long long m = m0 + g; m < m1; m += 64) {
      typedef T vecT __attribute__((ext_vector_type(V)));
      const vecT v = __builtin_bit_cast(vecT, (u32x4)*(const loose16*)(p + m * ld));
#pragma unroll
      for (int e = 0; e < V; e++) acc[e] += (float)v[e];
    }
  } else {
    for (long long m = m0 + g; m < m1; m += 64)
#pragma unroll
      for (int e = 0; e < V; e++)
        if (n + e < N) acc[e] += load_as_float(x + m * ld + n + e);
  }
#pragma unroll
  for (int e = 0; e < V; e++) sums[g][V * c + e] = acc[e];
  __syncthreads();
  if (threadIdx.x < LANES * V && n0 + threadIdx.x < N) {
    float v = 0.f;
#pragma unroll 16
    for (int i = 0; i < 64; i++) v += sums[i][threadIdx.x];
    if (part) part[blockIdx.y * N + n0 + threadIdx.x] = v;
    else store_from_float(out + n0 + threadIdx.x, v);
  }
}

// 64 columns per workgroup, the ranges among its four wavefronts
template <typename T>
__global__ __launch_bounds__(256) void colsum_merge_kernel(const float* part, int ranges, long long N, T* out) {
  __shared__ float sums[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long n = (long long)blockIdx.x * 64 + lane;
  float v = 0.f;
  if (n < N) {
#pragma unroll 8
    for (int i = wave; i < ranges; i += 4) v += part[i * N + n];
  }
  sums[wave][lane] = v;
  __syncthreads();
  if (wave == 0 && n < N) store_from_float(out + n, (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]));
}

template <typename T>
int launch_colsum_merge(const float* part, int ranges, long long N, void* out, hipStream_t stream) {
  hipLaunchKernelGGL((colsum_merge_kernel<T>), dim3((unsigned)((N + 63) / 64)), dim3(256), 0, stream, part, ranges, N, (T*)out);
  return (int)hipGetLastError();
}

// Row ranges: enough for two workgroups per CU, of no fewer than 1024 rows' worth of work each (16 loads per lane).
int colsum_ranges(long long M, long long N, int dtype) {
  const long long wide = dtype == TTSDPA_F32 ? 64 : 128, blocks = (N + wide - 1) / wide;
  long long want = (512 + blocks - 1) / blocks;
  const long long most = M / 512;
  if (want > most) want = most;
  return want > 1 ? (int)want : 1;
}

template <typename T>
int launch_colsum(const void* x, long long M, long long N, long long ld, void* out, float* part, int ranges, hipStream_t stream) {
  constexpr int wide = 16 * (16 / (int)sizeof(T));
  const long long rows = (M + ranges - 1) / ranges;
  if ((N + wide - 1) / wide > 0x7fffffffLL) return TTSDPA_ERR_SHAPE;
  hipLaunchKernelGGL((colsum_kernel<T>), dim3((unsigned)((N + wide - 1) / wide), (unsigned)ranges), dim3(1024), 0, stream, (const T*)x, M, N, ld,
                     rows, (T*)out, ranges > 1 ? part : nullptr);
  return ranges > 1 ? launch_colsum_merge<T>(part, ranges, N, out, stream) : (int)hipGetLastError();
}

bool aligned(const void* p, size_t n) { return ((uintptr_t)p % n) == 0; }

int check(int dtype, const void* x, const void* w, const void* out, long long M, long long N, long long K, long long ldx,
          long long ldw, long long ldo, int* route) {
  if (dtype != TTSDPA_F32 && dtype != TTSDPA_F16 && dtype != TTSDPA_BF16) return TTSDPA_ERR_DTYPE;
  if (M < 0 || N < 0 || K < 0) return TTSDPA_ERR_SHAPE;
  *route = TTLINEAR_ROUTE_NONE;
  if (M == 0 || N == 0) return TTSDPA_OK;
  if (!out || (K > 0 && (!x || !w))) return TTSDPA_ERR_NULL;
  if (ldx < K || ldw < K || ldo < N) return TTSDPA_ERR_STRIDE;
  const size_t esz = dtype == TTSDPA_F32 ? 4 : 2;
  if (!aligned(x, esz) || !aligned(w, esz) || !aligned(out, esz)) return TTSDPA_ERR_STRIDE;
  if ((M + 63) / 64 > 65535 || (N + 63) / 64 > 0x7fffffffLL) return TTSDPA_ERR_SHAPE;
  const long long kpc = 16 / (long long)esz;  // elements per 16 bytes
  const bool mfma = K > 0 && K % (8 * kpc) == 0 && N % 4 == 0 && ldx % kpc == 0 && ldw % kpc == 0 && ldo % 4 == 0 &&
                    aligned(x, 16) && aligned(w, 16) && aligned(out, 4 * esz) &&
                    ldx < (1 << 21) && ldw < (1 << 21);  // 256 rows are addressed with 32-bit byte offsets
  *route = mfma ? TTLINEAR_ROUTE_MFMA : TTLINEAR_ROUTE_GENERAL;
  return TTSDPA_OK;
}

// Workgroups that tile_of_block spreads over the 8 XCDs (the kernels count in 32 bits).
long long blocks_of_tiles(const LinArgs& a, int TM, int TN) {
  const long long tiles = ((a.M + TM - 1) / TM) * ((a.N + TN - 1) / TN);
  return (tiles + 7) / 8 * 8;
}

template <typename TR, int TM, int TN, int WN, int WM, int ST>
int launch_mfma_stages(const LinArgs& a, hipStream_t stream, unsigned entries) {
  constexpr int lds = ST * (TM + TN) * ROWB;
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  const hipError_t granted = grant_dynamic_lds((const void*)linear_mfma_kernel<TR, TM, TN, WN, WM, ST>, lds, state, done);
  if (granted != hipSuccess) return (int)granted;
  const long long nwg = blocks_of_tiles(a, TM, TN) * a.splits;
  if (nwg > 0x3fffffffLL) return TTSDPA_ERR_SHAPE;
  hipLaunchKernelGGL((linear_mfma_kernel<TR, TM, TN, WN, WM, ST>), dim3((unsigned)nwg, entries), dim3(WN * WM * 64), lds, stream, a);
  return (int)hipGetLastError();
}

// 128 x 128 tiles, one per CU at most: four k-tiles in LDS
bool tile_per_cu(const LinArgs& a, unsigned entries) { return ((a.M + 127) / 128) * ((a.N + 127) / 128) * entries <= 256; }

template <typename TR>
int launch_small_tiles(const LinArgs& a, hipStream_t stream, unsigned entries = 1) {
  return tile_per_cu(a, entries) ? launch_mfma_stages<TR, 128, 128, 4, 2, 4>(a, stream, entries) : launch_mfma_stages<TR, 128, 128, 4, 2, 2>(a, stream, entries);
}

// ... with the contraction divided (a.splits, a.part)
template <typename TR>
int launch_divided(const LinArgs& a, hipStream_t stream) {
  return launch_mfma_stages<TR, 128, 128, 4, 2, 4>(a, stream, 1);
}

template <typename TR, int T_, bool XT, bool WT>
int launch_mfma_t_tile(const LinArgs& a, hipStream_t stream) {
  constexpr int lds = 2 * (T_ + T_) * ROWB;
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  const hipError_t granted = grant_dynamic_lds((const void*)linear_mfma_t_kernel<TR, T_, T_, XT, WT>, lds, state, done);
  if (granted != hipSuccess) return (int)granted;
  const long long nwg = blocks_of_tiles(a, T_, T_);
  if (nwg > 0x3fffffffLL) return TTSDPA_ERR_SHAPE;
  hipLaunchKernelGGL((linear_mfma_t_kernel<TR, T_, T_, XT, WT>), dim3((unsigned)nwg), dim3(512), lds, stream, a);
  return (int)hipGetLastError();
}

// 256 x 256 tiles once they fill the chip, unless their last round over the 256 CUs would be under 85 % full: then four
// times as many 128 x 128 tiles (weight gradient of the QKV projection, 384 large tiles: 878 -> 936 TFLOP/s; its input
// gradient, 512 large tiles, runs 1063 against 795 on the small ones)
bool large_in_place(long long n256) { return n256 >= 256 && n256 * 100 >= (n256 + 255) / 256 * 256 * 85; }

// 16-bit operands read as they lie in memory (a.xt / a.wt: stored contraction-major)
template <typename TR>
int launch_mfma_t(const LinArgs& a, hipStream_t stream) {
  const bool big = large_in_place(((a.M + 255) / 256) * ((a.N + 255) / 256));
  if (a.xt && a.wt) return big ? launch_mfma_t_tile<TR, 256, true, true>(a, stream) : launch_mfma_t_tile<TR, 128, true, true>(a, stream);
  if (a.xt) return big ? launch_mfma_t_tile<TR, 256, true, false>(a, stream) : launch_mfma_t_tile<TR, 128, true, false>(a, stream);
  return big ? launch_mfma_t_tile<TR, 256, false, true>(a, stream) : launch_mfma_t_tile<TR, 128, false, true>(a, stream);
}

template <typename TR, int TM>
int launch_linear256(const LinArgs& a, hipStream_t stream) {
  constexpr int lds = kLin256Lds<TM>;
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  const hipError_t granted = grant_dynamic_lds((const void*)linear256_kernel<TR, TM>, lds, state, done);
  if (granted != hipSuccess) return (int)granted;
  const long long nwg = blocks_of_tiles(a, TM, 256);
  if (nwg > 0x3fffffffLL) return TTSDPA_ERR_SHAPE;
  hipLaunchKernelGGL((linear256_kernel<TR, TM>), dim3((unsigned)nwg), dim3(256), lds, stream, a);
  return (int)hipGetLastError();
}

// The large tiles of an XCD that are whole rounds of its CUs and what is left, where that makes at most one round of halves.
bool mixed_rounds(const LinArgs& a, long long* whole, long long* left) {
  const long long per = (((a.M + 255) / 256) * ((a.N + 255) / 256) + 7) / 8;
  *whole = per / kCusOfXcd * kCusOfXcd, *left = per - *whole;
  return *whole > 0 && *left > 0 && 2 * *left <= kCusOfXcd;
}

template <typename TR>
int launch_linear256_mixed(const LinArgs& a, hipStream_t stream) {
  constexpr int lds = kLin256Lds<256> > kLin256Lds<128> ? kLin256Lds<256> : kLin256Lds<128>;
  static hipError_t state[kMaxDevices];
  static bool done[kMaxDevices];
  const hipError_t granted = grant_dynamic_lds((const void*)linear256_mixed_kernel<TR>, lds, state, done);
  if (granted != hipSuccess) return (int)granted;
  long long whole, left;
  if (!mixed_rounds(a, &whole, &left)) return (int)hipErrorInvalidValue;
  const long long nwg = 8 * (whole + 2 * left);
  if (nwg > 0x3fffffffLL) return TTSDPA_ERR_SHAPE;
  hipLaunchKernelGGL((linear256_mixed_kernel<TR>), dim3((unsigned)nwg), dim3(256), lds, stream, a, (int)whole);
  return (int)hipGetLastError();
}

// Microseconds of the tiled kernels, from measurements, against each other's and the streaming kernel's.  A k-step is 128 bytes of
// k; a round, 256 tiles on the 256 CUs.  fp32 128 x 128: 2.2 us a k-step and round.  16-bit 128 x 128, two to a CU: 0.55 us (with
// weights from memory; 0.44 from the caches), and 0.54 for each further round (445 x 3072 x 8576, 96 tiles, 75 us; 1024 x 4096 x
// 4096, 256, 43; 1500 x 5120 x 5120, 480, 86; 6000 x 3000 x 1024, 1128, 56).
double small_tiles_cost(const LinArgs& a, int dtype, unsigned entries) {
  const double tiles = (double)((a.M + 127) / 128) * (double)((a.N + 127) / 128) * entries;
  const double steps = a.K * (dtype == TTSDPA_F32 ? 4 : 2) / 128.0, rounds = (double)(long long)((tiles + 255) / 256);
  if (dtype == TTSDPA_F32) return 3 + steps * 2.2 * rounds;
  const double fill = tiles / 256 - (rounds - 1);  // of the last round
  const double cold = steps < 16 ? 2 - steps / 8 : 0;  // few steps do not hide the first loads (192 of k into 3469 x 64: 7.0)
  return 1 + cold + 1.2 * rounds + steps * (rounds > 1 ? 0.54 * (rounds - 1) + 0.3 + 0.24 * fill : 0.54 + 0.06 * fill);
}
// The hand-ordered kernel's 256 x 256 tiles, 16-bit, one to a CU: 9 us a round for its first loads and its output and 1.5 a k-step, in
// a last round that is not full less, because the power is shared by fewer (1999 x 4096 x 14336, 128 tiles, 240 us; x 6144 x 4096,
// 192, 82; 4096 x 4096 x 4096, 256, 102; 4096 x 6144 x 8192, 384, 318).
// Few k-steps do not hide a tile's first loads (2495 x 4876, 3 steps: 22 us; on the small tiles 16).
double large_cold(const LinArgs& a) { return a.K < 1024 ? 5 * (2 - a.K / 512.0) : 0; }
double large_tiles_cost(const LinArgs& a) {
  const double tiles = (double)((a.M + 255) / 256) * (double)((a.N + 255) / 256), rounds = (double)(long long)((tiles + 255) / 256);
  const double fill = tiles / 256 - (rounds - 1);
  return 9 * rounds + large_cold(a) + a.K / 64.0 * (1.5 * (rounds - 1) + 1.04 + 0.46 * fill * fill);
}
// Its 128 x 256 tiles: more bytes through LDS for a product, so they are for what leaves large tiles' CUs idle (the same 1999 x 4096 x
// 14336, 256 tiles, 194 us; 1500 x 5120 x 5120, 240, 70, on the others 98 and 86; but 4096 x 4096 x 4096, 512, 121).
double half_tiles_cost(const LinArgs& a) {
  const double tiles = (double)((a.M + 127) / 128) * (double)((a.N + 255) / 256), rounds = (double)(long long)((tiles + 255) / 256);
  const double fill = tiles / 256 - (rounds - 1);
  return 6 * rounds + a.K / 64.0 * (0.9 * (rounds - 1) + 0.62 + 0.24 * fill);
}

// Whole rounds of large tiles and one of halves.
double mixed_tiles_cost(const LinArgs& a) {
  long long whole, left;
  if (!mixed_rounds(a, &whole, &left)) return 1e30;
  const double rounds = (double)(whole / kCusOfXcd);
  return 9 * rounds + 6 + large_cold(a) + a.K / 64.0 * (1.5 * rounds + 0.62 + 0.24 * (2 * left) / kCusOfXcd);
}

// 128 x 128 tiles whose contraction is divided among S workgroups each, one to a CU (of an XCD's: 826 x 1536 x 4160, 84 tiles in 3 shares,
// 33 on some, 36 us; 28 by this) at most: a launch more, and the shares' fp32 sums written and read at 5 TB/s.  What leaves most CUs
// idle otherwise, or goes to the streaming kernel, which takes in the operands of smaller tiles: 288 x 2048 x 6592, 48 tiles, 34.7 there
// -> 22.9 in 5 shares; 200 x 4096 x 14336, 64, 74 -> 48 in 4; 720 x 1536 x 4736, 72, 43 -> 24 in 3 (2: 26.6; 5, more than a round: 27.3).
// fp32: only what the streaming kernel does not take, contraction-major operands of fewer than 16 rows (6 x 768 x 28672 1740 -> 133).
// (Four wavefronts of 64 x 64 instead of eight of 64 x 32, fewer LDS reads: 3 to 8 % slower in every such call.)
double divided_cost(const LinArgs& a, int dtype, int S) {
  const double esz = dtype == TTSDPA_F32 ? 4 : 2, sums = 5.5 + 8.0 * S * a.M * a.N / 5e6;
  LinArgs share = a;
  share.K = (long long)((a.K * esz / 128 + S - 1) / S) * (long long)(128 / esz);
  const double work = small_tiles_cost(share, dtype, S), read = 2.2 + esz * (a.M + a.N) * a.K / 4.2e6;  // weights from memory: 69 x 6208 x 5440 29.5
  return (work > read ? work : read) + sums;
}
size_t divided_bytes(const LinArgs& a, int S) { return S > 1 ? ((size_t)S * (size_t)(a.M * a.N + a.M) * sizeof(float) + 255) / 256 * 256 : 0; }

// x . w^T on rows of whole k-tiles
double nt_cost(const LinArgs& a, int dtype, unsigned entries) {
  double us = small_tiles_cost(a, dtype, entries);
  if (dtype == TTSDPA_F32 || entries > 1) return us;
  const double large = large_tiles_cost(a), half = half_tiles_cost(a), mixed = mixed_tiles_cost(a);
  if (large < us) us = large;
  if (half < us) us = half;
  return mixed < us ? mixed : us;
}

// The tiles of a 16-bit product on rows of whole k-tiles: the cheapest by estimate.
int tiles_of(const LinArgs& a) {
  const double us = nt_cost(a, TTSDPA_BF16, 1);
  if (large_tiles_cost(a) <= us) return TTLINEAR_TILES_256x256;
  if (half_tiles_cost(a) <= us) return TTLINEAR_TILES_128x256;
  if (mixed_tiles_cost(a) <= us) return TTLINEAR_TILES_MIXED;
  return TTLINEAR_TILES_128x128;
}

template <typename TR>
int launch_mfma(const LinArgs& a, hipStream_t stream) {
  // (four wavefronts with 128 x 128 each — accumulators in AGPRs, half the LDS operand reads — measured 2-10 % slower
  // than eight with 64 x 128: one wavefront per SIMD hides too little)
  if constexpr (!std::is_same<TR, F32>::value) {
    switch (tiles_of(a)) {
      case TTLINEAR_TILES_256x256: return launch_linear256<TR, 256>(a, stream);  // the hand-ordered kernel
      case TTLINEAR_TILES_128x256: return launch_linear256<TR, 128>(a, stream);
      case TTLINEAR_TILES_MIXED: return launch_linear256_mixed<TR>(a, stream);
      default: return launch_small_tiles<TR>(a, stream);
    }
  } else {
    const long long big = ((a.M + 255) / 256) * ((a.N + 255) / 256);
    return big >= 256 ? launch_mfma_stages<TR, 256, 256, 4, 2, 2>(a, stream, 1) : launch_small_tiles<TR>(a, stream);
  }
}

// What the kernels of contraction-major operands take in place: the small tiles 0.6 us a k-step as long as every CU has one at most
// and with more in proportion, 10 % more where only w is contraction-major (a tile of the other form takes both kinds of LDS
// read), the large ones 2.3 us (8192 x 4096 x 6144, 512 tiles: 443 us).
double in_place_cost(const LinArgs& a, int dtype, unsigned entries) {
  if (!a.xt && !a.wt) return nt_cost(a, dtype, entries);
  const long long n256 = ((a.M + 255) / 256) * ((a.N + 255) / 256);
  if (large_in_place(n256)) return 3 + a.K / 64.0 * 2.3 * (double)((n256 + 255) / 256);
  if (dtype == TTSDPA_F32) return small_tiles_cost(a, dtype, entries) * (a.wt && !a.xt ? 1.1 : 1);
  const double tiles = (double)((a.M + 127) / 128) * (double)((a.N + 127) / 128) * entries;
  return (1.3 + (1.7 + a.K / 64.0 * 0.6) * (tiles > 256 ? tiles / 256 : 1)) * (a.wt && !a.xt ? 1.1 : 1);
}

bool streams(const LinArgs& a, int dtype, unsigned entries) {
  return stream_takes(a, dtype) && plan_stream(a, dtype, entries, false).us < in_place_cost(a, dtype, entries);
}

// What the tiled kernels' layout does not allow: the streaming kernel, or where one of its operands is too narrow for that (a
// k-major operand of fewer than 16 rows, an empty contraction) the vector ALUs.
template <typename T>
int launch_general_linear(const LinArgs& a, hipStream_t stream, unsigned entries = 1) {
  const int dtype = sizeof(T) == 4 ? TTSDPA_F32 : std::is_same<T, _Float16>::value ? TTSDPA_F16 : TTSDPA_BF16;
  if (stream_takes(a, dtype)) return launch_stream(a, dtype, stream, plan_stream(a, dtype, entries, false), entries);
  dim3 grid((unsigned)((a.N + 63) / 64), (unsigned)((a.M + 63) / 64), entries);
  hipLaunchKernelGGL((linear_general_kernel<T>), grid, dim3(256), 0, stream, a);
  return (int)hipGetLastError();
}

}  // namespace
}  // namespace ttsdpa

using namespace ttsdpa;

extern "C" {

int ttlinear_plan(int dtype, const void* x, const void* w, const void* bias, const void* out, int64_t M, int64_t N,
                  int64_t K, int64_t ldx, int64_t ldw, int64_t ldo, int* route) {
  (void)bias;
  int r = TTLINEAR_ROUTE_NONE;
  const int rc = check(dtype, x, w, out, M, N, K, ldx, ldw, ldo, &r);
  if (rc == TTSDPA_OK && route) *route = r;
  return rc;
}

// 16-bit operands that a matrix-core kernel reads in place, one of them contraction-major at least (no copies, no scratch).
static bool in_place_ok(const LinArgs& g, int dtype) {
  if (dtype == TTSDPA_F32 || g.K < 1 || g.K % 64 != 0 || g.N % 4 != 0 || g.ldo % 4 != 0 || !aligned(g.out, 8)) return false;
  auto operand_ok = [](const void* p, bool contraction_major, int64_t rows, int64_t ld) {
    if (!aligned(p, 16) || ld % 8 != 0) return false;
    // a tile's rows are addressed with 32-bit byte offsets: 64 k-rows of a contraction-major operand, 256 rows otherwise
    return contraction_major ? (rows % 8 == 0 && ld < (1 << 24)) : ld < (1 << 21);
  };
  return (g.xt || g.wt) && operand_ok(g.x, g.xt, g.M, g.ldx) && operand_ok(g.w, g.wt, g.N, g.ldw);
}

// x . w^T on the tiled kernels, with copies of the operands whose layout they do not take (contraction-major, rows that are
// not whole k-tiles, unaligned) in scratch: what the copies need and what the product is estimated to take with them.
// And the shares of its contraction, where that is divided (S > 1), whose sums lie behind the copies.
struct PackPlan {
  bool ok, x, w;
  long long kpad;
  size_t xbytes, copies, bytes;
  int S;
  double us;
};

// beat: what another way of the product is estimated to take.
static PackPlan plan_pack(const LinArgs& g, int dtype, size_t room, double beat) {
  const long long esz = dtype == TTSDPA_F32 ? 4 : 2, bk = ROWB / esz, kpc = 16 / esz;
  PackPlan p{};
  p.kpad = (g.K + bk - 1) / bk * bk;
  auto as_it_is = [&](const void* ptr, int kmajor, long long ld) { return !kmajor && g.K == p.kpad && ld % kpc == 0 && aligned(ptr, 16); };
  p.x = !as_it_is(g.x, g.xt, g.ldx);
  p.w = !as_it_is(g.w, g.wt, g.ldw);
  // rows of a tile are addressed with 32-bit byte offsets; grids
  p.ok = g.K > 0 && p.kpad < (1 << 21) && (p.x || g.ldx < (1 << 21)) && (p.w || g.ldw < (1 << 21)) && (g.M + 15) / 16 <= 65535 &&
         (!p.w || (g.N + 15) / 16 <= 65535);
  if (!p.ok) return p;
  auto bytes = [&](long long rows) { return ((size_t)rows * (size_t)p.kpad * (size_t)esz + 255) / 256 * 256; };
  p.xbytes = p.x ? bytes(g.M) : 0;
  p.copies = p.bytes = p.xbytes + (p.w ? bytes(g.N) : 0);
  LinArgs nt = g;
  nt.K = p.kpad, nt.xt = nt.wt = 0;
  const double whole = nt_cost(nt, dtype, 1);
  double us = whole;
  p.S = 1;
  // (copies for the alignment's sake alone: 804 x 1983 x 5329 64 us, undivided 57; fp32 that the streaming kernel takes: that adds a
  // contraction up in more and shorter chains)
  // And not worth a look where two shares' sums and the operands read once take longer than another way, at choose()'s margins.
  const bool may = (p.copies == 0 || g.xt || g.wt) && !(dtype == TTSDPA_F32 && stream_takes(g, dtype)) &&
                   7.7 + (double)esz * (double)(g.M + g.N) * (double)g.K / 4.2e6 + 16.0 * (double)g.M * (double)g.N / 5e6 < 1.03 * beat;
  const long long most = kCusOfXcd / ((((g.M + 127) / 128) * ((g.N + 127) / 128) + 7) / 8);  // a workgroup to a CU
  for (int S = 2; may && S <= 16 && S <= most && p.kpad / bk >= 4 * S; S++) {
    const double divided = divided_cost(nt, dtype, S);
    if (divided < us && divided < 0.9 * whole && p.copies + divided_bytes(nt, S) <= room) us = divided, p.S = S;
  }
  p.bytes += divided_bytes(nt, p.S);
  p.us = us + (double)p.copies * 2 / 5e6 + 5.5 * (p.x + p.w);  // read and written at 5 TB/s; a launch each, and the next one's wait
  // (262 x 866 x 2545: 6.5 and 5.0 us beside 5.2 MB's 1)
  return p;
}

// sums: the column sums of x's rows' parts, where x is packed from a contraction-major operand ([ranges][M])
static int launch_packed(const LinArgs& g, const PackPlan& p, int dtype, hipStream_t s, char* scratch, float* sums) {
  LinArgs nt = g;
  nt.K = p.kpad, nt.xt = nt.wt = 0;
  auto pack = [&](const void* src, void* dst, long long rows, long long ld, bool kmajor, float* part) {
    switch (dtype) {
      case TTSDPA_F32: return launch_pack<float>(src, dst, rows, g.K, ld, p.kpad, kmajor, part, s);
      case TTSDPA_F16: return launch_pack<_Float16>(src, dst, rows, g.K, ld, p.kpad, kmajor, part, s);
      default: return launch_pack<__bf16>(src, dst, rows, g.K, ld, p.kpad, kmajor, part, s);
    }
  };
  if (p.x) {
    const int rc = pack(g.x, scratch, g.M, g.ldx, g.xt, sums);
    if (rc != 0) return rc;
    nt.x = scratch, nt.ldx = p.kpad;
  }
  if (p.w) {
    const int rc = pack(g.w, scratch + p.xbytes, g.N, g.ldw, g.wt, nullptr);
    if (rc != 0) return rc;
    nt.w = scratch + p.xbytes, nt.ldw = p.kpad;
  }
  if (p.S > 1) {
    nt.splits = p.S, nt.part = (float*)(scratch + p.copies);
    const int rc = dtype == TTSDPA_F32 ? launch_divided<F32>(nt, s) : dtype == TTSDPA_F16 ? launch_divided<F16>(nt, s) : launch_divided<BF16>(nt, s);
    return rc != 0 ? rc : launch_linear_merge(nt, dtype, s);
  }
  return dtype == TTSDPA_F32 ? launch_mfma<F32>(nt, s) : dtype == TTSDPA_F16 ? launch_mfma<F16>(nt, s) : launch_mfma<BF16>(nt, s);
}

// How a product runs: the cheapest by estimate of the ways that take it.
enum class Way {
  General = TTLINEAR_WAY_GENERAL,
  Stream = TTLINEAR_WAY_STREAM,
  InPlace = TTLINEAR_WAY_IN_PLACE,
  Packed = TTLINEAR_WAY_TILED,
  Outer = TTLINEAR_WAY_OUTER
};
struct Choice {
  Way way = Way::General;
  double us = 1e30;
  PackPlan pack;
  StreamPlan stream{0, 1, 0};  // where the kernel takes the product
};

static Choice choose(const LinArgs& g, int dtype, bool scratch, size_t scratch_bytes) {
  Choice c;
  auto take = [&](Way w, double cost) {
    if (cost < c.us) c.way = w, c.us = cost;
  };
  if (in_place_ok(g, dtype)) take(Way::InPlace, in_place_cost(g, dtype, 1));
  if (stream_takes(g, dtype)) {
    c.stream = plan_stream(g, dtype, 1, scratch);
    take(Way::Stream, c.stream.us);
  }
  c.pack = plan_pack(g, dtype, scratch ? scratch_bytes : 0, c.us);
  // (margins for divided contractions: the estimates of the ways that read contraction-major operands as they lie miss by more, the
  // input gradient of 231 x 19072 x 3072 17 us shorter so than divided with its copies; those of the streaming kernel's small tiles and
  // shares by a tenth, of its large tiles less)
  const bool sure = c.way == Way::Stream && c.stream.R == 4 && c.stream.S == 1;
  if (c.pack.ok && c.pack.bytes <= (scratch ? scratch_bytes : 0))
    take(Way::Packed, c.pack.S == 1 ? c.pack.us : c.pack.us / (c.pack.copies > 0 ? 0.75 : sure ? 1.03 : 0.9));
  // (row sums, where wanted, come with the product, as on the streaming kernel; the tiled kernels need launches for them)
  if (outer_takes(g, dtype)) take(Way::Outer, outer_cost(g, dtype) - (g.rowsum && c.way != Way::Stream ? 4 : 0));
  return c;
}

static int run(const LinArgs& g, const Choice& c, int dtype, void* scratch, size_t scratch_bytes, hipStream_t s) {
  switch (c.way) {
    case Way::Stream: return launch_stream(g, dtype, s, c.stream, 1, scratch, scratch_bytes);
    case Way::InPlace: return dtype == TTSDPA_F16 ? launch_mfma_t<F16>(g, s) : launch_mfma_t<BF16>(g, s);
    case Way::Packed: return launch_packed(g, c.pack, dtype, s, (char*)scratch, nullptr);
    case Way::Outer: return launch_outer(g, dtype, s);
    default: break;
  }
  switch (dtype) {
    case TTSDPA_F32: return launch_general_linear<float>(g, s);
    case TTSDPA_F16: return launch_general_linear<_Float16>(g, s);
    default: return launch_general_linear<__bf16>(g, s);
  }
}

static int product(const LinArgs& g, int dtype, void* scratch, size_t scratch_bytes, hipStream_t s) {
  return run(g, choose(g, dtype, scratch, scratch_bytes), dtype, scratch, scratch_bytes, s);
}

// x . w^T + bias; scratch (optional): lets the streaming kernel divide the contraction among workgroups, and holds copies
static int forward(int dtype, const void* x, const void* w, const void* bias, void* out, int64_t M, int64_t N, int64_t K, int64_t ldx,
                   int64_t ldw, int64_t ldo, void* scratch, size_t scratch_bytes, void* stream) {
  int route = TTLINEAR_ROUTE_NONE;
  const int rc = check(dtype, x, w, out, M, N, K, ldx, ldw, ldo, &route);
  if (rc != TTSDPA_OK || route == TTLINEAR_ROUTE_NONE) return rc;
  if (bias && !aligned(bias, dtype == TTSDPA_F32 ? 4 : 2)) return TTSDPA_ERR_STRIDE;
  return product(LinArgs{x, w, bias, out, M, N, K, ldx, ldw, ldo}, dtype, scratch, scratch_bytes, (hipStream_t)stream);
}

int ttlinear_forward(int dtype, const void* x, const void* w, const void* bias, void* out, int64_t M, int64_t N,
                     int64_t K, int64_t ldx, int64_t ldw, int64_t ldo, void* stream) {
  return forward(dtype, x, w, bias, out, M, N, K, ldx, ldw, ldo, nullptr, 0, stream);
}

// Sizes and layout alone: dense operands on aligned addresses.
static LinArgs flags_args(int64_t M, int64_t N, int64_t K, int trans_a, int trans_b) {
  return LinArgs{nullptr, nullptr, nullptr, nullptr, M, N, K, trans_a ? M : K, trans_b ? K : N, N, trans_a ? 1 : 0, trans_b ? 0 : 1};
}

// Room for the copies (where the product would be made on copies, or operands lie contraction-major) or the parts of a divided contraction.
// The latter also where aligned operands would go another way: sizes do not say how rows are aligned, and unaligned ones go to the
// streaming kernel.  (Some MB at most: only products of few tiles are divided.)
static size_t scratch_of(const LinArgs& g, const Choice& c, int dtype, size_t behind_copies = 0) {
  const size_t parts = stream_part_bytes(g, plan_stream_call(g, dtype, 1, true, c.stream));
  const size_t packed = c.way == Way::Packed ? c.pack.bytes + behind_copies : 0;
  return packed > parts ? packed : parts;
}

size_t ttlinear_matmul_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t K, int trans_a, int trans_b) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const LinArgs g = flags_args(M, N, K, trans_a, trans_b);
  return scratch_of(g, choose(g, dtype, true, ~(size_t)0), dtype);
}

int ttlinear_matmul_tiles(int dtype, int64_t M, int64_t N, int64_t K, int trans_a, int trans_b) {
  if ((dtype != TTSDPA_F16 && dtype != TTSDPA_BF16) || M <= 0 || N <= 0 || K <= 0) return TTLINEAR_TILES_OTHER;
  LinArgs g = flags_args(M, N, K, trans_a, trans_b);
  const Choice c = choose(g, dtype, true, ~(size_t)0);
  if (c.way != Way::Packed) return TTLINEAR_TILES_OTHER;
  g.K = c.pack.kpad, g.xt = g.wt = 0;
  return c.pack.S > 1 ? TTLINEAR_TILES_128x128 : tiles_of(g);
}

static ttlinear_kernel_info info_of(const LinArgs& g, const Choice& c, int dtype) {
  ttlinear_kernel_info info{(int32_t)c.way, 0, 0, 1, 1};
  if (c.way == Way::Packed) info.shares = c.pack.S;
  if (c.way != Way::Stream) return info;
  const StreamPlan call = plan_stream_call(g, dtype, 1, true, c.stream);
  const StreamTiles t = stream_tiles(g, dtype, 1, call);
  return {TTLINEAR_WAY_STREAM, t.rows, t.columns, t.per_workgroup, call.S};
}

int ttlinear_matmul_kernel(int dtype, int64_t M, int64_t N, int64_t K, int trans_a, int trans_b, ttlinear_kernel_info* info) {
  if (!info) return TTSDPA_ERR_NULL;
  if (dtype != TTSDPA_F32 && dtype != TTSDPA_F16 && dtype != TTSDPA_BF16) return TTSDPA_ERR_DTYPE;
  if (M <= 0 || N <= 0 || K <= 0) return TTSDPA_ERR_SHAPE;
  const LinArgs g = flags_args(M, N, K, trans_a, trans_b);
  *info = info_of(g, choose(g, dtype, true, ~(size_t)0), dtype);
  return TTSDPA_OK;
}

int ttlinear_matmul(int dtype, const void* a, const void* b, const void* bias, void* out, int64_t M, int64_t N, int64_t K,
                    int trans_a, int trans_b, int64_t lda, int64_t ldb, int64_t ldo, void* workspace,
                    size_t workspace_bytes, void* stream) {
  if (!workspace || !aligned(workspace, 256)) workspace = nullptr, workspace_bytes = 0;
  if (!trans_a && trans_b) return forward(dtype, a, b, bias, out, M, N, K, lda, ldb, ldo, workspace, workspace_bytes, stream);
  if (dtype != TTSDPA_F32 && dtype != TTSDPA_F16 && dtype != TTSDPA_BF16) return TTSDPA_ERR_DTYPE;
  if (M < 0 || N < 0 || K < 0) return TTSDPA_ERR_SHAPE;
  if (M == 0 || N == 0) return TTSDPA_OK;
  if (!out || (K > 0 && (!a || !b))) return TTSDPA_ERR_NULL;
  if (lda < (trans_a ? M : K) || ldb < (trans_b ? K : N) || ldo < N) return TTSDPA_ERR_STRIDE;
  const size_t esz = dtype == TTSDPA_F32 ? 4 : 2;
  if (!aligned(a, esz) || !aligned(b, esz) || !aligned(out, esz) || (bias && !aligned(bias, esz))) return TTSDPA_ERR_STRIDE;
  if ((M + 63) / 64 > 65535 || (N + 63) / 64 > 0x7fffffffLL) return TTSDPA_ERR_SHAPE;
  return product(LinArgs{a, b, bias, out, M, N, K, lda, ldb, ldo, trans_a ? 1 : 0, trans_b ? 0 : 1}, dtype, workspace, workspace_bytes,
                 (hipStream_t)stream);
}

int ttlinear_matmul_batched(int dtype, const void* a, const void* b, const void* bias, void* out, int64_t M, int64_t N,
                            int64_t K, int trans_a, int trans_b, int64_t lda, int64_t ldb, int64_t ldo, int nbatch_dims,
                            const int64_t* batch_shape, const int64_t* a_batch_stride, const int64_t* b_batch_stride,
                            int64_t out_batch_stride, void* workspace, size_t workspace_bytes, void* stream) {
  if (dtype != TTSDPA_F32 && dtype != TTSDPA_F16 && dtype != TTSDPA_BF16) return TTSDPA_ERR_DTYPE;
  if (nbatch_dims < 0 || nbatch_dims > TTLINEAR_MAX_BATCH_DIMS) return TTSDPA_ERR_SHAPE;
  if (nbatch_dims > 0 && (!batch_shape || !a_batch_stride || !b_batch_stride)) return TTSDPA_ERR_NULL;
  long long entries = 1;
  for (int d = 0; d < nbatch_dims; d++) {
    if (batch_shape[d] < 0 || a_batch_stride[d] < 0 || b_batch_stride[d] < 0) return TTSDPA_ERR_SHAPE;
    entries *= batch_shape[d];
  }
  if (out_batch_stride < 0) return TTSDPA_ERR_STRIDE;
  const size_t esz = dtype == TTSDPA_F32 ? 4 : 2;
  auto offsets = [&](long long i, long long* ao, long long* bo) {
    // offsets of entry i: the reference's index walk from the innermost batch dimension outwards
    long long rest = i;
    *ao = 0, *bo = 0;
    for (int d = nbatch_dims - 1; d >= 0; d--) {
      const long long idx = rest % batch_shape[d];
      rest /= batch_shape[d];
      *ao += idx * a_batch_stride[d];
      *bo += idx * b_batch_stride[d];
    }
  };
  // One grid for all entries (the reference's strided-batched product, src/Operation/OpLinalg.cpp:113-150) when the
  // entries' offsets are a multiple of the entry index in both operands (no broadcast pattern that breaks the stride)
  // and an entry is small enough that a launch each would be launch-bound; x . w^T on the tiled matrix-core kernel when
  // the layout allows and its tiles are worth it, else on the general route, which reads the operands in place.
  if (entries > 1 && entries <= 65535 && M > 0 && N > 0 && K > 0 && a && b && out && (double)M * N * K <= (double)(1 << 27)) {
    long long sa = 0, sb = 0;
    offsets(1, &sa, &sb);
    bool uniform = true;
    for (long long i = 2; i < entries && uniform; i++) {
      long long ao, bo;
      offsets(i, &ao, &bo);
      uniform = ao == i * sa && bo == i * sb;
    }
    if (uniform && lda >= (trans_a ? M : K) && ldb >= (trans_b ? K : N) && ldo >= N && aligned(a, esz) && aligned(b, esz) &&
        aligned(out, esz) && (!bias || aligned(bias, esz)) && (M + 63) / 64 <= 65535) {
      hipStream_t s = (hipStream_t)stream;
      LinArgs g{a, b, bias, out, M, N, K, lda, ldb, ldo, trans_a ? 1 : 0, trans_b ? 0 : 1};
      g.bsx = sa, g.bsw = sb, g.bso = out_batch_stride;
      int route = TTLINEAR_ROUTE_NONE;
      const long long kpc = 16 / (long long)esz;
      if (!trans_a && trans_b && check(dtype, a, b, out, M, N, K, lda, ldb, ldo, &route) == TTSDPA_OK && route == TTLINEAR_ROUTE_MFMA &&
          sa % kpc == 0 && sb % kpc == 0 && out_batch_stride % 4 == 0 && !streams(g, dtype, (unsigned)entries)) {
        g.xt = g.wt = 0;
        switch (dtype) {
          case TTSDPA_F32: return launch_small_tiles<F32>(g, s, (unsigned)entries);
          case TTSDPA_F16: return launch_small_tiles<F16>(g, s, (unsigned)entries);
          default: return launch_small_tiles<BF16>(g, s, (unsigned)entries);
        }
      }
      switch (dtype) {
        case TTSDPA_F32: return launch_general_linear<float>(g, s, (unsigned)entries);
        case TTSDPA_F16: return launch_general_linear<_Float16>(g, s, (unsigned)entries);
        default: return launch_general_linear<__bf16>(g, s, (unsigned)entries);
      }
    }
  }
  for (long long i = 0; i < entries; i++) {
    // offsets of entry i: the reference's index walk from the innermost batch dimension outwards
    long long ao = 0, bo = 0, rest = i;
    for (int d = nbatch_dims - 1; d >= 0; d--) {
      const long long idx = rest % batch_shape[d];
      rest /= batch_shape[d];
      ao += idx * a_batch_stride[d];
      bo += idx * b_batch_stride[d];
    }
    const int rc = ttlinear_matmul(dtype, a ? (const char*)a + ao * esz : nullptr, b ? (const char*)b + bo * esz : nullptr, bias,
                                   out ? (char*)out + i * out_batch_stride * esz : nullptr, M, N, K, trans_a, trans_b, lda, ldb,
                                   ldo, workspace, workspace_bytes, stream);
    if (rc != 0) return rc;
  }
  return TTSDPA_OK;
}

// Ranges of rows that a packed grad^T's column sums come in.
static long long pack_ranges(long long kpad) { return (kpad + kPackRows - 1) / kPackRows; }

size_t ttlinear_backward_least_workspace_bytes(int dtype, int64_t M, int64_t N) {
  return M <= 0 || N <= 0 ? 0 : (size_t)colsum_ranges(M, N, dtype) * (size_t)N * sizeof(float);
}

// The two products of a layer's backward, and whether they run in one launch.
struct BackwardPlan {
  Choice w, i;
  PairPlan pair;
  bool paired, joint;  // pair is filled in; and is the way
};

// Small layers: both products, and the column sums with the weight's, in one launch.  Where the two would be launched
// on the streaming kernel anyway and the launches saved (5 us, the column sums' among them) are worth more than what
// the common workgroup size may cost (64 x 784 x 500 fp32: 10 us in two launches and 5 for the column sums); fp32, which
// the products bound, wherever it is estimated faster (1501 x 1999 x 2501: 322 us, on tiles with copies 381).
static BackwardPlan plan_backward(const LinArgs& gw, const LinArgs& gi, int dtype, size_t workspace_bytes) {
  BackwardPlan p;
  p.w = choose(gw, dtype, true, workspace_bytes);
  p.i = choose(gi, dtype, true, workspace_bytes);
  const bool takes = stream_takes(gw, dtype) && stream_takes(gi, dtype);
  const bool streams = (p.w.way == Way::Stream || p.w.way == Way::Outer) && p.i.way == Way::Stream;
  p.joint = p.paired = takes && (streams || dtype == TTSDPA_F32);
  if (!p.paired) return p;
  p.pair = plan_stream_pair(gw, gi, dtype);
  // Against a launch each, the weight's gradient in 128 x 128 tiles: 16-bit 20 x 1024 x 1024 5.1 us in one, 7.5 in two, 20 x 2048 x 1024 9.7
  // and 8.4; 120 rows 7.8 and 8.7, 12.9 and 12.3.
  p.joint = p.pair.us() < (p.w.way == Way::Outer ? outer_cost(gw, dtype) - 0.2 : p.w.us + 5) + p.i.us && stream_part_bytes(gw, p.pair.gw) <= workspace_bytes;
  return p;
}

size_t ttlinear_backward_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const LinArgs gw = flags_args(N, K, M, 1, 0), gi = flags_args(M, K, N, 0, 0);
  const BackwardPlan p = plan_backward(gw, gi, dtype, ~(size_t)0);
  // one after the other on the same scratch; sizes do not say how rows are aligned (above)
  const size_t of_i = scratch_of(gi, p.i, dtype), of_w = scratch_of(gw, p.w, dtype, (size_t)pack_ranges(p.w.pack.kpad) * (size_t)N * sizeof(float));
  const size_t of_b = ttlinear_backward_least_workspace_bytes(dtype, M, N);
  size_t most = of_i > of_w ? of_i : of_w;
  if (stream_takes(gw, dtype) && stream_takes(gi, dtype)) {
    const size_t of_pair = stream_part_bytes(gw, (p.paired ? p.pair : plan_stream_pair(gw, gi, dtype)).gw);
    if (of_pair > most) most = of_pair;
  }
  return most > of_b ? most : of_b;
}

int ttlinear_backward_kernels(int dtype, int64_t M, int64_t N, int64_t K, int with_bias, ttlinear_kernel_info* of_weight,
                              ttlinear_kernel_info* of_input, int* one_launch) {
  if (!of_weight || !of_input || !one_launch) return TTSDPA_ERR_NULL;
  if (dtype != TTSDPA_F32 && dtype != TTSDPA_F16 && dtype != TTSDPA_BF16) return TTSDPA_ERR_DTYPE;
  if (M <= 0 || N <= 0 || K <= 0) return TTSDPA_ERR_SHAPE;
  LinArgs gw = flags_args(N, K, M, 1, 0);
  int sum;  // (never written: whether the row sums are wanted decides)
  gw.rowsum = with_bias ? &sum : nullptr;
  const LinArgs gi = flags_args(M, K, N, 0, 0);
  const BackwardPlan p = plan_backward(gw, gi, dtype, ~(size_t)0);
  *one_launch = p.joint;
  *of_weight = info_of(gw, p.w, dtype), *of_input = info_of(gi, p.i, dtype);
  if (p.joint) {
    const StreamTiles w = stream_tiles(gw, dtype, 1, p.pair.gw, &gi, p.pair.gi.R);
    *of_weight = {TTLINEAR_WAY_STREAM, w.rows, w.columns, w.per_workgroup, p.pair.gw.S};
    *of_input = {TTLINEAR_WAY_STREAM, 16 * p.pair.gi.R, 16 * p.pair.gi.R, 1, 1};
  }
  return TTSDPA_OK;
}

int ttlinear_backward(int dtype, const void* grad, const void* x, const void* w, void* grad_x, void* grad_w, void* grad_b, int64_t M,
                      int64_t N, int64_t K, int64_t ldg, int64_t ldx, int64_t ldw, void* workspace, size_t workspace_bytes,
                      void* stream) {
  if (dtype != TTSDPA_F32 && dtype != TTSDPA_F16 && dtype != TTSDPA_BF16) return TTSDPA_ERR_DTYPE;
  if (M <= 0 || N <= 0 || K <= 0) return TTSDPA_ERR_SHAPE;
  if (!grad || !x || !w || !grad_x || !grad_w) return TTSDPA_ERR_NULL;
  if (ldg < N || ldx < K || ldw < K) return TTSDPA_ERR_STRIDE;
  const size_t esz = dtype == TTSDPA_F32 ? 4 : 2;
  if (!aligned(grad, esz) || !aligned(x, esz) || !aligned(w, esz) || !aligned(grad_x, esz) || !aligned(grad_w, esz) || !aligned(grad_b, esz))
    return TTSDPA_ERR_STRIDE;
  if (workspace_bytes < ttlinear_backward_least_workspace_bytes(dtype, M, N) || !workspace || !aligned(workspace, 256))
    return TTSDPA_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  // grad_w [N,K] = grad^T . x, grad_x [M,K] = grad . w
  LinArgs gw{grad, x, nullptr, grad_w, N, K, M, ldg, ldx, K, 1, 1};
  gw.rowsum = grad_b;
  const LinArgs gi{grad, w, nullptr, grad_x, M, K, N, ldg, ldw, K, 0, 1};
  const BackwardPlan p = plan_backward(gw, gi, dtype, workspace_bytes);
  if (p.joint) return launch_stream_pair(gw, gi, dtype, s, p.pair, workspace);
  int rc = run(gi, p.i, dtype, workspace, workspace_bytes, s);
  if (rc != 0) return rc;
  if (p.w.way == Way::Stream || p.w.way == Way::Outer) return run(gw, p.w, dtype, workspace, workspace_bytes, s);
  gw.rowsum = nullptr;  // a launch of its own, or with the copies
  const PackPlan& pw = p.w.pack;
  const long long sums = pack_ranges(pw.kpad);
  if (p.w.way == Way::Packed && pw.x && workspace_bytes >= pw.bytes + (size_t)sums * (size_t)N * sizeof(float)) {
    // the column sums come with the transposed copy
    float* part = grad_b ? (float*)((char*)workspace + pw.bytes) : nullptr;
    rc = launch_packed(gw, pw, dtype, s, (char*)workspace, part);
    if (rc != 0 || !grad_b) return rc;
    switch (dtype) {
      case TTSDPA_F32: return launch_colsum_merge<float>(part, (int)sums, N, grad_b, s);
      case TTSDPA_F16: return launch_colsum_merge<_Float16>(part, (int)sums, N, grad_b, s);
      default: return launch_colsum_merge<__bf16>(part, (int)sums, N, grad_b, s);
    }
  }
  rc = run(gw, p.w, dtype, workspace, workspace_bytes, s);
  if (rc != 0 || !grad_b) return rc;
  const int ranges = colsum_ranges(M, N, dtype);
  switch (dtype) {
    case TTSDPA_F32: return launch_colsum<float>(grad, M, N, ldg, grad_b, (float*)workspace, ranges, s);
    case TTSDPA_F16: return launch_colsum<_Float16>(grad, M, N, ldg, grad_b, (float*)workspace, ranges, s);
    default: return launch_colsum<__bf16>(grad, M, N, ldg, grad_b, (float*)workspace, ranges, s);
  }
}

}  // extern "C"
