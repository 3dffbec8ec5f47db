// Shared device-side definitions for the gfx950 attention kernels.
#pragma once

#include <float.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace ttsdpa {

// Kernel argument block: the validated contents of ttsdpa_params plus derived values.
struct KArgs {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  const void* mask;
  const int* kv_len;  // per-batch valid key count (device), or nullptr
  const int* block_table;  // paged cache: page of key j of batch b = block_table[b * bt_stride + (j >> page_shift)], or nullptr
  int page_shift, bt_stride;
  int B, Hq, Hkv, L, S, D;
  int G;  // Hq / Hkv: query heads per KV head
  int causal;     // key j is visible to query i iff j <= i + offset
  int causal_br;  // offset: 0 (top-left aligned, the reference's mask) or max(0, keys of the batch entry - L) (bottom-right)
  int mask_kind;
  float scale;
  long long qs[3], ks[3], vs[3], os[3];  // element strides: batch, head, sequence
  long long ms[4];                       // mask element strides: batch, head, query row, key (0 = broadcast)
  // Packed query heads (4-wavefront prefill kernel only): the G query heads of a KV head are presented as one head of
  // G * pack_L rows (dense q / out make that a plain reshape); row x is query position x % pack_L.  0 = not packed.
  int pack_L;
  // Split keys (prefill kernels): workgroup (.., split) covers keys split * kv_chunk .. + kv_chunk - 1 of its row tile and leaves a
  // record per row in ws (store_split_record) for split_merge_kernel, or the output itself where the row tile's keys end in the
  // first split (the pipelined kernel of head_dim 64: a record then too).  kv_splits <= 1: no split.
  int kv_splits, kv_chunk;
  float* ws;
  int full_p;  // 4-wavefront prefill kernel with an attnMask: probabilities reach the matrix cores with all their fp32 bits
  int mask_vec4;  // keys are contiguous in the mask and groups of 4 keys starting at a multiple of 4 are naturally aligned
  // Pipelined prefill kernels under a causal mask: 0 = a workgroup takes a row tile and its mirror (equal work for all),
  // 1 = one row tile per workgroup, longest first (launches whose pairs would leave CUs without a workgroup).
  int single_tiles;
};

// Offset of the causal diagonal in key coordinates for a batch entry with S keys.
__device__ __forceinline__ int causal_offset(const KArgs& a, int S) {
  const int d = S - (a.pack_L ? a.pack_L : a.L);
  return (a.causal_br && d > 0) ? d : 0;
}

// Element offset of key tile kv0 (a multiple of the tile length, which divides the page size) from the K or V pointer
// of a (batch, kv head): `table` is the batch entry's row of the block table, or nullptr for a contiguous cache.  For
// paged caches the (batch, kv head) pointer carries the head offset only: pstride is the pool's page stride.
__device__ __forceinline__ long long kv_tile_offset(const KArgs& a, const int* table, int kv0, long long rstride, long long pstride) {
  if (!table) return (long long)kv0 * rstride;
  const int page = __builtin_amdgcn_readfirstlane(table[kv0 >> a.page_shift]);
  return (long long)page * pstride + (long long)(kv0 & ((1 << a.page_shift) - 1)) * rstride;
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr float kLog2e = 1.4426950408889634f;

// Kernels that use more than 64 KiB of dynamic LDS need that granted per kernel and per device.  Done on the first
// launch on a device (the device is the current one of the calling thread) and remembered; safe from several host
// threads (the worst case is granting twice).
constexpr int kMaxDevices = 64;
constexpr int kCusPerXcd = 32;  // MI355X: 256 compute units in 8 XCDs, each XCD with an L2 of its own
inline hipError_t grant_dynamic_lds(const void* kernel, int bytes, hipError_t (&state)[kMaxDevices], bool (&done)[kMaxDevices]) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (!__atomic_load_n(&done[dev], __ATOMIC_ACQUIRE)) {
    state[dev] = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    __atomic_store_n(&done[dev], true, __ATOMIC_RELEASE);
  }
  return state[dev];
}

// Element-type traits: storage is 16-bit (or fp32 for the general kernel), arithmetic is fp32.
struct BF16 {
  typedef __bf16 elem;
  typedef bf16x8 vec8;
  typedef bf16x4 vec4;
  static __device__ __forceinline__ f32x16 mfma32(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma16(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static constexpr int kParts = 3;  // parts that hold an fp32 number
  // the leading bits of eight numbers, which are left with the rest (exactly)
  static __device__ __forceinline__ vec8 take_part(f32x8& x) {
    u32x4 w;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float x0 = x[2 * i], x1 = x[2 * i + 1];
      const uint32_t a = __builtin_bit_cast(uint32_t, x0), b = __builtin_bit_cast(uint32_t, x1);
      w[i] = __builtin_amdgcn_perm(b, a, 0x07060302u);  // their upper halves
      x[2 * i] = x0 - __builtin_bit_cast(float, a & 0xffff0000u);
      x[2 * i + 1] = x1 - __builtin_bit_cast(float, b & 0xffff0000u);
    }
    return __builtin_bit_cast(vec8, w);
  }
  // fp32 value of the low / high 16-bit half of a packed pair
  static __device__ __forceinline__ float lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
  static __device__ __forceinline__ float hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
};

struct F16 {
  typedef _Float16 elem;
  typedef f16x8 vec8;
  typedef f16x4 vec4;
  static __device__ __forceinline__ f32x16 mfma32(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma16(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  static constexpr int kParts = 2;  // to 2^-22 of it
  static __device__ __forceinline__ vec8 take_part(f32x8& x) {
    vec8 y;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const auto w = __builtin_amdgcn_cvt_pkrtz(x[2 * i], x[2 * i + 1]);  // (towards zero)
      y[2 * i] = w[0], y[2 * i + 1] = w[1];
      x[2 * i] = fmaf(-1.f, (float)w[0], x[2 * i]);
      x[2 * i + 1] = fmaf(-1.f, (float)w[1], x[2 * i + 1]);
    }
    return y;
  }
  static __device__ __forceinline__ float lo(uint32_t w) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xffffu));
  }
  static __device__ __forceinline__ float hi(uint32_t w) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
  }
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ float load_as_float(const float* p) { return *p; }
__device__ __forceinline__ float load_as_float(const __bf16* p) { return (float)*p; }
__device__ __forceinline__ float load_as_float(const _Float16* p) { return (float)*p; }
__device__ __forceinline__ void store_from_float(float* p, float x) { *p = x; }
__device__ __forceinline__ void store_from_float(__bf16* p, float x) { *p = (__bf16)x; }
__device__ __forceinline__ void store_from_float(_Float16* p, float x) { *p = (_Float16)x; }

// The scores of a call with an attnMask, and what turns a difference of two of them into a power of two (scores_unit).  Bool:
// raw products, hidden keys at -inf.  Additive: score = raw * scale + bias, an fp32 number as in the reference's chain
// (src/Function/FuncNNLayer.h:237,249-260), whatever the bias: every finite value of the type is a key that counts.  A row may
// therefore lie at the lowest value altogether, and a kernel's maximum starts at -FLT_MAX (hidden keys only: -inf - -FLT_MAX
// gives weight 0) and is subtracted before anything is multiplied: with the bias divided by the scale and
// exp2(fma(s, c, -m*c)), rows at fp32's lowest value were NaN (an overflow; every weight 0 against a start at -1e30), and at
// -1e9 the rounding of m*c alone is a factor of 2^+-64.
__device__ __forceinline__ float scores_unit(const KArgs& a) { return a.mask_kind == 2 ? kLog2e : a.scale * kLog2e; }

// attnMask applied to the 32 x 32 score block of an MFMA accumulator (reference src/Function/FuncNNLayer.h:249-260):
// a lane holds one query row (mask row offset `mrow`, in elements) and, in register group rg, the four consecutive
// keys kv0 + 8*rg + 4*lh .. +3.  Element strides of 0 broadcast an axis.  Keys at or beyond S are left
// alone (masked by the caller).  Here the pipelined kernels' Bool masks (bool_mask_streams_ok: four keys at a time, S a multiple
// of 4) in their general steps, which have few registers to spare.
__device__ __forceinline__ void apply_bool_mask(const KArgs& a, f32x16& s, long long mrow, int kv0, int lh, int S) {
#pragma unroll
  for (int rg = 0; rg < 4; rg++) {
    const int key0 = kv0 + 8 * rg + 4 * lh;
    if (key0 < S) {
      const uint32_t w = *(const uint32_t*)((const uint8_t*)a.mask + mrow + key0);
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (((w >> (8 * e)) & 0xffu) == 0) s[4 * rg + e] = -INFINITY;
    }
  }
}

// Any attnMask, in two halves, so that a kernel can request a tile's mask ahead of the scores.  What is loaded: additive, the
// block's 16 values; Bool, four bytes in each of the first four words.  With contiguous keys a group of four is one load
// at whatever byte its row begins (rows of an odd length; global loads take any alignment), and the loads of a block
// are in flight together; a group that runs past the last key is read from key S - 4 on and shifted.  Other masks are read
// key by key.  S >= 1; values of keys at or beyond S are arbitrary: the caller hides those keys after the mask is applied.
// RAW (Bool): such a group is shifted when the mask is applied, not where it is read, where the wavefront waits for it.
template <typename T>
using MaskBlock = uint32_t __attribute__((ext_vector_type(4 * sizeof(T))));

template <typename T, bool RAW = false>
__device__ __forceinline__ MaskBlock<T> load_attn_mask(const KArgs& a, long long mrow, int kv0, int lh, int S) {
  constexpr int WPG = sizeof(T);  // words per group of four keys, additive
  typedef uint32_t loose32 __attribute__((aligned(1)));
  typedef uint32_t looseg __attribute__((ext_vector_type(WPG), aligned(sizeof(T))));
  MaskBlock<T> m = {};
  if (a.ms[3] == 1 && kv0 + 32 <= S) {
    const long long at = mrow + kv0 + 4 * lh;
    if (a.mask_kind == 1) {
      const uint8_t* p = (const uint8_t*)a.mask + at;
#pragma unroll
      for (int rg = 0; rg < 4; rg++) m[rg] = *(const loose32*)(p + 8 * rg);
    } else {
      const T* p = (const T*)a.mask + at;
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        const looseg w = *(const looseg*)(p + 8 * rg);
#pragma unroll
        for (int i = 0; i < WPG; i++) m[WPG * rg + i] = w[i];
      }
    }
  } else if (a.ms[3] == 1 && S >= 4) {
#pragma unroll
    for (int rg = 0; rg < 4; rg++) {
      const int key0 = kv0 + 8 * rg + 4 * lh;
      const int past = key0 > S - 4 ? key0 - (S - 4) : 0;
      if (a.mask_kind == 1) {
        m[rg] = *(const loose32*)((const uint8_t*)a.mask + mrow + (key0 - past)) >> (RAW ? 0 : 8 * (past & 3));
      } else {
        looseg w = *(const looseg*)((const T*)a.mask + mrow + (key0 - past));
        if constexpr (WPG == 2) {
          if (past & 2) w = looseg{w[1], 0};
          if (past & 1) w = looseg{(w[0] >> 16) | (w[1] << 16), w[1] >> 16};
        } else {
          if (past & 2) w = looseg{w[2], w[3], 0, 0};
          if (past & 1) w = looseg{w[1], w[2], w[3], 0};
        }
#pragma unroll
        for (int i = 0; i < WPG; i++) m[WPG * rg + i] = w[i];
      }
    }
  } else {
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int key = kv0 + 8 * (r >> 2) + 4 * lh + (r & 3);
      const long long at = mrow + (key < S ? key : S - 1) * a.ms[3];
      if (a.mask_kind == 1)
        m[r >> 2] |= (uint32_t)((const uint8_t*)a.mask)[at] << (8 * (r & 3));
      else if (WPG == 4)
        m[r] = ((const uint32_t*)a.mask)[at];
      else
        m[r >> 1] |= (uint32_t)((const uint16_t*)a.mask)[at] << (16 * (r & 1));
    }
  }
  return m;
}

// Whether a Bool mask's block lets any row of the wavefront see any of its keys (raw bytes, and those beyond the last key, may
// say so wrongly), and whether it hides none of them (told for the bytes 1 of a Bool tensor; other masks are applied).
template <typename T>
__device__ __forceinline__ bool mask_sees_any(const MaskBlock<T>& m) {
  return __builtin_amdgcn_ballot_w64((m[0] | m[1] | m[2] | m[3]) != 0) != 0;
}
template <typename T>
__device__ __forceinline__ bool mask_sees_all(const MaskBlock<T>& m) {
  return __builtin_amdgcn_ballot_w64((m[0] & m[1] & m[2] & m[3]) != 0x01010101u) == 0;
}

template <typename T, bool RAW = false>
__device__ __forceinline__ void apply_attn_mask(const KArgs& a, f32x16& s, MaskBlock<T> m, int kv0 = 0, int lh = 0, int S = 0) {
  if (RAW && a.ms[3] == 1 && kv0 + 32 > S && S >= 4) {
#pragma unroll
    for (int rg = 0; rg < 4; rg++) {
      const int key0 = kv0 + 8 * rg + 4 * lh;
      const int past = key0 > S - 4 ? key0 - (S - 4) : 0;
      m[rg] >>= 8 * (past & 3);
    }
  }
  constexpr int WPG = sizeof(T);
  if (a.mask_kind == 1) {
#pragma unroll
    for (int r = 0; r < 16; r++)
      if (((m[r >> 2] >> (8 * (r & 3))) & 0xffu) == 0) s[r] = -INFINITY;
  } else {
    typedef T vec16t __attribute__((ext_vector_type(16)));
    const vec16t b = __builtin_bit_cast(vec16t, m);
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = fmaf(s[r], a.scale, (float)b[r]);
  }
}

// Backward call: the forward's arguments (f.out holds the forward's result, an input here) plus the upstream gradient
// and the three gradients to write.  stats is scratch [B,Hq,L,2] floats: per query row a statistic of its scores and delta =
// dout . out.  Without an attnMask, in the MFMA kernels, the statistic is log2 of the sum of exponentials of the scaled
// scores.  With one, and in the vector-ALU kernels, it is the row's maximum, in the scores' own units (scores_unit), and
// log_sums ([B,Hq,L]) has the log of the sum relative to that maximum (log2 in the MFMA kernels, natural in the others; the
// two kernels of a call are always of one family): next to a maximum of -1e9 the sum's logarithm is lost to rounding, and
// such a row's weights were 1 each instead of 1 / keys.
struct BwdArgs {
  KArgs f;
  const void* dout;
  void* dq;
  void* dk;
  void* dv;
  long long dos[3], dqs[3], dks[3], dvs[3];  // element strides: batch, head, sequence
  float* stats;
  float* log_sums = nullptr;
  // matrix-core pairs only: with dkv_splits > 1 the query stream of every key block is dealt out to that many
  // workgroups, which leave partial dk / dv in `partial` ([split][dk | dv][B][Hkv][S][D] floats) for a third kernel to add.
  float* partial;
  int dkv_splits;
  // matrix-core pairs only: with dq_splits > 1 the key range of every 128-row query block is dealt out to that many
  // workgroups of the dq kernel, which leave their unnormalised fp32 sums in `dq_partial` ([split][B][Hq][L][D] floats,
  // then [split][B][Hq][L] pairs (maximum in log2 units, or with an attnMask the scores' own; sum of exponentials)) for
  // backward_dq_merge_kernel.
  float* dq_partial;
  int dq_splits;
  // dk/dv kernels under a causal mask: workgroups of an XCD that run together (CUs per XCD x workgroups per CU), or 0.
  // The workgroups of every second such round walk their query tiles upwards (dkv_walks_up).
  int dkv_round;
  // fp32 pair: the tiles of 32 rows' (keys') streams are dealt out to a workgroup's wavefronts (no splits then)
  bool dq_dealt = false, dkv_dealt = false;
};

// Splits of a backward launch that would leave half of the chip idle with `n`: its workgroups walk their streams tile by tile,
// tile_us each, however few they are.  The number, up to 16, whose longest stream, second launch and partial records (record_us
// for each split, written and read at 2 TB/s, in fp32, whose tiles hide half of it, 4) take least by estimate: bf16 2 x 4 heads on
// 1 x 199 rows, head_dim 128: whole backward 50 -> 37 us; fp32 8 heads on 1 x 2000 x 2000, head_dim 64: 665 -> 257.
inline int cheapest_backward_splits(int n, long long wgs, long long tiles, long long slots, double tile_us, double record_us) {
  if (wgs * n * 2 > slots) return n;
  auto us = [&](int k) {
    const double rounds = wgs * k > slots ? (double)(wgs * k) / (double)slots : 1.0;
    return (double)((tiles + k - 1) / k) * tile_us * rounds + (k > 1 ? 4.5 + k * record_us : 0.0);
  };
  int best = n;
  for (int k = n + 1; k <= 16; k++)
    if (us(k) < 0.9 * us(best)) best = k;
  return best;
}

// fp32: whether dealing a stream's tiles out to the four wavefronts of workgroups of 32 rows is shorter than n splits (`narrow`: such
// workgroups; one to a CU).
inline bool backward_tiles_dealt(int n, long long narrow, long long tiles, double tile_us, double record_us) {
  if (narrow > 256) return false;
  const double dealt = ((double)((tiles + 3) / 4) + 0.5) * tile_us, split = (double)((tiles + n - 1) / n) * tile_us + (n > 1 ? 4.5 + n * record_us : 0.0);
  return dealt < 0.8 * split;  // (a margin: one wavefront per SIMD hides less; 4 x 64 heads on 8 x 251 x 128 at 0.91: 313 us against 297)
}

// Workgroups that share a key block in the matrix-core dk/dv kernels (1: none, the kernel writes dk / dv itself): fp32, calls with an attnMask, and
// 16-bit head sizes other than 64 and 128 (those, without a mask: backward_splits_16bit).
// A dk/dv workgroup owns 128 keys and about one runs per CU at a time; under a causal mask its length varies
// 1 : (number of key blocks), and below about four workgroups per CU the longest ones set the time.  Without a causal
// mask all are equally long and splitting only serves to give every CU one (256 equal workgroups with an attnMask split further: 13-20 %
// slower).  A split must still get a few tiles.  `per_cu`: workgroups of the kernel that fit a CU (2 up to head_dim 64 without an attnMask, else 1).
inline int backward_dkv_splits(int B, int Hkv, int Hq, int L, int S, int D, bool causal, int per_cu, bool f32, bool* dealt) {
  const long long wgs = (long long)B * Hkv * ((S + 127) / 128);
  const long long tiles = (long long)(Hq / Hkv) * ((L + 31) / 32);  // the longest query stream, in 32-row tiles
  // causal: two rounds of the workgroups a CU holds at a time.  fp32 head_dim 128, 512 workgroups (B2 32q/8kv 4096 x 4096): splitting
  // them in two measured the same time, 60 % more bytes read and a third kernel for the partial sums; 256 of them (2048 x 2048) two
  // splits 76.5, four 74.1 TFLOP/s.
  const long long enough = causal ? 512LL * per_cu : 256 * per_cu;
  int n = 1;
  while (n < 4 && wgs * n < enough && tiles >= 16 * n && (D == 64 || D == 128)) n *= 2;  // (measured for these two sizes)
  const double record_us = (double)B * Hkv * S * D * 16 / (f32 ? 4e6 : 2e6), tile_us = f32 ? (D <= 64 ? 5.0 : 10.0) : D <= 64 ? 1.15 : 2.0;
  n = cheapest_backward_splits(n, wgs, tiles, 256 * per_cu, tile_us, record_us);
  *dealt = f32 && backward_tiles_dealt(n, (long long)B * Hkv * ((S + 31) / 32), tiles, tile_us, record_us);
  return *dealt ? 1 : n;
}

// Workgroups that share a 128-row query block in the matrix-core dq kernels (1: none, the kernel writes dq itself).
// The same calls.  A launch of fewer workgroups than the chip holds is split: that gives every slot a workgroup, and under a causal mask,
// where their lengths vary 1 : (number of row blocks) and they start longest first, a second round to end evenly.  A split must still get
// a few hundred keys.
// `slots`: workgroups of the kernel the chip holds at a time (512; 256 for the fp32 kernel at head_dim 128).
inline int backward_dq_splits(int B, int Hq, int L, int S, int D, bool causal, int slots, bool f32, bool* dealt) {
  *dealt = false;
  const long long wgs = (long long)B * Hq * ((L + 127) / 128);
  const long long tiles = (S + 31) / 32;  // the longest key range, in 32-key tiles
  if (wgs >= slots) return 1;
  const long long enough = causal ? 2 * slots : slots;
  int n = 1;
  while (n < 8 && wgs * n < enough && tiles >= 16 * n && (D == 64 || D == 128)) n *= 2;
  const double record_us = (double)B * Hq * L * D * 8 / (f32 ? 4e6 : 2e6), tile_us = f32 ? (D <= 64 ? 4.0 : 8.0) : D <= 64 ? 0.9 : 1.4;
  n = cheapest_backward_splits(n, wgs, tiles, slots, tile_us, record_us);
  *dealt = f32 && backward_tiles_dealt(n, (long long)B * Hq * ((L + 31) / 32), tiles, tile_us, record_us);
  return *dealt ? 1 : n;
}

// Splits of the 16-bit pair's kernels at head_dim 64 and 128 without an attnMask.  A launch of n splits takes, us, `launch` + a tile's time
// times the longest chain of tiles that a place for a workgroup runs, + (n > 1) the second launch and the partial records at `per_mb`.
// Fitted to 480 calls of 1 to 8 sequences, 1 to 64 heads, 100 to 4096 rows with the number of either kernel forced to 1 .. 8
// (the estimates' differences miss by 4 to 8 % of the call's time; the numbers they choose give 1 % less than the best ones).
// Records cost more than an uneven end: 4 x 8 heads x 1545 rows, head_dim 128, causal, dq in 4 splits 192 us, whole 143 (whole backward).
// Up to 16 pieces, where few blocks have long streams: 70 drawn calls of 9 to 16 pieces take 2 % more than with their best number, with
// 8 instead 6 % more (1 x 16 heads (2) x 1031, head_dim 64, dk/dv in 8 71 us, in 14 59); but dq at head_dim 64, in up to 16 instead of 8, lost 5 %
// (1 x 8 x 263 rows on 4859 keys in 14 52.4 us, in 8 49.4; 4 x 2 (1) x 424 on 3598 in 10 57.5, in 8 54.4).
// Records of keys that no row sees are zeros and cost half, while all records are `cached` MB or less (80 top-left causal calls on 2 to 12 times
// as many keys as rows: 4 % from their best, 1.5 % so; 4 x 64 heads (8) x 211 rows on 1711 keys, head_dim 64, dk/dv whole 85 us, in 3 pieces 67;
// beyond that not: 2 x 64 (8) x 841 on 7870, head_dim 128, whole 217, in two pieces, 259 MB, 248).
struct BackwardCost {
  double start, tile_us, launch, per_mb;  // start: what a workgroup costs beside its tiles, in tiles, where another one has its place before
  double cached = 0;
};
inline int backward_splits_16bit(const BackwardCost& c, bool of_keys, int B, int Hq, int Hkv, int L, int S, int D, bool causal, int offset) {
  const int slots = of_keys && D == 128 ? 256 : 512;  // workgroups side by side
  const int group = of_keys ? Hq / Hkv : 1, halves = of_keys && D == 128 ? 2 : 1;  // heads of a stream; wavefront groups that share it
  const int nblk = ((of_keys ? S : L) + 127) / 128;
  const long long heads = (long long)B * (of_keys ? Hkv : Hq);
  auto tiles = [&](int t) {  // of the t-th longest block
    if (!causal) return group * (((of_keys ? L : S) + 31) / 32);
    if (of_keys) {
      const int first = 128 * t - offset > 0 ? (128 * t - offset) / 32 : 0, all = (L + 31) / 32;
      return first < all ? group * (all - first) : 0;
    }
    const int row = 128 * (nblk - t) < L ? 128 * (nblk - t) : L, last = row + offset < S ? row + offset : S;
    return (last + 31) / 32;
  };
  // Tiles of all blocks of a head, in closed form (block by block, 65536 rows took 2.2 us of the host's time): under a causal mask a whole row
  // block has four more than the one above it, up to all keys, and a key block four less than the one before it, from the first that starts
  // behind the first row's keys on.
  double sum;
  if (!causal) {
    sum = (double)nblk * tiles(0);
  } else if (of_keys) {
    const long long all = ((long long)L + 31) / 32, o = ((long long)offset + 31) / 32, full = o / 4 + 1 < nblk ? o / 4 + 1 : nblk;
    const long long end = (all + o - 1) / 4 < nblk - 1 ? (all + o - 1) / 4 : nblk - 1;  // the last block that rows see
    const long long n = end >= full ? end - full + 1 : 0;
    sum = (double)group * (full * all + n * (all + o) - 2 * n * (full + end));
  } else {
    const long long all = ((long long)S + 31) / 32, ends = S > offset ? ((long long)S - offset - 1) / 128 : 0;
    const long long n = ends < nblk - 1 ? ends : nblk - 1;  // whole blocks that end before the keys do
    sum = (double)(n * (4 + ((long long)offset + 31) / 32) + 2 * n * (n - 1) + (nblk - 1 - n) * all + tiles(0));
  }
  const int longest = tiles(0);
  const long long blocks = heads * nblk;
  const double mb_each = of_keys ? 8e-6 * heads * S * D : 4e-6 * heads * L * (D + 2);  // records of a piece
  const long long end = (((long long)L + offset + 127) & ~127ll), seen = causal && end < S ? end : S;
  auto record_us = [&](int n) {
    const double mb = n * mb_each;
    return c.launch + c.per_mb * (mb <= c.cached ? mb * (seen + S) / (2.0 * S) : mb);
  };
  auto us = [&](int n, double most) {  // (`most` or more: it is not less)
    const double per = n * halves, more = n > 1 ? record_us(n) : 0;
    const long long wgs = blocks * n;
    double chain = ceil(longest / per);
    if (n > 1 && c.tile_us * chain + more >= most) return most;
    if (wgs > slots) {
      double next;
      if (!causal) {
        next = (wgs + slots - 1) / slots * (chain + c.start) - c.start;
      } else if (wgs <= 2 * slots) {
        const int each = (int)(heads * n);
        next = ceil(tiles((slots - 1) / each) / per) + ceil(tiles(slots / each) / per) + c.start;
      } else {
        next = heads * sum / halves / slots + 0.5 * tiles(nblk - 1) / per + c.start * ((double)wgs / slots - 1);
      }
      chain = next > chain ? next : chain;
    }
    return c.tile_us * chain + more;
  };
  int best = 1;
  double least = us(1, 0);
  const double even = heads * sum / halves / slots;
  const int most = of_keys || D == 128 ? 16 : 8;
  for (int n = 2; n <= most; n++) {
    // (in more than two rounds a place's chain is its share of all tiles at least, and more pieces only leave more records)
    if (blocks * n > 2 * slots && c.tile_us * even + record_us(n) > 0.951 * least) break;
    const double t = us(n, 0.95 * least);
    if (t < 0.95 * least) best = n, least = t;
  }
  return best;
}

// Workgroup id of a dk/dv launch with split query streams -> (key-block workgroup n, split).  The hardware hands
// workgroup id to XCD id % 8 and map_workgroup places n by n % 8: the splits of eight consecutive n follow each other in
// groups of eight, so that n % 8 == id % 8 and the order (longest key blocks first) is kept.
__device__ __forceinline__ void split_of_workgroup(int id, int nsplit, int npair, int* n, int* split) {
  if ((npair & 7) == 0) {
    const int r = id % (8 * nsplit);
    *split = r >> 3;
    *n = (id / (8 * nsplit)) * 8 + (r & 7);
  } else {
    *split = id % nsplit;
    *n = id / nsplit;
  }
}

// dk / dv = sum of the partials, split 0 first (a fixed order), converted to the tensors' element type.
template <typename T>
__global__ __launch_bounds__(256) void backward_dkv_sum_kernel(BwdArgs a, long long nvec) {
  typedef T vec4t __attribute__((ext_vector_type(4)));
  const KArgs& f = a.f;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;  // one group of four elements of dk and of dv
  if (i >= nvec) return;
  const int dvec = f.D / 4;
  const int d = 4 * (int)(i % dvec);
  long long row = i / dvec;
  const int key = (int)(row % f.S);
  row /= f.S;
  const int hk = (int)(row % f.Hkv), b = (int)(row / f.Hkv);
  const long long plane = (long long)f.B * f.Hkv * f.S * f.D;
  const float* p = a.partial + 4 * i;
  f32x4 x = *(const f32x4*)p, y = *(const f32x4*)(p + plane);
  for (int s = 1; s < a.dkv_splits; s++) {
    x += *(const f32x4*)(p + 2 * s * plane);
    y += *(const f32x4*)(p + (2 * s + 1) * plane);
  }
  *(vec4t*)((T*)a.dk + b * a.dks[0] + hk * a.dks[1] + key * a.dks[2] + d) = __builtin_convertvector(x, vec4t);
  *(vec4t*)((T*)a.dv + b * a.dvs[0] + hk * a.dvs[1] + key * a.dvs[2] + d) = __builtin_convertvector(y, vec4t);
}
template <typename T>
int launch_backward_dkv_sum(const BwdArgs& a, hipStream_t stream) {
  const long long nvec = (long long)a.f.B * a.f.Hkv * a.f.S * (a.f.D / 4);
  hipLaunchKernelGGL(backward_dkv_sum_kernel<T>, dim3((unsigned)((nvec + 255) / 256)), dim3(256), 0, stream, a, nvec);
  return (int)hipGetLastError();
}
// A lane's share of a query row's unnormalised dq sums (accumulator layout of the 32 x 32 matrix instructions: registers 4rg .. 4rg+3 of block db are
// elements 32db + 8rg + 4lh .. +3) and the row's (maximum, sum of exponentials) as this split's partial record; split 0 also
// leaves delta for the dk/dv kernel.
template <int D, bool PAD = false>
__device__ __forceinline__ void store_dq_partial(const BwdArgs& a, int piece, long long row_id, int lh, const f32x16 (&dqacc)[D / 32],
                                                 float m, float l_tot, float delta) {
  const long long rows = (long long)a.f.B * a.f.Hq * a.f.L;
  const int have = PAD ? a.f.D : D;
  float* dst = a.dq_partial + (piece * rows + row_id) * have;
#pragma unroll
  for (int db = 0; db < D / 32; db++)
#pragma unroll
    for (int rg = 0; rg < 4; rg++) {
      f32x4 x;
#pragma unroll
      for (int i = 0; i < 4; i++) x[i] = dqacc[db][4 * rg + i];
      if (!PAD || 32 * db + 8 * rg + 4 * lh < have) *(f32x4*)(dst + 32 * db + 8 * rg + 4 * lh) = x;
    }
  if (lh == 0) {
    float* ml = a.dq_partial + a.dq_splits * rows * have;
    *(float2*)(ml + 2 * (piece * rows + row_id)) = make_float2(m, l_tot);
    if (piece == 0) a.stats[2 * row_id + 1] = delta;
  }
}

// A row's statistics in a call with an attnMask (matrix-core pairs); a row whose keys are all hidden gets a maximum and a
// logarithm that give it weight 0 in the dk/dv kernel, and a delta of 0: its own is NaN (the forward's output there), which 0
// times would leave in dk.
__device__ __forceinline__ void store_masked_stat(const BwdArgs& a, long long row_id, bool seen, float m, float l, float delta) {
  *(float2*)(a.stats + 2 * row_id) = make_float2(seen ? m : FLT_MAX, seen ? delta : 0.f);
  a.log_sums[row_id] = seen ? __log2f(l) : 1e30f;
}

// dq of a call whose key ranges were split: the splits' sums brought to the common maximum, added in a fixed order (split
// 0 first) and normalised; the row statistic for the dk/dv kernel.  One thread per four elements of a row.
template <typename T>
__global__ __launch_bounds__(256) void backward_dq_merge_kernel(BwdArgs a, long long nvec) {
  typedef T vec4t __attribute__((ext_vector_type(4)));
  const KArgs& f = a.f;
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= nvec) return;
  const int dvec = f.D / 4;
  const int d = 4 * (int)(i % dvec);
  const long long row_id = i / dvec;  // (b * Hq + h) * L + qi
  const int qi = (int)(row_id % f.L);
  const long long bh = row_id / f.L;
  const int h = (int)(bh % f.Hq), b = (int)(bh / f.Hq);
  const long long rows = (long long)f.B * f.Hq * f.L;
  const float* ml = a.dq_partial + (long long)a.dq_splits * rows * f.D;
  vec4t* out = (vec4t*)((T*)a.dq + b * a.dqs[0] + h * a.dqs[1] + qi * a.dqs[2] + d);
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
  int S = f.S;
  if (f.kv_len) {
    const int len = f.kv_len[b];
    S = len < 0 ? 0 : (len < S ? len : S);
  }
  if (S == 0) {  // no keys: the dq kernel's workgroups returned at once
    *out = __builtin_convertvector(x, vec4t);
    return;
  }
  const float unit = f.mask_kind != 0 ? scores_unit(f) : 1.f;
  float m = -INFINITY;
  for (int s = 0; s < a.dq_splits; s++) m = fmaxf(m, ml[2 * (s * rows + row_id)]);
  float l = 0.f;
  for (int s = 0; s < a.dq_splits; s++) {
    const float2 st = *(const float2*)(ml + 2 * (s * rows + row_id));
    const float w = fast_exp2((st.x - m) * unit);
    l += st.y * w;
    x += *(const f32x4*)(a.dq_partial + (s * rows + row_id) * f.D + d) * w;
  }
  // a row whose keys are all hidden: dq = 0, and a statistic that gives it weight 0 in the dk/dv kernel
  const bool seen = l > 0.f;
  const float w = seen ? f.scale / l : 0.f;
#pragma unroll
  for (int e = 0; e < 4; e++) x[e] = seen ? x[e] * w : 0.f;
  *out = __builtin_convertvector(x, vec4t);
  if (d == 0) {
    if (f.mask_kind != 0) store_masked_stat(a, row_id, seen, m, l, a.stats[2 * row_id + 1]);
    else a.stats[2 * row_id] = seen ? m + __log2f(l) : 1e30f;
  }
}
template <typename T>
int launch_backward_dq_merge(const BwdArgs& a, hipStream_t stream) {
  const long long nvec = (long long)a.f.B * a.f.Hq * a.f.L * (a.f.D / 4);
  hipLaunchKernelGGL(backward_dq_merge_kernel<T>, dim3((unsigned)((nvec + 255) / 256)), dim3(256), 0, stream, a, nvec);
  return (int)hipGetLastError();
}
int launch_backward_general(const BwdArgs& a, int dtype, hipStream_t stream);
int launch_backward_mfma(const BwdArgs& a, int dtype, hipStream_t stream);  // fp16/bf16, head_dim 64 or 128
int launch_backward_dq_d128(const BwdArgs& a, bool bf16, hipStream_t stream);   // its kernels at head_dim 128 without an attnMask
int launch_backward_dkv_d128(const BwdArgs& a, bool bf16, hipStream_t stream);
int launch_backward_f32(const BwdArgs& a, int dtype, hipStream_t stream);   // on the fp32 matrix cores, head_dim 64 or 128: fp32, and fp16/bf16 with an attnMask

// Workgroup n -> (pair, block) for npair (batch, head) pairs of nblk blocks each, block 0 the longest under a causal
// mask.  Workgroups are handed to the 8 XCDs round-robin (n % 8) and start in order: every XCD gets whole pairs (a
// contiguous range, so the heads of a group share its L2) and takes their blocks longest first across all its pairs,
// which keeps the XCDs evenly loaded and the short blocks for the end.  Without a multiple of 8 pairs: longest first
// over all pairs.
__device__ __forceinline__ void map_workgroup(int n, int npair, int nblk, int* pair, int* blk) {
  if ((npair & 7) == 0) {
    const int xcd = n & 7, slot = n >> 3, ppx = npair >> 3;
    *blk = slot / ppx;
    *pair = xcd * ppx + slot % ppx;
  } else {
    *blk = n / npair;
    *pair = n % npair;
  }
}

// head_dim 128 needs more than 256 registers per lane: one wavefront per SIMD, the gradient accumulators in the
// accumulation registers.  Pinning them there at the end of every iteration keeps the loop-carried values in that
// register class, so the matrix instructions accumulate in place instead of being fed through copies (128 moves each
// way per tile otherwise).
template <bool PIN>
__device__ __forceinline__ void pin_accumulator(f32x16& acc) {
  if constexpr (PIN) asm volatile("" : "+a"(acc));
}

// A lane's share of the dk / dv rows of key `key` (accumulator layout: registers 4rg .. 4rg+3 of block db are elements
// 32db + 8rg + 4lh .. +3) goes to the gradient tensors, or — when the key block's query stream is split over several
// workgroups — as fp32 to this split's partial sums, dense [split][dk | dv][B][Hkv][S][D].
// PAD: the tensors' head_dim a.f.D is a multiple of 8 below D; only its columns are written.
template <typename TR, int D, bool PAD = false>
__device__ __forceinline__ void store_key_grads(const BwdArgs& a, int split, int b, int hk, int key, int lh,
                                                const f32x16 (&dkacc)[D / 32], const f32x16 (&dvacc)[D / 32], float scale) {
  typedef typename TR::elem T;
  if (key >= a.f.S) return;
  if (a.dkv_splits > 1) {
    const int have = PAD ? a.f.D : D;
    const long long plane = (long long)a.f.B * a.f.Hkv * a.f.S * have;
    float* dkp = a.partial + 2 * split * plane + (((long long)b * a.f.Hkv + hk) * a.f.S + key) * have;
#pragma unroll
    for (int db = 0; db < D / 32; db++)
#pragma unroll
      for (int rg = 0; rg < 4; rg++) {
        f32x4 x, y;
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = dkacc[db][4 * rg + i] * scale, y[i] = dvacc[db][4 * rg + i];
        if (PAD && 32 * db + 8 * rg + 4 * lh >= have) continue;
        *(f32x4*)(dkp + 32 * db + 8 * rg + 4 * lh) = x;
        *(f32x4*)(dkp + plane + 32 * db + 8 * rg + 4 * lh) = y;
      }
    return;
  }
  T* dkp = (T*)a.dk + b * a.dks[0] + hk * a.dks[1] + key * a.dks[2];
  T* dvp = (T*)a.dv + b * a.dvs[0] + hk * a.dvs[1] + key * a.dvs[2];
#pragma unroll
  for (int db = 0; db < D / 32; db++)
#pragma unroll
    for (int rg = 0; rg < 4; rg++) {
      f32x4 x, y;
#pragma unroll
      for (int i = 0; i < 4; i++) x[i] = dkacc[db][4 * rg + i] * scale, y[i] = dvacc[db][4 * rg + i];
      if (PAD && 32 * db + 8 * rg + 4 * lh >= a.f.D) continue;
      *(typename TR::vec4*)(dkp + 32 * db + 8 * rg + 4 * lh) = __builtin_convertvector(x, typename TR::vec4);
      *(typename TR::vec4*)(dvp + 32 * db + 8 * rg + 4 * lh) = __builtin_convertvector(y, typename TR::vec4);
    }
}

// dk and dv rows of a key no query row attends to (at or beyond the batch entry's key count): zeros.
template <typename TR, int D, bool PAD = false>
__device__ __forceinline__ void zero_key_rows(const BwdArgs& a, int split, int b, int hk, int key, int lh) {
  f32x16 zero[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) zero[i][r] = 0.f;
  store_key_grads<TR, D, PAD>(a, split, b, hk, key, lh, zero, zero, 0.f);
}

// Direction in which a dk/dv workgroup walks the query tiles it0 .. ntq-1 that see its key block.  The workgroups of an XCD
// start longest first (map_workgroup), `dkv_round` of them at a time.  Those of the first round start together at the last
// tile and walk down in step (the tile one fetches is in the XCD's L2 for the others); the workgroup of key block kb ends
// after ntq - it0(kb) tiles, and the CU it frees takes the longest block left, which has as many tiles as the first had
// few.  Walking UP from its first tile, that workgroup is at the same tile at the same time as every other one of the
// second round (all arrive at the last tile together); walking down, each would be alone with its position and fetch
// its tiles from memory itself.  The third round starts together again: rounds alternate.  (bf16 head_dim 128, B2 32q/8kv
// 4096 x 4096: 458 -> 240 MB read per launch of the dk/dv kernel.)
// The splits of a key block walk alike, whatever round each is in: wg, its place without splits.
__device__ __forceinline__ bool dkv_walks_up(const BwdArgs& a, bool causal, int wg) {
  return causal && a.dkv_round > 0 && ((a.f.B * a.f.Hkv) & 7) == 0 && (((wg >> 3) * a.dkv_splits / a.dkv_round) & 1) != 0;
}

// Workgroups of `kernel` that fit one CU, times the CUs of an XCD: the dkv_round of a launch (looked up once per device).
inline int dkv_round_of(const void* kernel, int threads, int lds_bytes, int (&cache)[kMaxDevices]) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
  if (cache[dev] == 0) {
    int n = 0;
    cache[dev] = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, (size_t)lds_bytes) == hipSuccess && n > 0 ? n * kCusPerXcd : -1;
  }
  return cache[dev] > 0 ? cache[dev] : 0;
}

// A Bool attnMask the pipelined prefill kernels' streams can apply: four keys per aligned dword, row offsets of a
// (batch, head) within 32 bits, no causal flag, per-batch key counts, pages or key splits beside it.
inline bool bool_mask_streams_ok(const KArgs& a) {
  return !a.causal && a.mask_kind == 1 && a.mask_vec4 && (a.S % 4) == 0 && !a.kv_len && !a.block_table && a.kv_splits <= 1 &&
         (long long)(a.L - 1) * a.ms[2] + 8 < (1ll << 32);
}

// Host-side launchers (one per kernel family); each returns a hipError_t as int.
int launch_general(const KArgs& a, int dtype, hipStream_t stream);
int launch_prefill(const KArgs& a, int dtype, hipStream_t stream);       // 128-row workgroups; head_dim 64 or 128
int launch_prefill_d128(const KArgs& a, int dtype, hipStream_t stream);  // 256-row workgroups, pipelined; head_dim 128
int launch_prefill_d64(const KArgs& a, int dtype, hipStream_t stream);   // the same at head_dim 64 (no attnMask, no pages)
int launch_prefill_dealt(const KArgs& a, int dtype, hipStream_t stream);  // 128-row workgroups, keys dealt out to two groups of wavefronts; head_dim 128 or 64
int launch_prefill_f32(const KArgs& a, hipStream_t stream);              // fp32 tensors on the fp32 matrix cores; head_dim 64 or 128
// key tiles (of 32) that an unsplit launch takes one after the other; dealt: its wavefronts share a row tile's
double prefill_f32_tiles(const KArgs& a, bool* dealt = nullptr);
int heads_rows(const KArgs& a, int dtype);                                     // whether, and how, launch_heads is the way for a call
int launch_heads(const KArgs& a, int dtype, hipStream_t stream);            // with an attnMask, up to 256 keys, 16-bit tensors (sdpa_heads.hip)
int launch_short_forward(const KArgs& a, int dtype, hipStream_t stream);    // short sequences, any element type (sdpa_short.hip)
int launch_short_backward(const BwdArgs& a, int dtype, bool joint, hipStream_t stream);  // joint: in one launch
int launch_decode(const KArgs& a, int dtype, void* workspace, hipStream_t stream);

// Keys of batch entry b: all S of them, or the filled prefix of a cache / the unpadded length (kv_len).
__device__ __forceinline__ int keys_of_batch(const KArgs& f, int b) {
  int S = f.S;
  if (f.kv_len) {
    const int len = __builtin_amdgcn_readfirstlane(f.kv_len[b]);
    S = len < 0 ? 0 : (len < S ? len : S);
  }
  return S;
}

// The last key that any row of the row tile q0 .. q0 + rows - 1 sees in a batch entry with S keys (-1: none).
__device__ __forceinline__ int last_key_of_rows(const KArgs& a, int q0, int rows, int S) {
  int last = S - 1;
  if (a.causal) {
    const int v = (a.pack_L ? a.pack_L - 1 : (q0 + rows < a.L ? q0 + rows : a.L) - 1) + causal_offset(a, S);
    last = v < last ? v : last;
  }
  return last;
}

// XCD-aware order of the (batch, KV head) pairs: workgroup n runs on XCD n % 8, and with gq = gcd(pairs, 8) the XCDs form gq classes of
// 8 / gq, class x % gq serves the pairs congruent to it and deals their work items out to its XCDs in turn.
__host__ __device__ inline int pair_classes(int npair) { return (npair & 7) == 0 ? 8 : ((npair & 3) == 0 ? 4 : ((npair & 1) == 0 ? 2 : 1)); }
// ... of a split launch: entries of unlike lengths are all in every class.
__host__ __device__ inline int split_classes(const KArgs& a) { return pair_classes(a.kv_len && a.B > 1 ? a.Hkv : a.B * a.Hkv); }

// The piece of a split launch of a prefill kernel (row tiles of `rows` rows) that this workgroup takes.  A class's pieces start in
// this order: every row tile's first split, longest row tile first, then every row tile's second one ... (those that run together
// read the same keys), and without gaps: a workgroup with nothing to do among the others leaves CUs empty (workgroups go to the
// parts of an XCD in turn: 2 heads on 1 of 8192 rows, head_dim 128, 68 us with gaps, 42 so; the merge takes 5 more).
// False: nothing is left for this one.
// in: the head in its group and the row tile (longest first under a causal mask).
__device__ __forceinline__ bool find_piece(const KArgs& a, int rows, bool causal, int* pair, int* in, int* split) {
  const int gq = split_classes(a), ppc = a.B * a.Hkv / gq;
  const int xcd = blockIdx.x & 7, cls = xcd % gq;
  int q = (int)(blockIdx.x >> 3) * (8 / gq) + xcd / gq;
  const int ntile = (a.L + rows - 1) / rows;
  const bool alike = !a.kv_len || a.B == 1;
  const int own = alike ? 1 : ppc, same = alike ? a.G * ppc : a.G;  // pairs of unlike lengths one by one, else all together
  // every split has all row tiles, or is beyond the keys: the caller returns; and launches of 128-row workgroups that fit the
  // CUs in one go, or nearly with one row tile a head, which gaps do not slow (the 4-wavefront kernels: 3 heads x 136 rows on 1115 keys, ragged, 10.2
  // us with the search below, 8.6 so; 9 x 8 heads x 16 rows on 10495, 792 pieces, 36.2 and 35.0; 8 x 4 x 512 on 5000 35.5 and 37.6; the
  // kernel with dealt keys: 60 drawn calls 2 % faster so, -1 to 5)
  const bool few = rows <= 128 && a.B * a.Hkv * a.G * ntile * a.kv_splits <= (ntile == 1 ? 1024 : 256);
  if (few || (alike && (!causal || a.pack_L))) {
    const int same = a.G * ppc;
    const int s = q / (same * ntile), w = q - s * (same * ntile), t = w / same, h = w - t * same;
    *split = __builtin_amdgcn_readfirstlane(s), *pair = __builtin_amdgcn_readfirstlane(cls + gq * (h % ppc));
    *in = __builtin_amdgcn_readfirstlane(t * a.G + h / ppc);
    return *split < a.kv_splits;
  }
  // a lane to each (split, pair): how many pieces it has, and where they begin
  const int lane = threadIdx.x & 63;
  for (int at = 0; at < a.kv_splits * own; at += 64) {
    const int s = (at + lane) / own, i = (at + lane) - s * own;
    int S = a.S;
    if (a.kv_len) {
      const int len = a.kv_len[(cls + gq * i) / a.Hkv];
      S = len < 0 ? 0 : (len < S ? len : S);
    }
    const int first = s * a.kv_chunk;
    int tiles = s < a.kv_splits && first < S ? ntile : 0;  // row tiles that see the split's first key: the last ones under a causal mask
    if (causal && tiles) {
      const int row = first - causal_offset(a, S);  // the first row that does
      if (a.pack_L) tiles = row >= a.pack_L ? 0 : ntile;  // (a row tile of packed heads has rows of all positions)
      else tiles = row >= a.L ? 0 : ntile - (row > 0 ? row / rows : 0);
    }
    int end = same * tiles;
#pragma unroll
    for (int off = 1; off < 64; off *= 2) {
      const int x = __shfl_up(end, off);
      end += lane >= off ? x : 0;
    }
    const unsigned long long later = __builtin_amdgcn_ballot_w64(end > q);
    if (later != 0) {
      const int l = __builtin_ctzll(later), before = l ? __builtin_amdgcn_readlane(end, l ? l - 1 : 0) : 0;
      const int t = (q - before) / same, w = (q - before) - t * same, p = alike ? w % ppc : __builtin_amdgcn_readlane(i, l);
      *split = __builtin_amdgcn_readlane(s, l), *pair = __builtin_amdgcn_readfirstlane(cls + gq * p);
      *in = __builtin_amdgcn_readfirstlane(t * a.G + (alike ? w / ppc : w));
      return true;
    }
    q -= __builtin_amdgcn_readlane(end, 63);
  }
  return false;
}
// Workgroups of such a launch: the most pieces there can be.
inline long long split_grid(const KArgs& a, int rows) {
  const int gq = split_classes(a);
  const long long per_class = (long long)(a.B * a.Hkv / gq) * a.G * ((a.L + rows - 1) / rows) * a.kv_splits;
  return (per_class + 8 / gq - 1) / (8 / gq) * 8;
}

// What a split leaves of 32 rows (a wavefront's, row0 a multiple of 32; W: the kernel's head_dim): the unnormalised accumulators as
// the lanes hold them, [W/32][4][64 lanes] groups of four, then the rows' maxima and sums.  Every store covers whole lines (a lane
// its own row's 8-byte pieces: 1 TB/s).
template <int W>
__device__ __forceinline__ void store_split_record(const KArgs& a, long long bh, int split, int row0, int lane, const f32x16 (&acc)[W / 32],
                                                   float m, float l) {
  if (row0 >= a.L) return;
  float* rec = a.ws + ((bh * a.kv_splits + split) * ((a.L + 31) / 32) + row0 / 32) * (32 * (W + 2));
#pragma unroll
  for (int db = 0; db < W / 32; db++)
#pragma unroll
    for (int rg = 0; rg < 4; rg++)
      *(f32x4*)(rec + 256 * (4 * db + rg) + 4 * lane) = (f32x4){acc[db][4 * rg], acc[db][4 * rg + 1], acc[db][4 * rg + 2], acc[db][4 * rg + 3]};
  rec[32 * W + lane] = lane < 32 ? m : l;
}
inline size_t split_record_bytes(long long heads, int L, int splits, int W) {
  return (size_t)heads * splits * ((L + 31) / 32) * 32 * (W + 2) * sizeof(float);
}

// The records of a split launch of a prefill kernel -> out; W: the kernel's head_dim >= a.D, `rows`: of its row tiles.  A workgroup
// takes 32 columns of 32 rows: each row's splits up to its last visible key, brought to their common maximum, added in split order,
// normalised, and through LDS into whole pieces of rows.  Row tiles whose keys end in the first split are in the output already
// (rows = 0: none are).
// Rows of a batch entry without keys: zeros (weightless rows: ttsdpa.h).
template <typename T>
__global__ __launch_bounds__(256) void split_merge_kernel(KArgs a, int W, int rows) {
  constexpr int E = 16 / sizeof(T), PITCH = 32 + E;
  __shared__ __attribute__((aligned(16))) T tile[32 * PITCH];
  const int nblk = (a.L + 31) / 32;
  const int blk = blockIdx.x % nblk;
  const long long bh = blockIdx.x / nblk;
  const int h = (int)(bh % a.Hq), b = (int)(bh / a.Hq);
  const int t = threadIdx.x, lane = t & 63, rg = t >> 6, db = blockIdx.y;
  const int r = lane & 31, row = 32 * blk + r;
  int S = a.S;
  if (a.kv_len) {
    const int len = a.kv_len[b];
    S = len < 0 ? 0 : (len < S ? len : S);
  }
  const int last = rows ? last_key_of_rows(a, 32 * blk / rows * rows, rows, S) : S - 1;
  if (rows && last >= 0 && last < a.kv_chunk) return;
  int own = S - 1;  // the row's last key (packed heads: of any position)
  if (a.causal && !a.pack_L) {
    const int v = row + causal_offset(a, S);
    own = v < own ? v : own;
  }
  int n = last < 0 ? 0 : (own < last ? own : last) / a.kv_chunk + 1;
  n = n < a.kv_splits ? n : a.kv_splits;
  const float c = scores_unit(a);
  const long long step = (long long)nblk * (32 * (W + 2));
  const float* rec = a.ws + (bh * a.kv_splits * nblk + blk) * (32 * (W + 2));
  const float* ml = rec + 32 * W + r;
  const float* acc = rec + 256 * (4 * db + rg) + 4 * lane;
  float m = -FLT_MAX, l = 0.f;
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
  // the loads of a batch of splits are in flight together; a batch's places beyond the last split re-read that one
  auto add_up = [&](auto batch) __attribute__((always_inline)) {
    constexpr int N = decltype(batch)::value;
    if (n > N) {  // (one batch: with its sums and values, below)
      for (int s = 0; s < n; s += N) {
        float v[N];
#pragma unroll
        for (int j = 0; j < N; j++) v[j] = ml[(s + j < n ? s + j : n - 1) * step];
#pragma unroll
        for (int j = 0; j < N; j++) m = fmaxf(m, v[j]);
      }
    }
    for (int s = 0; s < n; s += N) {
      float v[N], sums[N];
      f32x4 y[N];
#pragma unroll
      for (int j = 0; j < N; j++) {
        const long long at = (s + j < n ? s + j : n - 1) * step;
        v[j] = ml[at], sums[j] = ml[at + 32], y[j] = *(const f32x4*)(acc + at);
        if (s + j >= n) sums[j] = 0.f, y[j] = (f32x4){0.f, 0.f, 0.f, 0.f};  // (not a weight of 0: the sums may be infinite)
      }
      if (n <= N) {
#pragma unroll
        for (int j = 0; j < N; j++) m = fmaxf(m, v[j]);
      }
#pragma unroll
      for (int j = 0; j < N; j++) {
        const float w = fast_exp2((v[j] - m) * c);
        l = fmaf(w, sums[j], l);
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = fmaf(w, y[j][e], x[e]);
      }
    }
  };
  if (n <= 2) add_up(std::integral_constant<int, 2>{});
  else if (n <= 4) add_up(std::integral_constant<int, 4>{});
  else add_up(std::integral_constant<int, 8>{});
  const float inv = n > 0 ? 1.f / l : 0.f;
#pragma unroll
  for (int e = 0; e < 4; e++) tile[r * PITCH + 8 * rg + 4 * (lane >> 5) + e] = (T)(x[e] * inv);
  __syncthreads();
  constexpr int CH = 32 / E;  // 16-byte pieces of a row's 32 columns
  if (t < 32 * CH) {
    const int orow = 32 * blk + t / CH, d = 32 * db + E * (t % CH);
    if (orow < a.L && d < a.D)
      *(u32x4*)((T*)a.out + b * a.os[0] + h * a.os[1] + orow * a.os[2] + d) = *(const u32x4*)(tile + t / CH * PITCH + E * (t % CH));
  }
}

int launch_split_merge(const KArgs& a, int dtype, int W, int rows, hipStream_t stream);  // split_merge_kernel (sdpa_prefill.hip)
int launch_zero(const KArgs& a, int dtype, hipStream_t stream);
struct KvAppendArgs {
  void* kc;
  void* vc;
  const void* kn;
  const void* vn;
  const int* positions;
  const int* block_table;  // paged caches, as in KArgs
  int page_shift, bt_stride;
  int B, Hkv, Smax, Lnew, D, position, esz;
  long long kcs[3], vcs[3], kns[3], vns[3];
};
int launch_kv_append(const KvAppendArgs& a, hipStream_t stream);

// Decode tiling, shared by the workspace-size query and the launcher.
struct DecodePlan {
  int splits;      // KV splits per (batch, kv head)
  int chunk;       // keys per split (multiple of the per-wave key block)
  int rows;        // query rows handled together per KV head: L * G
  size_t ws_bytes; // workspace: per (batch, kv head, split): rows * (D + 2) floats
  int waves;  // wavefronts of a workgroup: 4, or 8 (up to 8 query rows)
};
DecodePlan plan_decode(const KArgs& a, bool f32);

constexpr int kDecodeMaxRows = 16;  // L * (Hq/Hkv) handled by one MFMA row block

}  // namespace ttsdpa
