// KV-cache append: writes the new tokens' K and V rows into preallocated caches [B,Hkv,Smax,D] (or page pools
// [pages,Hkv,page_size,D] addressed through a block table) at per-batch positions.
// The reference grows K/V with op::concat on the sequence axis (reference src/Operation/OpTransform.cpp:306-357), which
// copies the whole history for every generated token; here only the new rows move.  HBM-bound by construction:
// 2 * B*Hkv*Lnew*D elements read and written once, 16 bytes per lane when rows allow it.

#include "sdpa_common.h"

namespace ttsdpa {

namespace {

// A decode step's call is a few rows and all latency: the new rows are requested beside the positions, not behind them, and the
// indices are divided in 32 bits where they fit (I; 64-bit divisions are some 60 instructions each).  In a layer's step, head_dim 128,
// medians under the profiler: 8 heads x 1 row 2.7 -> 2.0 us, 24 sequences x 4 heads 3.7 -> 2.9 (with cold positions 4.8 both ways).
template <int VEC, typename I>  // bytes per lane and access
__global__ __launch_bounds__(256) void kv_append_kernel(KvAppendArgs a) {
  typedef uint32_t word_t __attribute__((ext_vector_type(VEC >= 4 ? VEC / 4 : 1)));
  typedef typename std::conditional<VEC == 2, uint16_t, word_t>::type piece_t;
  const int row_bytes = a.D * a.esz;
  const int per_row = row_bytes / VEC;
  const I total = (I)((long long)a.B * a.Hkv * a.Lnew * per_row);
  for (I e = (I)blockIdx.x * 256 + threadIdx.x; e < total; e += (I)gridDim.x * 256) {
    I r = e / (I)per_row;
    const int piece = (int)(e - r * (I)per_row);
    I q = r / (I)a.Lnew;
    const int l = (int)(r - q * (I)a.Lnew);
    const int b = (int)(q / (I)a.Hkv), hk = (int)(q - (I)b * (I)a.Hkv);
    const char* ksrc = (const char*)a.kn + (b * a.kns[0] + hk * a.kns[1] + l * a.kns[2]) * a.esz + piece * VEC;
    const char* vsrc = (const char*)a.vn + (b * a.vns[0] + hk * a.vns[1] + l * a.vns[2]) * a.esz + piece * VEC;
    const piece_t kx = *(const piece_t*)ksrc, vx = *(const piece_t*)vsrc;
    const int pos = (a.positions ? a.positions[b] : a.position) + l;
    if (pos < 0 || pos >= a.Smax) continue;  // no room: the row is dropped
    long long slab = b;  // contiguous cache: the batch entry; paged cache: the page that holds row pos
    int row = pos;
    if (a.block_table) {
      slab = a.block_table[(long long)b * a.bt_stride + (pos >> a.page_shift)];
      row = pos & ((1 << a.page_shift) - 1);
    }
    *(piece_t*)((char*)a.kc + (slab * a.kcs[0] + hk * a.kcs[1] + row * a.kcs[2]) * a.esz + piece * VEC) = kx;
    *(piece_t*)((char*)a.vc + (slab * a.vcs[0] + hk * a.vcs[1] + row * a.vcs[2]) * a.esz + piece * VEC) = vx;
  }
}

bool aligned_for(const KvAppendArgs& a, int vec) {
  auto ok = [&](const void* p, const long long* st) {
    if (((uintptr_t)p % vec) != 0) return false;
    for (int i = 0; i < 3; i++)
      if ((st[i] * a.esz) % vec != 0) return false;
    return true;
  };
  return (a.D * a.esz) % vec == 0 && ok(a.kc, a.kcs) && ok(a.vc, a.vcs) && ok(a.kn, a.kns) && ok(a.vn, a.vns);
}

}  // namespace

int launch_kv_append(const KvAppendArgs& a, hipStream_t stream) {
  const int vec = aligned_for(a, 16) ? 16 : aligned_for(a, 4) ? 4 : 2;
  const long long total = (long long)a.B * a.Hkv * a.Lnew * (a.D * a.esz / vec);
  long long nwg = (total + 255) / 256;
  if (nwg > 256 * 16) nwg = 256 * 16;
  if (nwg < 1) return 0;
  dim3 grid((unsigned)nwg), block(256);
  const bool narrow = total < 0x40000000LL;  // (the index goes past it by one grid)
#define TT_KVA(VEC)                                                                                        \
  if (narrow) hipLaunchKernelGGL((kv_append_kernel<VEC, uint32_t>), grid, block, 0, stream, a);            \
  else hipLaunchKernelGGL((kv_append_kernel<VEC, unsigned long long>), grid, block, 0, stream, a)
  if (vec == 16) {
    TT_KVA(16);
  } else if (vec == 4) {
    TT_KVA(4);
  } else {
    TT_KVA(2);
  }
#undef TT_KVA
  return (int)hipGetLastError();
}

}  // namespace ttsdpa
