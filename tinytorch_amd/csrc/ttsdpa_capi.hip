// C ABI of the attention library (declarations and contract: include/ttsdpa.h).
// Validates a call, picks the kernel family, and enqueues it on the caller's stream.  Nothing here allocates device
// memory, synchronises, throws or aborts.

#include <math.h>
#include <string.h>

#include "../../include/ttsdpa.h"
#include "sdpa_common.h"

using namespace ttsdpa;

namespace {

bool dense_last_ok(const int64_t* st, int align) { return st[0] % align == 0 && st[1] % align == 0 && st[2] % align == 0; }

bool ptr_aligned(const void* p, size_t a) { return ((uintptr_t)p % a) == 0; }

// The causal mode a call reduces to.  Bottom-right alignment with one query row hides nothing; without per-batch key
// counts and with S <= L its offset is 0, which is the top-left aligned mask.
int effective_causal(const ttsdpa_params* p) {
  if (p->causal != TTSDPA_CAUSAL_BOTTOM_RIGHT) return p->causal;
  if (p->L == 1) return TTSDPA_CAUSAL_NONE;
  if (!p->kv_len && p->S <= p->L) return TTSDPA_CAUSAL_TOP_LEFT;
  return TTSDPA_CAUSAL_BOTTOM_RIGHT;
}

// Groups of four consecutive keys of the mask (starting at multiples of 4) can be read with one aligned load.
bool mask_vec4_ok(const ttsdpa_params* p) {
  if (p->mask_kind != TTSDPA_MASK_BOOL && p->mask_kind != TTSDPA_MASK_ADD) return false;
  const size_t mesz = p->mask_kind == TTSDPA_MASK_BOOL ? 1 : (p->dtype == TTSDPA_F32 ? 4 : 2);
  return p->mask_stride[3] == 1 && p->mask_stride[0] % 4 == 0 && p->mask_stride[1] % 4 == 0 && p->mask_stride[2] % 4 == 0 &&
         ptr_aligned(p->mask, 4 * mesz);
}

// Validation shared by every entry point; fills the kernel argument block.
int validate(const ttsdpa_params* p, KArgs* a) {
  if (!p) return TTSDPA_ERR_NULL;
  if (p->struct_size != sizeof(ttsdpa_params)) return TTSDPA_ERR_ABI;
  if (p->dtype != TTSDPA_F32 && p->dtype != TTSDPA_F16 && p->dtype != TTSDPA_BF16) return TTSDPA_ERR_DTYPE;
  if (p->B < 0 || p->Hq < 1 || p->Hkv < 1 || p->L < 0 || p->S < 0 || p->D < 1 || p->D > 256) return TTSDPA_ERR_SHAPE;
  if (p->Hq % p->Hkv != 0) return TTSDPA_ERR_SHAPE;
  if (p->mask_kind < TTSDPA_MASK_NONE || p->mask_kind > TTSDPA_MASK_ADD) return TTSDPA_ERR_MASK;
  if (p->causal < TTSDPA_CAUSAL_NONE || p->causal > TTSDPA_CAUSAL_BOTTOM_RIGHT) return TTSDPA_ERR_MASK;
  if (p->mask_kind != TTSDPA_MASK_NONE && p->causal) return TTSDPA_ERR_MASK;  // reference FuncNNLayer.h:242
  const bool empty_out = p->B == 0 || p->L == 0;
  if (!empty_out) {
    if (!p->q || !p->out) return TTSDPA_ERR_NULL;
    if (p->S > 0 && (!p->k || !p->v)) return TTSDPA_ERR_NULL;
    if (p->mask_kind != TTSDPA_MASK_NONE && !p->mask) return TTSDPA_ERR_NULL;
  }
  for (int i = 0; i < 3; i++) {
    if (p->q_stride[i] < 0 || p->k_stride[i] < 0 || p->v_stride[i] < 0 || p->o_stride[i] < 0) return TTSDPA_ERR_STRIDE;
  }
  if (p->q_stride[2] < p->D && p->L > 1) return TTSDPA_ERR_STRIDE;
  if (p->o_stride[2] < p->D && p->L > 1) return TTSDPA_ERR_STRIDE;
  if ((p->k_stride[2] < p->D || p->v_stride[2] < p->D) && p->S > 1) return TTSDPA_ERR_STRIDE;
  const size_t esz = p->dtype == TTSDPA_F32 ? 4 : 2;
  if (!ptr_aligned(p->q, esz) || !ptr_aligned(p->k, esz) || !ptr_aligned(p->v, esz) || !ptr_aligned(p->out, esz))
    return TTSDPA_ERR_STRIDE;
  for (int i = 0; i < 4; i++) {
    if (p->mask_kind != TTSDPA_MASK_NONE && p->mask_stride[i] < 0) return TTSDPA_ERR_STRIDE;
    a->ms[i] = p->mask_kind != TTSDPA_MASK_NONE ? p->mask_stride[i] : 0;
  }
  if (p->mask_kind == TTSDPA_MASK_ADD && !ptr_aligned(p->mask, esz)) return TTSDPA_ERR_STRIDE;
  a->mask_vec4 = mask_vec4_ok(p) ? 1 : 0;
  a->single_tiles = 0, a->full_p = 0;
  a->pack_L = 0, a->kv_splits = 1, a->kv_chunk = 0, a->ws = nullptr;
  if (p->kv_len && !ptr_aligned(p->kv_len, 4)) return TTSDPA_ERR_STRIDE;
  a->kv_len = p->kv_len;
  a->block_table = p->block_table, a->page_shift = 0, a->bt_stride = p->block_table_stride;
  if (p->block_table) {
    if (!ptr_aligned(p->block_table, 4) || p->block_table_stride < 0) return TTSDPA_ERR_STRIDE;
    if (p->page_size < 1 || (p->page_size & (p->page_size - 1)) != 0) return TTSDPA_ERR_SHAPE;
    while ((1 << a->page_shift) < p->page_size) a->page_shift++;
    if ((long long)p->block_table_stride * p->page_size < p->S && p->B > 1) return TTSDPA_ERR_STRIDE;  // tables would overlap
  }
  a->q = p->q, a->k = p->k, a->v = p->v, a->out = p->out, a->mask = p->mask;
  a->B = p->B, a->Hq = p->Hq, a->Hkv = p->Hkv, a->L = p->L, a->S = p->S, a->D = p->D;
  a->G = p->Hq / p->Hkv;
  a->causal = effective_causal(p) != TTSDPA_CAUSAL_NONE ? 1 : 0;
  a->causal_br = effective_causal(p) == TTSDPA_CAUSAL_BOTTOM_RIGHT ? 1 : 0;
  a->mask_kind = p->mask_kind;
  a->scale = p->scale;
  for (int i = 0; i < 3; i++) {
    a->qs[i] = p->q_stride[i], a->ks[i] = p->k_stride[i], a->vs[i] = p->v_stride[i], a->os[i] = p->o_stride[i];
  }
  return TTSDPA_OK;
}

// The MFMA prefill kernels stage key tiles of up to 64 rows: over a paged cache a tile must lie in one page.
constexpr int kPrefillMinPage = 64;

// 16-bit tensors the MFMA kernels can read with 16-byte loads and write with 8-byte stores.
bool fast_layout_ok(const ttsdpa_params* p, bool masks_ok = false, bool pages_ok = false) {
  if (p->block_table && !pages_ok) return false;
  if (p->dtype != TTSDPA_F16 && p->dtype != TTSDPA_BF16) return false;
  if (p->mask_kind != TTSDPA_MASK_NONE && !masks_ok) return false;
  if (!(p->scale > 0.f) || !isfinite(p->scale)) return false;  // the row maximum is taken on unscaled scores
  if (!dense_last_ok(p->q_stride, 8) || !dense_last_ok(p->k_stride, 8) || !dense_last_ok(p->v_stride, 8) ||
      !dense_last_ok(p->o_stride, 8))
    return false;
  return ptr_aligned(p->q, 16) && ptr_aligned(p->k, 16) && ptr_aligned(p->v, 16) && ptr_aligned(p->out, 16);
}

// What the MFMA routes take: attnMasks readable four keys at a time (aligned groups, whole groups only).  The kernels
// themselves apply any attnMask: any_mask = true in the tests below admits the others, which the general route hands
// to them (a general-route call of 16 x 12 heads x 197 rows, head_dim 64, fp16, with a key-padding mask: 124 us on the
// vector ALUs, 18 us there).
bool simple_mask_ok(const ttsdpa_params* p, bool any_mask = false) {
  return any_mask || p->mask_kind == TTSDPA_MASK_NONE || (mask_vec4_ok(p) && p->S % 4 == 0 && !p->kv_len);
}

// fp32 tensors the fp32 MFMA kernel can read and write with 16-byte accesses.
bool f32_prefill_ok(const ttsdpa_params* p, bool any_mask = false) {
  if (p->dtype != TTSDPA_F32 || (p->block_table && p->page_size < kPrefillMinPage) || !simple_mask_ok(p, any_mask)) return false;
  if (p->D < 4 || p->D > 128 || p->D % 4 != 0) return false;  // 64 and 128; other multiples of 4 on the next one up with zero columns
  if (!(p->scale > 0.f) || !isfinite(p->scale) || p->S < 1 || p->L < 1) return false;
  if (!dense_last_ok(p->q_stride, 4) || !dense_last_ok(p->k_stride, 4) || !dense_last_ok(p->v_stride, 4) ||
      !dense_last_ok(p->o_stride, 4))
    return false;
  return ptr_aligned(p->q, 16) && ptr_aligned(p->k, 16) && ptr_aligned(p->v, 16) && ptr_aligned(p->out, 16);
}

// A Bool attnMask the pipelined kernels apply inside their instruction streams (bool_mask_streams_ok on the kernels' side).
bool bool_mask_streams_param_ok(const ttsdpa_params* p) {
  return p->mask_kind == TTSDPA_MASK_BOOL && !p->causal && mask_vec4_ok(p) && p->S % 4 == 0 && !p->kv_len && !p->block_table &&
         (long long)(p->L - 1) * p->mask_stride[2] + 8 < (1ll << 32);
}

// Whether they are the faster kernels for it: against the 4-wavefront kernel, which takes rows in tiles of half the size and divides
// the keys when row tiles are few, 8 x 12 heads x 512 rows, key padding, take 16.0 to 19.7 us (head_dim 128: 21.2 to 29.4), but
// 1 x 8 x 1024 24.8 to 17.1 (31.0 to 24.7; 2 x 8 x 1024 31.2 to 35.8), and at head_dim 64 16 x 12 x 196
// 13.7 to 11.7.
bool mask_streams_best(const ttsdpa_params* p) {
  const bool few = (long long)p->B * p->Hq * ((p->L + 255) / 256) <= 32 && p->S >= 1024;
  return bool_mask_streams_param_ok(p) && !few && (p->D != 64 || p->L >= 256);
}

// Calls of the shape that the pipelined head_dim-128 kernel is for.
bool long_d128(const ttsdpa_params* p) {
  // the kernel addresses the 64 rows of a K / V tile and the 256 rows of a Q tile with 32-bit byte offsets
  return p->D == 128 && p->L > 128 && p->k_stride[2] < (1 << 24) && p->v_stride[2] < (1 << 24) && p->q_stride[2] < (1 << 22);
}

// It runs them unless an attnMask is not for its streams (additive, or a Bool one that is not read four keys at a time): the
// 4-wavefront kernel applies those in variants of its own.  Against the general form of the pipelined kernel's steps: 8 x 12
// heads x 777 rows, key padding 156 -> 68 us, additive 312 -> 95; 32 x 8 x 135, key padding 23.1 -> 18.1; 16 x 8 x 256, additive
// 22.5 -> 18.5; 2 x 16 x 4096, additive 574 -> 484; 1 x 16 x 905, additive, its keys divided, 186 -> 50.
bool pipelined_ok(const ttsdpa_params* p) {
  return long_d128(p) && (p->mask_kind == TTSDPA_MASK_NONE || mask_streams_best(p));
}

// 256-row tiles in all.
long long row_tiles(const ttsdpa_params* p) { return (long long)p->B * p->Hq * ((p->L + 255) / 256); }

// Keys that a row can see: under a top-left aligned causal mask no more than there are rows.
long long visible_keys(const ttsdpa_params* p) {
  return effective_causal(p) == TTSDPA_CAUSAL_TOP_LEFT && p->L < p->S ? p->L : p->S;
}

// The pipelined kernel at head_dim 64: no pages, and of attnMasks only Bool masks its streams can apply.  Against the 4-wavefront
// kernel (128-row tiles) it measured level or up to 30 % faster from 512 query rows on; shorter calls take it when they fill half of
// the chip's CUs, or on many keys with up to 64 row tiles (causal: 128).  Both kernels divide the keys of these among workgroups; us
// on the 4-wavefront kernel and on this one, rows by keys, no mask:
//   130 x 512:    8 heads  9.2 and 11.1    32 heads 11.0 and 11.1    100 heads  11.7 and  11.6
//   256 x 2048:   8       12.8     14.5    32       18.9     23.4    100        31.7      28.4
//   400 x 4096:   8       20.5     20.8    32       31.0     28.7
//   256 x 16384:  8       25.6     25.4    32       56.6     48.4    100       183.8     148.6
// so that neither line is sharp: few heads on 2048 to 4096 keys lose up to a fifth here, 65 to 128 row tiles without a mask on 4096
// keys or more up to a third there.
bool pipelined64_ok(const ttsdpa_params* p) {
  if (p->D != 64 || p->L <= 128 || p->block_table) return false;
  if (p->mask_kind != TTSDPA_MASK_NONE && !mask_streams_best(p)) return false;
  if (!(p->k_stride[2] < (1 << 24) && p->v_stride[2] < (1 << 24) && p->q_stride[2] < (1 << 22))) return false;
  const long long tiles = (p->L + 255) / 256;
  if ((long long)p->B * p->Hq * (p->causal ? (tiles + 1) / 2 : tiles) >= 128) return true;
  if (p->L >= 512) return true;
  const long long units = row_tiles(p), keys = visible_keys(p);
  return p->mask_kind == TTSDPA_MASK_NONE && keys >= 2048 && (units <= 64 || (units <= 128 && p->causal && keys >= 4096));
}

// Few query rows per head against many keys on the 4-wavefront kernel: the G heads of a KV head share one row tile
// (dense q / out make [B,Hq,L,D] a [B,Hkv,G*L,D] tensor), so K/V are streamed once per KV head instead of once per
// query head and the tile is not mostly padding.
bool pack_heads_ok(const ttsdpa_params* p) {
  const int G = p->Hq / p->Hkv;
  if (pipelined_ok(p) || G < 2 || p->mask_kind != TTSDPA_MASK_NONE || p->L > 64 || p->S < 256) return false;
  if (p->dtype == TTSDPA_F32 && !f32_prefill_ok(p)) return false;
  return p->q_stride[1] == (int64_t)p->L * p->q_stride[2] && p->o_stride[1] == (int64_t)p->L * p->o_stride[2];
}

void pack_heads(KArgs* a) {
  a->pack_L = a->L;
  a->L = a->L * a->G, a->Hq = a->Hkv;
  a->qs[1] *= a->G, a->os[1] *= a->G;
  a->G = 1;
}

// Key splits.  A workgroup walks its row tile's keys one tile after another, 2 us (fp32: 3 to 5) each however few workgroups there
// are; when batch x heads x row tiles leave CUs idle, the keys are divided among several workgroups whose partial results a
// second kernel combines.  The number is the one whose estimated time is least: the longest workgroup's tiles, in as
// many rounds as the workgroups need; and with splits the second launch and its records, written and read (fp32: half as fast, beside
// matrix cores that are never idle).
struct SplitPlan {
  int splits, chunk;
  size_t ws_bytes;
};

// heads, L: with records of L rows each; share: of the keys, that a row sees on average; tile_us, tile: of one key tile; slots:
// workgroups that run side by side; step: a chunk is a multiple of it; whole_us: of the unsplit call, where it does not follow from
// the rest
SplitPlan cheapest_split(long long wgs, long long keys, long long heads, int L, int width, double share, double tile_us, int tile, int slots, int step,
                         double whole_us = 0) {
  SplitPlan best{1, 0, 0};
  double least = 0;
  for (long long want = 1; want <= 64; want++) {  // (64: more have not been measured)
    long long chunk = (keys + want - 1) / want;
    chunk = (chunk + step - 1) / step * step;
    const long long n = (keys + chunk - 1) / chunk;
    if (n < want) continue;  // the same as fewer
    double busy = (double)(wgs * n) * share / slots;
    if (slots <= 256 && busy > 1 && busy < 4) busy = (double)(long long)(busy + 0.999);  // one to a CU: whole rounds
    const double per = (double)((n > 1 ? chunk : keys) + tile - 1) / tile;
    const size_t bytes = n > 1 ? split_record_bytes(heads, L, (int)n, width) : 0;
    const double us = (double)(long long)per * tile_us * (busy > 1 ? busy : 1) + (n > 1 ? 5 + bytes / (tile == 32 ? 0.8e6 : 1.6e6) : 0);
    if (n > 1 && us > 0.9 * least) continue;
    if (n == 1 && whole_us > 0) {
      least = whole_us;
      continue;
    }
    if (n == 1 || us < least) least = us, best = SplitPlan{(int)n, n > 1 ? (int)chunk : 0, bytes};
  }
  return best;
}

// Head_dim of the 4-wavefront kernel that runs a call: its records' width.
int tile_width(int dtype, int D) {
  if (dtype == TTSDPA_F32) return D <= 64 ? 64 : 128;
  return D <= 32 ? 32 : D <= 64 ? 64 : D <= 96 ? 96 : D <= 128 ? 128 : D <= 192 ? 192 : 256;
}

// The 4-wavefront kernels (128-row tiles; possibly after packing): fp32 tiles of 32 keys are bound by the matrix cores (2 heads x
// 777 rows, head_dim 80, causal 118 -> 24 us), 16-bit ones of 64 keys by latency (4 heads x 449 rows, head_dim 64, key-padding mask
// 18 -> 12 us, 2 x 8 x 927 rows, head_dim 80, 128 workgroups 37 -> 33).
SplitPlan plan_prefill_splits(const ttsdpa_params* p, const KArgs& a /* after packing */) {
  const bool f32 = p->dtype == TTSDPA_F32;
  if (!f32 && (pipelined_ok(p) || pipelined64_ok(p))) return SplitPlan{1, 0, 0};
  const int W = tile_width(p->dtype, a.D);
  const long long heads = (long long)a.B * a.Hq, wgs = heads * ((a.L + 127) / 128);
  const double us = f32 ? (W == 64 ? 2.7 : 4.6) : W <= 64 ? 1.8 : W <= 128 ? 2.2 : 4.0;
  const long long keys = effective_causal(p) == TTSDPA_CAUSAL_TOP_LEFT && !a.pack_L && a.L < a.S ? a.L : a.S;
  if (f32 && keys <= 512) return SplitPlan{1, 0, 0};  // short walks are dealt out to a workgroup's wavefronts instead, in one launch
  KArgs whole = a;
  whole.kv_splits = 1;
  // under a causal mask a row sees half of the last L keys, and all before them
  const double share = !a.causal ? 1.0 : a.L >= keys ? 0.6 : a.pack_L ? 1.0 : 1.0 - 0.5 * a.L / keys;
  // workgroups side by side: by registers and LDS; fp32 ones are bound by the matrix cores, but entries of unlike lengths end early
  const int slots = W > 128 ? 256 : f32 ? (a.kv_len && a.B > 1 ? 448 : 256) : W > 64 ? 512 : 768;
  return cheapest_split(wgs, keys, heads, a.L, W, share, us, f32 ? 32 : 64, slots, 64,
                        f32 ? us * prefill_f32_tiles(whole) : 0);
}

// What a launch of the pipelined kernels takes with splits of `chunk` key tiles, estimated from its row tiles' lengths (add: `count`
// row tiles of `tiles` key tiles).  Whole pieces fill rounds of the 256 CUs, the row tiles' last pieces what those leave free and
// then rounds of their own.  A tile takes 1.4 us, 1.85 with every CU busy (power); a piece that is not all of its row tile leaves a
// record, 133 KB, which all CUs write at about the same time and the merge kernel reads: 1 x 32 heads x 500 rows on 6000 keys in
// 4 pieces 54 + 9 us, on 16000 127 + 9.  Few records cost little beside the merge's launch: 2 heads x 777 rows, whole 23.5 us, in 4
// pieces, 32 records, 18.6 (head_dim 64: 17.0, 13.0); 1 x 300 on 600 keys 19.9, 16.7.  Many cost what shorter pieces gain: 1 x 4096
// in 8 pieces, 128 records, 30.5, in 16 31.0 (head_dim 64: 21.1, 25.4).
struct SplitCost {
  double chunk, whole = 0, rests = 0, rest = 0, longest_rest = 0, records = 0;
  void add(double count, int tiles) {
    const double pieces = floor(tiles / chunk), last = tiles - pieces * chunk;
    whole += count * pieces, rest += count * last;
    if (last > 0) rests += count;
    if (last > longest_rest) longest_rest = last;
    if (tiles > chunk) records += count * (pieces + (last > 0));
  }
  // add(count, first + step * i), i = 0 .. n-1, of a step that divides the chunk: in pieces of p = chunk / step places, place i + first / step
  // (first % step key tiles further: a rest, if not zero, even where a place is the first of its piece)
  void add_series(double count, unsigned first, unsigned step, unsigned n) {
    if (n < 1) return;
    const unsigned c = (unsigned)chunk, p = c / step, lo = first / step, hi = lo + n, over = first % step;  // places lo .. hi-1
    const unsigned q0 = lo / p, r0 = lo % p, q1 = hi / p, r1 = hi % p;
    auto below = [&](double q, double r) { return p * (0.5 * q * (q - 1)) + q * r; };  // pieces before the places up to p q + r, added up
    const double pieces = below(q1, r1) - below(q0, r0), sum = (double)n * first + step * (0.5 * n * (n - 1.0));
    const double even = over ? 0 : (q1 + (r1 > 0)) - (q0 + (r0 > 0));  // places that end with a piece
    const double longest = step * (double)(q1 > q0 ? p - 1 : r1 - 1) + over;
    const unsigned undivided = first > c ? 0 : (c - first) / step + 1;
    whole += count * pieces, rest += count * (sum - chunk * pieces), rests += count * (n - even);
    if (longest > longest_rest) longest_rest = longest;
    records += count * (pieces + (n - even) - (undivided < n ? undivided : n));
  }
  double longest() const {  // a CU's tiles
    const double rounds = ceil(whole / 256), room = 256 * rounds - whole, left = rest - room * chunk;
    double tiles = rounds * chunk;
    if (rests > room) {  // the longest of them go first: lengths taken to be spread evenly, or all the same
      const double spread = 2 * rest / rests * (1 - room / rests), longest = spread < longest_rest ? spread : longest_rest;
      tiles += left / 256 > longest ? left / 256 : longest;
    }
    return tiles;
  }
  double us() const {
    const double tiles = longest(), busy = (whole * chunk + rest) / (256 * tiles);
    const double many = 12 + 0.035 * records, few = 6 + 0.1 * records;
    return tiles * (1.4 + 0.45 * busy) + (records > 0 ? (few < many ? few : many) : 0);
  }
};

// Key splits for the pipelined kernels (head_dim 128 and 64): a call with half as many 256-row tiles as the chip has CUs, or fewer (a
// chunk of a sequence's rows against a long cache, paged or not, a few heads of a tensor-parallel share), leaves CUs without work.
// Its row tiles then share their keys among workgroups of `chunk` keys (a multiple of 256: four key tiles, so the kernel's stages
// keep their constants), as many as SplitCost finds shortest, and split_merge_kernel combines the records.  More row tiles are
// left whole: their lengths may differ (key counts), but balancing them gains what the records cost (3 x 32 heads x 500 rows on
// 6000, 5392 and 4062 keys: 134 us whole, 128 with 68-tile pieces, 141 with 64, 151 with 32).
SplitPlan plan_pipelined_splits(const ttsdpa_params* p) {
  SplitPlan s{1, 0, 0};
  if (p->dtype == TTSDPA_F32 || !(pipelined_ok(p) || pipelined64_ok(p)) || p->mask_kind != TTSDPA_MASK_NONE) return s;
  const long long units = row_tiles(p), keys = visible_keys(p);
  if (units > 128 || keys < 512) return s;
  const long long heads = (long long)p->B * p->Hq;
  const int ntile = (p->L + 255) / 256, causal = effective_causal(p);
  const int offset = causal == TTSDPA_CAUSAL_BOTTOM_RIGHT && p->S > p->L ? p->S - p->L : 0;
  const int longest = (int)((keys + 63) / 64);
  // row tiles that end before the keys do, each 256 keys behind the one above; the others see all keys
  const long long ends = causal == TTSDPA_CAUSAL_NONE || p->S <= offset ? 0 : ((long long)p->S - offset - 1) / 256, rising = ends < ntile ? ends : ntile;
  double least = 0;
  for (int n = 1; n <= 64 && (n == 1 || units * n <= 1024); n++) {
    const int chunk = ((longest + n - 1) / n + 3) & ~3;
    if ((longest + chunk - 1) / chunk < n) continue;  // the same as fewer
    SplitCost cost{(double)chunk};
    if (rising > 0) cost.add_series((double)heads, 4 + (unsigned)(offset + 63ll) / 64, 4, (unsigned)rising);
    if (rising < ntile) cost.add((double)(heads * (ntile - rising)), (int)(((long long)p->S + 63) / 64));
    const double us = cost.us();
    if (n == 1 || us < 0.95 * least) least = us, s.splits = n, s.chunk = 64 * chunk;
  }
  if (s.splits < 2) return SplitPlan{1, 0, 0};
  s.ws_bytes = split_record_bytes(heads, p->L, s.splits, p->D);
  return s;
}

// ---- 256 rows to a workgroup, or 128 with the keys dealt out (sdpa_prefill_dealt.hip) ------------------------------------------
// What a launch of either kernel takes, us, from the lengths of its row tiles (in 64 keys: a tile of the one, a step of both groups of
// the other).  Fitted to 600 calls (1 to 8 sequences, 1 to 64 query heads, 129 to 8192 rows on as many keys or a chunk's on up to 16384,
// paged or not, causal or not); they miss by 4 to 7 % on average.  A workgroup costs `start` lengths beside its own (its launch, the
// first loads, the output), which shows where a CU has several; a length costs `each`, and `busy` more where all CUs are at work (power).
struct PipelinedCost {
  double base, each, busy, start;              // undivided launches
  double split_base, split_each, split_busy, split_more, record;  // divided keys: with the merge's launch; per round beyond the first; per record
};
constexpr PipelinedCost kRows256[2] = {{7.2, 0.74, 0.30, 6, 11.2, 0.63, 0.33, 0.0, 0.027}, {8.9, 1.02, 0.58, 7, 14.9, 0.60, 0.83, 8.2, 0.039}};
constexpr PipelinedCost kRows128[2] = {{6.6, 0.47, 0.09, 10, 8.2, 0.53, 0.0, 1.9, 0.027}, {7.6, 0.68, 0.20, 9, 11.8, 0.69, 0.17, 4.0, 0.026}};

// Row tiles of `rows` rows (256, 128), longest first: length of the t-th, and of all.  Under a causal mask their lengths rise from the last one by rows /
// 64 up to that of all keys; the first one may have fewer rows.  Sums over them are closed forms: tile by tile, a plan of one head on
// 16384 rows took 9.6 us of the host's time.
template <int rows>
struct RowTiles {
  int ntile, S, offset, L;
  bool causal;
  long long heads, rising = 0, first = 0, sum = 0;  // rising: whole tiles that end before the keys do, the shortest `first` long
  explicit RowTiles(const ttsdpa_params* p) : ntile((p->L + rows - 1) / rows), S(p->S), L(p->L), heads((long long)p->B * p->Hq) {
    const int c = effective_causal(p);
    causal = c != TTSDPA_CAUSAL_NONE, offset = c == TTSDPA_CAUSAL_BOTTOM_RIGHT && S > L ? S - L : 0;
    const long long all = ((long long)S + 63) / 64;
    if (!causal) {
      sum = heads * ntile * all;
      return;
    }
    const long long ends = S > offset ? ((long long)S - offset - 1) / rows : 0;
    rising = ends < ntile - 1 ? ends : ntile - 1, first = rows / 64 + ((long long)offset + 63) / 64;
    sum = heads * (rising * first + rows / 64 * (rising * (rising - 1) / 2) + (ntile - 1 - rising) * all + length(0));
  }
  int length(int t) const {
    long long last = S;
    if (causal) {
      const long long end = (long long)rows * (ntile - t), v = (end < L ? end : L) + offset;
      last = v < last ? v : last;
    }
    return (int)((last + 63) / 64);
  }
  double whole_us(const PipelinedCost& c) const {
    const long long n = heads * ntile, rounds = (n + 255) / 256, pairs = heads * ((ntile + 1) / 2), pair_rounds = (pairs + 255) / 256;
    double longest = length(0);
    if (n > 256) {
      if (!causal) longest = rounds * longest + (rounds - 1) * c.start;
      else if (rows == 256 && ntile > 1 && pairs >= 256 && pairs * 10 >= pair_rounds * 256 * 9)  // mirrored pairs (launch_prefill_d128)
        longest = ntile % 2 == 0 ? pair_rounds * (longest + length(ntile - 1) + c.start) - c.start
                                 : sum / 256.0 + c.start * (pairs / 256.0 - 1) + 0.25 * longest;  // (the middle ones are single)
      else {
        // the CU with the shortest of the first 256 takes the next one
        const double next = n <= 512 ? length(255 / (int)heads) + length(256 / (int)heads) + c.start
                                     : sum / 256.0 + 0.5 * length(ntile - 1) + c.start * (n / 256.0 - 1);
        longest = next > longest ? next : longest;
      }
    }
    return c.base + c.each * longest + c.busy * sum / 256.0;
  }
  // with pieces of `chunk` (64 keys); 0: none that is shorter than the longest row tile
  double split_us(const PipelinedCost& c, int chunk) const {
    SplitCost s{(double)chunk};
    if (!causal) {
      s.add((double)(heads * ntile), length(0));
    } else {
      s.add_series((double)heads, (unsigned)first, rows / 64, (unsigned)rising);
      if (rising < ntile - 1) s.add((double)(heads * (ntile - 1 - rising)), (int)(((long long)S + 63) / 64));
      s.add((double)heads, length(0));
    }
    const double pieces = (s.whole + s.rests) / 256 - 1;
    return c.split_base + c.split_each * s.longest() + c.split_busy * (s.whole * chunk + s.rest) / 256 + (pieces > 0 ? c.split_more * pieces : 0) + c.record * s.records;
  }
};

// The call's way through the pipelined kernels: which of them, and the division of its keys.  dealt: the kernel of 128-row workgroups, with
// the number of pieces that is shortest there, where that is shorter by these estimates: 2 x 8 x 756 rows, head_dim 128, causal 24.3 -> 16.5
// us, 16 x 1327 34.4 -> 22.9, 32 x 1539 41 -> 33, 6 x 32 x 326 on 3781 keys, paged, 162 -> 126; head_dim 64, 4 x 8 x 727 18.1 -> 12.8.  Where
// row tiles fill the chip evenly its keys cost more (2 x 32 x 4096, no mask, 454 and 511): a barrier for 32 of them.
struct PipelinedPlan {
  bool dealt;
  SplitPlan split;
};
PipelinedPlan plan_pipelined(const ttsdpa_params* p, bool divided = true, double* us = nullptr) {
  PipelinedPlan plan{false, divided ? plan_pipelined_splits(p) : SplitPlan{1, 0, 0}};
  if (p->dtype == TTSDPA_F32 || p->mask_kind != TTSDPA_MASK_NONE || !(pipelined_ok(p) || pipelined64_ok(p)) || p->S < 1) return plan;
  const RowTiles<256> wide(p);
  const RowTiles<128> narrow(p);
  const PipelinedCost &c256 = kRows256[p->D == 128], &c128 = kRows128[p->D == 128];
  double least = plan.split.splits > 1 ? wide.split_us(c256, plan.split.chunk / 64) : wide.whole_us(c256);
  const double whole = narrow.whole_us(c128);
  // (sequences of unlike lengths: the estimates take them all for the longest, which is too much for a divided launch)
  if (whole < (p->kv_len && p->B > 1 ? 0.9 : 0.95) * least) least = whole, plan.dealt = true, plan.split = SplitPlan{1, 0, 0};
  const int longest = narrow.length(0);
  // least of any division: a CU has its share of all lengths, and a whole piece; a row tile is a piece or more
  const double even = narrow.sum / 256.0, rounds = narrow.heads * narrow.ntile / 256.0 - 1;
  const double further = c128.split_busy * even + (rounds > 0 ? c128.split_more * rounds : 0);
  for (int n = 2; divided && n <= 16 && narrow.heads * narrow.ntile * n <= 1024; n++) {
    const int chunk = ((longest + n - 1) / n + 3) & ~3;
    if ((longest + chunk - 1) / chunk < n) continue;  // the same as fewer
    const double most = (plan.dealt ? 1.0 : 0.95) * least;
    if (c128.split_base + c128.split_each * (even > chunk ? even : chunk) + further > 1.001 * most) continue;
    const double t = narrow.split_us(c128, chunk);
    if (t < most)
      least = t, plan.dealt = true, plan.split = SplitPlan{n, 64 * chunk, split_record_bytes(narrow.heads, p->L, n, p->D)};
  }
  if (us) *us = least;
  return plan;
}

// ---- short sequences (sdpa_short.hip) -----------------------------------------------------------------------------------
// Calls whose other kernels are a wavefront's chain of a few tiles on part of the chip.  Which way is shorter follows from estimates,
// each fitted to 128 calls of its element type and head_dim (64, or 128 for those above it): 1 to 4 sequences, 2 to 64 query heads,
// groups of 1, 2 and 4, 64 to 1024 rows on as many keys, causal or not, us.  They miss by 8 to 10 % on average and by a third at
// worst, mostly where a second workgroup shares a CU, so that more of those ask for a wider margin.
struct ShortShape {
  int rows, keys;         // units of 16
  double heads, kv, avg;  // query heads and KV heads of all sequences; key units that a row unit sees on average
  bool causal, f32, wide;
  int group, L;
  ShortShape(const ttsdpa_params* p) {
    const int c = effective_causal(p);
    rows = (p->L + 15) / 16, keys = ((c == TTSDPA_CAUSAL_TOP_LEFT && p->L < p->S ? p->L : p->S) + 15) / 16;
    heads = (double)p->B * p->Hq, kv = (double)p->B * p->Hkv, group = p->Hq / p->Hkv, L = p->L;
    causal = c != TTSDPA_CAUSAL_NONE, f32 = p->dtype == TTSDPA_F32, wide = p->D > 64;
    const double tri = 0.5 * ((rows < keys ? rows : keys) - 1);
    avg = !causal ? keys : keys - tri;
  }
  // what the workgroups beyond the first on each CU add, in key units (row units)
  static double more(double wgs, double each) { return wgs > 256 ? (ceil(wgs / 256) - 1) * each : 0; }
  double least_margin() const { return heads * rows > 256 ? 0.8 : 0.92; }

  double forward_us() const {
    static const double fit[2][2][3] = {{{4.2, 0.57, 0.11}, {4.2, 1.2, 0.23}}, {{3.9, 1.7, 0.25}, {5.3, 2.8, 0.58}}};
    const double* c = fit[f32][wide];
    return c[0] + c[1] * ((keys + 7) / 8) + c[2] * more(heads * rows, avg);
  }
  // Whether an fp32 forward call is one of those that the two estimates get wrong: a single long head, which the other kernel divides (892
  // rows 14.5 us, 15.8 here; 918 x 128 20.0 and 27.3), and causal ones of several rounds of workgroups on shared KV heads, whose loads then bound this
  // kernel and whose end the other one's wavefronts share (256 heads x 76 x 64 12.1 and 14.6; 128 x 107 x 128 21.3 and 24.5, 32 x 435 x 128
  // 33.5 and 38.6; but 32 x 328 x 128, each with its own keys, 32.7 and 27.1).
  bool forward_misses(const ttsdpa_params* p, double f32_tiles, bool dealt) const {
    if (heads == 1) return rows > 52;
    if (!wide) return heads * rows > 1152;
    if (p->D <= 96 || group == 1 || !causal || heads * rows <= 512 || L > 512) return false;
    const double other = dealt && heads * ((L + 31) / 32) > 256 ? 17 + 1.1 * f32_tiles : 6.5 + 4.1 * f32_tiles;
    return forward_us() + more(heads * rows, 2.7) > other;
  }
  // of the other kernels: 16-bit ones by 64-key tiles, up to eight in a row (more are divided); fp32 ones by the tiles of 32 that their
  // own rule for dealing them out finds
  double other_forward_us(double f32_tiles) const {
    const int tiles = (keys + 3) / 4;
    const double work = heads * ((L + 127) / 128) * tiles * (causal ? 0.6 : 1.0) / 512, row = tiles < 8 ? tiles : 8;
    if (f32) return wide ? 5.8 + 2.96 * f32_tiles : 4.0 + 2.3 * f32_tiles;
    return wide ? 4.8 + 1.47 * row + 0.33 * work + (L > 128 ? 1.5 : 0) : 4.1 + 1.05 * row + 0.48 * work;
  }
  // workgroups that share a dk / dv workgroup's units: as many as have a CU, each with a unit for its wavefronts
  int splits() const {
    const double wgs = kv * keys;
    const int most = (group * rows + 7) / 8, room = wgs < 256 ? (int)(256 / wgs) : 1, n = most < room ? most : room;
    return n < 1 ? 1 : n > 16 ? 16 : n;
  }
  double backward_us(bool joint) const {
    static const double two[2][2][6] = {{{9.6, 1.2, 0.28, 1.3, 0.16, 3.8}, {11.9, 2.5, 0.68, 2.2, 0.30, 4.4}},
                                        {{11.8, 2.8, 0.74, 2.7, 0.34, 4.3}, {16.8, 5.8, 1.5, 5.2, 0.58, 4.9}}};
    static const double one[2][2][6] = {{{7.6, 0.163, 0.062, 0.31, 0.71, 3.8}, {10.3, 0.258, 0.132, 0.54, 1.07, 5.1}},
                                        {{10.7, 0.37, 0.134, 0.46, 1.57, 5.4}, {}}};
    const int n = splits(), turns = ((group * rows + n - 1) / n + 7) / 8;
    const double per_key = heads * rows * avg / (kv * keys * n);  // units of a dk / dv workgroup on average
    const double q = more(heads * rows, avg), k = more(kv * keys * n, per_key), sum = n > 1 ? 1 : 0;
    if (!joint) {
      const double* c = two[f32][wide];
      return c[0] + c[1] * ((keys + 7) / 8) + c[2] * q + c[3] * turns + c[4] * k + c[5] * sum;
    }
    if (f32 && wide) return 1e9;  // (its registers do not hold both roles)
    const double* c = one[f32][wide];
    const double stats = heads * rows * keys * keys * (causal ? 1.0 / 3 : 1.0) / 256;  // score products for the statistics
    return c[0] + c[1] * turns * keys + c[2] * stats + c[3] * q + c[4] * k + c[5] * sum;
  }
};

// Calls the kernels take, of a length that the estimates are for.
bool short_ok(const ttsdpa_params* p) {
  return p->mask_kind == TTSDPA_MASK_NONE && !p->block_table && p->D <= 128 && p->L >= 16 && p->S >= 16 && p->L <= 1024 && p->S <= 1024 &&
         p->L <= 2 * p->S && p->S <= 2 * p->L && (long long)p->B * p->Hq <= 1024;
}

bool prefill_ok(const ttsdpa_params* p, bool any_mask = false) {
  if (f32_prefill_ok(p, any_mask)) return true;
  // any attnMask at head_dim 128 with more than 128 rows; else those that can be read four keys at a time
  // head sizes between the 4-wavefront kernel's (32, 64, 96, 128, 192, 256) run on the next one up with zero columns
  const bool mfma_head_dim = p->D >= 8 && p->D <= 256 && p->D % 8 == 0;
  if (p->block_table && p->page_size < kPrefillMinPage) return false;
  // the 16-bit kernels address the rows of a K / V tile with 32-bit byte offsets (the fp32 kernel returned above does not)
  const bool tile_offsets_ok = p->k_stride[2] < (1 << 24) && p->v_stride[2] < (1 << 24);
  return fast_layout_ok(p, true, true) && mfma_head_dim && p->S >= 1 && p->L >= 1 && tile_offsets_ok &&
         (long_d128(p) || simple_mask_ok(p, any_mask));
}

bool decode_ok(const ttsdpa_params* p) {
  // a top-left aligned causal mask leaves a few keys per row: not the streaming kernel's case
  // head_dim 64 and 128; other multiples of 8 up to 128 on the next one up with zero columns
  if (!fast_layout_ok(p, false, true) || p->D < 8 || p->D > 128 || p->D % 8 != 0 || effective_causal(p) == TTSDPA_CAUSAL_TOP_LEFT ||
      p->S < 1 || p->L < 1)
    return false;
  if (p->block_table && p->page_size < 32) return false;  // a 32-key block of a wavefront must lie in one page
  return (long long)p->L * (p->Hq / p->Hkv) <= kDecodeMaxRows;
}

// fp32 calls of the prefill route that the split-KV streaming kernel runs when it has its scratch: few query rows per KV head
// (4 sequences of 1000 keys, 16 query heads on 4, head_dim 128, strided q: 145 us on the fp32 MFMA kernel's 128-row
// tiles, which such a q keeps from sharing heads and splitting keys).
bool f32_decode_ok(const ttsdpa_params* p) {
  return f32_prefill_ok(p) && p->mask_kind == TTSDPA_MASK_NONE && effective_causal(p) != TTSDPA_CAUSAL_TOP_LEFT &&
         (long long)p->L * (p->Hq / p->Hkv) <= kDecodeMaxRows;
}

// ... where that is the shortest way forward (of a call of the prefill route).
bool short_forward_best(const ttsdpa_params* p, const KArgs& a) {
  if (!short_ok(p) || pack_heads_ok(p) || !prefill_ok(p)) return false;
  const ShortShape s(p);
  bool dealt = false;
  const double tiles = s.f32 ? prefill_f32_tiles(a, &dealt) : 0;
  if (s.forward_us() >= s.least_margin() * s.other_forward_us(tiles) || (s.f32 && s.forward_misses(p, tiles, dealt))) return false;
  double pipelined = 0;
  return s.f32 || !plan_pipelined(p, true, &pipelined).dealt || s.forward_us() < pipelined;
}

int pick_route(const ttsdpa_params* p) {
  if (p->B == 0 || p->L == 0) return TTSDPA_ROUTE_NONE;
  if (p->S == 0) return TTSDPA_ROUTE_ZERO;
  // Few query rows against many keys: streaming the cache once for the whole head group beats a 128-row tile.
  if (decode_ok(p) && p->S >= 256) {
    // 9-16 rows per KV head: the streaming kernel does P.V on the vector ALUs and measures 5.5 TB/s there; the
    // 4-wavefront MFMA kernel with packed heads and split keys 5.85 TB/s, when the call allows it
    const long long rows = (long long)p->L * (p->Hq / p->Hkv);
    // (measured at head_dim 64 / 128; the sizes between keep to the streaming kernel)
    if (rows > 8 && (p->D == 64 || p->D == 128) && prefill_ok(p) && !pipelined_ok(p) && (p->Hq == p->Hkv || pack_heads_ok(p)))
      return TTSDPA_ROUTE_PREFILL;
    return TTSDPA_ROUTE_DECODE;
  }
  if (prefill_ok(p) && p->L >= 16) return TTSDPA_ROUTE_PREFILL;
  if (decode_ok(p)) return TTSDPA_ROUTE_DECODE;
  if (prefill_ok(p)) return TTSDPA_ROUTE_PREFILL;
  return TTSDPA_ROUTE_GENERAL;
}

// ---- backward ---------------------------------------------------------------------------------------------------------
int validate_backward(const ttsdpa_backward_params* p, BwdArgs* a) {
  if (!p) return TTSDPA_ERR_NULL;
  if (p->struct_size != sizeof(ttsdpa_backward_params)) return TTSDPA_ERR_ABI;
  int rc = validate(&p->fwd, &a->f);
  if (rc != TTSDPA_OK) return rc;
  const ttsdpa_params* f = &p->fwd;
  if (f->block_table) return TTSDPA_ERR_UNSUPPORTED;
  const size_t esz = f->dtype == TTSDPA_F32 ? 4 : 2;
  if (f->B > 0 && f->L > 0 && (!p->dout || !p->dq)) return TTSDPA_ERR_NULL;
  if (f->B > 0 && f->S > 0 && (!p->dk || !p->dv || !f->k || !f->v)) return TTSDPA_ERR_NULL;
  if (!ptr_aligned(p->dout, esz) || !ptr_aligned(p->dq, esz) || !ptr_aligned(p->dk, esz) || !ptr_aligned(p->dv, esz))
    return TTSDPA_ERR_STRIDE;
  for (int i = 0; i < 3; i++) {
    if (p->dout_stride[i] < 0 || p->dq_stride[i] < 0 || p->dk_stride[i] < 0 || p->dv_stride[i] < 0) return TTSDPA_ERR_STRIDE;
    a->dos[i] = p->dout_stride[i], a->dqs[i] = p->dq_stride[i], a->dks[i] = p->dk_stride[i], a->dvs[i] = p->dv_stride[i];
  }
  if ((p->dout_stride[2] < f->D || p->dq_stride[2] < f->D) && f->L > 1) return TTSDPA_ERR_STRIDE;
  if ((p->dk_stride[2] < f->D || p->dv_stride[2] < f->D) && f->S > 1) return TTSDPA_ERR_STRIDE;
  a->dout = p->dout, a->dq = p->dq, a->dk = p->dk, a->dv = p->dv, a->stats = nullptr, a->partial = nullptr, a->dkv_splits = 1, a->dq_partial = nullptr, a->dq_splits = 1, a->dkv_round = 0;
  return TTSDPA_OK;
}

// The MFMA backward kernels: 16-bit tensors they can read and write with 16-byte / 8-byte accesses, head_dim 64 or
// 128, attnMasks the forward's 4-wavefront kernel takes (keys readable four at a time, no kv_len beside them).
bool backward_mfma_ok(const ttsdpa_backward_params* p, bool any_mask = false) {
  const ttsdpa_params* f = &p->fwd;
  // head_dim 64 and 128; other multiples of 8 up to 128 on the register-staged kernels of the next one up (zero columns)
  if (!fast_layout_ok(f, true) || !simple_mask_ok(f, any_mask) || f->D < 8 || f->D > 128 || f->D % 8 != 0 || f->L < 1 || f->S < 1) return false;
  if (!dense_last_ok(p->dout_stride, 8) || !dense_last_ok(p->dq_stride, 8) || !dense_last_ok(p->dk_stride, 8) ||
      !dense_last_ok(p->dv_stride, 8))
    return false;
  // the head_dim-128 dk/dv kernel addresses the rows of a tile with 32-bit byte offsets from the tile's first row
  if (f->D == 128 && (f->q_stride[2] >= (1 << 24) || f->k_stride[2] >= (1 << 24) || f->v_stride[2] >= (1 << 24) ||
                      p->dout_stride[2] >= (1 << 24)))
    return false;
  return ptr_aligned(p->dout, 16) && ptr_aligned(p->dq, 16) && ptr_aligned(p->dk, 16) && ptr_aligned(p->dv, 16);
}

// The fp32 matrix-core backward kernels: fp32 tensors with 16-byte aligned rows, head_dim 64 or 128, attnMasks as for
// the 16-bit pair.
bool backward_f32_ok(const ttsdpa_backward_params* p, bool any_mask = false) {
  const ttsdpa_params* f = &p->fwd;
  if (f->dtype != TTSDPA_F32 || f->block_table || !simple_mask_ok(f, any_mask) || f->D < 4 || f->D > 128 || f->D % 4 != 0) return false;
  if (!(f->scale > 0.f) || !isfinite(f->scale) || f->L < 1 || f->S < 1) return false;  // the row maximum is taken on unscaled scores
  if (!dense_last_ok(f->q_stride, 4) || !dense_last_ok(f->k_stride, 4) || !dense_last_ok(f->v_stride, 4) ||
      !dense_last_ok(f->o_stride, 4) || !dense_last_ok(p->dout_stride, 4) || !dense_last_ok(p->dq_stride, 4) ||
      !dense_last_ok(p->dk_stride, 4) || !dense_last_ok(p->dv_stride, 4))
    return false;
  return ptr_aligned(f->q, 16) && ptr_aligned(f->k, 16) && ptr_aligned(f->v, 16) && ptr_aligned(f->out, 16) &&
         ptr_aligned(p->dout, 16) && ptr_aligned(p->dq, 16) && ptr_aligned(p->dk, 16) && ptr_aligned(p->dv, 16);
}

int pick_backward_route(const ttsdpa_backward_params* p) {
  const ttsdpa_params* f = &p->fwd;
  if (f->B == 0 || (f->L == 0 && f->S == 0)) return TTSDPA_ROUTE_NONE;
  return backward_mfma_ok(p) || backward_f32_ok(p) ? TTSDPA_ROUTE_PREFILL : TTSDPA_ROUTE_GENERAL;
}

// The matrix-core pairs run the call: the MFMA route, and of the general route what only its attnMask keeps off it (16-bit tensors
// then on the fp32 pair: that route's arithmetic is fp32).
bool backward_on_mfma(const ttsdpa_backward_params* p) {
  return pick_backward_route(p) != TTSDPA_ROUTE_NONE && (backward_mfma_ok(p, true) || backward_f32_ok(p, true));
}

bool backward_on_f32_pair(const ttsdpa_backward_params* p) {
  return backward_on_mfma(p) && (p->fwd.dtype == TTSDPA_F32 || !simple_mask_ok(&p->fwd));
}

// The rows' statistics: (statistic, delta) pairs, then log_sums where the kernels keep one (BwdArgs).
size_t backward_rows(const ttsdpa_backward_params* p) { return (size_t)p->fwd.B * p->fwd.Hq * p->fwd.L; }
bool backward_log_sums(const ttsdpa_backward_params* p) { return p->fwd.mask_kind != TTSDPA_MASK_NONE || !backward_on_mfma(p); }
size_t backward_stats_bytes(const ttsdpa_backward_params* p) { return backward_rows(p) * (backward_log_sums(p) ? 3 : 2) * sizeof(float); }

// How the matrix-core pairs divide a call (made once for a call): the dk / dv kernel's query streams and the dq kernel's key ranges.
struct PairSplits;
int short_backward_splits(const ttsdpa_backward_params* p, const PairSplits& n, bool* joint = nullptr);
struct PairSplits {
  int dkv = 1, dq = 1;
  bool dkv_dealt = false, dq_dealt = false;
  int own = -1;  // 16-bit calls: the answer of short_backward_splits, found on the way
  bool own_joint = false;
  PairSplits(const ttsdpa_backward_params* p) {
    const ttsdpa_params* f = &p->fwd;
    if (!backward_on_mfma(p)) return;
    const bool f32 = backward_on_f32_pair(p), causal = effective_causal(f) != TTSDPA_CAUSAL_NONE;
    if (f->dtype != TTSDPA_F32 && f->mask_kind == TTSDPA_MASK_NONE && (f->D == 64 || f->D == 128)) {
      static constexpr BackwardCost kDq[2] = {{0, 0.59, 3.6, 0.47}, {4.5, 0.53, 2.9, 0.37}}, kDkv[2] = {{0, 0.95, 2.5, 0.40, 120}, {0, 1.75, 1.8, 0.41, 80}};
      own = short_backward_splits(p, *this, &own_joint);
      if (own > 0) return;  // (whole: with less scratch than those kernels ask for)
      const int offset = effective_causal(f) == TTSDPA_CAUSAL_BOTTOM_RIGHT && f->S > f->L ? f->S - f->L : 0;
      dq = backward_splits_16bit(kDq[f->D == 128], false, f->B, f->Hq, f->Hkv, f->L, f->S, f->D, causal, offset);
      dkv = backward_splits_16bit(kDkv[f->D == 128], true, f->B, f->Hq, f->Hkv, f->L, f->S, f->D, causal, offset);
      return;
    }
    const int per_cu = f->D <= 64 && f->mask_kind == TTSDPA_MASK_NONE ? 2 : 1;
    dkv = backward_dkv_splits(f->B, f->Hkv, f->Hq, f->L, f->S, f->D, causal, per_cu, f32, &dkv_dealt);
    dq = backward_dq_splits(f->B, f->Hq, f->L, f->S, f->D, causal, f32 && f->D > 64 ? 256 : 512, f32, &dq_dealt);
  }
};

// Scratch layout: the statistics, then (a split query stream) the partial dk / dv, then (split key ranges) the partial dq records,
// each 256-byte aligned.
size_t backward_partial_offset(const ttsdpa_backward_params* p) { return (backward_stats_bytes(p) + 255) & ~(size_t)255; }
size_t backward_dq_partial_offset(const ttsdpa_backward_params* p, const PairSplits& n) {
  if (n.dkv == 1) return backward_partial_offset(p);
  const size_t end = backward_partial_offset(p) + (size_t)n.dkv * 2 * p->fwd.B * p->fwd.Hkv * p->fwd.S * p->fwd.D * sizeof(float);
  return (end + 255) & ~(size_t)255;
}
// Estimated time of a call on the matrix-core pairs, by the longest stream of each kernel.  (16-bit: fitted to the head_dim-128 pair as the compiler
// orders it and to its splits of then; of 104 drawn calls that go to the short sequences' kernels by it, the pair of now is shorter for one, 45.2 us and
// 48.0, 1 x 4 heads (2) x 592 on 760, head_dim 128.)
double pair_backward_us(const ttsdpa_params* f, const ShortShape& s, const PairSplits& n) {
  if (!s.f32) {
    const int tiles = (s.keys + 3) / 4, stream = s.group * ((f->L + 31) / 32);
    const double work = s.heads * ((f->L + 127) / 128) * tiles * (s.causal ? 0.6 : 1.0) / 512, row = tiles < 8 ? tiles : 8, st = stream < 32 ? stream : 32;
    return s.wide ? 16.6 + 2.2 * row + 6.9 * work + 0.37 * st : 11.6 + 1.7 * row + 4.3 * work + 0.27 * st;
  }
  auto us = [&](int n, bool dealt, double wgs, int tiles, double slots, double tile_us) {
    if (dealt) return ((tiles + 3) / 4 + 0.5) * tile_us;
    const double rounds = (s.causal ? 0.6 : 1.0) * wgs * n / slots;
    return (tiles + n - 1) / n * tile_us * (rounds > 1 ? rounds : 1) + (n > 1 ? 4.5 : 0);
  };
  const double dkv = us(n.dkv, n.dkv_dealt, s.kv * ((f->S + 127) / 128), s.group * ((f->L + 31) / 32), s.wide ? 256 : 512, s.wide ? 10 : 5);
  const double dq = us(n.dq, n.dq_dealt, s.heads * ((f->L + 127) / 128), (f->S + 31) / 32, s.wide ? 256 : 512, s.wide ? 8 : 4);
  return s.wide ? 18.5 + 0.54 * dq + 1.08 * dkv : 5.5 + 1.5 * dq + 1.0 * dkv;
}

// The short sequences' backward: splits of its dk / dv workgroups, 0 where the pairs are the shorter way.
int short_backward_splits(const ttsdpa_backward_params* p, const PairSplits& n, bool* joint) {
  if (n.own >= 0) {
    if (joint) *joint = n.own_joint;
    return n.own;
  }
  const ttsdpa_params* f = &p->fwd;
  if (!short_ok(f) || !(backward_mfma_ok(p) || backward_f32_ok(p))) return 0;
  const ShortShape s(f);
  const double one = s.backward_us(true), two = s.backward_us(false);
  if (joint) *joint = one < two;
  // (the joint launch takes longer than its estimate by a tenth for each round of workgroups beyond the first: with more than three of
  // them it lost up to 24 %, 256 heads x 64 x 64 fp32 34.9 us on the pairs, 45.6 here; bf16 x 75 24.3 and 28.2)
  const double us = one < two ? one : two, pair = pair_backward_us(f, s, n), rounds = s.heads * s.rows / 256;
  const bool padded = s.wide && f->D <= 96;  // (of 128 columns: less than the estimate, 64 heads x 111 x 80 18.0 us, 27.4 on the pairs)
  if (one < two && rounds > 1 && !padded && us * (1 + 0.1 * (rounds - 1)) >= 0.85 * pair) return 0;
  return us < s.least_margin() * pair ? s.splits() : 0;
}
size_t short_backward_bytes(const ttsdpa_backward_params* p, int splits) {
  return backward_partial_offset(p) + (splits > 1 ? (size_t)splits * 2 * p->fwd.B * p->fwd.Hkv * p->fwd.S * p->fwd.D * sizeof(float) : 0);
}

// ... with that much scratch (less than the query asks for: the pairs).
int short_backward_taken(const ttsdpa_backward_params* p, const PairSplits& pair, size_t workspace_bytes, bool* joint) {
  const int n = short_backward_splits(p, pair, joint);
  return n > 0 && workspace_bytes >= short_backward_bytes(p, n) ? n : 0;
}

// of the pairs
size_t backward_scratch_bytes(const ttsdpa_backward_params* p, const PairSplits& n) {
  if (n.dq > 1)
    return backward_dq_partial_offset(p, n) + (size_t)n.dq * p->fwd.B * p->fwd.Hq * p->fwd.L * (p->fwd.D + 2) * sizeof(float);
  if (n.dkv == 1) return backward_stats_bytes(p);
  return backward_partial_offset(p) + (size_t)n.dkv * 2 * p->fwd.B * p->fwd.Hkv * p->fwd.S * p->fwd.D * sizeof(float);
}

int check_grid(long long nwg) { return nwg > 0x7fffffffLL ? TTSDPA_ERR_SHAPE : TTSDPA_OK; }

// Scratch of ttsdpa_decode_static: the split-KV partial records of one decode call.  Every GPU the library runs on holds
// its own copy of this array, at its own address, until the process ends.  In host code the array's name is only a
// handle for hipGetSymbolAddress: kernels and memory calls get the address that call returns, never the name.
constexpr size_t kStaticScratchBytes = TTSDPA_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

// Address of the current device's copy of `scratch`, looked up once per device (with that device current) and kept.
// Safe from several host threads: the worst case is two identical look-ups.
int static_scratch_of_current_device(void** out) {
  static void* ptr[kMaxDevices];
  static bool done[kMaxDevices];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return (int)hipErrorInvalidDevice;
  if (!__atomic_load_n(&done[dev], __ATOMIC_ACQUIRE)) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!p) return (int)hipErrorInvalidSymbol;
    __atomic_store_n(&ptr[dev], p, __ATOMIC_RELAXED);
    __atomic_store_n(&done[dev], true, __ATOMIC_RELEASE);
  }
  *out = __atomic_load_n(&ptr[dev], __ATOMIC_RELAXED);
  return TTSDPA_OK;
}

}  // namespace

extern "C" {

int ttsdpa_abi_version(void) { return TTSDPA_ABI_VERSION; }

const char* ttsdpa_status_string(int status) {
  switch (status) {
    case TTSDPA_OK: return "ok";
    case TTSDPA_ERR_NULL: return "required pointer is NULL";
    case TTSDPA_ERR_DTYPE: return "unsupported dtype";
    case TTSDPA_ERR_SHAPE: return "invalid or unsupported shape";
    case TTSDPA_ERR_STRIDE: return "unsupported stride or alignment";
    case TTSDPA_ERR_MASK: return "invalid mask arguments";
    case TTSDPA_ERR_WORKSPACE: return "workspace missing or too small";
    case TTSDPA_ERR_UNSUPPORTED: return "arguments outside this kernel's domain";
    case TTSDPA_ERR_ABI: return "ttsdpa_params.struct_size mismatch";
    case TTSDPA_ERR_STATIC_SCRATCH: return "call needs more scratch than the library's static buffer holds (TTSDPA_STATIC_SCRATCH_BYTES)";
    default: return status > 0 ? hipGetErrorString((hipError_t)status) : "unknown status";
  }
}

void ttsdpa_params_init(ttsdpa_params* p, int dtype, int B, int Hq, int Hkv, int L, int S, int D) {
  memset(p, 0, sizeof(*p));
  p->struct_size = sizeof(*p);
  p->dtype = dtype;
  p->B = B, p->Hq = Hq, p->Hkv = Hkv, p->L = L, p->S = S, p->D = D;
  p->q_stride[0] = (int64_t)Hq * L * D, p->q_stride[1] = (int64_t)L * D, p->q_stride[2] = D;
  p->k_stride[0] = (int64_t)Hkv * S * D, p->k_stride[1] = (int64_t)S * D, p->k_stride[2] = D;
  p->v_stride[0] = p->k_stride[0], p->v_stride[1] = p->k_stride[1], p->v_stride[2] = D;
  p->o_stride[0] = p->q_stride[0], p->o_stride[1] = p->q_stride[1], p->o_stride[2] = D;
  p->scale = D > 0 ? 1.f / sqrtf((float)D) : 1.f;
  p->causal = 0;
  p->mask_kind = TTSDPA_MASK_NONE;
  p->mask = nullptr;
  p->mask_stride[0] = 0, p->mask_stride[1] = 0, p->mask_stride[2] = S, p->mask_stride[3] = 1;
  p->kv_len = nullptr;
  p->block_table = nullptr, p->page_size = 0, p->block_table_stride = 0;
}

int ttsdpa_plan(const ttsdpa_params* p, int* route) {
  KArgs a;
  int rc = validate(p, &a);
  if (rc != TTSDPA_OK) return rc;
  if (route) *route = pick_route(p);
  return TTSDPA_OK;
}

size_t ttsdpa_workspace_bytes(const ttsdpa_params* p) {
  KArgs a;
  if (validate(p, &a) != TTSDPA_OK) return 0;
  if (p->B == 0 || p->L == 0 || p->S == 0) return 0;
  // enough for ttsdpa_forward's route and for an explicit ttsdpa_decode of the same call
  size_t need = decode_ok(p) ? plan_decode(a, p->dtype == TTSDPA_F32).ws_bytes : 0;
  const int route = pick_route(p);
  if (route == TTSDPA_ROUTE_PREFILL || (route == TTSDPA_ROUTE_GENERAL && p->mask_kind != TTSDPA_MASK_NONE && prefill_ok(p, true))) {
    if (f32_decode_ok(p)) {
      const size_t decode = plan_decode(a, p->dtype == TTSDPA_F32).ws_bytes;
      need = decode > need ? decode : need;
    }
    if (pack_heads_ok(p)) pack_heads(&a);
    size_t split = plan_prefill_splits(p, a).ws_bytes;
    need = split > need ? split : need;
    split = plan_pipelined(p).split.ws_bytes;
    need = split > need ? split : need;
  }
  return need;
}

int ttsdpa_general(const ttsdpa_params* p, void* stream) {
  KArgs a;
  int rc = validate(p, &a);
  if (rc != TTSDPA_OK) return rc;
  if (p->B == 0 || p->L == 0) return TTSDPA_OK;
  if (p->S == 0) return launch_zero(a, p->dtype, (hipStream_t)stream);
  if ((rc = check_grid((long long)a.B * a.Hq * ((a.L + 63) / 64))) != TTSDPA_OK) return rc;
  return launch_general(a, p->dtype, (hipStream_t)stream);
}

// Which of the kernels for short sequences a call of the prefill route (or of the general one whose masks the matrix-core kernels
// apply) runs on.
static int short_kernel_of(const ttsdpa_params* p, const KArgs& a) {
  const int rows = heads_rows(a, p->dtype);
  if (rows > 0) return rows == 16 ? TTSDPA_KERNEL_HEADS_16 : TTSDPA_KERNEL_HEADS_32;
  return short_forward_best(p, a) ? TTSDPA_KERNEL_SHORT : TTSDPA_KERNEL_OTHER;
}
// masked calls of the general route: fp32 probabilities
static int full_probabilities(const ttsdpa_params* p) { return p->mask_kind != TTSDPA_MASK_NONE && !long_d128(p) && !simple_mask_ok(p); }

// ttsdpa_prefill with optional scratch: with it, a short-L call may divide its keys among workgroups.
static int prefill_impl(const ttsdpa_params* p, void* workspace, size_t workspace_bytes, void* stream, bool any_mask = false) {
  KArgs a;
  int rc = validate(p, &a);
  if (rc != TTSDPA_OK) return rc;
  if (p->B == 0 || p->L == 0) return TTSDPA_OK;
  if (!prefill_ok(p, any_mask)) return TTSDPA_ERR_UNSUPPORTED;
  if ((rc = check_grid((long long)a.B * a.Hq * ((a.L + 127) / 128))) != TTSDPA_OK) return rc;
  a.full_p = full_probabilities(p);  // (any_mask: the general route's calls, its arithmetic)
  const int kind = short_kernel_of(p, a);
  if (kind == TTSDPA_KERNEL_SHORT) return launch_short_forward(a, p->dtype, (hipStream_t)stream);
  if (kind != TTSDPA_KERNEL_OTHER) return launch_heads(a, p->dtype, (hipStream_t)stream);
  // head_dim 128 with enough rows to fill 256-row workgroups takes the software-pipelined kernel (its tile loads
  // address 64 rows with 32-bit byte offsets)
  if (p->dtype != TTSDPA_F32 && (pipelined_ok(p) || pipelined64_ok(p))) {
    PipelinedPlan plan = plan_pipelined(p);
    if (plan.split.splits > 1 && !(workspace && workspace_bytes >= plan.split.ws_bytes && ptr_aligned(workspace, 16))) plan = plan_pipelined(p, false);
    if (plan.split.splits > 1) {
      a.kv_splits = plan.split.splits, a.kv_chunk = plan.split.chunk, a.ws = (float*)workspace;
      if ((rc = check_grid((long long)a.B * a.Hq * ((a.L + (plan.dealt ? 127 : 255)) / (plan.dealt ? 128 : 256) + 8) * a.kv_splits)) != TTSDPA_OK) return rc;
    } else {
      a.kv_splits = 1, a.kv_chunk = 0, a.ws = nullptr;
    }
    // with splits: the kernel and the merge of its records
    if (plan.dealt) return launch_prefill_dealt(a, p->dtype, (hipStream_t)stream);
    return p->D == 128 ? launch_prefill_d128(a, p->dtype, (hipStream_t)stream) : launch_prefill_d64(a, p->dtype, (hipStream_t)stream);
  }
  if (f32_decode_ok(p)) {
    const DecodePlan pl = plan_decode(a, p->dtype == TTSDPA_F32);
    if ((pl.ws_bytes == 0 || (workspace && workspace_bytes >= pl.ws_bytes && ptr_aligned(workspace, 16))) &&
        check_grid((long long)a.B * a.Hkv * pl.splits) == TTSDPA_OK)
      return launch_decode(a, p->dtype, workspace, (hipStream_t)stream);
  }
  auto launch = [&](const KArgs& k) {
    return p->dtype == TTSDPA_F32 ? launch_prefill_f32(k, (hipStream_t)stream) : launch_prefill(k, p->dtype, (hipStream_t)stream);
  };
  if (pack_heads_ok(p)) pack_heads(&a);
  a.kv_splits = 1, a.kv_chunk = 0, a.ws = nullptr;
  const SplitPlan sp = plan_prefill_splits(p, a);
  if (sp.splits > 1 && workspace && workspace_bytes >= sp.ws_bytes && ptr_aligned(workspace, 16) && p->S > 0) {
    a.kv_splits = sp.splits, a.kv_chunk = sp.chunk, a.ws = (float*)workspace;
    if ((rc = check_grid((long long)a.B * a.Hq * ((a.L + 127) / 128 + 8) * sp.splits)) != TTSDPA_OK) return rc;
    rc = launch(a);
    if (rc != 0) return rc;
    return launch_split_merge(a, p->dtype, tile_width(p->dtype, a.D), 128, (hipStream_t)stream);
  }
  return launch(a);
}

int ttsdpa_prefill(const ttsdpa_params* p, void* stream) { return prefill_impl(p, nullptr, 0, stream); }

int ttsdpa_decode(const ttsdpa_params* p, void* workspace, size_t workspace_bytes, void* stream) {
  KArgs a;
  int rc = validate(p, &a);
  if (rc != TTSDPA_OK) return rc;
  if (p->B == 0 || p->L == 0) return TTSDPA_OK;
  if (!decode_ok(p)) return TTSDPA_ERR_UNSUPPORTED;
  DecodePlan pl = plan_decode(a, p->dtype == TTSDPA_F32);
  if (pl.ws_bytes > 0 && (!workspace || workspace_bytes < pl.ws_bytes || !ptr_aligned(workspace, 16)))
    return TTSDPA_ERR_WORKSPACE;
  if ((rc = check_grid((long long)a.B * a.Hkv * pl.splits)) != TTSDPA_OK) return rc;
  return launch_decode(a, p->dtype, workspace, (hipStream_t)stream);
}

int ttsdpa_decode_static(const ttsdpa_params* p, void* stream) {
  KArgs a;
  int rc = validate(p, &a);
  if (rc != TTSDPA_OK) return rc;
  if (p->B == 0 || p->L == 0) return TTSDPA_OK;
  if (!decode_ok(p)) return TTSDPA_ERR_UNSUPPORTED;
  const DecodePlan pl = plan_decode(a, p->dtype == TTSDPA_F32);
  if (pl.ws_bytes > kStaticScratchBytes) return TTSDPA_ERR_STATIC_SCRATCH;
  if ((rc = check_grid((long long)a.B * a.Hkv * pl.splits)) != TTSDPA_OK) return rc;
  void* ws = nullptr;
  if ((rc = static_scratch_of_current_device(&ws)) != TTSDPA_OK) return rc;
  // Nothing in the records has to start at zero: every split writes its whole record (an empty split a weight of
  // zero) before the merge kernel, later on the same stream, reads it.
  return launch_decode(a, p->dtype, ws, (hipStream_t)stream);
}

int ttsdpa_forward(const ttsdpa_params* p, void* workspace, size_t workspace_bytes, void* stream) {
  KArgs a;
  int rc = validate(p, &a);
  if (rc != TTSDPA_OK) return rc;
  switch (pick_route(p)) {
    case TTSDPA_ROUTE_NONE: return TTSDPA_OK;
    case TTSDPA_ROUTE_ZERO: return launch_zero(a, p->dtype, (hipStream_t)stream);
    case TTSDPA_ROUTE_DECODE: return ttsdpa_decode(p, workspace, workspace_bytes, stream);
    case TTSDPA_ROUTE_PREFILL: return prefill_impl(p, workspace, workspace_bytes, stream);
    default: break;
  }
  // the general route: what only its attnMask keeps off the MFMA kernels runs on them, the rest on the vector ALUs
  if (p->mask_kind != TTSDPA_MASK_NONE && prefill_ok(p, true)) return prefill_impl(p, workspace, workspace_bytes, stream, true);
  return ttsdpa_general(p, stream);
}

int ttsdpa_kernel(const ttsdpa_params* p, int* kind) {
  KArgs a;
  const int rc = validate(p, &a);
  if (rc != TTSDPA_OK) return rc;
  const int route = pick_route(p);
  a.full_p = full_probabilities(p);
  const bool prefill = route == TTSDPA_ROUTE_PREFILL || (route == TTSDPA_ROUTE_GENERAL && p->mask_kind != TTSDPA_MASK_NONE && prefill_ok(p, true));
  int k = prefill ? short_kernel_of(p, a) : TTSDPA_KERNEL_OTHER;
  if (prefill && k == TTSDPA_KERNEL_OTHER && plan_pipelined(p).dealt) k = TTSDPA_KERNEL_DEALT;
  if (kind) *kind = k;
  return TTSDPA_OK;
}

int ttsdpa_division(const ttsdpa_params* p, int* key_pieces, int* wavefronts) {
  KArgs a;
  const int rc = validate(p, &a);
  if (rc != TTSDPA_OK) return rc;
  int n = 1, w = 0;
  const int route = pick_route(p);
  a.full_p = full_probabilities(p);
  const bool prefill = route == TTSDPA_ROUTE_PREFILL || (route == TTSDPA_ROUTE_GENERAL && p->mask_kind != TTSDPA_MASK_NONE && prefill_ok(p, true));
  if (route == TTSDPA_ROUTE_DECODE || (prefill && f32_decode_ok(p))) {
    const DecodePlan pl = plan_decode(a, p->dtype == TTSDPA_F32);
    n = pl.splits, w = pl.waves;
  } else if (prefill && short_kernel_of(p, a) == TTSDPA_KERNEL_OTHER) {
    if (p->dtype != TTSDPA_F32 && (pipelined_ok(p) || pipelined64_ok(p))) {
      n = plan_pipelined(p).split.splits;
    } else {
      if (pack_heads_ok(p)) pack_heads(&a);
      n = plan_prefill_splits(p, a).splits;
    }
  }
  if (key_pieces) *key_pieces = n;
  if (wavefronts) *wavefronts = w;
  return TTSDPA_OK;
}

void ttsdpa_backward_params_init(ttsdpa_backward_params* p, int dtype, int B, int Hq, int Hkv, int L, int S, int D) {
  memset(p, 0, sizeof(*p));
  p->struct_size = sizeof(*p);
  ttsdpa_params_init(&p->fwd, dtype, B, Hq, Hkv, L, S, D);
  for (int i = 0; i < 3; i++) {
    p->dout_stride[i] = p->dq_stride[i] = p->fwd.q_stride[i];
    p->dk_stride[i] = p->dv_stride[i] = p->fwd.k_stride[i];
  }
}

int ttsdpa_backward_plan(const ttsdpa_backward_params* p, int* route) {
  BwdArgs a;
  int rc = validate_backward(p, &a);
  if (rc != TTSDPA_OK) return rc;
  if (route) *route = pick_backward_route(p);
  return TTSDPA_OK;
}

int ttsdpa_backward_kernel(const ttsdpa_backward_params* p, size_t workspace_bytes, int* kind) {
  BwdArgs a;
  const int rc = validate_backward(p, &a);
  if (rc != TTSDPA_OK) return rc;
  bool joint = false;
  const int n = pick_backward_route(p) == TTSDPA_ROUTE_NONE ? 0 : short_backward_taken(p, PairSplits(p), workspace_bytes, &joint);
  if (kind) *kind = n == 0 ? TTSDPA_KERNEL_OTHER : joint ? TTSDPA_KERNEL_SHORT_JOINT : TTSDPA_KERNEL_SHORT;
  return TTSDPA_OK;
}

int ttsdpa_backward_division(const ttsdpa_backward_params* p, int* query_pieces, int* key_pieces) {
  BwdArgs a;
  const int rc = validate_backward(p, &a);
  if (rc != TTSDPA_OK) return rc;
  int n = 1, m = 1;
  if (pick_backward_route(p) != TTSDPA_ROUTE_NONE) {
    const PairSplits pair(p);
    const int own = short_backward_splits(p, pair);
    n = own > 0 ? own : pair.dkv, m = own > 0 ? 1 : pair.dq;
  }
  if (query_pieces) *query_pieces = n;
  if (key_pieces) *key_pieces = m;
  return TTSDPA_OK;
}

size_t ttsdpa_backward_workspace_bytes(const ttsdpa_backward_params* p) {
  BwdArgs a;
  if (validate_backward(p, &a) != TTSDPA_OK) return 0;
  const PairSplits pair(p);
  const size_t pairs = backward_scratch_bytes(p, pair);
  const int n = short_backward_splits(p, pair);
  const size_t own = n > 0 ? short_backward_bytes(p, n) : 0;
  return own > pairs ? own : pairs;
}

int ttsdpa_backward(const ttsdpa_backward_params* p, void* workspace, size_t workspace_bytes, void* stream) {
  BwdArgs a;
  int rc = validate_backward(p, &a);
  if (rc != TTSDPA_OK) return rc;
  const int route = pick_backward_route(p);
  if (route == TTSDPA_ROUTE_NONE) return TTSDPA_OK;
  const PairSplits pair(p);
  const size_t need = backward_scratch_bytes(p, pair);
  if (need > 0 && (!workspace || workspace_bytes < need || !ptr_aligned(workspace, 16))) return TTSDPA_ERR_WORKSPACE;
  a.stats = (float*)workspace;
  a.log_sums = backward_log_sums(p) ? a.stats + 2 * backward_rows(p) : nullptr;
  bool joint = false;
  const int n = short_backward_taken(p, pair, workspace_bytes, &joint);
  if (n > 0) {
    a.dkv_splits = n, a.partial = n > 1 ? (float*)((char*)workspace + backward_partial_offset(p)) : nullptr;
    return launch_short_backward(a, p->fwd.dtype, joint, (hipStream_t)stream);
  }
  a.dkv_splits = pair.dkv, a.dkv_dealt = pair.dkv_dealt;
  a.partial = a.dkv_splits > 1 ? (float*)((char*)workspace + backward_partial_offset(p)) : nullptr;
  a.dq_splits = pair.dq, a.dq_dealt = pair.dq_dealt;
  a.dq_partial = a.dq_splits > 1 ? (float*)((char*)workspace + backward_dq_partial_offset(p, pair)) : nullptr;
  if (backward_on_mfma(p)) {
    const long long g1 = (long long)a.f.B * a.f.Hq * ((a.f.L + 127) / 128) * a.dq_splits, g2 = (long long)a.f.B * a.f.Hkv * ((a.f.S + 127) / 128);
    if (check_grid(g1) != TTSDPA_OK || check_grid(g2) != TTSDPA_OK) return TTSDPA_ERR_SHAPE;
    if (backward_on_f32_pair(p)) return launch_backward_f32(a, p->fwd.dtype, (hipStream_t)stream);
    return launch_backward_mfma(a, p->fwd.dtype, (hipStream_t)stream);
  }
  {  // the vector-ALU pair: 64 rows per workgroup up to head_dim 128, 32 beyond
    const int rows = a.f.D <= 128 ? 64 : 32;
    const long long g1 = (long long)a.f.B * a.f.Hq * ((a.f.L + rows - 1) / rows), g2 = (long long)a.f.B * a.f.Hkv * ((a.f.S + rows - 1) / rows);
    if (check_grid(g1) != TTSDPA_OK || check_grid(g2) != TTSDPA_OK) return TTSDPA_ERR_SHAPE;
  }
  return launch_backward_general(a, p->fwd.dtype, (hipStream_t)stream);
}

void ttsdpa_kv_append_params_init(ttsdpa_kv_append_params* p, int dtype, int B, int Hkv, int Smax, int Lnew, int D) {
  memset(p, 0, sizeof(*p));
  p->struct_size = sizeof(*p);
  p->dtype = dtype;
  p->B = B, p->Hkv = Hkv, p->Smax = Smax, p->Lnew = Lnew, p->D = D;
  p->kc_stride[0] = (int64_t)Hkv * Smax * D, p->kc_stride[1] = (int64_t)Smax * D, p->kc_stride[2] = D;
  p->kn_stride[0] = (int64_t)Hkv * Lnew * D, p->kn_stride[1] = (int64_t)Lnew * D, p->kn_stride[2] = D;
  for (int i = 0; i < 3; i++) p->vc_stride[i] = p->kc_stride[i], p->vn_stride[i] = p->kn_stride[i];
}

int ttsdpa_kv_append(const ttsdpa_kv_append_params* p, void* stream) {
  if (!p) return TTSDPA_ERR_NULL;
  if (p->struct_size != sizeof(ttsdpa_kv_append_params)) return TTSDPA_ERR_ABI;
  if (p->dtype != TTSDPA_F32 && p->dtype != TTSDPA_F16 && p->dtype != TTSDPA_BF16) return TTSDPA_ERR_DTYPE;
  if (p->B < 0 || p->Hkv < 1 || p->Smax < 0 || p->Lnew < 0 || p->D < 1) return TTSDPA_ERR_SHAPE;
  if (p->B == 0 || p->Lnew == 0 || p->Smax == 0) return TTSDPA_OK;
  if (!p->k_cache || !p->v_cache || !p->k_new || !p->v_new) return TTSDPA_ERR_NULL;
  const size_t esz = p->dtype == TTSDPA_F32 ? 4 : 2;
  if (!ptr_aligned(p->k_cache, esz) || !ptr_aligned(p->v_cache, esz) || !ptr_aligned(p->k_new, esz) ||
      !ptr_aligned(p->v_new, esz) || (p->positions && !ptr_aligned(p->positions, 4)))
    return TTSDPA_ERR_STRIDE;
  KvAppendArgs a;
  for (int i = 0; i < 3; i++) {
    if (p->kc_stride[i] < 0 || p->vc_stride[i] < 0 || p->kn_stride[i] < 0 || p->vn_stride[i] < 0) return TTSDPA_ERR_STRIDE;
    a.kcs[i] = p->kc_stride[i], a.vcs[i] = p->vc_stride[i], a.kns[i] = p->kn_stride[i], a.vns[i] = p->vn_stride[i];
  }
  if ((p->kc_stride[2] < p->D || p->vc_stride[2] < p->D) && p->Smax > 1) return TTSDPA_ERR_STRIDE;
  if ((p->kn_stride[2] < p->D || p->vn_stride[2] < p->D) && p->Lnew > 1) return TTSDPA_ERR_STRIDE;
  a.kc = p->k_cache, a.vc = p->v_cache, a.kn = p->k_new, a.vn = p->v_new, a.positions = p->positions;
  a.block_table = p->block_table, a.page_shift = 0, a.bt_stride = p->block_table_stride;
  if (p->block_table) {
    if (!ptr_aligned(p->block_table, 4) || p->block_table_stride < 0) return TTSDPA_ERR_STRIDE;
    if (p->page_size < 1 || (p->page_size & (p->page_size - 1)) != 0) return TTSDPA_ERR_SHAPE;
    while ((1 << a.page_shift) < p->page_size) a.page_shift++;
  }
  a.B = p->B, a.Hkv = p->Hkv, a.Smax = p->Smax, a.Lnew = p->Lnew, a.D = p->D, a.position = p->position, a.esz = (int)esz;
  return launch_kv_append(a, (hipStream_t)stream);
}

}  // extern "C"
