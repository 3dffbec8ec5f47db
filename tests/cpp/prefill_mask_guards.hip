// Calls of the pipelined prefill launchers with attnMasks that their kernels cannot apply: each has to be refused before anything is
// launched.  Exit code: how many were not.
#include <stdio.h>

#include "sdpa_common.h"

using namespace ttsdpa;

static KArgs bool_mask_call(int D) {
  KArgs a{};
  a.B = 1, a.Hq = a.Hkv = 2, a.G = 1, a.L = 512, a.S = 1024, a.D = D;
  a.scale = 1.f, a.kv_splits = 1;
  a.mask_kind = 1, a.mask_vec4 = 1;
  a.ms[2] = a.S, a.ms[3] = 1;
  return a;
}

int main() {
  int wrong = 0;
  auto refused = [&](const char* what, KArgs a) {
    for (int dtype = 1; dtype <= 2; dtype++) {
      const int rc = a.D == 128 ? launch_prefill_d128(a, dtype, nullptr) : launch_prefill_d64(a, dtype, nullptr);
      printf("head_dim %d, dtype %d, %s: %d\n", a.D, dtype, what, rc);
      wrong += rc != (int)hipErrorInvalidValue;
    }
  };
  static int lens[1], table[16];
  for (int D = 64; D <= 128; D += 64) {
    KArgs a = bool_mask_call(D);
    a.mask_kind = 2;
    refused("additive", a);
    a = bool_mask_call(D), a.mask_vec4 = 0;
    refused("keys not in aligned groups of four", a);
    a = bool_mask_call(D), a.S = 1022;
    refused("an odd group at the end", a);
    a = bool_mask_call(D), a.kv_len = lens;
    refused("key counts", a);
    a = bool_mask_call(D), a.block_table = table, a.page_shift = 6;
    refused("pages", a);
    a = bool_mask_call(D), a.kv_splits = 2, a.kv_chunk = 512;
    refused("divided keys", a);
    a = bool_mask_call(D), a.ms[2] = 1ll << 32;
    refused("rows beyond 32-bit offsets", a);
    a = bool_mask_call(D), a.causal = 1;
    refused("a causal mask beside it", a);
  }
  return wrong;
}
