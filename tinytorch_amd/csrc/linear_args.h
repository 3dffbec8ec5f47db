// Argument block of the linear-layer kernels (linear.hip, linear_stream.hip).
#pragma once

#include "sdpa_common.h"

namespace ttsdpa {

struct LinArgs {
  const void* x;
  const void* w;
  const void* bias;
  void* out;
  long long M, N, K, ldx, ldw, ldo;
  // x is stored [K, M] (x(m,k) = x[k*ldx + m]) / w is stored [K, N] (w(n,k) = w[k*ldw + n])
  int xt = 0, wt = 0;
  // batch entries of one launch: entry e reads x + e*bsx, w + e*bsw and writes out + e*bso (elements; 0 = the operand is
  // shared by all entries)
  long long bsx = 0, bsw = 0, bso = 0;
  // linear_stream.hip: the sums of x over the contraction ([M], or nullptr: not wanted; only with both operands k-major), and the division of the contraction
  // among `splits` workgroups per tile, whose sums go to part ([splits][M*N + M] floats) to be added by another kernel
  void* rowsum = nullptr;
  int splits = 1;
  float* part = nullptr;
};

// linear_stream.hip: products whose wavefronts divide the contraction among themselves, for any alignment of the operands.
bool stream_takes(const LinArgs& a, int dtype);                             // sizes and strides are in its range
double stream_cost(const LinArgs& a, int dtype, unsigned entries, bool may_split);  // estimated microseconds
double stream_call_cost(const LinArgs& a, int dtype, bool may_split);        // of the plan that a call has
int stream_chains(const LinArgs& a, int dtype, bool may_split);              // chains that it adds a contraction up in
size_t stream_scratch(const LinArgs& a, int dtype);                         // bytes that let it divide the contraction
int launch_stream(const LinArgs& a, int dtype, hipStream_t stream, unsigned entries = 1, void* scratch = nullptr, size_t scratch_bytes = 0);
// out = bias + the sums of a.splits shares of a product in a.part (and the row sums)
int launch_linear_merge(const LinArgs& a, int dtype, hipStream_t stream);
// a layer's two backward products in one launch (gw: both operands k-major; gi: w k-major), each in the kernel's range
double stream_pair_cost(const LinArgs& gw, const LinArgs& gi, int dtype);
size_t stream_pair_scratch(const LinArgs& gw, const LinArgs& gi, int dtype);
int launch_stream_pair(const LinArgs& gw, const LinArgs& gi, int dtype, hipStream_t stream, void* scratch);

// linear_outer.hip: both operands k-major, a short contraction (and the row sums, as above).
bool outer_takes(const LinArgs& a, int dtype);
double outer_cost(const LinArgs& a, int dtype);  // estimated microseconds
int launch_outer(const LinArgs& a, int dtype, hipStream_t stream);

}  // namespace ttsdpa
