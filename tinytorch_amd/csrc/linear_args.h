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
  int tile_waves = 0;  // linear_stream.hip: wavefronts that share a tile (0: a workgroup's all)
  float* part = nullptr;
};

// linear_stream.hip: products whose wavefronts divide the contraction among themselves, for any alignment of the operands.
// A plan: tiles of 16 R rows of either operand, the contraction divided among S workgroups, estimated microseconds.  Planning is host
// time of every call, so that a call's plan is made once and handed on.
struct StreamPlan {
  int R, S;
  double us;
};
bool stream_takes(const LinArgs& a, int dtype);                                               // sizes and strides are in its range
StreamPlan plan_stream(const LinArgs& a, int dtype, unsigned entries, bool may_split);        // the estimate that chooses a product's way
StreamPlan plan_stream_call(const LinArgs& a, int dtype, unsigned entries, bool may_split, const StreamPlan& p);  // what a call with that plan runs on
size_t stream_part_bytes(const LinArgs& a, const StreamPlan& call);                           // scratch for its shares
struct StreamTiles {
  int rows, columns, per_workgroup;  // of the output in a tile; tiles of a workgroup
};
// other, RI: another product in the launch, on tiles of 16 RI rows
StreamTiles stream_tiles(const LinArgs& a, int dtype, unsigned entries, const StreamPlan& call, const LinArgs* other = nullptr, int RI = 0);
int launch_stream(const LinArgs& a, int dtype, hipStream_t stream, const StreamPlan& p, unsigned entries = 1, void* scratch = nullptr,
                  size_t scratch_bytes = 0);
// out = bias + the sums of a.splits shares of a product in a.part (and the row sums)
int launch_linear_merge(const LinArgs& a, int dtype, hipStream_t stream);
// a layer's two backward products in one launch (gw: both operands k-major; gi: w k-major), each in the kernel's range
struct PairPlan {
  StreamPlan gw, gi;
  double us() const { return gw.us + gi.us - 3; }  // one launch
};
PairPlan plan_stream_pair(const LinArgs& gw, const LinArgs& gi, int dtype);
int launch_stream_pair(const LinArgs& gw, const LinArgs& gi, int dtype, hipStream_t stream, const PairPlan& p, void* scratch);

// linear_outer.hip: both operands k-major, a short contraction (and the row sums, as above).
bool outer_takes(const LinArgs& a, int dtype);
double outer_cost(const LinArgs& a, int dtype);  // estimated microseconds
int launch_outer(const LinArgs& a, int dtype, hipStream_t stream);

}  // namespace ttsdpa
