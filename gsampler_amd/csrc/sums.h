// sums.h -- row sums over a column slice that is not written (internal interface).
#ifndef GSAMPLER_CSRC_SUMS_H_
#define GSAMPLER_CSRC_SUMS_H_

#include "common.h"

namespace gs {

// out[id + key_offset] += the edge's value squared, for the edges of the view; an entry
// that holds -0 before is -0 afterwards if no edge has its key, and not -0 if one has.
// The workspace (sliced_square_sum_bytes, which may be none) is optional.
// onto.fresh: `out` holds nothing yet and counts as onto.base everywhere.
struct SumsOnto {
  bool fresh = false;
  float base = 0.f;
};
int sliced_square_sum(SliceView view, const int64_t* indices, const int32_t* indices32,
                      int64_t nnz, const int64_t* edge_map, const float* efeat, float* out,
                      int64_t num_out, void* workspace, size_t workspace_bytes, hipStream_t s,
                      SumsOnto onto = {});
size_t sliced_square_sum_bytes(int64_t nnz, int64_t num_out);
// Whether such a sum goes by ranges of rows (else by an atomic per tile and row).
bool sums_by_range(int64_t nnz, int64_t num_out);

}  // namespace gs

#endif  // GSAMPLER_CSRC_SUMS_H_
