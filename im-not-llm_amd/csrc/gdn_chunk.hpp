// The chunked gated delta rule (gdn_chunk.hip) behind inl_gdn_rule_fwd.
#pragma once

#include <type_traits>

#include "inl_common.hpp"

namespace inl {

struct GdnChunkParams {
  const void* mixed;
  int64_t ms;
  const float* g;
  const float* beta;
  int64_t gs;
  float* out;
  int64_t os;
  const int32_t* cu;
  int64_t n;
  int32_t n_texts, nk, nv, dk, dv;
};

// Whether a call takes the chunked form.
bool gdn_chunk_fits(const GdnChunkParams& p, int32_t dtype);
int gdn_chunk_launch(const GdnChunkParams& p, int32_t dtype, hipStream_t st);

}  // namespace inl
