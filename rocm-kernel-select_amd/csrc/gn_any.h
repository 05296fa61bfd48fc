// GroupNorm kernels for shapes outside the aligned fast paths of group_norm.hip.
#pragma once
#include "atk_common.h"

namespace atk {

// NC[S] forward: rows of any length >= one 16-byte vector and any element alignment.  ATK_UNSUPPORTED
// for shorter rows.  partials: ngroups * NS (mean, M2) pairs, used when a group exceeds one
// workgroup's registers; slice: elements per slice, a multiple of a vector.
int gn_any_fwd(const void* x, const void* gamma, const void* beta, void* y, int64_t ngroups, int G, int64_t cpg,
               int64_t S, float eps, int silu, int dtype, int pdt, float* partials, int NS, int64_t slice,
               hipStream_t s);

// Channels-last forward for any C that is a multiple of a 16-byte vector, C <= 256 vectors, any
// channels per group, G <= 256.
bool gn_cl_any_takes(int64_t C, int G, int dtype);
size_t gn_cl_any_workspace_bytes(int64_t N, int64_t C, int64_t S, int G);
int gn_cl_any_fwd(const void* x, const void* gamma, const void* beta, void* y, int64_t N, int64_t C, int64_t S, int G,
                  float eps, int silu, int dtype, int pdt, void* workspace, hipStream_t s);

}  // namespace atk
