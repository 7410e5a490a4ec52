// Two independent bf16 products at once (llattn_gemm.hip, llattn_gemm_tile.hip): in one launch where that is expected to
// pay, else one after the other.
#pragma once

#include <cstddef>
#include <cstdint>

#include "llattn.h"

namespace llattn {
namespace gemm {

size_t pair_workspace(const llattn_gemm_desc* d0, const llattn_gemm_desc* d1);
int32_t run_pair(const llattn_gemm_desc* d0, const llattn_gemm_desc* d1, void* workspace, size_t workspace_bytes,
                 void* stream);

}  // namespace gemm
}  // namespace llattn
