// The general GEMM kernels (gemm_general.hip), for the launcher in gemm.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "runtime_abi.h"

/// Runs any shape and dtype mix (m, n > 0); p->work may hold partial sums.
int mlkdLaunchGemmGeneral(const mlkd_gemm* p, hipStream_t st);

/// Workspace bytes with which a launch splits its K range over more
/// workgroups; 0 when it does not.
int64_t mlkdGemmGeneralBytes(const mlkd_gemm* p);

/// The kernels a launch runs, joined by '+', as mlkd_gemm_kernel_name names
/// them (p->work as the launch will have it).
const char* mlkdGemmGeneralName(const mlkd_gemm* p);

/// The output tile of a workgroup of that launch.
void mlkdGemmGeneralTile(const mlkd_gemm* p, int64_t* rows, int64_t* cols);
