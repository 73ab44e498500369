// Entries of gemm_wide.hip for gemm.hip: validated problems of a 16-bit type.
#pragma once
#include <hip/hip_runtime.h>
#include "../../include/mi355_layer.h"

struct MiGemmPlan {
    double us;              // expected time
    int tile;               // blocks of 128 or 256 rows and columns
    int splits;             // of the contraction (a single problem of one segment)
    size_t workspace_bytes;
    int cut;                // rows, or columns, that go in a launch of whole rounds, in front of the rest; 0: all in one launch
    bool columns;
    int apart;              // several problems: 0 in one launch, -1 in a launch (and with a plan) each, i + 1 problem i alone and the rest in one
};
// the fastest plan that takes no more than workspace_bytes
MiGemmPlan mi_gemm_wide_plan(const mi_gemm_problem* problems, int count, size_t workspace_bytes, int compute_units);
int mi_gemm_wide(const mi_gemm_problem* problems, int count, int dtype, const MiGemmPlan& plan, void* workspace, int compute_units, hipStream_t stream);
