// What the recurrences' launches on the vector ALU (state_scan.hip) and on the matrix cores (scan_mfma.hip) share.
#pragma once
#include "fmt_dev.h"

namespace NVX_NS {

enum { SCAN_DECAY = 0, SCAN_GLA = 1, SCAN_MLSTM = 2 };

// One launch of a recurrence over a memory per head (see state_scan.hip for the operands of each; what a recurrence does not have is null).
struct ScanArgs {
    const void* x;                     // rows with q, k and v at their offsets
    int64_t x_stride;
    int q_off, k_off, v_off, act, heads, dim, vdim, chunk, n_chunk_max, half, vec;
    float q_mul, k_mul, cap;
    const float *decay, *alpha, *gates, *gate_bias;
    float* S;                          // the pool, and the chunks' own memories
    float* ws;
    const float *N_in, *M_in;          // mlstm: normaliser and maximum as read, as written, of the chunks; the chunks' forget sums
    float *N, *M, *N_ws, *M_ws, *F_ws;
    float* keep_ws;                    // gla: the chunks' products of decays
    const int32_t* qo_indptr;
    const int64_t* pos0;
    const int32_t* state_slot;
    float* out;
    TurnRows turn;
};

}  // namespace NVX_NS

// phases: 0 a whole portion, 1 a chunk's own memory, 3 a chunk's read-out; defined in scan_mfma.hip
void nvx_launch_scan_mfma(const NVX_NS::ScanArgs& args, int fmt, int mode, int phase, int64_t n_seq, hipStream_t stream);
int nvx_scan_mfma_columns();           // value columns of one of its workgroups
