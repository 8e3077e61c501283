// tq_encode.h -- the prefill encoders' launch interface (tq_encode.hip), shared by the plain
// (tq_quantize.hip) and the channel-group (tq_group.hip) entry points.
#pragma once

#include "tq_mfma.h"

namespace tqenc {

struct EncodeArgs {
    const uint16_t* x;
    int heads;
    int64_t tokens;
    int64_t n_vec;  // < 2^31
    int64_t x_sb, x_sh, x_st;
    const float* R;           // [D][D], a group's in channel space
    const float* centers;     // Q_prod only
    const float* boundaries;  // [2^bits - 1]
    const float* S;           // Q_prod only, nullptr for Q_mse
    uint8_t* codes;
    uint16_t* norms;
    uint8_t* signs;
    uint16_t* rnorms;
    int64_t out_cap, out_offset;
    uint32_t mask[TQ_DIM / 32];  // channels of the group (all of them for a plain call)
    int sub_dim;                 // rows of R and S that count; TQ_DIM for a plain call
    tqmx::FastDiv tok_div, head_div;
};

// Encodes a call of the prefill sizes: codes and norms, then (S given) signs and residual norms.
// `group`: rows of any alignment, bits 1..8; otherwise bits 1..4 and 16-byte aligned rows.
int launch_encode(EncodeArgs a, int bits, bool group, hipStream_t s);

}  // namespace tqenc
