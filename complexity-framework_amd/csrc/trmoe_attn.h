// Argument blocks and launchers of the decoder's attention kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "trmoe_common.h"

namespace trmoe {

struct RopeArgs {
    const bf16_t* kqv;       // [rows, (kvh + heads + kvh) * 64]: k heads, q heads, v heads
    int64_t ldkqv;
    int64_t rows, T;         // rows = sequences * T
    int heads, kvh;
    const bf16_t* qw;        // norm weights [64]
    const bf16_t* kw;
    float eps;
    const float* cos;        // [positions >= L, 64]
    const float* sin;
    bf16_t* q;               // [rows, heads, 64]
    bf16_t* k;               // [sequences, kvh, L, 64]
    bf16_t* v;
    int64_t L;
    int64_t pos0;            // position of t = 0 (plus *pos when given)
    const int64_t* pos;
};

struct PrefillAttnArgs {
    const bf16_t* q;         // [sequences, T, heads, 64]
    const bf16_t* k;         // [sequences, kvh, L, 64], positions 0 .. T - 1 filled
    const bf16_t* v;
    int64_t T, L;
    int heads, kvh;
    float scale;
    bf16_t* out;             // [sequences, T, heads * 64]
};

struct DecodeAttnArgs {
    const bf16_t* x;         // [B, H] hidden rows
    int64_t ldx;
    int B, H, kvh, n_qkv;
    const bf16_t* norm_w;
    float norm_eps;
    const bf16_t* w_kqv;     // [n_qkv, H]
    const bf16_t* qn_w;
    const bf16_t* kn_w;
    float qk_eps, scale;
    const float* cos;
    const float* sin;
    const int64_t* pos;      // device: the token's position
    bf16_t* k_cache;         // [B, kvh, L, 64]
    bf16_t* v_cache;
    int64_t L;
    float* qkv;              // scratch [B, n_qkv]
    int* counters;           // scratch [B * kvh]
    float* part;             // scratch [B * kvh, splits, group, 66]
    bf16_t* attn;            // [B, heads * 64]
};

int launch_qk_rope(const RopeArgs& a, hipStream_t stream);
int launch_prefill_attn(const PrefillAttnArgs& a, int64_t sequences, hipStream_t stream);
int64_t decode_attn_splits(int64_t L, int pairs);
int launch_decode_attn(const DecodeAttnArgs& a, int group, hipStream_t stream);

}  // namespace trmoe
