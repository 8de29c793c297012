// Shared by the attention kernels (attention.hip, attention_f32.hip).
#pragma once

#include "common.h"

namespace idolq {

struct AttnParams {
    const void* q;
    const void* k;
    const void* v;
    void* out;
    int dt, out_dt;
    int64_t lq, lk, heads, head_dim;
    int64_t ldq, ldkv, q_bs, kv_bs, ldo, o_bs;
    float scale_log2;  // log2(e) / sqrt(head_dim)
    // V staged ahead of attn_mfma_hd64<bf16, true> by attn_v_tiles: fp16 V^T tiles and their exponents
    const uint16_t* vt;
    const int* vexps;
    int64_t ntiles;
    int out_vec;  // out has the input dtype and 16-byte aligned rows and batches: rows go out as 16-byte stores
    int64_t batch;
};

// attention_f32.hip: fp32 inputs, head_dim 32 or 64, 16-byte aligned rows, 32 key rows within 2^31 bytes.
struct AttnF32Plan {
    int waves;  // per workgroup, 32 queries each; 0: attn_f32_mfma is cheaper
    int parts;  // the key range is cut into (1: no workspace is used)
};
AttnF32Plan attn_f32_plan(int64_t batch, int64_t lq, int64_t lk, int64_t heads, int64_t head_dim);
size_t attn_f32_workspace_bytes(int64_t batch, int64_t lq, int64_t heads, int64_t head_dim, int parts);
int launch_attn_f32_split(const AttnParams& p, AttnF32Plan plan, float* workspace, hipStream_t s);

}  // namespace idolq
