// What the two forms of the FP32 tree attention share: tv_attention_fp32.hip (matrix instructions)
// and tv_attention_rows.hip (a wave per packed row, for short requests).
#pragma once

#include <math.h>
#include <stdint.h>

#include "tv_internal.h"

namespace tv {

struct Fp32Params {
    const void* q;
    int64_t q_s0, q_s1;
    const void* k;
    const void* v;
    int64_t k_s0, k_s1, k_s2, k_s3;
    int64_t v_s0, v_s1, v_s2, v_s3;
    int64_t num_blocks;
    void* out;
    int64_t o_s0, o_s1;
    int32_t out_dtype;
    const int32_t* cu;
    const int32_t* q2r;
    const int32_t* local;
    const int32_t* plen;
    const int32_t* cnt;
    const int32_t* tables;
    int64_t t_s0;
    const int64_t* tree_slots;
    const float* bias;
    const int64_t* bias_off;
    const void* pslots;
    int64_t ps_s0;
    int32_t ps_i64;
    int32_t num_requests;
    int32_t total_queries;
    int32_t groups;       // query heads per KV head
    int32_t head_dim;
    int32_t block_size;
    float scale;          // softmax scale in the form's score units
    int32_t splits;       // chunks a row block's keys may be cut into
    int32_t slots;        // workgroups the chip runs at a time
    int32_t places;       // workgroups of a launch by list (a cut one has room for their partial rows); 0: by number
    int32_t min_chunk;    // tiles of the shortest chunk a block is cut into
    int32_t kv_heads;
    int32_t vec;          // K/V rows take vector loads
    int32_t q_vec;        // Q rows do
    int64_t unit0;        // first (row block, KV head) of this launch
    float* ws_o;          // partial rows [chunk, KV head, 32, head_dim] (splits > 1)
    float2* ws_ml;        // their (maximum, sum) [chunk, KV head, 32]
    int32_t rows_keys;    // > 0: both forms are launched, and the row form takes a batch whose requests
                          // have at most this many live keys
    int32_t* status;
};

constexpr int kWave = 64;

__device__ __forceinline__ float to_float(float x) { return x; }
__device__ __forceinline__ float to_float(__bf16 x) { return static_cast<float>(x); }
__device__ __forceinline__ float to_float(_Float16 x) { return static_cast<float>(x); }

__device__ __forceinline__ void store_value(const Fp32Params& p, int64_t index, float x) {
    if (p.out_dtype == TV_F32) {
        static_cast<float*>(p.out)[index] = x;
    } else if (p.out_dtype == TV_BF16) {
        static_cast<__bf16*>(p.out)[index] = static_cast<__bf16>(x);
    } else {
        static_cast<_Float16*>(p.out)[index] = static_cast<_Float16>(x);
    }
}

// The longest request's live keys, in every lane.  Both forms decide by it where the host does not
// know the lengths, so a replayed graph takes the form an eager launch takes.
__device__ __forceinline__ int longest_request(const Fp32Params& p) {
    int keys = 0;
    for (int r = threadIdx.x & (kWave - 1); r < p.num_requests; r += kWave) {
        const int nodes = p.cnt[r], prefix = p.plen[r];
        if (nodes > 0 && prefix >= 0) keys = max(keys, prefix > INT32_MAX - nodes ? INT32_MAX : prefix + nodes);
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) keys = max(keys, __shfl_xor(keys, off));
    return keys;
}

// The row form; `p.scale` is the softmax scale itself.
void launch_rows(const Fp32Params& p, int32_t in_dtype, hipStream_t stream);

}  // namespace tv
