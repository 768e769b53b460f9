// FP32 tree attention for every geometry (include/treeverify.h: tv_tree_attention_fp32).
//
// The MI355X form of the reference's scalar FP32 kernel (paged_backend.py:116-213) and
// of its legacy slot-addressed form (paged_backend.py:20-113): the path for batches the
// MFMA kernel does not take (f32 operands, head sizes other than 64, 128 and 256, query
// groups the MFMA kernel is not built for, page sizes that are not multiples of 32, trees
// above 2048 nodes, finite qq_bias values).  The reference runs one program per (packed
// row, query head).
//
// Work split.  The T x G score rows of one request and KV head (row = node * G + query
// head) are cut into blocks of 32.  A workgroup of four waves owns one block and a range of
// the block's visible keys; its waves take the range's 32-key tiles in turn, each with its
// own online softmax, and meet once at the end (LDS).  A wave therefore needs no barrier
// and no staging of K/V: it loads its tiles straight into the operand registers of the
// matrix instructions, and the row blocks of one request find the K/V in L2.  Batches with
// few blocks cut the keys over up to kMaxSplits workgroups per block, whose partial rows a
// second kernel merges.  The cut depends on the live lengths and on the launch's shapes
// only, so a replayed graph computes what an eager launch computes.
//
// Products (per 32-key tile and 32-row block, written transposed so that every per-row
// quantity sits in the two lanes c, c + 32 of row c):
//   S^T[32 keys x 32 rows] = K . Q^T        A: lane (c, g) holds key c, B: score row c
//   O^T[dims x 32 rows]   += V^T . P^T      A: lane (c, g) holds dims 64j + 2c, 2c + 1
//   f32 operands: v_mfma_f32_32x32x2_f32, exact fp32 products with fp32 sums.  Contraction
//     slot g of step (j, i) of K.Q^T is dim 8j + 4g + i (16-byte loads of both); slot g of
//     step v of V^T.P^T is the key that S^T register v of half g holds, so the
//     probabilities feed the product from the registers the scores were computed in.
//   16-bit operands: v_mfma_f32_32x32x16; the fp32 probability is split into three terms of
//     the operand type (its rounding, the rounding of the remainder, and that of the rest),
//     one product each: all 24 bits of it in bf16; in f16 to 2^-39 of the row's reference
//     (Op<_Float16>), which is below what fp32 sums of it keep.
//
// Short requests take the row form (tv_attention_rows.hip; row_form_keys has the rule).
//
// What bounds it.  f32: the matrix core, 8192 cycles a tile and wave (a wave's tile takes 10.7 us
// with two waves a SIMD, 7 us at the core's rate), scratch traffic (16 to 66 spilled VGPRs at
// head sizes 80 to 128), and the uneven lengths of the workgroups.
// 16 bits: the loads and the softmax's vector work (3 us a tile) and the workgroup's fixed time
// (lookups 3, Q and first tile 3, waves' merge 3, partial rows 2.5 us).  Measured, before (a wave
// per packed row, fp32 vector products, K/V staged in LDS) -> now: 8 f32 requests of 310-3304
// keys and 18-64 nodes, 32/8 heads x 128: 525 -> 138 us (5.9 GFLOP; 42 us at the f32 matrix
// rate); 4 bf16 requests of 1204-1998 keys, 24/8 heads x 96, 16-token pages: 490 -> 34 us;
// 2 x 1500-row bf16 chunks, 32/8 x 128: 7.1 -> 0.69 ms; head size 512, bf16: 7.2 -> 0.87 ms.
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "tv_attention_fp32.h"

namespace tv {
namespace {

constexpr int kBlockRows = 32;      // score rows of a workgroup
constexpr int kTile = 32;           // keys of a tile
constexpr int kWaves = 4;           // waves of a workgroup: they take its tiles in turn
constexpr int kThreadsFp32 = kWave * kWaves;
constexpr int kMaxSplits = 16;
constexpr int kCus = 256;           // compute units of an MI355X
constexpr int64_t kCutRows = 4096;  // row blocks times chunks a batch is cut into at most
constexpr int kCutRequests = kWave; // requests of a batch that is cut at most (one lane each)
// Shortest chunk: a workgroup's fixed time (about 15 us: lookups, Q, the waves' merge, the partial
// rows) against its tiles' (a wave's takes 11 us in f32, 3 us in 16 bits).
constexpr int kMinChunk32 = 8, kMinChunk16 = 16;
constexpr int kWholeKeys = 1 << 30;   // as the shortest chunk: nothing is cut
constexpr int32_t kMaxRowKeys = 256;    // the most keys of a request the row form takes
constexpr int64_t kRowRequests = 1024;  // ... and requests (every workgroup reads the lengths of a captured launch)
// Scores and maxima are kept in units of two octaves (natural units * log2(e) / 2): the factor is
// below 1, so that the most negative bias a mask can hold stays a finite score (in log2 units
// torch.finfo(float32).min would become -inf and a row that sees nothing else a NaN).
constexpr float kUnit = 1.4426950408889634f / 2;
// The maximum is subtracted before the factor of two, which would overflow.
__device__ __forceinline__ float exp2_units(float x) { return __builtin_amdgcn_exp2f(2.f * x); }

// The launch numbers the row blocks of request r from start(r) = floor(cu[r] * G / 32) + r on:
// the ranges are disjoint and increasing (start(r + 1) - start(r) >= ceil(T_r * G / 32)), so a
// grid of floor(Q * G / 32) + R + 1 numbers covers every block with at most one idle number per
// request, whatever the (live) node counts.
__device__ __forceinline__ int64_t group_start(const int32_t* cu, int groups, int r) {
    return static_cast<int64_t>(cu[r]) * groups / kBlockRows + r;
}

// The request whose group range holds workgroup b: the last r with start(r) <= b, by a
// 64-way search of the wave (two rounds of loads up to 4096 requests).
__device__ int request_of_group(const int32_t* cu, int groups, int num_requests, int64_t b) {
    const int lane = threadIdx.x & (kWave - 1);
    int lo = 0, hi = num_requests;   // start(lo) <= b; the answer is in [lo, hi)
    while (hi - lo > 1) {
        const int step = (hi - lo + kWave - 1) / kWave;
        const int r = lo + lane * step;
        const bool le = r < hi && group_start(cu, groups, r) <= b;
        const uint64_t mask = __ballot(le);   // lanes 0 .. k set: start() increases with r
        const int last = 63 - __builtin_clzll(mask | 1ull);
        lo += last * step;
        hi = min(hi, lo + step);
    }
    return lo;
}

// One workgroup's work: a row block of a request, and the block's chunk of the visible keys.
struct RowBlock {
    int r, row0, rows, nodes, prefix;   // rows: score rows of the block (<= 32)
    int64_t tree0;                      // the request's first packed row
    int tiles;                          // 32-key tiles any row of the block can see
    int seq;                            // ... keys
    int chunk, part;                    // tiles of a chunk, this workgroup's chunk
    int first;                          // index of the block's first chunk, which places its partial rows
};

// Fills the block `index` of request r, whose live metadata are given; false for an index past
// the request's rows and for a request whose live lengths are malformed.
__device__ __forceinline__ bool block_of_request(const Fp32Params& p, int r, int index, int cu, int nodes, int prefix,
                                                 RowBlock& b, bool report) {
    b.r = r;
    b.row0 = index * kBlockRows;
    b.prefix = prefix;
    b.nodes = nodes;
    b.tree0 = cu;
    b.first = 0;
    const int64_t rows = static_cast<int64_t>(nodes) * p.groups;
    if (b.row0 >= rows) return false;
    const int last = static_cast<int>((min(static_cast<int64_t>(b.row0) + kBlockRows, rows) - 1) / p.groups);
    if (prefix < 0 || cu < 0 || b.tree0 + last >= p.total_queries) {
        if (report && threadIdx.x == 0) set_status(p.status, TV_STATUS_BAD_REQUEST);
        return false;
    }
    b.rows = static_cast<int>(min(static_cast<int64_t>(kBlockRows), rows - b.row0));
    b.seq = prefix + last + 1;
    b.tiles = (b.seq + kTile - 1) / kTile;
    b.chunk = b.tiles;
    b.part = 0;
    return true;
}

// Wave-wide sums and maxima in every lane, with DPP moves (shifts within rows of 16 lanes, then
// row broadcasts: lane 63 ends with the whole); a lane without a source reads 0.
template <int kCtrl, int kRowMask = 0xf>
__device__ __forceinline__ int dpp(int v) {
    return __builtin_amdgcn_update_dpp(0, v, kCtrl, kRowMask, 0xf, false);
}
__device__ __forceinline__ int prefix_sum(int x) {   // inclusive
    x += dpp<0x111>(x);
    x += dpp<0x112>(x);
    x += dpp<0x114>(x);
    x += dpp<0x118>(x);
    x += dpp<0x142, 0xa>(x);
    x += dpp<0x143, 0xc>(x);
    return x;
}
__device__ __forceinline__ int wave_total(int x) { return __builtin_amdgcn_readlane(prefix_sum(x), kWave - 1); }
__device__ __forceinline__ float wave_total(float x) {
    auto move = [](float v, auto f) { return __builtin_bit_cast(float, f(__builtin_bit_cast(int, v))); };
    x += move(x, dpp<0x111>);
    x += move(x, dpp<0x112>);
    x += move(x, dpp<0x114>);
    x += move(x, dpp<0x118>);
    x += move(x, dpp<0x142, 0xa>);
    x += move(x, dpp<0x143, 0xc>);
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), kWave - 1));
}
__device__ __forceinline__ int wave_max(int x) {   // of non-negative values
    x = max(x, dpp<0x111>(x));
    x = max(x, dpp<0x112>(x));
    x = max(x, dpp<0x114>(x));
    x = max(x, dpp<0x118>(x));
    x = max(x, dpp<0x142, 0xa>(x));
    x = max(x, dpp<0x143, 0xc>(x));
    return __builtin_amdgcn_readlane(x, kWave - 1);
}

// The cut of a batch launched by list (p.places > 0, at most kCutRequests requests), the same in
// every wave that computes it: chunks of at most `target` tiles (cut_target), so that
// the workgroups fill the chip once (p.slots of them run at a time: a part-filled second round
// would double the launch), or as many times as the row blocks alone do.  Lane l holds request l.
struct Cut {
    int cu, nodes, prefix;   // the request's live metadata
    int blocks, tiles;       // its row blocks and the tiles of its keys
    int target;
};

__host__ __device__ __forceinline__ int chunks_of(int tiles, int target) {
    return static_cast<int>((static_cast<uint32_t>(tiles) + target - 1) / static_cast<uint32_t>(target));
}
// Tiles of one of `parts` even chunks, in whole turns of the waves.
__device__ __forceinline__ int chunk_tiles(int tiles, int parts) {
    return ((tiles + parts - 1) / parts + kWaves - 1) / kWaves * kWaves;
}

// Shortest chunk, in whole turns of the waves, whose workgroups fit `limit`: count(target) is
// their number, which falls as the target grows and fits for an uncut batch.  The shortest is
// the most even one.  `work` block-tiles over `limit` workgroups are a share no target goes
// below, and the answer is mostly that share or little above it: every wave of the launch
// searches upwards from there, about four counts.
template <class Count>
__host__ __device__ __forceinline__ int cut_target(int longest, int splits, int min_chunk, float work, int limit,
                                                   Count count) {
    const int even = static_cast<int>(fminf(work / limit, 1e9f));
    const int floor = max(max(min_chunk, even), (longest + splits - 1) / splits);
    const int most = (longest + kWaves - 1) / kWaves;   // uncut
    int lo = (floor + kWaves - 1) / kWaves, hi = lo;
    for (int step = 1; hi < most && count(hi * kWaves) > limit; step *= 2) {
        lo = hi + 1;
        hi = min(most, hi + step);
    }
    while (lo < hi) {
        const int mid = lo + (hi - lo) / 2;
        if (count(mid * kWaves) <= limit) hi = mid; else lo = mid + 1;
    }
    return lo * kWaves;
}

__device__ __forceinline__ Cut plan_cut(const Fp32Params& p) {
    Cut cut = {0, 0, 0, 0, 0, 1};
    const int r = threadIdx.x & (kWave - 1);
    if (r < p.num_requests) {
        cut.cu = p.cu[r];
        cut.nodes = p.cnt[r];
        cut.prefix = p.plen[r];
        if (cut.nodes > 0 && cut.prefix >= 0 && cut.nodes <= p.total_queries) {
            cut.blocks = static_cast<int>((static_cast<int64_t>(cut.nodes) * p.groups + kBlockRows - 1) / kBlockRows);
            cut.tiles = static_cast<int>((static_cast<int64_t>(cut.prefix) + cut.nodes + kTile - 1) / kTile);
        } else if (blockIdx.x == 0 && cut.nodes != 0) {
            set_status(p.status, TV_STATUS_BAD_REQUEST);
        }
    }
    const int units = wave_total(cut.blocks) * p.kv_heads;
    const int longest = wave_max(cut.tiles);
    const int slots = p.slots * max(1, (units + p.slots - 1) / p.slots);
    const float work = wave_total(static_cast<float>(cut.blocks) * static_cast<float>(cut.tiles)) * p.kv_heads;
    cut.target = cut_target(longest, p.splits, p.min_chunk, work, slots, [&](int target) {
        return wave_total(cut.blocks * chunks_of(cut.tiles, target)) * p.kv_heads;
    });
    return cut;
}

// The block and chunk of index u (blocks and chunks of request 0 first, chunk fastest); false
// past the last.
__device__ __forceinline__ bool cut_block(const Fp32Params& p, const Cut& cut, int u, RowBlock& b, bool& live) {
    const int parts = chunks_of(cut.tiles, cut.target);
    const int mine = cut.blocks * parts, sum = prefix_sum(mine);
    const uint64_t past = __ballot(sum > u);
    if (!past) return false;
    const int l = __builtin_ctzll(past);
    const int np = __builtin_amdgcn_readlane(parts, l);
    const int index = u - __builtin_amdgcn_readlane(sum - mine, l), block = index / np;
    live = block_of_request(p, l, block, __builtin_amdgcn_readlane(cut.cu, l), __builtin_amdgcn_readlane(cut.nodes, l),
                            __builtin_amdgcn_readlane(cut.prefix, l), b, true);
    if (live) {
        b.chunk = chunk_tiles(__builtin_amdgcn_readlane(cut.tiles, l), np);
        b.part = index - block * np;
        b.first = u - b.part;
        live = b.part * b.chunk < b.tiles;   // an early block sees fewer keys than its request holds
    }
    return true;
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

// The same value, computed where it is used: keeps the many addresses of a rare or strided path
// from being held in registers across the tile loop.
__device__ __forceinline__ int opaque(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

template <typename T>
struct Op;
template <>
struct Op<__bf16> {
    typedef bf16x8_t vec;
    static __device__ __forceinline__ f32x16 mfma(vec a, vec b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    // log2 of the factor the probabilities carry (it cancels against the row sum).
    static constexpr float kShift = 0.f;
    static constexpr float kMargin = 4.f;
};
template <>
struct Op<_Float16> {
    typedef f16x8_t vec;
    static __device__ __forceinline__ f32x16 mfma(vec a, vec b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    // The three terms end at f16's smallest step, 2^-24, so probabilities are scaled up to it as
    // far as f16's range allows: at most 2 before the maximum is raised, 2^15 with the factor.  One
    // is then held to 2^-39 of the row's reference, all 24 bits down to 2^-15 of it, and even 2^15
    // keys rounded the same way shift the sum by no more than fp32's own rounding of it.
    static constexpr float kShift = 14.f;
    static constexpr float kMargin = 0.5f;
};
template <>
struct Op<float> {
    static constexpr float kShift = 0.f;
    static constexpr float kMargin = 4.f;
};

// A score more than Op::kMargin (4: 2^8 in probability) above a row's reference maximum raises
// the maximum; below it probabilities stay <= 2^8, which fp32 holds with its full relative
// precision, so the result is the same online softmax with rare rescales.

// T: operand type; DIM: the head size, or (EXACT false) an upper bound of it in {64, 128, 256,
// 512} with loads and products past p.head_dim left out, and element loads where the rows do not
// take vector ones.
template <typename T, int DIM, bool EXACT>
__device__ __forceinline__ void attend_block(const Fp32Params& p, const RowBlock& b, const int kvh) {
    constexpr bool F32 = sizeof(T) == 4;
    constexpr int DP = (DIM + 63) / 64 * 64;               // padded head size
    constexpr int NB = DP / 32;                            // 32-dim output blocks
    constexpr int SLAB = DP == 128 ? 128 : 64;             // dims of K and V held in registers at a time
    constexpr int SLABS = DP / SLAB;
    constexpr int KSTEP = F32 ? 8 : 16;                    // dims of a 16-byte K load of both lane halves
    constexpr int KV4 = SLAB / KSTEP;                      // K loads per lane and slab
    constexpr int SB = SLAB / 64;                          // 64-dim output pairs per slab
    constexpr int QPITCH = F32 ? DP + 4 : DP / 2 + 4;      // LDS row of Q in 4-byte words: 16-byte reads conflict free
    constexpr int OPITCH = DP + 2;                         // LDS row of O: 8-byte accesses conflict free
    constexpr int Q_WORDS = kBlockRows * QPITCH, O_WORDS = kBlockRows * OPITCH;
    __shared__ __attribute__((aligned(16))) uint32_t smem[Q_WORDS > 2 * O_WORDS ? Q_WORDS : 2 * O_WORDS];
    __shared__ uint64_t rows_lds[kWaves][2][2][kTile];     // addresses of the tile's K and V rows
    __shared__ float2 ml_lds[kWaves][kBlockRows];

    const int tid = threadIdx.x, lane = tid & (kWave - 1), c = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int D = EXACT ? DIM : p.head_dim;
    const int B = p.block_size, G = p.groups;
    const int tbeg = b.part * b.chunk, tend = min(b.tiles, tbeg + b.chunk);

    // This lane's score row.  Its metadata, the first tile's slots and the Q rows are loaded before
    // any of them is used: one round trip instead of four.
    const int row = b.row0 + c;
    const int local = row / G;
    const int64_t packed = b.tree0 + local;
    const int P = b.prefix;
    const bool in_block = c < b.rows;
    const int row_request = in_block ? p.q2r[packed] : b.r, row_local = in_block ? p.local[packed] : local;
    const int64_t bias_base = p.bias_off[b.r];
    const int64_t pool_slots = p.num_blocks * B;
    const float cs = p.scale;

    // Slot of key t0 + c of a tile.  Lanes of half 0 follow the key's K row, those of half 1 its V row.
    const bool pow2 = (B & (B - 1)) == 0;
    const int bshift = __builtin_ctz(B);
    auto slot_load = [&](int t0) __attribute__((always_inline)) -> int64_t {
        const int pos = t0 + c;
        if (pos >= b.seq) return -1;
        if (pos >= P) return p.tree_slots[b.tree0 + (pos - P)];
        if (p.pslots) {
            const int64_t at = static_cast<int64_t>(b.r) * p.ps_s0 + pos;
            return p.ps_i64 ? static_cast<const int64_t*>(p.pslots)[at]
                            : static_cast<int64_t>(static_cast<const int32_t*>(p.pslots)[at]);
        }
        return p.tables[static_cast<int64_t>(b.r) * p.t_s0 + (pow2 ? pos >> bshift : pos / B)];   // the page
    };
    const int64_t s0 = (g ? p.v_s0 : p.k_s0) * static_cast<int64_t>(sizeof(T));
    const int64_t s1 = (g ? p.v_s1 : p.k_s1) * static_cast<int64_t>(sizeof(T));
    const uint64_t head0 = reinterpret_cast<uint64_t>(g ? p.v : p.k) +
                           static_cast<uint64_t>(kvh * (g ? p.v_s2 : p.k_s2) * static_cast<int64_t>(sizeof(T)));
    // The tile's K and V row addresses into the wave's LDS list; returns the tile's present keys,
    // one bit each.
    auto resolve = [&](int t0, int64_t s, int buf) __attribute__((always_inline)) -> uint32_t {
        const int pos = t0 + c;
        int64_t blk = 0, off = 0;
        bool ok = false;
        if (pos < b.seq) {
            if (pos < P && !p.pslots) {
                blk = s;
                off = pow2 ? pos & (B - 1) : pos % B;
                ok = s >= 0 && s < p.num_blocks;
            } else {
                ok = s >= 0 && s < pool_slots;
                if (static_cast<uint64_t>(s) < (1ull << 32)) {
                    blk = static_cast<uint32_t>(s) / static_cast<uint32_t>(B);
                } else {
                    blk = ok ? s / B : 0;
                }
                off = s - blk * B;
            }
            if (!ok && g == 0) set_status(p.status, TV_STATUS_BAD_PAGE);
        }
        // A missing key reads the pool's first row: its score is hidden, and the loads need no
        // conditions.
        uint64_t at = head0;
        if (ok) at += static_cast<uint64_t>(blk * s0 + off * s1);
        rows_lds[wave][buf][g][c] = at;
        return static_cast<uint32_t>(__ballot(ok));
    };

    // K operand registers of one slab: 16 bytes per step (f32: dims 8j + 4g, 16-bit: 16j + 8g).
    u32x4 kr[KV4];
    auto k_load = [&](int buf, int slab) __attribute__((always_inline)) {
        const uint64_t at = rows_lds[wave][buf][0][c];
        const T* k = reinterpret_cast<const T*>(at) + (KSTEP / 2) * g;
#pragma unroll
        for (int j = 0; j < KV4; ++j) {
            const int d = SLAB * slab + KSTEP * j;
            if (EXACT ? d < DIM : d < D) {
                if (EXACT || p.vec) {
                    kr[j] = *reinterpret_cast<const u32x4*>(k + d);
                } else {
                    T e[16 / sizeof(T)];
                    const int dl = d + (KSTEP / 2) * opaque(g);
                    const T* row = reinterpret_cast<const T*>(at);
#pragma unroll
                    for (int i = 0; i < static_cast<int>(16 / sizeof(T)); ++i) {
                        e[i] = dl + i < D ? row[(dl + i) * p.k_s3] : static_cast<T>(0.f);
                    }
                    kr[j] = __builtin_bit_cast(u32x4, e);
                }
            }
        }
    };
    // V operand registers of one slab: for S^T register r the two dims 64j + 2c, + 1 of its key
    // (past D: the last ones again, for output dims that are not stored).
    typedef typename std::conditional<F32, u32x2, uint32_t>::type VPair;
    VPair vr[16][SB];
    auto v_load = [&](int buf, int slab) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const T* v = reinterpret_cast<const T*>(rows_lds[wave][buf][1][8 * (r >> 2) + 4 * g + (r & 3)]);
#pragma unroll
            for (int j = 0; j < SB; ++j) {
                const int d0 = SLAB * slab + 64 * j;
                if (EXACT ? d0 < DIM : d0 < D) {
                    if (EXACT || p.vec) {
                        vr[r][j] = *reinterpret_cast<const VPair*>(v + (EXACT && d0 + 64 <= DIM ? d0 + 2 * c
                                                                                                : min(d0 + 2 * c, D - 2)));
                    } else {
                        const int d = d0 + 2 * opaque(c);
                        T e[2];
                        e[0] = v[min(d, D - 1) * p.v_s3];
                        e[1] = v[min(d + 1, D - 1) * p.v_s3];
                        vr[r][j] = __builtin_bit_cast(VPair, e);
                    }
                }
            }
        }
    };

    f32x16 acc[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) acc[i] = f32x16{};
    float m = -INFINITY, l = 0.f;

    // V values that are not finite would reach rows the product multiplies by zero (keys hidden
    // from a row) or, split into three terms, turn an infinity into a NaN: such keys leave the
    // operand and are added one at a time, to the rows that give them weight.
    auto finite_v = [&](const f32x16& pr, int buf, int slab) __attribute__((always_inline)) {
        // Magnitude bits of a pair: two words (f32) or two halves of one.
        typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
        typedef typename std::conditional<F32, uint32_t, u16x2>::type Mag;
        constexpr uint32_t kInf = F32 ? 0x7f800000u : (std::is_same<T, __bf16>::value ? 0x7f80u : 0x7c00u);
        auto magnitude = [&](int r, int j) __attribute__((always_inline)) -> Mag {
            if constexpr (F32) return max(vr[r][j][0] & 0x7fffffffu, vr[r][j][1] & 0x7fffffffu);
            else return __builtin_bit_cast(u16x2, vr[r][j] & 0x7fff7fffu);
        };
        auto over = [&](Mag x) __attribute__((always_inline)) -> bool {
            if constexpr (F32) return x >= kInf;
            else return x[0] >= kInf || x[1] >= kInf;
        };
        Mag top = magnitude(0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
#pragma unroll
            for (int j = 0; j < SB; ++j) {
                if (EXACT ? SLAB * slab + 64 * j < DIM : SLAB * slab + 64 * j < D) {
                    top = __builtin_elementwise_max(top, magnitude(r, j));
                }
            }
        }
        if (!__any(over(top))) return;
        uint32_t bad = 0;   // the tile's keys with such a value
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            bool here = false;
#pragma unroll
            for (int j = 0; j < SB; ++j) here |= SLAB * slab + 64 * j < D && over(magnitude(r, j));
            const uint64_t both = __ballot(here);
            const int key = 8 * (r >> 2) + (r & 3);
            if (both & 0xffffffffull) bad |= 1u << key;
            if (both >> 32) bad |= 1u << (key + 4);
            if (g ? (both >> 32) != 0 : (both & 0xffffffffull) != 0) {
#pragma unroll
                for (int j = 0; j < SB; ++j) vr[r][j] = VPair{};
            }
        }
        for (; bad; bad &= bad - 1) {
            const int key = __builtin_ctz(bad), reg = 4 * (key >> 3) + (key & 3), half = (key >> 2) & 1;
            float w = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) w = r == reg ? pr[r] : w;
            w = __shfl(w, c + 32 * half);
            const T* v = reinterpret_cast<const T*>(rows_lds[wave][buf][1][key]);
            const int d0 = opaque(8 * g);
#pragma unroll
            for (int n = 0; n < SLAB / 32; ++n) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int d = d0 + SLAB * slab + 64 * (n >> 1) + 16 * (r >> 2) + 2 * (r & 3) + (n & 1);
                    const float x = to_float(v[min(d, D - 1) * p.v_s3]);
                    acc[SLAB / 32 * slab + n][r] += w != 0.f ? w * x : 0.f;
                }
            }
        }
    };

    // Software pipeline of a wave: while tile i is computed, its V loads, the K loads of its next
    // tile and the slot lookup of the one after are in flight.
    const int first = tbeg + wave;
    // A pool without pages has no row to read: the rows come out empty.
    const bool empty = p.num_blocks < 1;
    if (empty && tid == 0) set_status(p.status, TV_STATUS_BAD_PAGE);
    const int count = first < tend && !empty ? (tend - first + kWaves - 1) / kWaves : 0;
    int64_t next_slot = count > 0 ? slot_load(kTile * first) : -1;
    // Q block into LDS (zeros past the block's rows and past D): eight threads a row.
    {
        const int rr = tid >> 3, part = tid & 7;
        constexpr int PER = 16 / sizeof(T), LOADS = (DP + 8 * PER - 1) / (8 * PER);
        const bool here = rr < b.rows;
        const int node = (b.row0 + rr) / G, head = kvh * G + (b.row0 + rr) - node * G;
        const T* q = static_cast<const T*>(p.q) +
                     (here ? (b.tree0 + node) * p.q_s0 + static_cast<int64_t>(head) * p.q_s1 : 0);
        u32x4 x[LOADS];
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int d = PER * (8 * i + part);
            x[i] = u32x4{0u, 0u, 0u, 0u};
            if (p.q_vec) {
                if (here && d < D) x[i] = *reinterpret_cast<const u32x4*>(q + d);
            } else {
                T e[PER];
#pragma unroll
                for (int n = 0; n < PER; ++n) e[n] = here && d + n < D ? q[d + n] : static_cast<T>(0.f);
                x[i] = __builtin_bit_cast(u32x4, e);
            }
        }
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int d = PER * (8 * i + part);
            if (d < DP) *reinterpret_cast<u32x4*>(smem + rr * QPITCH + d * static_cast<int>(sizeof(T)) / 4) = x[i];
        }
    }
    // The metadata must place a request's rows consecutively.
    bool row_ok = in_block;
    if (row_request != b.r || row_local != local) {
        set_status(p.status, TV_STATUS_BAD_REQUEST);
        row_ok = false;
    }
    const int my_end = row_ok ? P + local + 1 : 0;         // this row's visible range
    const float* bias_row = p.bias + (row_ok ? bias_base + static_cast<int64_t>(local) * b.nodes : 0);
    uint32_t valid = 0;
    if (count > 0) {
        valid = resolve(kTile * first, next_slot, 0);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the wave's own list
        k_load(0, 0);
        if (count > 1) next_slot = slot_load(kTile * (first + kWaves));
    }
    __syncthreads();   // Q staged
    for (int i = 0; i < count; ++i) {
        const int t0 = kTile * (first + kWaves * i), buf = i & 1;
        const uint32_t here = valid;
        v_load(buf, 0);
        __builtin_amdgcn_sched_barrier(0);
        // Scores.
        f32x16 s = f32x16{};
#pragma unroll
        for (int slab = 0; slab < SLABS; ++slab) {
            if (slab > 0) k_load(buf, slab);
#pragma unroll
            for (int j = 0; j < KV4; ++j) {
                if (EXACT ? SLAB * slab + KSTEP * j < DIM : SLAB * slab + KSTEP * j < D) {
                    const u32x4 qw = *reinterpret_cast<const u32x4*>(
                        smem + c * QPITCH + (F32 ? SLAB * slab + 8 * j + 4 * g : (SLAB * slab + 16 * j + 8 * g) / 2));
                    if constexpr (F32) {
                        const f32x4 a = __builtin_bit_cast(f32x4, kr[j]), q4 = __builtin_bit_cast(f32x4, qw);
#pragma unroll
                        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], q4[e], s, 0, 0, 0);
                    } else {
                        typedef typename Op<T>::vec V8;
                        s = Op<T>::mfma(__builtin_bit_cast(V8, kr[j]), __builtin_bit_cast(V8, qw), s);
                    }
                }
            }
        }
        if (i + 1 < count) {
            valid = resolve(t0 + kTile * kWaves, next_slot, buf ^ 1);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            k_load(buf ^ 1, 0);
            if (i + 2 < count) next_slot = slot_load(t0 + 2 * kTile * kWaves);
        }
        __builtin_amdgcn_sched_barrier(0);
        // Softmax of the 16 keys this lane holds (key 8 * (r / 4) + 4 * g + r % 4).
        const bool masked = here != ~0u || t0 + kTile > P;
        const float mul = masked ? 1.f : cs;   // masked tiles hold finished scores, the others K.Q
        float mx = -INFINITY;
        if (masked) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = 8 * (r >> 2) + 4 * g + (r & 3), pos = t0 + key;
                bool visible = pos < my_end && ((here >> key) & 1u);
                float x = s[r] * cs;
                if (visible && pos >= P) {
                    const float bias = bias_row[pos - P];
                    visible = bias != -INFINITY;
                    x = fmaf(bias, kUnit, x);
                }
                s[r] = visible ? x : -INFINITY;
                mx = fmaxf(mx, s[r]);
            }
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r] * cs);
        }
        if (__any(mx > m + Op<T>::kMargin)) {   // rare after the first tile
            // Both halves of a row decide on the whole row; rows that do not ask keep their maximum.
            const float row_max = fmaxf(mx, __shfl_xor(mx, 32));
            if (row_max > m + Op<T>::kMargin) {
                const float alpha = exp2_units(m - row_max);   // 0 while m is -inf
                l *= alpha;
#pragma unroll
                for (int n = 0; n < NB; ++n) acc[n] *= alpha;
                m = row_max;
            }
        }
        const float ref = m == -INFINITY ? 0.f : -m;   // a score of -inf gives 0, whatever m
        float l0 = 0.f, l1 = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float pr = __builtin_amdgcn_exp2f(fmaf(fmaf(s[r], mul, ref), 2.f, Op<T>::kShift));
            s[r] = pr;
            if (r & 1) l1 += pr; else l0 += pr;
        }
        l += l0 + l1;
        // P.V.
#pragma unroll
        for (int slab = 0; slab < SLABS; ++slab) {
            if (!EXACT && SLAB * slab >= D) continue;
            if (slab > 0) v_load(buf, slab);
            // f32: a key that no row of a tile is denied needs no care, its infinities and NaNs enter
            // as they would one key at a time.
            if (!F32 || masked) finite_v(s, buf, slab);
#pragma unroll
            for (int j = 0; j < SB; ++j) {
                if (EXACT ? SLAB * slab + 64 * j < DIM : SLAB * slab + 64 * j < D) {
                    f32x16& even = acc[SLAB / 32 * slab + 2 * j];
                    f32x16& odd = acc[SLAB / 32 * slab + 2 * j + 1];
                    if constexpr (F32) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const f32x2 a = __builtin_bit_cast(f32x2, vr[r][j]);
                            even = __builtin_amdgcn_mfma_f32_32x32x2f32(a[0], s[r], even, 0, 0, 0);
                            odd = __builtin_amdgcn_mfma_f32_32x32x2f32(a[1], s[r], odd, 0, 0, 0);
                        }
                    } else {
                        typedef typename Op<T>::vec V8;
#pragma unroll
                        for (int kk = 0; kk < 2; ++kk) {
                            V8 hi, mid, lo;
                            uint32_t we[4], wo[4];
#pragma unroll
                            for (int e = 0; e < 8; ++e) {
                                const float pr = s[8 * kk + e];
                                hi[e] = static_cast<T>(pr);
                                const float r1 = pr - static_cast<float>(hi[e]);
                                mid[e] = static_cast<T>(r1);
                                lo[e] = static_cast<T>(r1 - static_cast<float>(mid[e]));
                            }
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const uint32_t x = vr[8 * kk + 2 * e][j], y = vr[8 * kk + 2 * e + 1][j];
                                we[e] = __builtin_amdgcn_perm(y, x, 0x05040100u);   // low halves of x, y
                                wo[e] = __builtin_amdgcn_perm(y, x, 0x07060302u);   // high halves
                            }
                            const V8 ae = __builtin_bit_cast(V8, we), ao = __builtin_bit_cast(V8, wo);
                            even = Op<T>::mfma(ae, lo, even);
                            odd = Op<T>::mfma(ao, lo, odd);
                            even = Op<T>::mfma(ae, mid, even);
                            odd = Op<T>::mfma(ao, mid, odd);
                            even = Op<T>::mfma(ae, hi, even);
                            odd = Op<T>::mfma(ao, hi, odd);
                        }
                    }
                }
            }
        }
    }

    // Merge of the four waves' softmaxes: the row's maximum and sum, then the O rows in LDS.
    l += __shfl_xor(l, 32);
    if (g == 0) ml_lds[wave][c] = make_float2(m, l);
    __syncthreads();   // every wave is past its Q reads
    float row_m = ml_lds[0][c].x;
#pragma unroll
    for (int w = 1; w < kWaves; ++w) row_m = fmaxf(row_m, ml_lds[w][c].x);
    const float scale_w = m == -INFINITY ? 0.f : exp2_units(m - row_m);
    float* o_lds = reinterpret_cast<float*>(smem);
    // acc block 2j + i, register r of half g: dim 64j + 2 * (8 * (r / 4) + 4 * g + r % 4) + i.
    auto o_at = [&](int buf, int j, int r) __attribute__((always_inline)) -> f32x2* {
        return reinterpret_cast<f32x2*>(o_lds + buf * O_WORDS + c * OPITCH + 64 * j +
                                        2 * (8 * (r >> 2) + 4 * g + (r & 3)));
    };
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[n] *= scale_w;
    auto put = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NB / 2; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) *o_at(buf, j, r) = f32x2{acc[2 * j][r], acc[2 * j + 1][r]};
        }
    };
    auto take = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NB / 2; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const f32x2 x = *o_at(buf, j, r);
                acc[2 * j][r] += x[0];
                acc[2 * j + 1][r] += x[1];
            }
        }
    };
    if (wave >= 2) put(wave - 2);
    __syncthreads();
    if (wave < 2) take(wave);
    if (wave == 1) put(1);   // its own buffer: only wave 1 read it
    __syncthreads();
    if (wave == 0) {
        take(1);
        put(0);
    }
    __syncthreads();
    const bool split = b.tiles > b.chunk;   // this block has further chunks
    const int64_t part = (static_cast<int64_t>(b.first + b.part) * p.kv_heads + kvh) * kBlockRows;
    if (split && tid < kBlockRows) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float2 x = ml_lds[w][tid];
            sum += x.x == -INFINITY ? 0.f : x.y * exp2_units(x.x - row_m);
        }
        p.ws_ml[part + tid] = make_float2(row_m, sum);   // tid < 32: lane tid holds row tid's maximum
    }
    for (int rr = tid / kWave; rr < b.rows; rr += kWaves) {
        float inv = 0.f;
        int64_t base = 0;
        if (!split) {
            float top = ml_lds[0][rr].x, sum = 0.f;
#pragma unroll
            for (int w = 1; w < kWaves; ++w) top = fmaxf(top, ml_lds[w][rr].x);
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const float2 x = ml_lds[w][rr];
                sum += x.x == -INFINITY ? 0.f : x.y * exp2_units(x.x - top);
            }
            inv = 1.f / sum;
            const int node = (b.row0 + rr) / G, head = kvh * G + (b.row0 + rr) % G;
            const int64_t at = b.tree0 + node;
            if (p.q2r[at] != b.r || p.local[at] != node) continue;   // reported above
            base = at * p.o_s0 + static_cast<int64_t>(head) * p.o_s1;
        }
        for (int d = lane; d < D; d += kWave) {
            const float x = o_lds[rr * OPITCH + d];
            if (split) {
                p.ws_o[(part + rr) * D + d] = x;
            } else {
                store_value(p, base + d, x * inv);
            }
        }
    }
}

template <typename T, int DIM, bool EXACT>
__global__ void __launch_bounds__(kThreadsFp32, DIM <= 128 ? 2 : 1)
tree_attention_fp32_kernel(const Fp32Params p) {
    if (p.rows_keys > 0 && longest_request(p) <= p.rows_keys) return;   // the row form's batch
    // Index -> (block, chunk) and KV head, head fastest: with 8 KV heads the blocks and chunks of one
    // head share an XCD (workgroup i runs on XCD i % 8), and so its K/V in that L2.
    RowBlock b;
    if (p.places == 0) {
        const int64_t unit = p.unit0 + blockIdx.x;
        const int64_t number = unit / p.kv_heads;
        const int r = __builtin_amdgcn_readfirstlane(request_of_group(p.cu, p.groups, p.num_requests, number));
        const int index = __builtin_amdgcn_readfirstlane(static_cast<int>(number - group_start(p.cu, p.groups, r)));
        if (block_of_request(p, r, index, p.cu[r], p.cnt[r], p.plen[r], b, true)) {
            attend_block<T, DIM, EXACT>(p, b, static_cast<int>(unit - number * p.kv_heads));
        }
        return;
    }
    // The cut has at most p.places workgroups unless the live metadata hold more row blocks than
    // the launch's shapes allow.
    const Cut cut = plan_cut(p);
    const int u = blockIdx.x / p.kv_heads;
    if (blockIdx.x == 0) {
        const int chunks = wave_total(cut.blocks * chunks_of(cut.tiles, cut.target));
        if (static_cast<int64_t>(chunks) * p.kv_heads > p.places) set_status(p.status, TV_STATUS_BAD_REQUEST);
    }
    bool live;
    if (!cut_block(p, cut, u, b, live) || !live) return;
    attend_block<T, DIM, EXACT>(p, b, blockIdx.x - u * p.kv_heads);
}

// Combines the chunks of the row blocks that were cut: one wave per score row, its partial
// rows read coalesced and all in flight together.
__global__ void __launch_bounds__(kThreadsFp32)
merge_fp32_kernel(const Fp32Params p) {
    const Cut cut = plan_cut(p);
    const int number = blockIdx.x / p.kv_heads, kvh = blockIdx.x % p.kv_heads;
    const int lane = threadIdx.x & (kWave - 1);
    // The request whose numbers hold this one: the last that starts at or before it.
    const bool before = lane < p.num_requests &&
                        static_cast<int64_t>(cut.cu) * p.groups / kBlockRows + lane <= number;
    const int r = 63 - __builtin_clzll(__ballot(before) | 1ull);
    const int cu = __builtin_amdgcn_readlane(cut.cu, r), tiles = __builtin_amdgcn_readlane(cut.tiles, r);
    const int np = chunks_of(tiles, cut.target), mine = cut.blocks * chunks_of(cut.tiles, cut.target);
    const int before_r = __builtin_amdgcn_readlane(prefix_sum(mine) - mine, r);   // chunks of the earlier requests
    const int index = number - static_cast<int>(static_cast<int64_t>(cu) * p.groups / kBlockRows + r);
    RowBlock b;
    if (!block_of_request(p, r, index, cu,
                          __builtin_amdgcn_readlane(cut.nodes, r), __builtin_amdgcn_readlane(cut.prefix, r), b, false) ||
        tiles == 0) {
        return;
    }
    const int chunk = chunk_tiles(tiles, np);
    if (b.tiles <= chunk) return;   // one chunk: the attention kernel wrote the rows
    const int parts = (b.tiles + chunk - 1) / chunk;
    const int64_t step = static_cast<int64_t>(p.kv_heads) * kBlockRows;   // rows from a chunk to the next
    const int64_t first = (static_cast<int64_t>(before_r) + static_cast<int64_t>(index) * np) * step + kvh * kBlockRows;
    if (first + (parts - 1) * step >= static_cast<int64_t>(p.places) * kBlockRows) return;   // reported: no such workgroup
    const int rr = blockIdx.y * kWaves + threadIdx.x / kWave;
    if (rr >= b.rows) return;
    const int node = (b.row0 + rr) / p.groups, head = kvh * p.groups + (b.row0 + rr) % p.groups;
    const int64_t at = b.tree0 + node;
    if (p.q2r[at] != r || p.local[at] != node) return;
    // Lane s holds partial s's maximum and sum.
    const float2 ml = lane < parts ? p.ws_ml[first + lane * step + rr] : make_float2(-INFINITY, 0.f);
    float top = ml.x;
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off));
    const float w = ml.x == -INFINITY ? 0.f : exp2_units(ml.x - top);
    float sum = ml.y * w;
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    const float inv = 1.f / sum;
    const int64_t base = at * p.o_s0 + static_cast<int64_t>(head) * p.o_s1;
    for (int d0 = 0; d0 < p.head_dim; d0 += kWave) {   // every lane takes part in the exchange
        const int d = d0 + lane, dl = min(d, p.head_dim - 1);
        float o = 0.f;
#pragma unroll
        for (int s0 = 0; s0 < kMaxSplits; s0 += 8) {
            float x[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                x[s] = s0 + s < parts ? p.ws_o[(first + (s0 + s) * step + rr) * p.head_dim + dl] : 0.f;
            }
#pragma unroll
            for (int s = 0; s < 8; ++s) o = fmaf(x[s], __shfl(w, s0 + s), o);   // w is 0 past the parts
        }
        if (d < p.head_dim) store_value(p, base + d, o * inv);
    }
}

// Row-block numbers of a launch (group_start) and the chunks its blocks may be cut into, from
// the launch's shapes alone: a batch of kCutRows row blocks or more is not cut.
int64_t row_groups(int64_t total_queries, int64_t num_requests, int64_t groups) {
    return total_queries * groups / kBlockRows + num_requests + 1;
}
int split_count(int64_t total_queries, int64_t num_requests, int64_t groups, int64_t kv_heads) {
    const int64_t units = row_groups(total_queries, num_requests, groups) * kv_heads;
    if (num_requests > kCutRequests) return 1;
    return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(kMaxSplits, kCutRows / units)));
}
int64_t blocks_of(int64_t nodes, int64_t groups) { return (nodes * groups + kBlockRows - 1) / kBlockRows; }
// Workgroups the chip runs at a time (the kernel's launch bounds) and the shortest chunk.
int chip_slots(int32_t head_dim) { return head_dim <= 128 ? 2 * kCus : kCus; }
int min_chunk_tiles(int32_t in_dtype) { return in_dtype == TV_F32 ? kMinChunk32 : kMinChunk16; }
// Head sizes with an instance of their own (vector rows only).
bool own_instance(int32_t d) {
    return d == 64 || d == 80 || d == 96 || d == 112 || d == 128 || d == 192 || d == 256;
}
// Keys of the longest request up to which a batch takes the row form (0: never), from the launch's
// shapes.  The row form's time grows with 64-key tiles (f32, head size 128, one query head a KV
// head: 5 + 5.5 us a tile; four: 7 + 7.5; eight: 11 + 19, always behind), the matrix form's hardly
// within 128 keys (14 us with one score row a request, 20 with 32).  us, row / matrix form, one
// request of 8 KV heads: f32 x 128, 64 keys, 24 rows 10.3 / 20.2; 192 keys, 64 rows 22 / 29; 248
// keys, 8 rows 27 / 24; four heads a KV head, 120 keys, 40 nodes 20.7 / 23.3; 192 keys 29.5 / 29.5;
// f32 x 64, 64 keys, 24 rows 8 / 16.  In 16 bits the instances of their own are ahead from a few
// dozen keys on (x 96, three heads: always; x 80, one head, 64 keys, 24 rows 13 / 18), the shared
// ones, with their padding and element loads, behind for longer (x 72, 192 keys, 64 rows 28 / 35).
// Beyond one round of its workgroups (two a CU, four packed rows each) the row form loses its lead:
// 48 requests of 2 nodes, four heads, 32 keys 15 / 19; of 8 nodes, 64 keys 36 / 32.
int32_t row_form_keys(int64_t total_queries, int64_t num_requests, int64_t groups, int64_t kv_heads, int32_t in_dtype,
                      int32_t head_dim, bool vec) {
    if (groups > 4 || num_requests > kRowRequests) return 0;
    if ((total_queries / 4 + num_requests / 2) * kv_heads > 2 * kCus) return 0;
    const bool own = vec && own_instance(head_dim), f32 = in_dtype == TV_F32, few_heads = groups <= 2;
    const bool full = total_queries * groups >= 20 * num_requests;   // score rows of the average request
    if (!f32 && own) return few_heads ? (full ? (head_dim <= 128 ? 64 : 0) : 32) : 0;
    if (head_dim > 128) return few_heads ? 64 : (full ? 0 : 32);
    const bool longer = f32 && (head_dim > 64 || !own);
    if (few_heads) return longer ? (full ? 256 : 128) : (full ? 192 : 64);
    return full ? (longer ? (own ? 128 : 192) : 64) : 32;
}
// Workgroups of a cut launch: the chip's slots, as many times as the row blocks fill them.
int64_t cut_places(int64_t units, int32_t head_dim) {
    const int64_t slots = chip_slots(head_dim);
    return slots * ((units + slots - 1) / slots);
}
int64_t partial_bytes(int64_t places, int32_t head_dim) {
    return places * kBlockRows * (static_cast<int64_t>(head_dim) * 4 + static_cast<int64_t>(sizeof(float2)));
}

// Rows the vector loads take: unit element stride, 16-byte aligned rows, and a head size
// that divides into steps of two 16-byte pieces (one per lane half).
bool vector_rows(const void* base, const int64_t* stride, int64_t elem, int32_t head_dim) {
    const int64_t per = 16 / elem;
    return stride[3] == 1 && head_dim % (2 * per) == 0 && aligned(base, 16) && stride[0] % per == 0 &&
           stride[1] % per == 0 && stride[2] % per == 0;
}

template <typename T, int DIM, bool EXACT>
void launch_for_dims(const Fp32Params& p, const dim3& grid, hipStream_t s) {
    hipLaunchKernelGGL((tree_attention_fp32_kernel<T, DIM, EXACT>), grid, dim3(kThreadsFp32), 0, s, p);
}

// The head sizes models use are compiled in; the others share an instance per power of two.
template <typename T>
void launch_for_type(const Fp32Params& p, uint32_t units, hipStream_t s) {
    const dim3 grid(p.places == 0 ? units : static_cast<uint32_t>(p.places));
    const int d = p.head_dim;
    if (p.vec && d == 64) {
        launch_for_dims<T, 64, true>(p, grid, s);
    } else if (p.vec && d == 80) {
        launch_for_dims<T, 80, true>(p, grid, s);
    } else if (p.vec && d == 96) {
        launch_for_dims<T, 96, true>(p, grid, s);
    } else if (p.vec && d == 112) {
        launch_for_dims<T, 112, true>(p, grid, s);
    } else if (p.vec && d == 128) {
        launch_for_dims<T, 128, true>(p, grid, s);
    } else if (p.vec && d == 192) {
        launch_for_dims<T, 192, true>(p, grid, s);
    } else if (p.vec && d == 256) {
        launch_for_dims<T, 256, true>(p, grid, s);
    } else if (d <= 64) {
        launch_for_dims<T, 64, false>(p, grid, s);
    } else if (d <= 128) {
        launch_for_dims<T, 128, false>(p, grid, s);
    } else if (d <= 256) {
        launch_for_dims<T, 256, false>(p, grid, s);
    } else {
        launch_for_dims<T, 512, false>(p, grid, s);
    }
    if (p.splits > 1) {
        hipLaunchKernelGGL(merge_fp32_kernel, dim3(units, kBlockRows / kWaves), dim3(kThreadsFp32), 0, s,
                           p);
    }
}

bool valid_dtype(int32_t code) { return code == TV_F32 || code == TV_BF16 || code == TV_F16; }

}  // namespace
}  // namespace tv

using namespace tv;

extern "C" int64_t tv_sizeof_tree_attention_fp32_args(void) { return sizeof(tv_tree_attention_fp32_args); }

extern "C" int64_t tv_tree_attention_fp32_workspace_bytes(int32_t total_queries, int32_t num_requests,
                                                          int32_t num_q_heads, int32_t num_kv_heads,
                                                          int32_t head_dim) {
    if (total_queries < 1 || num_requests < 1 || num_kv_heads < 1 || num_q_heads < num_kv_heads || head_dim < 1) return 0;
    const int64_t groups = num_q_heads / num_kv_heads;
    const int splits = split_count(total_queries, num_requests, groups, num_kv_heads);
    if (splits == 1) return 0;
    return partial_bytes(cut_places(row_groups(total_queries, num_requests, groups) * num_kv_heads, head_dim), head_dim);
}

extern "C" int64_t tv_tree_attention_fp32_keys_workspace_bytes(int32_t total_queries, int32_t num_requests,
                                                               int32_t num_q_heads, int32_t num_kv_heads,
                                                               int32_t head_dim, int32_t in_dtype, int32_t max_keys) {
    if (max_keys > 0 && max_keys <= min_chunk_tiles(in_dtype) * kTile) return 0;   // never cut
    return tv_tree_attention_fp32_workspace_bytes(total_queries, num_requests, num_q_heads, num_kv_heads, head_dim);
}

extern "C" int tv_tree_attention_fp32_chunk_keys(const int32_t* prefix_lens_host, const int32_t* node_counts_host,
                                                 int32_t num_requests, int32_t num_q_heads, int32_t num_kv_heads,
                                                 int32_t head_dim, int32_t in_dtype, int32_t* chunk_keys,
                                                 int32_t* workgroups) {
    clear_error();
    if (!prefix_lens_host || !node_counts_host || !chunk_keys || !workgroups) {
        return fail(TV_ERR_INVALID, "tree_attention_fp32_chunk_keys: null argument");
    }
    if (num_requests < 1 || num_kv_heads < 1 || num_q_heads < num_kv_heads || num_q_heads % num_kv_heads ||
        head_dim < 1 || !valid_dtype(in_dtype)) {
        return fail(TV_ERR_INVALID, "tree_attention_fp32_chunk_keys: invalid geometry");
    }
    const int64_t groups = num_q_heads / num_kv_heads;
    int64_t queries = 0, units = 0, longest = 0;
    double work = 0;
    for (int32_t r = 0; r < num_requests; ++r) {
        const int64_t keys = static_cast<int64_t>(prefix_lens_host[r]) + node_counts_host[r];
        if (prefix_lens_host[r] < 0 || node_counts_host[r] < 0 || keys > INT32_MAX - kTile) {
            return fail(TV_ERR_INVALID, "tree_attention_fp32_chunk_keys: invalid lengths of request %d", r);
        }
        queries += node_counts_host[r];
        if (node_counts_host[r] == 0) continue;
        units += blocks_of(node_counts_host[r], groups) * num_kv_heads;
        longest = std::max(longest, (keys + kTile - 1) / kTile);
        work += static_cast<double>(blocks_of(node_counts_host[r], groups) * num_kv_heads) * ((keys + kTile - 1) / kTile);
    }
    *chunk_keys = 0;
    *workgroups = static_cast<int32_t>(units);
    const int splits = split_count(queries, num_requests, groups, num_kv_heads);
    if (splits == 1 || longest == 0) return TV_OK;
    auto count = [&](int target) {
        int64_t n = 0;
        for (int32_t r = 0; r < num_requests; ++r) {
            if (node_counts_host[r] == 0) continue;
            const int tiles = static_cast<int>((static_cast<int64_t>(prefix_lens_host[r]) + node_counts_host[r] + kTile - 1) / kTile);
            n += blocks_of(node_counts_host[r], groups) * chunks_of(tiles, target);
        }
        return static_cast<int>(n * num_kv_heads);
    };
    const int slots = chip_slots(head_dim);
    const int limit = static_cast<int>(slots * std::max<int64_t>(1, (units + slots - 1) / slots));
    const int target = cut_target(static_cast<int>(longest), splits, min_chunk_tiles(in_dtype),
                                  static_cast<float>(work), limit, count);
    *chunk_keys = target * kTile;
    *workgroups = count(target);
    return TV_OK;
}

extern "C" int tv_tree_attention_fp32(const tv_tree_attention_fp32_args* a, void* stream) {
    return tv_tree_attention_fp32_keys(a, 0, nullptr, 0, stream);
}

extern "C" int tv_tree_attention_fp32_split(const tv_tree_attention_fp32_args* a, void* workspace,
                                            int64_t workspace_bytes, void* stream) {
    return tv_tree_attention_fp32_keys(a, 0, workspace, workspace_bytes, stream);
}

extern "C" int tv_tree_attention_fp32_keys(const tv_tree_attention_fp32_args* a, int32_t max_keys, void* workspace,
                                           int64_t workspace_bytes, void* stream) {
    clear_error();
    if (!a) return fail(TV_ERR_INVALID, "tree_attention_fp32: null args");
    if (a->num_requests < 1 || a->total_queries < 0) return fail(TV_ERR_INVALID, "tree_attention_fp32: invalid counts");
    if (a->num_kv_heads < 1 || a->num_q_heads < a->num_kv_heads || a->num_q_heads % a->num_kv_heads) {
        return fail(TV_ERR_INVALID, "tree_attention_fp32: %d query heads over %d KV heads", a->num_q_heads,
                    a->num_kv_heads);
    }
    if (a->num_kv_heads > 65535) return fail(TV_ERR_UNSUPPORTED, "tree_attention_fp32: more than 65535 KV heads");
    const int64_t units = row_groups(a->total_queries, a->num_requests, a->num_q_heads / a->num_kv_heads) *
                          a->num_kv_heads;
    if (a->head_dim < 1 || a->head_dim > 512) {
        return fail(TV_ERR_UNSUPPORTED, "tree_attention_fp32: head_dim %d (implemented: 1..512)", a->head_dim);
    }
    if (a->block_size < 1 || a->num_blocks < 0 || a->num_blocks > (int64_t{1} << 62) / a->block_size) {
        return fail(TV_ERR_INVALID, "tree_attention_fp32: invalid pool geometry");
    }
    if (!valid_dtype(a->in_dtype) || !valid_dtype(a->out_dtype)) {
        return fail(TV_ERR_INVALID, "tree_attention_fp32: dtypes must be TV_F32, TV_BF16 or TV_F16");
    }
    if (!isfinite(a->scale)) return fail(TV_ERR_INVALID, "tree_attention_fp32: softmax scale must be finite");
    if (a->prefix_slots && a->prefix_slots_stride < 0) {
        return fail(TV_ERR_INVALID, "tree_attention_fp32: negative prefix slot stride");
    }
    if (max_keys < 0) return fail(TV_ERR_INVALID, "tree_attention_fp32: negative key count");
    if (a->total_queries == 0) return TV_OK;
    if (!a->q || !a->k_pool || !a->v_pool || !a->out || !a->cu_seqlens_q || !a->query_to_request ||
        !a->query_local_row || !a->prefix_lens || !a->node_counts || !a->tree_slots || !a->qq_bias ||
        !a->qq_bias_offsets || (!a->prefix_slots && !a->block_tables)) {
        return fail(TV_ERR_INVALID, "tree_attention_fp32: null pointer");
    }
    Fp32Params p;
    p.q = a->q;
    p.q_s0 = a->q_stride_row;
    p.q_s1 = a->q_stride_head;
    p.k = a->k_pool;
    p.v = a->v_pool;
    p.k_s0 = a->k_stride[0];
    p.k_s1 = a->k_stride[1];
    p.k_s2 = a->k_stride[2];
    p.k_s3 = a->k_stride[3];
    p.v_s0 = a->v_stride[0];
    p.v_s1 = a->v_stride[1];
    p.v_s2 = a->v_stride[2];
    p.v_s3 = a->v_stride[3];
    p.num_blocks = a->num_blocks;
    p.out = a->out;
    p.o_s0 = a->out_stride_row;
    p.o_s1 = a->out_stride_head;
    p.out_dtype = a->out_dtype;
    p.cu = a->cu_seqlens_q;
    p.q2r = a->query_to_request;
    p.local = a->query_local_row;
    p.plen = a->prefix_lens;
    p.cnt = a->node_counts;
    p.tables = a->block_tables;
    p.t_s0 = a->block_table_stride;
    p.tree_slots = a->tree_slots;
    p.bias = a->qq_bias;
    p.bias_off = a->qq_bias_offsets;
    p.pslots = a->prefix_slots;
    p.ps_s0 = a->prefix_slots_stride;
    p.ps_i64 = a->prefix_slots_is_int64 != 0;
    p.num_requests = a->num_requests;
    p.total_queries = a->total_queries;
    p.groups = a->num_q_heads / a->num_kv_heads;
    p.head_dim = a->head_dim;
    p.block_size = a->block_size;
    p.scale = a->scale * kUnit;
    p.status = a->status;
    p.kv_heads = a->num_kv_heads;
    p.splits = 1;
    p.places = 0;
    p.ws_o = nullptr;
    p.ws_ml = nullptr;
    if (workspace && (max_keys == 0 || max_keys > min_chunk_tiles(a->in_dtype) * kTile)) {
        const int splits = split_count(a->total_queries, a->num_requests, p.groups, a->num_kv_heads);
        if (splits > 1) {
            if (!aligned(workspace, 16)) return fail(TV_ERR_INVALID, "tree_attention_fp32: unaligned workspace");
            const int64_t places = cut_places(units, a->head_dim), bytes = partial_bytes(places, a->head_dim);
            if (workspace_bytes < bytes) {
                return fail(TV_ERR_CAPACITY, "tree_attention_fp32: workspace of %lld bytes, %lld needed",
                            (long long)workspace_bytes, (long long)bytes);
            }
            p.places = static_cast<int32_t>(places);
            p.splits = splits;
            p.slots = chip_slots(a->head_dim);
            p.min_chunk = min_chunk_tiles(a->in_dtype);
            // (maximum, sum) pairs first: 8-byte aligned whatever the head size.
            p.ws_ml = static_cast<float2*>(workspace);
            p.ws_o = reinterpret_cast<float*>(p.ws_ml + places * kBlockRows);
        }
    }
    // Whole keys, but more numbers than the chip takes at once: the idle numbers between the requests'
    // blocks (group_start) would alternate with live ones and leave places empty, so the blocks are
    // listed as a cut batch's are (48 f32 requests of 8 nodes and 248 keys, 32/8 heads x 128: 92 us
    // by number, 55 listed; up to one round the search costs a microsecond for nothing, and beyond
    // 2048 numbers most are live: of 60 nodes at head size 64, 154 by number, 165 listed).
    if (p.places == 0 && a->num_requests <= kCutRequests && units > chip_slots(a->head_dim) &&
        units <= kCutRows / 2) {
        p.places = static_cast<int32_t>(units);
        p.slots = chip_slots(a->head_dim);
        p.min_chunk = kWholeKeys;
    }
    const int64_t elem = a->in_dtype == TV_F32 ? 4 : 2;
    p.vec = vector_rows(a->k_pool, a->k_stride, elem, a->head_dim) &&
            vector_rows(a->v_pool, a->v_stride, elem, a->head_dim);
    const int64_t per = 16 / elem;
    p.q_vec = aligned(a->q, 16) && a->q_stride_row % per == 0 && a->q_stride_head % per == 0 && a->head_dim % per == 0;
    // A batch whose lengths the host knows takes its form here; otherwise both are launched and
    // the one that is not the batch's exits (4 to 5 us of empty launches for a short batch).
    hipStream_t s = as_stream(stream);
    const int32_t rows_keys = row_form_keys(a->total_queries, a->num_requests, p.groups, a->num_kv_heads, a->in_dtype,
                                            a->head_dim, p.vec);
    static_assert(kMaxRowKeys <= kTile * kMinChunk32 && kMaxRowKeys <= kTile * kMinChunk16, "such a batch is never cut");
    p.rows_keys = 0;
    if (rows_keys > 0 && max_keys <= rows_keys) {
        Fp32Params rows = p;
        rows.scale = a->scale;
        if (max_keys == 0) rows.rows_keys = p.rows_keys = rows_keys;
        launch_rows(rows, a->in_dtype, s);
        if (max_keys > 0) return check_launch("tree_attention_fp32");
    }
    // A grid holds 2^32 threads: a huge batch takes several launches.
    constexpr int64_t kLaunchUnits = int64_t{1} << 23;
    for (p.unit0 = 0; p.unit0 < units; p.unit0 += kLaunchUnits) {
        const uint32_t count = static_cast<uint32_t>(std::min(kLaunchUnits, units - p.unit0));
        if (a->in_dtype == TV_F32) {
            launch_for_type<float>(p, count, s);
        } else if (a->in_dtype == TV_BF16) {
            launch_for_type<__bf16>(p, count, s);
        } else {
            launch_for_type<_Float16>(p, count, s);
        }
    }
    return check_launch("tree_attention_fp32");
}
