// Causal attention over a KV cache, the step after the qkv projection of a
// decode or prefill pass (reference: cuda_attention.h:8-39, attention_single
// and attention_split in cuda_attention.cu:39-285, attention_cuda :339-362).
//
// Row i of a call sits at position *pos + i and attends to cached positions
// [0, *pos + i]; query head h reads kv head h / (n_heads / n_kv_heads).
// out[i][h*hs + d] = sum_t softmax_t(q . k_t / sqrt(hs)) v_t[d]. The position
// is read on the device, so one captured graph serves every position.
//
// Two kernels, both for 256-thread workgroups of four wave64s:
//
//  * split (decode, few rows): workgroup (head group, row, chunk) covers one
//    chunk of the context for the G query heads that share a kv head, so a
//    key or value row is loaded once for all G. A position's key and value
//    are read by a power-of-two group of lanes, float4 each, contiguous
//    across the group; every key and value of a 64-position round is loaded
//    before any is used, and the dot products are finished with xor shuffles
//    inside the wave. Each lane group keeps an online softmax of its
//    positions in registers; the groups are merged in LDS in a fixed order.
//    The chunk's softmax is left unnormalised (max m, sum l, exp-weighted
//    values o) in scratch, and a second kernel merges the chunks of each
//    (row, head) in chunk order. The merge is a separate launch rather than a
//    "last workgroup merges" arrival: on gfx950 every cross-workgroup arrival
//    measured slower than a second launch, and the fixed merge order keeps
//    results bit-identical across calls. A context that fits one chunk is
//    normalised and written by the first kernel; the merge kernel then exits.
//    With more rows (prefill), automatic runs the tile kernel (16
//    query rows per wave on fp32 MFMA), split over the context as well when
//    its grid is small, or for large grids the 64-row kernel (bf16 MFMA, keys
//    and values shared through LDS); for head sizes it is not built for, the same split
//    kernel with one chunk per row: the whole context in rounds, no merge.
//  * single_block (on request): workgroup (head, row) holds the query and
//    the scores of the whole context in LDS; any head size.
//
// The grid is sized for seq_len, never for the position: chunks past the end
// of a row's context return at once.
#include <algorithm>
#include <cmath>
#include <string>

#include "common.hpp"
#include "internal.hpp"

namespace em {
namespace {

// Chunks per (row, head group), at most: past 128 the merge's extra chunks
// cost more than the shorter chunks save (context 16384, 32 heads / 8 kv
// heads: 105.4 / 39.3 us at 256, 103.5 / 36.5 at 128; shorter contexts
// never reach the cap).
constexpr int kMaxSplits = 128;
constexpr std::size_t kSplitMaxRows = 12;  // automatic: split up to this many rows, at most
constexpr std::size_t kMaxLds = 64 * 1024;  // dynamic LDS per workgroup

// Query heads per split workgroup: the most of 8, 4, 2, 1 that divides the
// heads sharing a kv head.
int heads_per_block(const AttnShape& s) {
    const int group = s.n_heads / s.n_kv_heads;
    for (int g : {8, 4, 2})
        if (group % g == 0) return g;
    return 1;
}

// Positions per split workgroup, at least (split_chunk).
int min_chunk(const AttnShape& s) {
    return heads_per_block(s) > 1 ? kSplitMinChunkGrouped : kSplitMinChunk;
}

int split_count(const AttnShape& s) {
    const int mc = min_chunk(s);
    const int n = (s.seq_len + mc - 1) / mc;
    return n < kMaxSplits ? n : kMaxSplits;
}

int split_chunk_cap(const AttnShape& s) {
    return split_chunk(s.seq_len, split_count(s), min_chunk(s));
}

std::size_t single_lds(const AttnShape& s) {
    return (static_cast<std::size_t>(s.head_size) + s.seq_len + kThreads) * sizeof(float);
}

// Lanes per position of the split kernel: head_size / 4 rounded up to a
// power of two in [4, 64]; F float4 columns per lane.
int split_lanes(const AttnShape& s) {
    const int hs4 = s.head_size / 4;
    int l = 4;
    while (l < hs4 && l < kWave) l <<= 1;
    return l;
}
int split_f(const AttnShape& s) { return (s.head_size / 4 + split_lanes(s) - 1) / split_lanes(s); }

// LDS of the in-kernel merge (merge_chunks): one float4 and one (max, sum)
// pair per thread.
constexpr std::size_t kMergeLds = kThreads * (sizeof(floatx4) + sizeof(float2));

// Slot merge buffers, plus with RoPE fused the G queries, key and value (and
// at least the in-kernel merge's buffers when it merges its own chunks).
std::size_t split_lds(const AttnShape& s, bool rope = false, bool merge_inside = false) {
    const std::size_t G = heads_per_block(s), hs = s.head_size;
    const std::size_t ns = kThreads / split_lanes(s);
    const std::size_t lds = (G * ns * hs + 2 * G * ns + (rope ? (G + 2) * hs : 0)) * sizeof(float);
    return merge_inside && lds < kMergeLds ? kMergeLds : lds;
}

struct SplitScratch {
    std::size_t o, ml, total;  // offsets and size in floats
};

SplitScratch split_scratch(const AttnShape& s, std::size_t rows) {
    const std::size_t blocks = rows * s.n_heads * split_count(s);
    auto up4 = [](std::size_t x) { return (x + 3) / 4 * 4; };
    SplitScratch l{};
    l.o = 0;
    l.ml = up4(blocks * s.head_size);
    l.total = l.ml + up4(2 * blocks);
    return l;
}

// automatic: the split kernel with chunks across workgroups for few rows,
// beyond that the tile kernel (16 query rows per wave on fp32 MFMA, each key
// and value row loaded once per 16 rows, split over the context when its
// grid is small) for head sizes it is built for; other head sizes run the
// split kernel with one chunk per row (the whole context, in rounds of 64
// positions, no merge) from 13 rows. The split kernel's cost grows with the
// rows (each reads its chunks' keys and values); the split tile kernel's
// hardly does below 16. Measured at 7B shapes (MHA / 8 kv heads), split
// against split tile, us:
//   context  256, 2-12 rows: 10.0-14.5 / 15.4-15.7, 12.0-14.8 / 14.2-15.4
//   context 1024, 4 rows:    18.2 / 18.5, 14.9 / 17.4; 8 rows: 25.1 / 19.0, 20.9 / 17.9
//   context 4096, 4 rows:    48.4 / 41.0, 31.6 / 33.7; 8 rows: 75.4 / 41.1, 51.8 / 33.9
// The context is read on the device, so the cut goes by seq_len: up to 5
// rows split when seq_len exceeds 512, up to 12 otherwise (and for head
// sizes the tile kernel does not take).
constexpr int kAttnWhole = 3;
constexpr int kAttnTile = 4;
constexpr int kTileRows = 16;        // query rows per tile wave
constexpr int kTileMaxHeadSize = 128;

bool tile_supports(const AttnShape& s) {
    return s.head_size % 16 == 0 && s.head_size <= kTileMaxHeadSize;
}

// A tile grid of a few row tiles has one workgroup per (head, 16 rows): 32
// workgroups for 16 rows of a 32-head model, which took 108-114 us at
// context 4096 whatever the row count. Such a grid is split over the
// context as well, into chunks of at least kTileChunkMin positions, enough
// to bring it near kTileTargetGroups workgroups; each chunk leaves its
// unnormalised softmax for the merge kernel, as the split kernel's do.
// Grids of 512 workgroups or more are not split.
constexpr int kTileChunkMin = 256;
constexpr long long kTileTargetGroups = 1024;

int tile_splits(const AttnShape& s, std::size_t rows) {
    const long long tiles = static_cast<long long>(s.n_heads) *
                            static_cast<long long>((rows + kTileRows - 1) / kTileRows);
    if (tiles >= kTileTargetGroups / 2) return 1;
    const long long want = (kTileTargetGroups + tiles - 1) / tiles;
    const long long cap = (s.seq_len + kTileChunkMin - 1) / kTileChunkMin;
    return static_cast<int>(std::max(1LL, std::min(want, cap)));
}

// Positions per chunk: a multiple of 64, so chunks are whole 16-position
// blocks, and splits chunks cover seq_len.
int tile_chunk(const AttnShape& s, int splits) {
    const int c = (s.seq_len + splits - 1) / splits;
    return (c + 63) / 64 * 64;
}

SplitScratch tile_scratch(const AttnShape& s, std::size_t rows, int splits) {
    const std::size_t blocks = rows * s.n_heads * static_cast<std::size_t>(splits);
    auto up4 = [](std::size_t x) { return (x + 3) / 4 * 4; };
    SplitScratch l{};
    l.o = 0;
    l.ml = up4(blocks * s.head_size);
    l.total = l.ml + up4(2 * blocks);
    return l;
}

std::size_t split_max_rows(const AttnShape& s) {
    return tile_supports(s) && s.seq_len > 512 ? 5 : kSplitMaxRows;
}

int resolve(int kernel, std::size_t rows, const AttnShape& s) {
    if (kernel != kAttnAutomatic) return kernel;
    if (rows <= split_max_rows(s)) return kAttnSplit;
    return tile_supports(s) ? kAttnTile : kAttnWhole;
}

struct AttnArgs {
    int n_heads, head_size, group, seq_len, splits, chunk_cap, rows;
    int min_chunk;   // split_chunk's least chunk for this shape
    int whole;       // contexts of up to this many positions are one chunk
    int group_chunk_min;  // grouped tile kernel: least positions per chunk (0: not it)
    int merge_from;  // the merge kernel takes rows of at least this many chunks (>= 2)
    int tile_chunk;  // tile kernel split over the context: positions per chunk (0: no split)
    int q_stride, kv_stride, out_stride;
    const int* pos;
    const float* q;
    const float* kc;
    const float* vc;
    float* part_o;
    float2* part_ml;
    float* out;
    // One-row decode with RoPE fused (attn_split_kernel<..., true>): the qkv
    // product as its consumers read it (q at column 0, k at dim, v at
    // dim + kv_dim), the rotation tables, and the caches to write.
    Summed src;
    int dim, kv_dim;
    const float* cos_t;
    const float* sin_t;
    float* kc_w;
    float* vc_w;
    // Non-null: a row split over several chunks is merged by the last of
    // its chunks' workgroups to finish (one counter per row and head group,
    // zero between calls), not by a merge launch.
    unsigned* merge_count;
};

// Positions per chunk of the grouped tile kernel for a call whose last row has
// n_ctx: whole 16-position blocks.
__device__ __forceinline__ int group_chunk(int n_ctx, int splits, int least) {
    const int c = (n_ctx + splits - 1) / splits;
    return ((c > least ? c : least) + 15) / 16 * 16;
}

// Lanes per key row: hs4 rounded up to a power of two, at most one wave.
__device__ __forceinline__ int lanes_per_row(int n) {
    int l = 1;
    while (l < n && l < kWave) l <<= 1;
    return l;
}

// Positions a lane group loads per round, at most: all of a round's key and
// value loads are issued before any is used.
constexpr int kRoundPerSlot = 8;

constexpr int kMergeDims = 8;
constexpr int kSc1 = 16;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));  // the cache-policy operand's sc1 bit (device-coherent access)

// The merge of the n chunks of heads h0 .. h0 + G - 1 of row i, inside the
// split launch by the last of the row's chunk workgroups: the arithmetic of
// attn_merge_kernel (below), which a merge launch would run, in the same
// slots and order, so the result has its bits. Each (head, group of dpw
// float4 columns) the merge kernel gives a workgroup is given a team of
// used x dpw threads here, as many teams at once as 256 threads hold. The
// chunks' partials, stored by other workgroups of this launch, are read with
// device-coherent (sc1) loads.
__device__ void merge_chunks(const AttnArgs& a, int i, int h0, int G, int n, float* lds) {
    const int hs4 = a.head_size / 4;
    const int dpw = hs4 < kMergeDims ? hs4 : kMergeDims, groups = (hs4 + dpw - 1) / dpw;
    const int slots = kThreads / dpw, used = min(slots, (n + 7) / 8);
    const int T = used * dpw, teams = kThreads / T, combos = G * groups;
    floatx4* red4 = reinterpret_cast<floatx4*>(lds);
    float2* red_ml = reinterpret_cast<float2*>(red4 + kThreads);
    const __amdgpu_buffer_rsrc_t ors =
        __builtin_amdgcn_make_buffer_rsrc(a.part_o, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t mrs =
        __builtin_amdgcn_make_buffer_rsrc(a.part_ml, 0, 0x7fffffff, 0x00020000);
    const int tid = threadIdx.x, team = tid / T, w = tid % T, r = w / dpw, dd = w % dpw;
    for (int base = 0; base < combos; base += teams) {
        const int combo = base + team;
        const bool active = team < teams && combo < combos;
        const int g = active ? combo / groups : 0;
        const int d = (active ? combo % groups : 0) * dpw + dd;
        const bool dok = d < hs4;
        const int dl = dok ? d : hs4 - 1;  // past the head: computed, not stored
        const uint32_t b = static_cast<uint32_t>((i * a.n_heads + h0 + g) * a.splits);
        if (active) {
            float m = -INFINITY, l = 0.0f;
            floatx4 acc{0.f, 0.f, 0.f, 0.f};
            for (int c0 = r; c0 < n; c0 += 8 * used) {
                float2 ml[8];
                floatx4 o[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint32_t c = b + min(c0 + u * used, n - 1);
                    ml[u] = __builtin_bit_cast(
                        float2, __builtin_amdgcn_raw_buffer_load_b64(mrs, c * 8, 0, kSc1));
                    o[u] = __builtin_bit_cast(
                        floatx4, __builtin_amdgcn_raw_buffer_load_b128(ors, (c * hs4 + dl) * 16, 0, kSc1));
                }
                merge_batch8(m, l, acc, ml, o, c0, used, n);
            }
            red4[team * T + r * dpw + dd] = acc;
            if (dd == 0) red_ml[team * used + r] = make_float2(m, l);
        }
        __syncthreads();
        if (active && w < dpw && dok) {
            reinterpret_cast<floatx4*>(a.out + static_cast<std::size_t>(i) * a.out_stride +
                                       static_cast<std::size_t>(h0 + g) * a.head_size)[d] =
                merge_combine(used, floatx4{0.f, 0.f, 0.f, 0.f},
                              [&](int rr) { return red_ml[team * used + rr]; },
                              [&](int rr) { return red4[team * T + rr * dpw + w]; });
        }
        __syncthreads();
    }
}

// Split workgroup: (head group hg, row i, chunk s). Thread = (slot, sub): the
// LPP lanes of a slot share a position and hold float4 columns
// d = sub + f * LPP of it (F per lane). Each slot keeps an online softmax of
// its positions in registers (running max m, sum l, weighted values o) for
// the G heads; the NS = 256 / LPP slots are then merged in LDS in slot order.
//
// ROPE (one row, the forward pass's decode step): the query is not read
// from a.q but formed here from the qkv product (a.src): summed, rotated as
// rope_cache_kernel rotates it (rope_pair), into LDS. The last chunk also
// forms the current position's key and value, writes them to the caches
// (the workgroup of the first head group of each kv head) and takes that
// position in slot 0 after its loop, from LDS: no workgroup reads a cache
// row written in the same launch.
//
// PIPE: the next round's keys are loaded once this round's are used, beside
// its softmax and values, and its values after them, in the same registers
// (up to four heads keep to 128, so four workgroups share a CU). split_pipes
// says where.
template <int G, int LPP, int F, bool ROPE = false, bool PIPE = false>
__global__ __launch_bounds__(kThreads, PIPE && G <= 4 ? 4 : 1) void attn_split_kernel(AttnArgs a) {
    constexpr int NS = kThreads / LPP;
    constexpr int MC = G > 1 ? kSplitMinChunkGrouped : kSplitMinChunk;  // min_chunk of the shape
    constexpr int PP = MC / NS < kRoundPerSlot ? (MC / NS > 0 ? MC / NS : 1) : kRoundPerSlot;
    constexpr int ROUND = NS * PP;
    extern __shared__ float lds[];

    const int hs = a.head_size, hs4 = hs / 4;
    const int hg = blockIdx.x, i = blockIdx.y, s = blockIdx.z;
    const int n_ctx = *a.pos + i + 1;
    // Only ROPE calls set `whole`. (Testing it in the others too cost heads of
    // 256 10 % by the registers that the compiler then gave their loads.)
    const int chunk = ROPE && n_ctx <= a.whole ? n_ctx : split_chunk(n_ctx, a.splits, a.min_chunk);
    const int t0 = s * chunk;
    if (t0 >= n_ctx) return;  // uniform across the workgroup
    const int len = min(chunk, n_ctx - t0);
    const int nchunks = (n_ctx + chunk - 1) / chunk;
    const int h0 = hg * G;
    const int kv_off = (h0 / a.group) * hs;
    const int tid = threadIdx.x, sub = tid % LPP, slot = tid / LPP;
    // With ROPE the last position (the current one) is not in the cache yet.
    const bool own_pos = ROPE && s == nchunks - 1;
    const int loop_len = own_pos ? len - 1 : len;
    float* rq = lds + G * NS * hs + 2 * G * NS;  // ROPE: G rotated queries, key, value

    // This lane's columns; lanes past hs4 read the last column with a zero
    // query and store nothing.
    int dcol[F];
    bool dok[F];
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const int d = sub + f * LPP;
        dok[f] = d < hs4;
        dcol[f] = dok[f] ? d : hs4 - 1;
    }
    const float* kbase = a.kc + static_cast<std::size_t>(t0) * a.kv_stride + kv_off;
    const float* vbase = a.vc + static_cast<std::size_t>(t0) * a.kv_stride + kv_off;
    // Every key and value of a round in flight; positions past the chunk
    // re-read its last position and are masked. (Issuing the first round
    // before the ROPE query is formed measured 1 us slower at ctx 512: the
    // query's loads then wait behind the whole chunk's.)
    floatx4 kv[PP][F], vv[PP][F];
    auto load_round = [&](floatx4 (&x)[PP][F], const float* base, int b0) {
#pragma unroll
        for (int pp = 0; pp < PP; ++pp) {
            const int t = min(b0 + slot + pp * NS, loop_len - 1);
            const floatx4* r = reinterpret_cast<const floatx4*>(base + static_cast<std::size_t>(t) * a.kv_stride);
#pragma unroll
            for (int f = 0; f < F; ++f) x[pp][f] = r[dcol[f]];
        }
    };

    if constexpr (ROPE) {
        const int pos = n_ctx - 1, half = hs / 2;
        const float* cs = a.cos_t + static_cast<std::size_t>(pos) * half;
        const float* sn = a.sin_t + static_cast<std::size_t>(pos) * half;
        const bool writer = h0 % a.group == 0;
        const int nq = G * hs4, total = nq + (own_pos ? 2 * hs4 : 0);
        for (int j = tid; j < total; j += kThreads) {
            int col, d;
            bool rot = true;
            if (j < nq) {
                d = j % hs4;
                col = h0 * hs + 4 * j;
            } else if (j < nq + hs4) {
                d = j - nq;
                col = a.dim + kv_off + 4 * d;
            } else {
                d = j - nq - hs4;
                col = a.dim + a.kv_dim + kv_off + 4 * d;
                rot = false;
            }
            // The angles are loaded for values too (d < hs4, so in range) and
            // before the product's slices: one wait covers every load here
            // and the first round of keys and values.
            const float c0 = cs[2 * d], s0 = sn[2 * d], c1 = cs[2 * d + 1], s1 = sn[2 * d + 1];
            const floatx4 x = summed4(a.src, 0, col);
            floatx4 y = x;
            if (rot) {
                const float2 r0 = rope_pair(x.x, x.y, c0, s0);
                const float2 r1 = rope_pair(x.z, x.w, c1, s1);
                y = floatx4{r0.x, r0.y, r1.x, r1.y};
            }
            reinterpret_cast<floatx4*>(rq)[j] = y;
            if (j >= nq && writer) {
                float* cache = j < nq + hs4 ? a.kc_w : a.vc_w;
                reinterpret_cast<floatx4*>(cache + static_cast<std::size_t>(pos) * a.kv_stride +
                                           kv_off)[d] = y;
            }
        }
        __syncthreads();
    }

    floatx4 q[G][F];
    const float* qrow = ROPE ? rq : a.q + static_cast<std::size_t>(i) * a.q_stride +
                                        static_cast<std::size_t>(h0) * hs;
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int f = 0; f < F; ++f)
            q[g][f] = dok[f] ? reinterpret_cast<const floatx4*>(qrow + g * hs)[dcol[f]]
                             : floatx4{0.f, 0.f, 0.f, 0.f};

    const float scale = 1.0f / sqrtf(static_cast<float>(hs));
    float m[G], l[G];
    floatx4 o[G][F];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        m[g] = -INFINITY;
        l[g] = 0.0f;
#pragma unroll
        for (int f = 0; f < F; ++f) o[g][f] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

    if (PIPE && loop_len > 0) {
        load_round(kv, kbase, 0);
        load_round(vv, vbase, 0);
    }
    for (int b0 = 0; b0 < loop_len; b0 += ROUND) {
        const bool more = PIPE && b0 + ROUND < loop_len;
        if constexpr (!PIPE) {
            load_round(kv, kbase, b0);
            load_round(vv, vbase, b0);
        }
        float sc[G][PP];
#pragma unroll
        for (int pp = 0; pp < PP; ++pp) {
            const bool valid = b0 + slot + pp * NS < loop_len;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                float dot = 0.0f;
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    const floatx4 x = q[g][f] * kv[pp][f];
                    dot += (x.x + x.y) + (x.z + x.w);
                }
#pragma unroll
                for (int off = LPP / 2; off > 0; off >>= 1) dot += __shfl_xor(dot, off, kWave);
                sc[g][pp] = valid ? dot * scale : -INFINITY;
            }
        }
        if (more) load_round(kv, kbase, b0 + ROUND);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float mb = sc[g][0];
#pragma unroll
            for (int pp = 1; pp < PP; ++pp) mb = fmaxf(mb, sc[g][pp]);
            const float mn = fmaxf(m[g], mb);
            if (mn == -INFINITY) continue;  // no position of this slot yet
            const float alpha = expf(m[g] - mn);
            l[g] *= alpha;
#pragma unroll
            for (int f = 0; f < F; ++f) o[g][f] *= alpha;
#pragma unroll
            for (int pp = 0; pp < PP; ++pp) {
                const float e = expf(sc[g][pp] - mn);
                l[g] += e;
#pragma unroll
                for (int f = 0; f < F; ++f) o[g][f] += e * vv[pp][f];
            }
            m[g] = mn;
        }
        if (more) load_round(vv, vbase, b0 + ROUND);
    }

    if (own_pos && slot == 0) {
        // The current position, in slot 0: its key and value from LDS.
        floatx4 kx[F], vx[F];
#pragma unroll
        for (int f = 0; f < F; ++f) {
            kx[f] = reinterpret_cast<const floatx4*>(rq + G * hs)[dcol[f]];
            vx[f] = reinterpret_cast<const floatx4*>(rq + G * hs + hs)[dcol[f]];
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float dot = 0.0f;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const floatx4 x = q[g][f] * kx[f];
                dot += (x.x + x.y) + (x.z + x.w);
            }
#pragma unroll
            for (int off = LPP / 2; off > 0; off >>= 1) dot += __shfl_xor(dot, off, kWave);
            const float sc = dot * scale;
            const float mn = fmaxf(m[g], sc);
            const float alpha = expf(m[g] - mn);
            const float e = expf(sc - mn);
            l[g] = l[g] * alpha + e;
#pragma unroll
            for (int f = 0; f < F; ++f) o[g][f] = o[g][f] * alpha + e * vx[f];
            m[g] = mn;
        }
    }

    // Merge the slots in slot order: o_s[g][slot][hs], ml_s[g][slot][2].
    float* o_s = lds;
    float* ml_s = lds + G * NS * hs;
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int f = 0; f < F; ++f)
            if (dok[f])
                reinterpret_cast<floatx4*>(o_s + (g * NS + slot) * hs)[dcol[f]] = o[g][f];
        if (sub == 0) {
            ml_s[(g * NS + slot) * 2] = m[g];
            ml_s[(g * NS + slot) * 2 + 1] = l[g];
        }
    }
    __syncthreads();

    const std::size_t head_row = static_cast<std::size_t>(i) * a.n_heads + h0;
    for (int j = tid; j < G * hs4; j += kThreads) {
        const int g = j / hs4, d = j % hs4;
        const float* mlg = ml_s + g * NS * 2;
        float M = -INFINITY;
        for (int sl = 0; sl < NS; ++sl) M = fmaxf(M, mlg[2 * sl]);
        float L = 0.0f;
        floatx4 O{0.f, 0.f, 0.f, 0.f};
        for (int sl = 0; sl < NS; ++sl) {
            const float w = expf(mlg[2 * sl] - M);  // 0 for a slot with no position
            L += w * mlg[2 * sl + 1];
            O += w * reinterpret_cast<const floatx4*>(o_s + (g * NS + sl) * hs)[d];
        }
        if (nchunks == 1) {
            reinterpret_cast<floatx4*>(a.out + static_cast<std::size_t>(i) * a.out_stride +
                                       static_cast<std::size_t>(h0 + g) * hs)[d] = O * (1.0f / L);
        } else if (a.merge_count) {
            // Device-coherent stores: the row's last workgroup reads them.
            const uint32_t c = static_cast<uint32_t>((head_row + g) * a.splits + s);
            __builtin_amdgcn_raw_buffer_store_b128(
                __builtin_bit_cast(u32x4, O),
                __builtin_amdgcn_make_buffer_rsrc(a.part_o, 0, 0x7fffffff, 0x00020000),
                (c * hs4 + d) * 16, 0, kSc1);
            if (d == 0)
                __builtin_amdgcn_raw_buffer_store_b64(
                    __builtin_bit_cast(u32x2, make_float2(M, L)),
                    __builtin_amdgcn_make_buffer_rsrc(a.part_ml, 0, 0x7fffffff, 0x00020000),
                    c * 8, 0, kSc1);
        } else {
            reinterpret_cast<floatx4*>(a.part_o)[((head_row + g) * a.splits + s) * hs4 + d] = O;
            if (d == 0) a.part_ml[(head_row + g) * a.splits + s] = make_float2(M, L);
        }
    }
    if (nchunks == 1 || !a.merge_count) return;
    // Counted in once every partial store above has landed; the last of the
    // row's chunks merges them and sets the counter back to zero.
    __shared__ unsigned arrived;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    unsigned* counter = a.merge_count + static_cast<std::size_t>(i) * gridDim.x + hg;
    if (tid == 0) arrived = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (arrived != static_cast<unsigned>(nchunks - 1)) return;
    merge_chunks(a, i, h0, G, nchunks, lds);
    if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Merges the chunks of one (head, row): m = max m_c,
// l = sum e^(m_c - m) l_c, out = sum e^(m_c - m) o_c / l. A workgroup takes
// kMergeDims float4s of the head's columns (blockIdx.x = head * groups +
// group), so a long context's chunks spread over more workgroups. As many
// slots work as eight chunks each need (up to 256 / dpw): the dpw threads of
// slot r take chunks r, r + used, ..., loaded in one batch, and keep their
// own max, sum and output over them; the slots are then combined in slot
// order, each scaled by e^(its max - m), after one barrier. The result is
// the same on every call. (One workgroup per head took 8.7 us for 32 heads
// x 256 chunks: four dependent batches in each of 32 workgroups; always
// using every slot made 64 chunks slower, a 32-step combine.)

__global__ __launch_bounds__(kThreads) void attn_merge_kernel(AttnArgs a) {
    extern __shared__ floatx4 red4[];  // slots x dpw outputs, then slots x (max, sum)
    const int hs4 = a.head_size / 4;
    const int dpw = hs4 < kMergeDims ? hs4 : kMergeDims, groups = (hs4 + dpw - 1) / dpw;
    const int h = blockIdx.x / groups, d0 = (blockIdx.x % groups) * dpw;
    const int i = blockIdx.y;
    const int n_ctx = *a.pos + i + 1;
    const int chunk = a.tile_chunk         ? a.tile_chunk
                      : a.group_chunk_min  ? group_chunk(*a.pos + a.rows, a.splits, a.group_chunk_min)
                      : n_ctx <= a.whole   ? n_ctx
                                         : split_chunk(n_ctx, a.splits, a.min_chunk);
    const int n = (n_ctx + chunk - 1) / chunk;
    if (n < a.merge_from) return;  // one chunk: written by the split kernel; few: by their consumer
    const std::size_t b = (static_cast<std::size_t>(i) * a.n_heads + h) * a.splits;
    const int tid = threadIdx.x;
    const int slots = kThreads / dpw, r = tid / dpw, dd = tid % dpw, d = d0 + dd;
    const bool dok = d < hs4;
    const int dl = dok ? d : hs4 - 1;  // past the head: computed, not stored
    const floatx4* po = reinterpret_cast<const floatx4*>(a.part_o);
    float2* red_ml = reinterpret_cast<float2*>(red4 + slots * dpw);
    const int used = min(slots, (n + 7) / 8);  // slots that take chunks

    if (r < used) {
        float m = -INFINITY, l = 0.0f;
        floatx4 acc{0.f, 0.f, 0.f, 0.f};
        for (int c0 = r; c0 < n; c0 += 8 * used) {
            float2 ml[8];
            floatx4 o[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int c = min(c0 + u * used, n - 1);
                ml[u] = a.part_ml[b + c];
                o[u] = po[(b + c) * hs4 + dl];
            }
            merge_batch8(m, l, acc, ml, o, c0, used, n);
        }
        red4[r * dpw + dd] = acc;
        if (dd == 0) red_ml[r] = make_float2(m, l);
    }
    __syncthreads();
    if (tid < dpw && dok) {
        reinterpret_cast<floatx4*>(a.out + static_cast<std::size_t>(i) * a.out_stride +
                                   static_cast<std::size_t>(h) * a.head_size)[d] =
            merge_combine(used, floatx4{0.f, 0.f, 0.f, 0.f},
                          [&](int rr) { return red_ml[rr]; },
                          [&](int rr) { return red4[rr * dpw + tid]; });
    }
}

// One workgroup per (head, row): query and scores in LDS, scalar loads, so
// any head size works.
__global__ __launch_bounds__(kThreads) void attn_single_kernel(AttnArgs a) {
    extern __shared__ float lds[];
    __shared__ float part[4];
    const int hs = a.head_size;
    float* q_s = lds;               // hs
    float* sc = lds + hs;           // seq_len
    float* red = sc + a.seq_len;    // kThreads
    const int h = blockIdx.x, i = blockIdx.y;
    const int n_ctx = *a.pos + i + 1;
    const int kv_off = (h / a.group) * hs;
    const int tid = threadIdx.x;

    const float* qg = a.q + static_cast<std::size_t>(i) * a.q_stride + static_cast<std::size_t>(h) * hs;
    for (int d = tid; d < hs; d += kThreads) q_s[d] = qg[d];
    __syncthreads();

    const int lpp = lanes_per_row(hs);
    const int sub = tid % lpp, slot = tid / lpp, nslots = kThreads / lpp;
    const float scale = 1.0f / sqrtf(static_cast<float>(hs));
    for (int base = 0; base < n_ctx; base += nslots) {
        const int t = base + slot;
        float dot = 0.0f;
        if (t < n_ctx) {
            const float* k = a.kc + static_cast<std::size_t>(t) * a.kv_stride + kv_off;
            for (int d = sub; d < hs; d += lpp) dot += q_s[d] * k[d];
        }
        for (int o = lpp / 2; o > 0; o >>= 1) dot += __shfl_xor(dot, o, kWave);
        if (t < n_ctx && sub == 0) sc[t] = dot * scale;
    }
    __syncthreads();

    float m = -INFINITY;
    for (int t = tid; t < n_ctx; t += kThreads) m = fmaxf(m, sc[t]);
    m = block_max(m, part);
    float l = 0.0f;
    for (int t = tid; t < n_ctx; t += kThreads) {
        const float e = expf(sc[t] - m);
        sc[t] = e;
        l += e;
    }
    l = block_sum(l, part);  // its barriers also publish the exponentials
    const float inv = 1.0f / l;

    float* oh = a.out + static_cast<std::size_t>(i) * a.out_stride + static_cast<std::size_t>(h) * hs;
    const float* vb = a.vc + kv_off;
    if (hs <= kThreads) {
        const int d = tid % hs, r = tid / hs, slots = kThreads / hs;
        if (r < slots) {
            float acc = 0.0f;
            for (int t = r; t < n_ctx; t += slots)
                acc += sc[t] * vb[static_cast<std::size_t>(t) * a.kv_stride + d];
            red[r * hs + d] = acc;
        }
        __syncthreads();
        if (tid < hs) {
            float o = red[tid];
            for (int rr = 1; rr < slots; ++rr) o += red[rr * hs + tid];
            oh[tid] = o * inv;
        }
    } else {
        for (int d = tid; d < hs; d += kThreads) {
            float acc = 0.0f;
            for (int t = 0; t < n_ctx; ++t)
                acc += sc[t] * vb[static_cast<std::size_t>(t) * a.kv_stride + d];
            oh[d] = acc * inv;
        }
    }
}

// --- prefill rows: tiles of 16 queries on fp32 MFMA ------------------------
//
// One wave per (query head, 16 consecutive rows). For each block of 16
// cached positions it forms S^T = K Q^T (positions x queries) with
// v_mfma_f32_16x16x4_f32, then O^T += V^T P^T. In lane l (g = l / 16,
// j = l % 16):
//  * S^T: the lane supplies K[position j][d] and Q[query j][d] for the head
//    dims d of its lane group's quarter (4E contiguous floats, E = hs / 16),
//    so its key and query loads are float4 runs; both operands take the
//    head dims in the same order.
//  * S^T's output layout leaves in the lane the scores of query j at
//    positions 4g + r (r = 0..3) of the block: exactly the B operand
//    P^T[position 4g + r][query j] of k-step r of the V product, so scores
//    never leave the lane's registers.
//  * V^T: lane j supplies rows d = E j + c (c = 0..E-1, one MFMA each), E
//    contiguous floats of a value row; output block c then holds
//    O[query j][E (4g + r) + c], so the lane ends with 4E contiguous head
//    dims of its query.
//  * Every accumulator of a lane belongs to query j: the online softmax
//    rescale is one factor per lane. The block max takes two xor shuffles
//    (the four lane groups of a query); the sum is combined once, at the end.
// Positions past a query's own are masked, and blocks past the tile's last
// row are never read; the next block's keys and values are loaded while
// this one is used (two register sets, alternating; a 32-position block
// measured no faster and needs twice the registers).
//
// A workgroup is four such waves on one (head, 16-row tile): wave w takes
// the w-th quarter of the tile's blocks, keeping its own online softmax, and
// the four are merged in LDS in wave order at the end. Causal tiles differ
// in length up to 32-fold at 512 rows, and with one wave per tile the
// longest set the kernel's time. A query with no position in a wave's
// quarter leaves that wave's m = -inf, l = 0, O = 0.
template <int E>
struct TileBlock {
    floatx4 k[E];   // K[t0 + j][4E g .. 4E g + 4E)
    float v[4][E];  // per r: V[t0 + 4g + r][E j .. E j + E)
};

template <int E>
__device__ __forceinline__ void load_run(const float* src, float* dst) {
    if constexpr (E % 4 == 0) {
#pragma unroll
        for (int u = 0; u < E / 4; ++u) {
            const floatx4 x = reinterpret_cast<const floatx4*>(src)[u];
            dst[4 * u] = x.x;
            dst[4 * u + 1] = x.y;
            dst[4 * u + 2] = x.z;
            dst[4 * u + 3] = x.w;
        }
    } else if constexpr (E % 2 == 0) {
#pragma unroll
        for (int u = 0; u < E / 2; ++u) {
            const float2 x = reinterpret_cast<const float2*>(src)[u];
            dst[2 * u] = x.x;
            dst[2 * u + 1] = x.y;
        }
    } else {
#pragma unroll
        for (int u = 0; u < E; ++u) dst[u] = src[u];
    }
}

constexpr int kTileWaves = 4;
constexpr int kGroupChunkMin = 64, kGroupWorkgroups = 512;

// One wave's online softmax over positions [first, wlast] (both ends of
// whole 16-position blocks) for 16 queries on the keys and values of one kv
// head; this lane's is row `row` of query head `h` (any of the kv head's):
// max m, this lane's part l of the sum, unnormalised output o. `last` is the
// last position that may be read. FINE keeps the chains of additions as short
// as the split kernel's: a score is a tree over four-product sums, the output
// a sum over blocks of two eight-product sums each.
template <int E, bool FINE = false>
__device__ __forceinline__ void tile_wave(const AttnArgs& a, int kvh, int h, int row, int last,
                                          int first, int wlast, float& m, float& l,
                                          floatx4 (&o)[E]) {
    constexpr int HS = 16 * E, Q4 = 4 * E;
    constexpr int KB = 16;  // positions per block
    const int lane = threadIdx.x % kWave, g = lane >> 4, j = lane & 15;
    const int pq = *a.pos + row;  // this lane's query position
    const float* kbase = a.kc + static_cast<std::size_t>(kvh * HS);
    const float* vbase = a.vc + static_cast<std::size_t>(kvh * HS);

    float q[Q4];
    load_run<Q4>(a.q + static_cast<std::size_t>(row) * a.q_stride + static_cast<std::size_t>(h) * HS + Q4 * g, q);

    // Positions past `last` re-read position `last` (in the cache: the
    // caller keeps *pos + rows <= seq_len) and are masked.
    auto load = [&](TileBlock<E>& b, int t0) {
        const int tk = min(t0 + j, last);
        const floatx4* kr = reinterpret_cast<const floatx4*>(
            kbase + static_cast<std::size_t>(tk) * a.kv_stride + Q4 * g);
#pragma unroll
        for (int u = 0; u < E; ++u) b.k[u] = kr[u];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int tv = min(t0 + 4 * g + r, last);
            load_run<E>(vbase + static_cast<std::size_t>(tv) * a.kv_stride + E * j, b.v[r]);
        }
    };

    const float scale = 1.0f / sqrtf(static_cast<float>(HS));
    m = -INFINITY;
    l = 0.0f;
#pragma unroll
    for (int c = 0; c < E; ++c) o[c] = floatx4{0.f, 0.f, 0.f, 0.f};

    auto use = [&](const TileBlock<E>& b, int t0) {
        // S^T in four accumulators (head-dim steps u mod 4), so consecutive
        // MFMAs are independent, added pairwise at the end.
        floatx4 sacc[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) sacc[c] = floatx4{0.f, 0.f, 0.f, 0.f};
        if constexpr (FINE) {
            floatx4 part[E];
#pragma unroll
            for (int u = 0; u < E; ++u) {
                floatx4 d[4];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    d[c] = mfma16x16x4(b.k[u][c], q[4 * u + c], floatx4{0.f, 0.f, 0.f, 0.f});
                part[u] = (d[0] + d[1]) + (d[2] + d[3]);
            }
#pragma unroll
            for (int n = 1; n < E; n *= 2) {
#pragma unroll
                for (int u = 0; u + n < E; u += 2 * n) part[u] += part[u + n];
            }
            sacc[0] = part[0];
        } else {
#pragma unroll
            for (int u = 0; u < Q4; ++u)
                sacc[u & 3] = mfma16x16x4(b.k[u / 4][u % 4], q[u], sacc[u & 3]);
        }
        float sv[4];
        float mb = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = t0 + 4 * g + r;
            const float x = ((sacc[0][r] + sacc[1][r]) + (sacc[2][r] + sacc[3][r])) * scale;
            sv[r] = t <= pq ? x : -INFINITY;
            mb = fmaxf(mb, sv[r]);
        }
        mb = fmaxf(mb, __shfl_xor(mb, 16, kWave));
        mb = fmaxf(mb, __shfl_xor(mb, 32, kWave));
        // mn = -inf: no position of this query yet (its position precedes
        // the wave's blocks so far); everything stays as it is.
        const float mn = fmaxf(m, mb);
        const bool none = mn == -INFINITY;
        const float alpha = none ? 1.0f : expf(m - mn);
        l *= alpha;
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p[r] = none ? 0.0f : expf(sv[r] - mn);
            l += p[r];
        }
        if constexpr (FINE) {
#pragma unroll
            for (int c = 0; c < E; ++c) {
                floatx4 d0 = mfma16x16x4(b.v[0][c], p[0], floatx4{0.f, 0.f, 0.f, 0.f});
                floatx4 d1 = mfma16x16x4(b.v[2][c], p[2], floatx4{0.f, 0.f, 0.f, 0.f});
                d0 = mfma16x16x4(b.v[1][c], p[1], d0);
                d1 = mfma16x16x4(b.v[3][c], p[3], d1);
                o[c] = o[c] * alpha + (d0 + d1);
            }
        } else {
#pragma unroll
            for (int c = 0; c < E; ++c) o[c] *= alpha;
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int c = 0; c < E; ++c) o[c] = mfma16x16x4(b.v[r][c], p[r], o[c]);
        }
        m = mn;
    };

    if (first <= wlast) {
        TileBlock<E> b0, b1;
        load(b0, first);
        for (int t0 = first; t0 <= wlast; t0 += 2 * KB) {
            if (t0 + KB <= wlast) load(b1, t0 + KB);
            use(b0, t0);
            if (t0 + KB > wlast) break;
            if (t0 + 2 * KB <= wlast) load(b0, t0 + 2 * KB);
            use(b1, t0 + KB);
        }
    }
}

// tile_wave position by position without matrix products, where a masked
// position (one past the lane's query) must not reach the output even as a
// product with zero: a value that is not finite. The output in tile_wave's
// layout: head dim 4E g + x in o[x % E][x / E].
template <int E>
__device__ void tile_wave_plain(const AttnArgs& a, int kvh, int h, int row, int last, int first,
                                int wlast, float& m, float& l, floatx4 (&o)[E]) {
    constexpr int HS = 16 * E;
    const int g = (threadIdx.x % kWave) >> 4, pq = *a.pos + row;
    const floatx4* q = reinterpret_cast<const floatx4*>(
        a.q + static_cast<std::size_t>(row) * a.q_stride + static_cast<std::size_t>(h) * HS + 4 * E * g);
    const std::size_t base = static_cast<std::size_t>(kvh * HS) + 4 * E * g;
    const float scale = 1.0f / sqrtf(static_cast<float>(HS));
    m = -INFINITY;
    l = 0.0f;
    for (int u = 0; u < E; ++u) o[u] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int t = first; t <= min(wlast, last); ++t) {
        const std::size_t off = base + static_cast<std::size_t>(t) * a.kv_stride;
        const floatx4* k = reinterpret_cast<const floatx4*>(a.kc + off);
        const floatx4* v = reinterpret_cast<const floatx4*>(a.vc + off);
        float x = 0.0f;
        for (int u = 0; u < E; ++u) {
            const floatx4 y = q[u] * k[u];
            x += (y[0] + y[1]) + (y[2] + y[3]);
        }
        x = sum32(sum16(x)) * scale;
        if (t > pq) continue;
        // A score of -inf has no weight, also where every one so far is.
        const float mn = fmaxf(m, x), alpha = m == mn ? 1.0f : expf(m - mn);
        const float p = x == -INFINITY ? 0.0f : expf(x - mn);
        l = l * alpha + p;
#pragma unroll
        for (int x = 0; x < 4 * E; ++x)
            o[x % E][x / E] = o[x % E][x / E] * alpha + p * v[x / 4][x % 4];
        m = mn;
    }
    // Each of a query's four lanes has the whole sum; the caller adds them.
    if (g) l = 0.0f;
}

// The result of row `row` of head h over positions from lo = cz * chunk on
// (chunk 0: the whole context): max M, whole sum l, unnormalised output.
// Split: a query whose context spans more than one chunk leaves this chunk's
// state for the merge kernel; one whose context fits chunk 0 is written here,
// as the split kernel writes it. run(u, f) is the float4 of f * the output at
// head dims run_at(u) .. + 3, u < E. Rows past the call store nothing.
template <int E, class At, class Run>
__device__ __forceinline__ void tile_store(const AttnArgs& a, int h, int row, int cz, int chunk,
                                           float M, float l, At run_at, Run run) {
    constexpr int HS = 16 * E;
    const int g = (threadIdx.x % kWave) >> 4;
    if (row >= a.rows) return;
    const int pq = *a.pos + row, lo = cz * chunk;
    if (chunk && pq >= chunk && lo <= pq) {
        const std::size_t b = (static_cast<std::size_t>(row) * a.n_heads + h) * a.splits + cz;
#pragma unroll
        for (int u = 0; u < E; ++u)
            *reinterpret_cast<floatx4*>(a.part_o + b * HS + run_at(u)) = run(u, 1.0f);
        if (g == 0) a.part_ml[b] = make_float2(M, l);
    } else if (cz == 0 && (chunk == 0 || pq < chunk)) {
        const float inv = 1.0f / l;
        float* dst = a.out + static_cast<std::size_t>(row) * a.out_stride +
                     static_cast<std::size_t>(h) * HS;
#pragma unroll
        for (int u = 0; u < E; ++u) *reinterpret_cast<floatx4*>(dst + run_at(u)) = run(u, inv);
    }
}

// tile_store of tile_wave's layout: o[c][r] is head dim E (4g + r) + c.
template <int E>
__device__ __forceinline__ void tile_store_wave(const AttnArgs& a, int h, int row, int cz, int chunk,
                                                float M, float l, const floatx4 (&o)[E]) {
    float flat[4 * E];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < E; ++c) flat[E * r + c] = o[c][r];
    const int g = (threadIdx.x % kWave) >> 4;
    tile_store<E>(a, h, row, cz, chunk, M, l, [&](int u) { return 4 * E * g + 4 * u; },
                  [&](int u, float f) {
                      return floatx4{flat[4 * u] * f, flat[4 * u + 1] * f, flat[4 * u + 2] * f,
                                     flat[4 * u + 3] * f};
                  });
}

// A tile workgroup: its waves take quarters of the blocks of positions [lo,
// hi] (lo a multiple of 16) for the same 16 queries, then merge in LDS.
template <int E, bool FINE = false>
__device__ __forceinline__ void tile_block(const AttnArgs& a, int kvh, int h, int row, int last,
                                           int lo, int hi, int cz, int chunk) {
    constexpr int KB = 16;  // positions per block
    __shared__ float ms[kTileWaves][kWave], ls[kTileWaves][kWave];
    __shared__ floatx4 os[kTileWaves][E][kWave];
    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // This wave's blocks: [nb * w / 4, nb * (w + 1) / 4) of the nb blocks
    // from lo through hi.
    const int b0i = lo / KB, nb = hi / KB + 1 - b0i;
    const int first = KB * (b0i + nb * wave / kTileWaves);
    const int wlast = KB * (b0i + nb * (wave + 1) / kTileWaves) - 1;  // < first: no blocks
    float m, l;
    floatx4 o[E];
    tile_wave<E, FINE>(a, kvh, h, min(row, a.rows - 1), last, first, wlast, m, l, o);
    if constexpr (FINE) {
        bool bad = !(l < INFINITY);
#pragma unroll
        for (int c = 0; c < E; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) bad |= !(fabsf(o[c][e]) < INFINITY);
        if (__ballot(bad))
            tile_wave_plain<E>(a, kvh, h, min(row, a.rows - 1), last, first, wlast, m, l, o);
    }

    // Merge the waves in order: lane l of every wave holds query j's state.
    ms[wave][lane] = m;
    ls[wave][lane] = l;
#pragma unroll
    for (int c = 0; c < E; ++c) os[wave][c][lane] = o[c];
    __syncthreads();
    if (wave != 0) return;
    // M is finite for every query with a position in [lo, hi] (the others
    // are not stored): some wave holds that position.
    float M = ms[0][lane];
#pragma unroll
    for (int w = 1; w < kTileWaves; ++w) M = fmaxf(M, ms[w][lane]);
    l = 0.0f;
#pragma unroll
    for (int c = 0; c < E; ++c) o[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kTileWaves; ++w) {
        const float mw = ms[w][lane];
        const float f = mw == -INFINITY ? 0.0f : expf(mw - M);
        l += f * ls[w][lane];
#pragma unroll
        for (int c = 0; c < E; ++c) o[c] += f * os[w][c][lane];
    }

    // The four lane groups of query j hold partial sums of its denominator;
    // the xor pairs add them in the same order in every lane.
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    tile_store_wave<E>(a, h, row, cz, chunk, M, l, o);
}

template <int E>
__global__ __launch_bounds__(kTileWaves * kWave) void attn_tile_kernel(AttnArgs a) {
    // Row tiles in reverse: the longest (causal) start first and the short
    // ones fill in behind them.
    const int h = blockIdx.x, r0 = (gridDim.y - 1 - blockIdx.y) * kTileRows;
    const int last = *a.pos + min(r0 + kTileRows - 1, a.rows - 1);  // the tile's last position
    // Split over the context: this workgroup takes positions [lo, hi] of
    // chunk blockIdx.z (none past last: the grid is sized for seq_len).
    const int cz = blockIdx.z, lo = cz * a.tile_chunk;
    if (lo > last) return;
    const int hi = a.tile_chunk ? min(last, lo + a.tile_chunk - 1) : last;
    tile_block<E>(a, h / a.group, h, r0 + static_cast<int>(threadIdx.x % 16), last, lo, hi, cz,
                  a.tile_chunk);
}

// A few rows of grouped heads: workgroup (kv head, 16 queries, chunk), the
// queries being the rows of the heads that share the kv head, so a key or
// value is read once for 16 of them and multiplied in the MFMAs that one would
// take. The split kernel reads it once a row and spends about 170 VALU ops a
// wave on two positions of four heads. 64 heads on 8 of 80, 4 rows at context
// 4096: 82 us there, 19.5 here. Bound by the latency of each wave's next
// block: 134 MB of 32 heads' 16384 positions (8 kv heads) in 40 us, 3.4 TB/s.
// kGroupWorkgroups fill two workgroups a CU (1024, at the registers of heads
// of 128: 43 us against 37; 128 positions at least instead of 64: 13 against
// 11 at context 1500, 32: 16).
template <int E>
__global__ __launch_bounds__(kTileWaves * kWave) void attn_group_kernel(AttnArgs a) {
    const int kvh = blockIdx.x, cz = blockIdx.z;
    const int last = *a.pos + a.rows - 1;
    const int chunk = group_chunk(last + 1, a.splits, a.group_chunk_min), lo = cz * chunk;
    if (lo > last) return;
    const int j = blockIdx.y * kTileRows + threadIdx.x % 16;
    tile_block<E, true>(a, kvh, kvh * a.group + j % a.group, j / a.group, last, lo,
                        min(last, lo + chunk - 1), cz, chunk);
}

// --- prefill rows: tiles of 64 queries on bf16 MFMA -------------------------
//
// Workgroup (query head, 64 rows): wave w has the 16 queries r0 + 16w + j.
// The tile kernel above reads every key and value once per 16 rows (1 GB of
// L2 reads for 1000 rows of 32 heads) and multiplies on fp32 MFMA at 32
// cycles per 16x16x4; here the four waves share each 32-position block
// through LDS, and both products are sums of six bf16 terms: every operand
// (Q, K, V and the softmax weights P) split exactly into three bf16 values,
// the products left out at most 2^-24 of the whole, hi * hi in an accumulator
// of its own (gemm_split.hip has the error argument; here 1.5e-7 off
// 64 bits against 1.9e-7). 1000 rows x 32 heads of 128
// at context 1000: 81 us against 134.
//
// A block's keys and values are loaded into registers one block ahead,
// split, and written to LDS between two barriers; two workgroups share a CU,
// so one's split and softmax run beside the other's MFMAs. In lane
// (g, j) of a wave:
//  * S^T = K Q^T (positions x queries): the keys are the first operand, in
//    16-position fragments of 32 head dims with the 16-byte units of a row
//    permuted by unit ^ (row / 2 % 4); Q's terms stay in registers. Head
//    dims past the head size (16, 48, 80, 112) are zeros.
//  * The lane ends with query j's scores at positions 4g + r of both halves
//    of the block, r < 4. They are its eight k values for O^T += V^T P^T
//    once V's fragments take the positions in that order (slot 8g + e is
//    position 4g + e, or 16 + 4g + e - 4 from e = 4), so scores never leave
//    the lane.
//  * O^T block c: head dims 16c + 4g + r of query j.
// The output is rescaled only when a maximum of the wave's queries moved.
//
// Small operands drop bits: a term is a multiple of 2^-133, so a value below
// 2^-109 is off by up to 2^-134, and exp_neg stops at e^-87, which drops bits
// too. Where that could show, the wave runs tile_wave instead:
//  * a query that dropped bits, whatever its keys, or one of 2^90 or more
//    (below it, keys' dropped bits add up to less than 2^7 2^-134 2^90 =
//    2^-37 of a score);
//  * dropped bits of V and an output's sum below 2^-50;
//  * dropped bits of a weight and an output's sum below 2^-99 positions times
//    the largest value, of which n weights off by 2^-125 are up to 2^-26;
//  * an output or sum that is not finite, or no sum at all.
constexpr int kRowsTile = 64;
constexpr int kRowsBlock = 32;

// e^x for x <= 0 (NaN stays; e^floor below floor, 0 past -88): 2^(x log2 e) with the
// rounding of the product and the rest of log2 e put back as a factor, within
// about 2 ulp in half of expf's instructions.
__device__ __forceinline__ float exp_neg(float x, float floor) {
    constexpr float kHi = 0x1.715476p+0f, kLo = 0x1.4ae0cp-26f, kLn2 = 0x1.62e43p-1f;
    const float t = x < floor ? floor : x;
    const float y = t * kHi;
    const float r = fmaf(t, kLo, fmaf(t, kHi, -y));
    const float p = __builtin_amdgcn_exp2f(y);
    return fmaf(p, r * kLn2, p);
}

template <int E>
__global__ __launch_bounds__(4 * kWave, 2) void attn_rows_kernel(AttnArgs a) {
    constexpr int HS = 16 * E, C = (HS + 31) / 32, T = 4 * kWave;
    constexpr int kKeys = C * 2 * 3 * 1024, kTerm = HS * 64;  // bytes; a term of V
    __shared__ __attribute__((aligned(1024))) char smem[kKeys + 3 * kTerm];
    const int tid = threadIdx.x, lane = tid % kWave, g = lane >> 4, j = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
    // Longest (causal) tiles first.
    const int h = blockIdx.x, r0 = (gridDim.y - 1 - blockIdx.y) * kRowsTile;
    const int pos0 = *a.pos;
    const int last = pos0 + min(r0 + kRowsTile - 1, a.rows - 1);
    const int wr0 = r0 + 16 * w;
    const int row = min(wr0 + j, a.rows - 1);  // rows past the call: computed, not stored
    const int pq = pos0 + row;                 // the lane's query position
    const int wlast = pos0 + min(wr0 + 15, a.rows - 1);  // the wave's last one
    const float* kbase = a.kc + static_cast<std::size_t>((h / a.group) * HS);
    const float* vbase = a.vc + static_cast<std::size_t>((h / a.group) * HS);

    uint32_t lost_q = 0, lost_v = 0, lost_p = 0, lost_k = 0;  // lost_k is not used: see above
    float top_q = 0.0f;
    bf16x8 q[C][3];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float* src = a.q + static_cast<std::size_t>(row) * a.q_stride +
                           static_cast<std::size_t>(h) * HS + min(32 * c + 8 * g, HS - 8);
        const floatx4 x0 = *reinterpret_cast<const floatx4*>(src);
        const floatx4 x1 = *reinterpret_cast<const floatx4*>(src + 4);
        const bool in = 32 * c + 8 * g < HS;
        float v[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = in ? x0[e] : 0.0f;
            v[4 + e] = in ? x1[e] : 0.0f;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) top_q = fmaxf(top_q, fabsf(v[e]));
        uint4 t[3];
        split3x8(v, t, lost_q);
#pragma unroll
        for (int x = 0; x < 3; ++x) q[c][x] = __builtin_bit_cast(bf16x8, t[x]);
    }

    // The block at t0 covers positions t0 .. t0 + 31; one that would pass
    // `last` starts at last - 31 instead (>= 0: the call has 32 rows or
    // more), its positions before t0 masked, so no load needs a bound.
    auto start = [&](int t0) { return min(t0, last - (kRowsBlock - 1)); };
    // Keys: wave-task x = w, w + 4, ... is (head dims 32 (x / 2), positions
    // 16 (x % 2)): lane l loads unit l % 4 of position l / 4.
    constexpr int NK = (2 * C + 3) / 4;
    const int jr = lane / 4, uu = lane % 4;
    int k_off[NK];
#pragma unroll
    for (int i = 0; i < NK; ++i) {
        const int x = min(w + 4 * i, 2 * C - 1);
        k_off[i] = (16 * (x % 2) + jr) * a.kv_stride + min(32 * (x / 2) + 8 * uu, HS - 8);
    }
    // Values: task t is (slot group t / HS, head dim t % HS).
    constexpr int NV = (4 * HS + T - 1) / T;
    int v_off[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int t = min(tid + i * T, 4 * HS - 1);
        v_off[i] = 4 * (t / HS) * a.kv_stride + t % HS;
    }
    floatx4 kr[NK][2];
    float vr[NV][8];
    auto load = [&](int t0) {
        const float* kp = kbase + static_cast<std::size_t>(start(t0)) * a.kv_stride;
        const float* vp = vbase + static_cast<std::size_t>(start(t0)) * a.kv_stride;
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            kr[i][0] = *reinterpret_cast<const floatx4*>(kp + k_off[i]);
            kr[i][1] = *reinterpret_cast<const floatx4*>(kp + k_off[i] + 4);
        }
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                vr[i][e] = vp[static_cast<std::size_t>(e < 4 ? e : 12 + e) * a.kv_stride + v_off[i]];
    };
    auto stash = [&] {
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int x = w + 4 * i;
            if ((2 * C) % 4 && x >= 2 * C) break;
            float v[8] = {kr[i][0].x, kr[i][0].y, kr[i][0].z, kr[i][0].w,
                          kr[i][1].x, kr[i][1].y, kr[i][1].z, kr[i][1].w};
            if (HS % 32 && x / 2 == C - 1) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = 32 * (C - 1) + 8 * uu < HS ? v[e] : 0.0f;
            }
            uint4 t[3];
            split3x8(v, t, lost_k);
            char* o = smem + x * 3072 + (jr * 4 + (uu ^ ((jr >> 1) & 3))) * 16;
#pragma unroll
            for (int y = 0; y < 3; ++y) *reinterpret_cast<uint4*>(o + y * 1024) = t[y];
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int x = tid + i * T;
            if ((4 * HS) % T && x >= 4 * HS) break;
            uint4 t[3];
            split3x8(vr[i], t, lost_v);
#pragma unroll
            for (int y = 0; y < 3; ++y)
                *reinterpret_cast<uint4*>(smem + kKeys + y * kTerm + x * 16) = t[y];
        }
    };

    const float scale = 1.0f / sqrtf(static_cast<float>(HS));
    float m = -INFINITY, l = 0.0f;
    floatx4 o[E], ol[E];  // the V hi * P hi products; the five smaller ones
#pragma unroll
    for (int c = 0; c < E; ++c) o[c] = ol[c] = floatx4{0.f, 0.f, 0.f, 0.f};
    const char* k_rd = smem + (j * 4 + (g ^ ((j >> 1) & 3))) * 16;
    const char* v_rd = smem + kKeys + (g * HS + j) * 16;

    auto use = [&](int t0) {
        // Scores of the block's two halves.
        floatx4 sh[2][2], sl[2];  // hi * hi in two accumulators, of even and odd dims' chunks
#pragma unroll
        for (int p = 0; p < 2; ++p) sh[0][p] = sh[1][p] = sl[p] = floatx4{0.f, 0.f, 0.f, 0.f};
        bf16x8 k[2][2][3], v[4][3];  // this step's fragments and the next's
        auto read_k = [&](int c) {
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int y = 0; y < 3; ++y)
                    k[c & 1][p][y] =
                        *reinterpret_cast<const bf16x8*>(k_rd + ((2 * c + p) * 3 + y) * 1024);
        };
        auto read_v = [&](int c0) {
#pragma unroll
            for (int c = c0; c < c0 + 2 && c < E; ++c)
#pragma unroll
                for (int y = 0; y < 3; ++y)
                    v[c & 3][y] = *reinterpret_cast<const bf16x8*>(v_rd + y * kTerm + c * 256);
        };
        read_k(0);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            if (c + 1 < C) read_k(c + 1);
            __builtin_amdgcn_sched_barrier(0);
            auto mma = [&](floatx4 (&d)[2], int tk, int tq) {
#pragma unroll
                for (int p = 0; p < 2; ++p) d[p] = mfma16x16x32(k[c & 1][p][tk], q[c][tq], d[p]);
            };
            mma(sh[c & 1], 0, 0);
            mma(sl, 2, 0);
            mma(sl, 1, 0);
            mma(sl, 0, 1);
            mma(sl, 1, 1);
            mma(sl, 0, 2);
        }
        read_v(0);
        float s[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) 
            s[e] = (sh[0][e / 4][e % 4] + sh[1][e / 4][e % 4] + sl[e / 4][e % 4]) * scale;
        const int ts = start(t0);
        // A masked position's weight is zero, so exp_neg may not stop short of
        // that here; another weight that becomes zero then counts as one that
        // dropped bits (found here, where it costs the other blocks nothing).
        float floor = -87.0f;
        if (ts != t0 || t0 + kRowsBlock - 1 > pos0 + wr0) {
            floor = -200.0f;
            float least = INFINITY, most = m;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int t = ts + 4 * g + (e < 4 ? e : 12 + e);
                const bool seen = t >= t0 && t <= pq;
                least = fminf(least, seen ? s[e] : INFINITY);
                s[e] = seen ? s[e] : -INFINITY;
                most = fmaxf(most, s[e]);
            }
            lost_p |= least - max32(max16(most)) < -87.0f;
        }
        float mb = s[0];
#pragma unroll
        for (int e = 1; e < 8; ++e) mb = fmaxf(mb, s[e]);
        mb = max32(max16(mb));
        // mn = -inf: no position of this query yet; everything stays.
        const float mn = fmaxf(m, mb);
        if (__ballot(mn > m)) {
            const float alpha = mn == -INFINITY ? 1.0f : expf(m - mn);
            l *= alpha;
#pragma unroll
            for (int c = 0; c < E; ++c) {
                o[c] *= alpha;
                ol[c] *= alpha;
            }
            m = mn;
        }
        const float base = mn == -INFINITY ? 0.0f : mn;
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            p[e] = exp_neg(s[e] - base, floor);
            l += p[e];
        }
        uint4 t[3];
        split3x8(p, t, lost_p);
        bf16x8 pt[3];
#pragma unroll
        for (int y = 0; y < 3; ++y) pt[y] = __builtin_bit_cast(bf16x8, t[y]);
        // Two output blocks at a time, so that an MFMA does not wait for the
        // one before it.
#pragma unroll
        for (int c = 0; c < E; c += 2) {
            if (c + 2 < E) read_v(c + 2);
            __builtin_amdgcn_sched_barrier(0);
            auto mma = [&](floatx4 (&d)[E], int tv, int tp) {
#pragma unroll
                for (int y = c; y < c + 2 && y < E; ++y) d[y] = mfma16x16x32(v[y & 3][tv], pt[tp], d[y]);
            };
            mma(o, 0, 0);
            mma(ol, 2, 0);
            mma(ol, 1, 0);
            mma(ol, 0, 1);
            mma(ol, 1, 1);
            mma(ol, 0, 2);
        }
    };

    load(0);
    // Not after the loop, where its operands would take registers through it.
    const bool redo_q = __ballot((lost_q & 0xffffu) != 0 || top_q >= 0x1p90f) != 0;
    for (int t0 = 0; t0 <= last; t0 += kRowsBlock) {
        __syncthreads();  // the previous block has been read
        stash();
        if (t0 + kRowsBlock <= last) load(t0 + kRowsBlock);
        __syncthreads();
        if (t0 <= wlast) use(t0);
    }

    // The four lane groups of query j hold parts of its sum.
    l = sum32(sum16(l));
    bool bad = redo_q || !(l < INFINITY && l > 0.0f);
    float low = INFINITY;
#pragma unroll
    for (int c = 0; c < E; ++c) {
        o[c] += ol[c];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float x = fabsf(o[c][e]);
            bad |= !(x < INFINITY);
            low = fminf(low, x);
        }
    }
    const bool v_lost = __syncthreads_or((lost_v & 0xffffu) != 0) != 0;
    bad |= v_lost && low < 0x1p-50f;
    if (__ballot((lost_p & 0xffffu) != 0)) {
        float top = 0.0f;
#pragma unroll 1
        for (int t = lane; t < (wlast + 1) * (HS / 4); t += kWave) {
            const floatx4 x = *reinterpret_cast<const floatx4*>(
                vbase + static_cast<std::size_t>(t / (HS / 4)) * a.kv_stride + t % (HS / 4) * 4);
            top = fmaxf(fmaxf(top, fmaxf(fabsf(x[0]), fabsf(x[1]))), fmaxf(fabsf(x[2]), fabsf(x[3])));
        }
        for (int d = 1; d < kWave; d *= 2) top = fmaxf(top, __shfl_xor(top, d, kWave));
        bad |= low < static_cast<float>(wlast + 1) * 0x1p-99f * top;
    }
    if (__ballot(bad)) {
        tile_wave<E>(a, h / a.group, h, row, wlast, 0, wlast / 16 * 16 + 15, m, l, o);
        l = sum32(sum16(l));
        tile_store_wave<E>(a, h, wr0 + j, 0, 0, m, l, o);
        return;
    }
    tile_store<E>(a, h, wr0 + j, 0, 0, m, l, [&](int u) { return 16 * u + 4 * g; },
                  [&](int u, float f) { return o[u] * f; });
}

// Where the 64-row kernel takes a tile-kernel call: one workgroup per CU and
// more without chunks of the context, as the position is not known here and a
// prompt's context may be no longer than its rows. 32 heads of 128, old / this
// kernel, us: 512 rows at context 512 / 1024 / 4096 46 / 42, 94 / 77, 380 /
// 301; 1024 rows 137 / 86 and at 4096 706 / 371; 256 rows at 1024 56 / 80.
// Heads of 64 (half the MFMAs beside the same softmax): 1024 rows at 1024 /
// 4096 54 / 49, 329 / 224, but 512 rows 47 / 54; of 48, 1024 rows of 6 heads
// 31 / 50. Heads of 112 pad their last 32 dims: 16 and 24 of them, 1057 and
// 775 rows at their own length 68 / 82, 54 / 60; from 1.5 workgroups a CU 0.9
// of the tile kernel's time and less.
bool rows_preferred(const AttnShape& s, int rows) {
    const long long tiles = static_cast<long long>(s.n_heads) * ((rows + kRowsTile - 1) / kRowsTile);
    const long long least = s.head_size >= 128   ? cu_count()
                            : s.head_size >= 112 ? cu_count() * 3 / 2
                                                 : 2 * cu_count();
    return rows >= kRowsBlock && s.head_size >= 64 && tiles >= least;
}

void launch_tile(const AttnShape& s, const AttnArgs& a, int rows, hipStream_t stream) {
    const dim3 grid(s.n_heads, (rows + kTileRows - 1) / kTileRows, a.tile_chunk ? a.splits : 1);
    const dim3 block(kTileWaves * kWave);
    switch (s.head_size / 16) {
        case 1: hipLaunchKernelGGL(attn_tile_kernel<1>, grid, block, 0, stream, a); break;
        case 2: hipLaunchKernelGGL(attn_tile_kernel<2>, grid, block, 0, stream, a); break;
        case 3: hipLaunchKernelGGL(attn_tile_kernel<3>, grid, block, 0, stream, a); break;
        case 4: hipLaunchKernelGGL(attn_tile_kernel<4>, grid, block, 0, stream, a); break;
        case 5: hipLaunchKernelGGL(attn_tile_kernel<5>, grid, block, 0, stream, a); break;
        case 6: hipLaunchKernelGGL(attn_tile_kernel<6>, grid, block, 0, stream, a); break;
        case 7: hipLaunchKernelGGL(attn_tile_kernel<7>, grid, block, 0, stream, a); break;
        default: hipLaunchKernelGGL(attn_tile_kernel<8>, grid, block, 0, stream, a); break;
    }
}

void launch_merge(const AttnShape& s, const AttnArgs& a, int rows, hipStream_t stream) {
    const int hs4 = s.head_size / 4;
    const int dpw = hs4 < kMergeDims ? hs4 : kMergeDims, groups = (hs4 + dpw - 1) / dpw;
    const std::size_t slots = kThreads / dpw;
    hipLaunchKernelGGL(attn_merge_kernel, dim3(s.n_heads * groups, rows), dim3(kThreads),
                       (slots * dpw * 4 + 2 * slots) * sizeof(float), stream, a);
}

// Where overlapping a chunk's rounds pays (us, apart / overlapped): four rows
// of 32 heads of 64 at context 4096 / 9000 38 / 32, 95 / 73, of 128 at 9000
// 135 / 121, of 32 on 8 kv heads of 128 82 / 77; one row of 32 heads of 64 at
// 9000 37.7 / 33.5. Not for one row of two or four heads of 128 a workgroup,
// whose four-deep grid already overlaps (8 kv heads at 9000 / 16384 28.2 /
// 29.6, 37.8 / 40.9), nor past 128 dims, where it spills, nor for a prompt's
// rows, which fill the card with workgroups (489 rows of 48 heads of 40 at
// context 5802 4397 / 6004).
template <int G, int LPP>
constexpr bool split_pipes(int rows) {
    return LPP <= 32 && rows <= static_cast<int>(kSplitMaxRows) &&
           (rows > 1 || G == 1 || G == 8 || LPP <= 16);
}

// Rows of fewer than a.merge_from chunks are left for the caller to merge;
// no merge launches when no row can have that many.
template <int G, int LPP, int F, bool ROPE>
void launch_split(const AttnShape& s, const AttnArgs& a, int rows, hipStream_t stream) {
    const dim3 grid(s.n_heads / G, rows, a.splits);
    const std::size_t lds = split_lds(s, ROPE, a.merge_count != nullptr);
    bool piped = false;
    if constexpr (split_pipes<G, LPP>(ROPE ? 1 : 2)) {
        piped = split_pipes<G, LPP>(rows);
        if (piped)
            hipLaunchKernelGGL((attn_split_kernel<G, LPP, F, ROPE, true>), grid, dim3(kThreads), lds,
                               stream, a);
    }
    if constexpr (!ROPE || !split_pipes<G, LPP>(1)) {
        if (!piped)
            hipLaunchKernelGGL((attn_split_kernel<G, LPP, F, ROPE>), grid, dim3(kThreads), lds, stream,
                               a);
    }
    if (a.merge_count) return;  // the kernel merges its own rows
    if (a.splits < a.merge_from) return;  // e.g. one chunk per row: written directly
    launch_merge(s, a, rows, stream);
}

template <int G, bool ROPE = false>
void launch_split_g(const AttnShape& s, const AttnArgs& a, int rows, hipStream_t stream) {
    switch (split_lanes(s) * 10 + split_f(s)) {
        case 41: launch_split<G, 4, 1, ROPE>(s, a, rows, stream); break;
        case 81: launch_split<G, 8, 1, ROPE>(s, a, rows, stream); break;
        case 161: launch_split<G, 16, 1, ROPE>(s, a, rows, stream); break;
        case 321: launch_split<G, 32, 1, ROPE>(s, a, rows, stream); break;
        case 641: launch_split<G, 64, 1, ROPE>(s, a, rows, stream); break;
        default: launch_split<G, 64, 2, ROPE>(s, a, rows, stream); break;
    }
}

// Where a few-row call runs on the grouped tile kernel, whose time follows the
// bytes of the context, not the columns (query rows times heads of a kv head):
// split / grouped kernel, us, heads of 128. 32 heads on 8 at context 16384: 1
// row 38 / 39 (4 columns), 2 rows 56 / 40, 4 rows 100 / 41; 48 on 8, 1 row 72 /
// 40; 32 on 16 at 1500 with 2 / 4 / 8 columns 13.5 / 16.4, 15.7 / 16.7, 22 /
// 17. Heads of 64, whose keys the split kernel has less work in flight for:
// 32 on 16 at 4096, 2 columns 16.7 / 14.2; 32 on 8, 4 columns 15.6 / 11.4. Odd
// groups the split kernel takes a head at a time: 24 on 8 of 96, 1 row at
// 16384 51 / 33. Short contexts, 2 to 4 rows: heads of 64 at 50 5.3 / 4.9, of 96
// and 112 at 50 5.2 / 6.3, at 300 the same, of 128 at 50 5.2 / 7.2, at 250 8.6 /
// 9.8, at 700 the same. The context is not known here, so a cache that holds
// no longer ones leaves the larger heads to the split kernel.
bool group_preferred(const AttnShape& s, int rows) {
    const int group = s.n_heads / s.n_kv_heads, columns = rows * group;
    const int cache = s.head_size <= 80 ? 0 : s.head_size <= 112 ? 256 : 1024;
    return group >= 2 && tile_supports(s) && s.seq_len > cache &&
           (columns >= (s.head_size > 64 ? 6 : 2) || heads_per_block(s) == 1);
}

// The call on the grouped tile kernel, its partials where the split kernel's
// would be (fewer chunks, so they fit).
void run_group(const AttnShape& s, AttnArgs a, int rows, hipStream_t stream) {
    a.group_chunk_min = kGroupChunkMin;
    a.splits = std::max(1, std::min(a.splits, kGroupWorkgroups / s.n_kv_heads));
    const int columns = rows * (s.n_heads / s.n_kv_heads);
    const dim3 grid(s.n_kv_heads, (columns + kTileRows - 1) / kTileRows, a.splits);
    const dim3 block(kTileWaves * kWave);
    switch (s.head_size / 16) {
        case 1: hipLaunchKernelGGL(attn_group_kernel<1>, grid, block, 0, stream, a); break;
        case 2: hipLaunchKernelGGL(attn_group_kernel<2>, grid, block, 0, stream, a); break;
        case 3: hipLaunchKernelGGL(attn_group_kernel<3>, grid, block, 0, stream, a); break;
        case 4: hipLaunchKernelGGL(attn_group_kernel<4>, grid, block, 0, stream, a); break;
        case 5: hipLaunchKernelGGL(attn_group_kernel<5>, grid, block, 0, stream, a); break;
        case 6: hipLaunchKernelGGL(attn_group_kernel<6>, grid, block, 0, stream, a); break;
        case 7: hipLaunchKernelGGL(attn_group_kernel<7>, grid, block, 0, stream, a); break;
        default: hipLaunchKernelGGL(attn_group_kernel<8>, grid, block, 0, stream, a); break;
    }
    if (a.splits > 1) launch_merge(s, a, rows, stream);
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace

std::string attention_reject(const AttnShape& s, int kernel) {
    if (kernel < kAttnAutomatic || kernel > kAttnSplit) return "attention: unknown kernel";
    if (s.n_heads <= 0 || s.n_kv_heads <= 0 || s.head_size <= 0 || s.seq_len <= 0 ||
        s.n_heads % s.n_kv_heads != 0)
        return "attention: bad shape";
    if (static_cast<std::size_t>(s.seq_len) * s.kv_stride >= (std::size_t{1} << 31) ||
        s.q_stride >= (std::size_t{1} << 31) || s.out_stride >= (std::size_t{1} << 31))
        return "attention: cache past 32-bit indexing";
    const bool single = kernel == kAttnSingle;
    // split loads float4s.
    if (!single && (s.head_size % 4 || s.head_size > 512 || s.q_stride % 4 ||
                    s.kv_stride % 4 || s.out_stride % 4))
        return "attention: split needs head_size and strides divisible by 4";
    const std::size_t need = single ? single_lds(s) : split_lds(s);
    if (need > kMaxLds)
        return "attention: seq_len " + std::to_string(s.seq_len) + " needs " +
               std::to_string(need) + " bytes of LDS, more than " + std::to_string(kMaxLds);
    return "";
}

// Enough for any call of up to `rows` rows, so that a buffer sized once for
// the most rows serves every smaller call: a split tile grid's chunk count
// grows as its row tiles shrink.
std::size_t attention_scratch_floats(const AttnShape& s, std::size_t rows, int kernel) {
    if (kernel == kAttnSingle) return 0;
    if (kernel != kAttnAutomatic) return split_scratch(s, rows).total;
    const std::size_t cut = split_max_rows(s);
    std::size_t need = split_scratch(s, rows < cut ? rows : cut).total;
    if (rows > cut && tile_supports(s)) {
        const std::size_t tiles = (rows + kTileRows - 1) / kTileRows;
        for (std::size_t rt = 1; rt <= tiles; ++rt) {
            const std::size_t m = std::min(rows, rt * kTileRows);
            if (m <= cut) continue;
            const int S = tile_splits(s, m);
            if (S == 1) break;  // more row tiles split no further
            need = std::max(need, tile_scratch(s, m, S).total);
        }
    }
    return need;
}

bool attention_uses_split(const AttnShape& s, std::size_t rows, int kernel) {
    return resolve(kernel, rows, s) != kAttnSingle;
}

bool attention_needs_scratch(const AttnShape& s, std::size_t rows, int kernel) {
    return resolve(kernel, rows, s) == kAttnSplit;
}

namespace {

AttnArgs base_args(const AttnShape& s, int rows, const int* pos, const float* q, const float* kc,
                   const float* vc, float* out) {
    AttnArgs a{};
    a.n_heads = s.n_heads;
    a.head_size = s.head_size;
    a.group = s.n_heads / s.n_kv_heads;
    a.seq_len = s.seq_len;
    a.q_stride = static_cast<int>(s.q_stride);
    a.kv_stride = static_cast<int>(s.kv_stride);
    a.out_stride = static_cast<int>(s.out_stride);
    a.pos = pos;
    a.q = q;
    a.kc = kc;
    a.vc = vc;
    a.out = out;
    a.rows = rows;
    a.merge_from = 2;
    a.min_chunk = min_chunk(s);
    return a;
}

void set_split(const AttnShape& s, int rows, float* scratch, AttnArgs& a) {
    const SplitScratch l = split_scratch(s, rows);
    a.splits = split_count(s);
    a.chunk_cap = split_chunk_cap(s);
    a.part_o = scratch + l.o;
    a.part_ml = reinterpret_cast<float2*>(scratch + l.ml);
}

}  // namespace

void run_attention(const AttnShape& s, int rows, const int* pos, const float* q, const float* kc,
                   const float* vc, float* out, float* scratch, int kernel, hipStream_t stream) {
    const bool automatic = kernel == kAttnAutomatic;
    kernel = resolve(kernel, rows, s);
    AttnArgs a = base_args(s, rows, pos, q, kc, vc, out);
    if (automatic && kernel == kAttnSplit && group_preferred(s, rows)) {
        set_split(s, rows, scratch, a);
        run_group(s, a, rows, stream);
        return;
    }
    if (kernel == kAttnTile && rows_preferred(s, rows)) {
        const dim3 grid(s.n_heads, (rows + kRowsTile - 1) / kRowsTile), block(4 * kWave);
        switch (s.head_size / 16) {
            case 4: hipLaunchKernelGGL(attn_rows_kernel<4>, grid, block, 0, stream, a); break;
            case 5: hipLaunchKernelGGL(attn_rows_kernel<5>, grid, block, 0, stream, a); break;
            case 6: hipLaunchKernelGGL(attn_rows_kernel<6>, grid, block, 0, stream, a); break;
            case 7: hipLaunchKernelGGL(attn_rows_kernel<7>, grid, block, 0, stream, a); break;
            default: hipLaunchKernelGGL(attn_rows_kernel<8>, grid, block, 0, stream, a); break;
        }
        return;
    }
    if (kernel == kAttnTile) {
        // The context split needs the caller's scratch (sized by
        // attention_scratch_floats); without it the grid stays whole.
        const int S = scratch && reinterpret_cast<uintptr_t>(scratch) % 16 == 0
                          ? tile_splits(s, static_cast<std::size_t>(rows))
                          : 1;
        if (S > 1) {
            const SplitScratch l = tile_scratch(s, static_cast<std::size_t>(rows), S);
            a.splits = S;
            a.tile_chunk = tile_chunk(s, S);
            a.part_o = scratch + l.o;
            a.part_ml = reinterpret_cast<float2*>(scratch + l.ml);
        }
        launch_tile(s, a, rows, stream);
        if (S > 1) launch_merge(s, a, rows, stream);
        return;
    }
    if (kernel == kAttnSingle) {
        hipLaunchKernelGGL(attn_single_kernel, dim3(s.n_heads, rows), dim3(kThreads),
                           single_lds(s), stream, a);
        return;
    }
    if (kernel == kAttnWhole) {
        a.splits = 1;
        a.chunk_cap = s.seq_len;
    } else {
        set_split(s, rows, scratch, a);
    }
    switch (heads_per_block(s)) {
        case 8: launch_split_g<8>(s, a, rows, stream); break;
        case 4: launch_split_g<4>(s, a, rows, stream); break;
        case 2: launch_split_g<2>(s, a, rows, stream); break;
        default: launch_split_g<1>(s, a, rows, stream); break;
    }
}

bool run_attention_rope(const AttnShape& s, const int* pos, const Summed& src, int dim,
                        int kv_dim, const float* cos_t, const float* sin_t, float* kc, float* vc,
                        float* out, float* scratch, hipStream_t stream, SplitRow* defer,
                        bool merge_inside, int whole) {
    if (resolve(kAttnAutomatic, 1, s) != kAttnSplit || split_lds(s, true, true) > kMaxLds)
        return false;
    if (src.n % 4 || src.mn % 4 || dim % 4 || kv_dim % 4) return false;
    if (!aligned16(src.slices == 1 ? src.c : src.partial) || (src.scale && !aligned16(src.scale)))
        return false;
    AttnArgs a = base_args(s, 1, pos, nullptr, kc, vc, out);
    set_split(s, 1, scratch, a);
    if (!defer) a.whole = whole;
    a.src = src;
    a.dim = dim;
    a.kv_dim = kv_dim;
    a.cos_t = cos_t;
    a.sin_t = sin_t;
    a.kc_w = kc;
    a.vc_w = vc;
    // Deferred: rows of up to kMergeInGemv chunks are merged by the consumer,
    // longer ones (a shape with more splits) by the merge kernel, into out.
    const bool hold = defer && a.splits > 1;
    if (hold) a.merge_from = kMergeInGemv + 1;
    if (!defer && merge_inside && a.splits > 1)
        a.merge_count = tile_counters(static_cast<std::size_t>(s.n_heads / heads_per_block(s)));
    switch (heads_per_block(s)) {
        case 8: launch_split_g<8, true>(s, a, 1, stream); break;
        case 4: launch_split_g<4, true>(s, a, 1, stream); break;
        case 2: launch_split_g<2, true>(s, a, 1, stream); break;
        default: launch_split_g<1, true>(s, a, 1, stream); break;
    }
    if (defer) {
        *defer = SplitRow{};
        if (hold) *defer = SplitRow{a.part_o, a.part_ml, out, pos, a.splits, s.n_heads, s.head_size, a.min_chunk};
    }
    return true;
}

bool attention_merge_inside_preferred(const AttnShape& s) { return heads_per_block(s) == 1; }

int attention_whole_context(const AttnShape& s) {
    return heads_per_block(s) == 1 && s.head_size <= 64 ? 256 : 0;
}

void run_attention_merge(const AttnShape& s, const SplitRow& r, float* out, hipStream_t stream) {
    AttnArgs a = base_args(s, 1, r.pos, nullptr, nullptr, nullptr, out);
    a.splits = r.splits;
    a.part_o = const_cast<float*>(r.o);
    a.part_ml = const_cast<float2*>(r.ml);
    launch_merge(s, a, 1, stream);
}

}  // namespace em
