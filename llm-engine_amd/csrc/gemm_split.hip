// fp32 products of many rows on bf16 matrix cores with fp32 results: what
// GpuKernel::automatic runs for fp32 B where gemm_split_preferred says so
// (reference: tiled / tiled_split, src/cuda_matmul.cu:49-125,
// 350-363).
//
// The split. An fp32 value x is exactly hi + mid + lo, three bf16 values:
// hi = x rounded to bf16 (8 significant bits, to nearest), mid = the exact
// remainder x - hi rounded to bf16, lo = what is left, which has at most
// seven significant bits. A product a * b is nine products of such terms,
// each exact in fp32 (8 x 8 bits). Six of them are summed by
// v_mfma_f32_16x16x32_bf16 into fp32 accumulators: hi*hi, hi*mid, mid*hi,
// hi*lo, lo*hi, mid*mid. The three left out are at most 2^-24 |a b| together
// (mid is up to 2^-8 of the value, lo 2^-17), one fp32 rounding of the
// product; over random operands 2^-27.4 rms and of either sign. (All operands
// 0x1.00ff8p+0, every left-out sum 2^-24.01 and of one sign: 5.9e-8 off at k =
// 32 to 4096, as the fp32 MFMA kernels are.) hi*hi has an accumulator of its own, so the sum at full magnitude is rounded
// once per 32 rows of k and the five small terms add nothing to that: the
// relative error against 64 bits at 4096 x 4096 x 4096 measured 4.0e-7,
// against 1.1e-6 for the fp32 MFMA chain of gemm_fast_kernel.
//
// Range. Every step above is exact while the terms are bf16 values, which on
// gfx950 (whose bf16 MFMA keeps subnormals) is |x| >= 2^-109 and zero; below
// that lo drops bits worth at most 2^-134. Each thread ORs what its lo terms
// could not hold. A tile whose sums hold a non-finite value (an infinity or
// NaN in the inputs, or an overflow), or which dropped bits and has a sum
// below 2^-50 in magnitude or an operand of 2^37 or more, is computed again
// by fp32 MFMAs straight from global memory (exact_tile). For the rest the
// k < 2^21 drops of either operand add up to less than 2^21 2^-133 2^37 =
// 2^-75, under a rounding of the sum. The operands are read again for their
// largest value only in a tile that dropped bits; 2048^3 does not notice the
// check (97.5 / 97.8 us), 300-row Llama-7B products take 775 -> 790.
//
// Speed. Six bf16 MFMAs stand for eight fp32 ones of twice the cycles each:
// 6/16 of the fp32 MFMA time. What paces the kernel is the card's power
// (random bf16 operands: 1.9 PFLOP/s from registers alone, 1.27 PFLOP/s for
// the vendor's 8192^3 product, so about 211 TFLOP/s here), then the VALU
// work of the split (6 ops per value, largely serial with the MFMAs) and LDS
// bandwidth. So tiles are as large as 256 registers a wave allow with two
// accumulator sets: a value of A is split once per column tile, one of B
// once per row tile. 4096^3 644 us (213 TFLOP/s) against 951 for
// gemm_fast_kernel; 300 x 4096 x 22016 352 us against 444.
//
// One workgroup of eight waves per CU, tile BM x BN, k in chunks of 32. A
// chunk's values are loaded into registers one chunk ahead, split and
// written as bf16 planes to the other of two LDS stages, then the next
// chunk's loads are issued and this chunk is multiplied; one barrier per
// chunk. A planes lie as 16-row fragments [term][row][unit], the four
// 16-byte units of a row (8 k each) permuted by unit ^ (row / 2 % 4) so that
// eight consecutive lanes of a read cover all banks; B planes as
// [term][8 k][column]. The weights are the MFMA's first operand, so a lane
// ends up with four consecutive columns of one row.
#include <algorithm>
#include <optional>

#include "common.hpp"
#include "internal.hpp"

namespace em {
namespace {

constexpr int kChunk = 32;  // k rows per step

struct GsParams {
    int m, n, k, span;  // span: chunks per k slice
    const float* A;
    const float* B;
    float* out;  // C (direct) or partials [slice][m][n]
    int direct, accumulate, vec;  // vec: float4 access to out
    int row_tiles, col_tiles;
};

// The wave's MB x NB blocks of 16 x 16 outputs over k in [kb, ke) by fp32
// MFMAs on operands from global memory, through put(mb, nb, sums) as the
// main path's sums: rows row0 + 16 mb + j, columns col0 + 16 nb + 4g .. + 3.
template <int MB, int NB, class Put>
__device__ __forceinline__ void exact_tile(const GsParams& p, int row0, int col0, int kb, int ke,
                                           Put put) {
    const int lane = threadIdx.x % kWave, g = lane >> 4, j = lane & 15;
    for (int nb = 0; nb < NB; ++nb) {
        floatx4 s[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) s[mb] = floatx4{0.f, 0.f, 0.f, 0.f};
        const float* b = p.B + min(col0 + 16 * nb + j, p.n - 1);
        for (int k0 = kb; k0 < ke; k0 += 4) {
            const int kk = k0 + g, kc = min(kk, p.k - 1);
            const bool in = kk < ke;
            const float bv = in ? b[static_cast<std::size_t>(kc) * p.n] : 0.0f;
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const int row = min(row0 + 16 * mb + j, p.m - 1);
                const float av = in ? p.A[static_cast<std::size_t>(row) * p.k + kc] : 0.0f;
                s[mb] = mfma16x16x4(bv, av, s[mb]);
            }
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) put(mb, nb, s[mb]);
    }
}

template <int MB, int NB, int WR, int WC>
__global__ __launch_bounds__(kWave * WR * WC, 2) void gemm_split_kernel(GsParams p) {
    constexpr int T = kWave * WR * WC, BM = 16 * MB * WR, BN = 16 * NB * WC;
    constexpr int kAStage = BM * 192, kBStage = BN * 192;  // bytes: three planes of 32 k
    __shared__ __attribute__((aligned(1024))) char smem[2 * (kAStage + kBStage)];

    const int tid = threadIdx.x, lane = tid % kWave, g = lane >> 4, j = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int wr = w / WC, wc = w % WC;
    const TileId place = tile_of(blockIdx.x, gridDim.x, p.row_tiles, p.col_tiles, true);
    const int m0 = place.row * BM, n0 = place.col * BN;
    const int chunks = (p.k + kChunk - 1) / kChunk;
    const int cb = place.slice * p.span, ce = min(chunks, cb + p.span);
    uint32_t lost = 0;

    // Chunk c covers k [32c, 32c + 32); the last one of a k that is not whole
    // chunks starts at k - 32 instead, its A values before 32c counted as
    // zero, so that no load needs a bound. Threads past a tile's last task
    // load that task again and store nothing.
    auto start = [&](int c) { return min(c * kChunk, p.k - kChunk); };

    // A: task t takes eight k (unit t % 4) of row t / 4; thread tid tasks
    // tid, tid + T, ... Rows past m read row m - 1; their sums are not
    // stored. k % 4 == 0.
    constexpr int kTasksA = BM * 4, NA = (kTasksA + T - 1) / T;
    const char* a_base = reinterpret_cast<const char*>(p.A + static_cast<std::size_t>(m0) * p.k);
    uint32_t a_off[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int t = min(tid + i * T, kTasksA - 1);
        a_off[i] = static_cast<uint32_t>((min(m0 + t / 4, p.m - 1) - m0) * p.k + (t % 4) * 8) * 4u;
    }
    floatx4 ra[NA][2];
    auto load_a = [&](int c) {
        const char* b = a_base + static_cast<std::size_t>(start(c)) * 4;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            ra[i][0] = *reinterpret_cast<const floatx4*>(b + a_off[i]);
            ra[i][1] = *reinterpret_cast<const floatx4*>(b + a_off[i] + 16);
        }
    };
    auto store_a = [&](int c, int s) {
        const int z = c * kChunk - start(c);
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            if (kTasksA % T && w + i * (T / kWave) >= kTasksA / kWave) break;
            const int t = tid + i * T, row = t / 4, jr = row % 16;
            char* o = smem + s * kAStage + (row / 16) * 3072 + (jr * 4 + ((t % 4) ^ ((jr >> 1) & 3))) * 16;
            float v[8] = {ra[i][0].x, ra[i][0].y, ra[i][0].z, ra[i][0].w,
                          ra[i][1].x, ra[i][1].y, ra[i][1].z, ra[i][1].w};
            if (z > 0) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = (t % 4) * 8 + e < z ? 0.0f : v[e];
            }
            uint4 x[3];
            split3x8(v, x, lost);
#pragma unroll
            for (int q = 0; q < 3; ++q) *reinterpret_cast<uint4*>(o + q * 1024) = x[q];
        }
    };
    // B: task t takes eight k (8 (t / BN) ..) of column t % BN. Columns past
    // n read column n - 1.
    constexpr int kTasksB = BN * 4, NT = (kTasksB + T - 1) / T;
    uint32_t b_off[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const int t = min(tid + i * T, kTasksB - 1);
        b_off[i] = static_cast<uint32_t>(8 * (t / BN) * p.n + min(n0 + t % BN, p.n - 1)) * 4u;
    }
    float rb[NT][8];
    auto load_b = [&](int c) {
        const char* b = reinterpret_cast<const char*>(p.B) + static_cast<std::size_t>(start(c)) * 4 * p.n;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                rb[i][e] = *reinterpret_cast<const float*>(
                    b + static_cast<std::size_t>(e) * p.n * 4 + b_off[i]);
    };
    auto store_b = [&](int s) {
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            if (kTasksB % T && w + i * (T / kWave) >= kTasksB / kWave) break;
            uint4 x[3];
            split3x8(rb[i], x, lost);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                *reinterpret_cast<uint4*>(smem + 2 * kAStage + s * kBStage + q * (BN * 64) +
                                          (tid + i * T) * 16) = x[q];
        }
    };

    // acc: hi * hi; low: the five smaller products.
    floatx4 acc[NB][MB], low[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = low[nb][mb] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int a_rd = wr * MB * 3072 + (j * 4 + (g ^ ((j >> 1) & 3))) * 16;
    const int b_rd = 2 * kAStage + (g * BN + wc * NB * 16 + j) * 16;
    auto multiply = [&](int s) {
        const char* as = smem + s * kAStage + a_rd;
        const char* bs = smem + s * kBStage + b_rd;
        bf16x8 a[MB][3], b[2][3];
#pragma unroll
        for (int t = 0; t < 3; ++t) b[0][t] = *reinterpret_cast<const bf16x8*>(bs + t * (BN * 64));
        // In the order of first use.
#pragma unroll
        for (int t = 0; t < 3; ++t)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                a[mb][t] = *reinterpret_cast<const bf16x8*>(as + (mb * 3 + t) * 1024);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (nb + 1 < NB) {
#pragma unroll
                for (int t = 0; t < 3; ++t)
                    b[(nb + 1) & 1][t] =
                        *reinterpret_cast<const bf16x8*>(bs + t * (BN * 64) + (nb + 1) * 256);
            }
            auto mma = [&](floatx4 (&d)[MB], int tb, int ta) {
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    d[mb] = mfma16x16x32(b[nb & 1][tb], a[mb][ta], d[mb]);
            };
            mma(acc[nb], 0, 0);
            mma(low[nb], 2, 0);
            mma(low[nb], 1, 0);
            mma(low[nb], 0, 1);
            mma(low[nb], 1, 1);
            mma(low[nb], 0, 2);
        }
    };

    if (cb < ce) {
        load_b(cb);
        load_a(cb);
        store_b(0);
        store_a(cb, 0);
        if (cb + 1 < ce) {
            load_b(cb + 1);
            load_a(cb + 1);
        }
        __syncthreads();
        for (int c = cb; c < ce; ++c) {
            const int s = (c - cb) & 1;
            if (c + 1 < ce) {
                store_b(s ^ 1);
                store_a(c + 1, s ^ 1);
                if (c + 2 < ce) {
                    load_b(c + 2);
                    load_a(c + 2);
                }
            }
            // The loads stay ahead of the MFMAs.
            __builtin_amdgcn_sched_barrier(0);
            multiply(s);
            __syncthreads();
        }
    }

    const int row0 = m0 + wr * MB * 16, col0 = n0 + wc * NB * 16;
    const float inf = __builtin_inff();
    bool bad = false, tiny = false;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            acc[nb][mb] += low[nb][mb];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = fabsf(acc[nb][mb][e]);
                bad |= !(x < inf);
                tiny |= x < 0x1p-50f;
            }
        }
    // Whether this thread's share of the tile's operands holds a value of 2^37
    // or more, by which a dropped bit could grow past that rounding.
    auto large = [&] {
        const int kb = cb * kChunk, ke = min(p.k, ce * kChunk);
        const int rows = min(BM, p.m - m0), cols = min(BN, p.n - n0);
        float top = 0.0f;
        for (int r = w; r < rows; r += T / kWave)
            for (int kk = kb + lane; kk < ke; kk += kWave)
                top = fmaxf(top, fabsf(p.A[static_cast<std::size_t>(m0 + r) * p.k + kk]));
        for (int kk = kb + w; kk < ke; kk += T / kWave)
            for (int c = lane; c < cols; c += kWave)
                top = fmaxf(top, fabsf(p.B[static_cast<std::size_t>(kk) * p.n + n0 + c]));
        return top >= 0x1p37f;
    };
    const bool dropped = __syncthreads_or((lost & 0xffffu) != 0) != 0;
    const bool redo = __syncthreads_or(bad || (dropped && (tiny || large()))) != 0;

    float* out = p.out + (p.direct ? 0 : static_cast<std::size_t>(place.slice) * p.m * p.n);
    const bool add = p.direct && p.accumulate;
    auto at = [&](int mb, int nb) {
        return out + static_cast<std::size_t>(row0 + 16 * mb + j) * p.n + col0 + 16 * nb + 4 * g;
    };
    // A sum whose columns reach past n, or whose rows are not float4s.
    auto put_scalar = [&](int mb, int nb, floatx4 v) {
        float* o = at(mb, nb);
        if (row0 + 16 * mb + j >= p.m) return;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (col0 + 16 * nb + 4 * g + e < p.n) o[e] = add ? o[e] + v[e] : v[e];
    };
    if (redo) {
        exact_tile<MB, NB>(p, row0, col0, cb * kChunk, min(p.k, ce * kChunk), put_scalar);
        return;
    }
    if (!p.vec) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) put_scalar(mb, nb, acc[nb][mb]);
        return;
    }
    // Prior values all loaded before the first store (in range: clamped), so
    // that no load waits behind a store it might alias.
    if (add) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const int row = min(row0 + 16 * mb + j, p.m - 1);
                const int col = min(col0 + 16 * nb + 4 * g, p.n - 4);
                low[nb][mb] = *reinterpret_cast<const floatx4*>(
                    p.out + static_cast<std::size_t>(row) * p.n + col);
            }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = low[nb][mb] + acc[nb][mb];
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        if (row0 + 16 * mb + j >= p.m) continue;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
            if (col0 + 16 * nb + 4 * g < p.n) *reinterpret_cast<floatx4*>(at(mb, nb)) = acc[nb][mb];
    }
}

// The tile shapes: rows, columns, and the time of one 32-deep step of a
// workgroup alone on its CU and of two sharing one (us; 0: two do not fit
// the LDS), measured with 240 and 480 workgroups at k = 4096.
struct Shape {
    int bm, bn;
    double one_us, two_us;
    void (*launch)(const GsParams&, int blocks, hipStream_t);
};

template <int MB, int NB, int WR, int WC>
void launch(const GsParams& p, int blocks, hipStream_t s) {
    hipLaunchKernelGGL((gemm_split_kernel<MB, NB, WR, WC>), dim3(blocks), dim3(kWave * WR * WC), 0,
                       s, p);
}

constexpr Shape kShapes[] = {
    {32, 128, 0.97, 1.41, launch<1, 2, 2, 4>}, {64, 128, 1.09, 1.90, launch<2, 2, 2, 4>},
    {96, 128, 1.34, 0, launch<3, 2, 2, 4>},    {128, 128, 1.62, 0, launch<4, 2, 2, 4>},
    {160, 128, 1.94, 0, launch<5, 2, 2, 4>},   {64, 64, 0.91, 1.20, launch<2, 1, 2, 4>},
    {128, 64, 1.07, 1.90, launch<2, 2, 4, 2>}, {192, 128, 2.19, 0, launch<3, 4, 4, 2>},
    {256, 128, 2.65, 0, launch<4, 4, 4, 2>},   {320, 96, 2.74, 0, launch<5, 3, 4, 2>},
    {320, 64, 2.16, 0, launch<5, 2, 4, 2>},
};

struct Plan {
    const Shape* shape;
    int slices, span;
    double us;
};

// The plan with the least estimated time: rounds of the grid over the CUs
// (two workgroups a CU where they fit) times the steps of one workgroup, 6 us
// of launch, first loads and last stores, 2 us a round; and for k slices
// the partials' traffic at 6 TB/s and a 2 us launch. Slices are at least
// four chunks deep. For the 300-row Llama-7B products it picks the fastest
// shape and slices of those measured.
// Past two workgroups a CU, more slices only add traffic. A few narrow tiles
// of a deep k take up to 64 (at most 16: 12 x 13000 x 256 25 us against 11.6
// now and 12.3 for tiled_split), every fourth past 16 to keep the search short.
Plan plan(int m, int n, int k, bool slices_ok) {
    const unsigned chunks = ceil_div(k, kChunk), cus = cu_count();
    Plan best{nullptr, 1, static_cast<int>(chunks), 0.0};
    for (const Shape& sh : kShapes) {
        const unsigned tiles = static_cast<unsigned>(ceil_div(m, sh.bm)) * ceil_div(n, sh.bn);
        const unsigned most =
            slices_ok ? std::max(1u, std::min({64u, chunks / 4, 2 * cus / tiles + 1})) : 1u;
        for (unsigned want = 1; want <= most; want += want < 16 ? 1 : 4) {
            const unsigned span = (chunks + want - 1) / want;
            const unsigned slices = (chunks + span - 1) / span;
            const unsigned groups = tiles * slices;
            double rounds_us;
            unsigned rounds;
            if (sh.two_us > 0) {
                const unsigned full = groups / (2 * cus), rest = groups % (2 * cus);
                rounds_us = full * sh.two_us + (rest > cus ? sh.two_us : rest > 0 ? sh.one_us : 0.0);
                rounds = full + (rest > 0);
            } else {
                rounds = (groups + cus - 1) / cus;
                rounds_us = rounds * sh.one_us;
            }
            double us = 6.0 + rounds_us * span + 2.0 * rounds;
            if (slices > 1) us += 2.0 + 4.0 * m * n * (2.0 * slices + 1.0) / 6e6;
            if (!best.shape || us < best.us) best = Plan{&sh, static_cast<int>(slices), static_cast<int>(span), us};
        }
    }
    return best;
}

}  // namespace

bool gemm_split_supports(const MatmulArgs& a) {
    return a.k % 4 == 0 && a.k >= kChunk && a.k < (1 << 21) && a.n < (1 << 24) &&
           reinterpret_cast<uintptr_t>(a.A) % 16 == 0;
}

// Measured through em_matmul_f32 against the fp32 MFMA kernels automatic ran
// before (us, before / this).
//  - 1024^2 weights at m = 24 .. 512 10.7-17.1 / 10.7-19.2 and 288 x 864
//    8.2-9.3 / 10.7-12.2: up to 2^20 weights the streamlined tiled kernel
//    keeps what it takes.
//  - 4096 x 512 at m = 24 / 300 / 2048 17.5 / 12.4, 25.7 / 21.9, 92 / 59;
//    4096^2 at m = 32 / 300 / 1024 25 / 22, 135 / 70, 263 / 177; 4096 x
//    11008 at m = 48 / 300 / 2048 80 / 55, 266 / 185, 1337 / 935; 3000 x
//    3001 at m = 17 / 700 42 / 15, 222 / 104.
//  - Without float4 stores past about 640 k^2 outputs the stores cost more than
//    the split gains: 956 x 64 x 3895 14.6 / 17.0, 1916 x 48 x 13122 47 / 92.
//    By n alone: an output off 16 bytes gives the same bits as one that is
//    not (so does 1100 x 32 x 40000, 49 / 67, which stays here).
//  - A shallow product whose 64 x 64 tiles are one round of the streamlined
//    tiled kernel (a quarter more up to k = 640): 298 x 448 x 3040 11.7 / 17.1,
//    440 x 512 x 2368 21.1 / 24.3, 302 x 896 x 2688 24.2 / 27.0, and a whole
//    round 295 x 1088 x 3264 27.1 / 31.2; with fewer than 5/8 of one, or
//    deeper, the split wins (k = 2048 and a round 0.85).
//  - At few rows tiled_split streams the weights with less work per byte:
//    m = 16 2048 x 4096 14.3 / 13.4 but 4096^2 20.1 / 22.0 and 4096 x 11008
//    35 / 41; m = 24 4096 x 11008 41.8 / 41.0, m = 17 5120 x 13824 53 / 57.
bool gemm_split_preferred(const MatmulArgs& a) {
    const long long w = static_cast<long long>(a.n) * a.k;
    if (a.m <= 8 || !gemm_split_supports(a)) return false;
    if (a.n % 4 && static_cast<long long>(a.m) * a.n > 640LL * a.k * a.k) return false;
    if (w <= (1LL << 20)) return !tiled_preferred(a);
    const int tiles = ceil_div(a.m, 64) * ceil_div(a.n, 64), cus = cu_count();
    if (a.k <= (16 * tiles > 15 * cus ? 1300 : 900) && 8 * tiles > 5 * cus && tiles <= cus + (a.k <= 640 ? cus / 4 : 0) &&
        tiled_preferred(a))
        return false;
    return w <= (1LL << 23) || a.m > 32 || (a.m > 16 && w < (1LL << 26)) ||
           !tiled_split_supports<float>(a);
}

void run_gemm_split(const MatmulArgs& a) {
    Plan pl = plan(a.m, a.n, a.k, true);
    float* partials = nullptr;
    std::optional<StreamWorkspace> workspace;  // held until both launches are queued
    if (pl.slices > 1) {
        workspace.emplace(a.stream, static_cast<std::size_t>(pl.slices) * a.m * a.n);
        partials = workspace->p();
        if (!partials) pl = plan(a.m, a.n, a.k, false);
    }
    GsParams p{};
    p.m = a.m;
    p.n = a.n;
    p.k = a.k;
    p.span = pl.span;
    p.A = a.A;
    p.B = static_cast<const float*>(a.B);
    p.direct = pl.slices == 1;
    p.accumulate = a.accumulate ? 1 : 0;
    p.out = p.direct ? a.C : partials;
    p.vec = a.n % 4 == 0 && reinterpret_cast<uintptr_t>(p.out) % 16 == 0;
    p.row_tiles = ceil_div(a.m, pl.shape->bm);
    p.col_tiles = ceil_div(a.n, pl.shape->bn);
    pl.shape->launch(p, p.row_tiles * p.col_tiles * pl.slices, a.stream);
    if (!p.direct)
        run_reduce_slices(a.m, a.n, pl.slices, partials, nullptr, a.C, a.accumulate, a.stream);
}

}  // namespace em
