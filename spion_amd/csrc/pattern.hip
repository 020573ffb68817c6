// Pattern discovery on the device: diagonal filter + block pooling in one pass over the score map,
// then (one work-group per map) the quantile threshold, the greedy path walks and the binarised mask.
//
// Restates what the reference does on the host CPU with PyTorch ops and a recursive Python function
// (main_conv_ff.py:35-62 and :254-278; top-k variant main_conv.py:236-256; pool-only main_ff.py:253-272).
#include "common.h"
#include "tile_ops.h"
#include "../../include/spion_hip.h"

#include <algorithm>
#include <climits>
#include <cmath>
#include <mutex>
#include <vector>

namespace spion {

constexpr int POOL_THREADS = 256;
constexpr int WALK_THREADS = 1024;
constexpr int POOLED_LDS = 36864;  // block grids up to 192 x 192 are walked from LDS (144 KB of the CU's 160)

// The score maps of one launch, wherever they lie (the reference's attn_lst holds one tensor per layer,
// models/model_transformer.py:137): reading them in place spares the copy that stacks them, a quarter of the whole
// discovery at four maps of 2048 x 2048.  More maps take further launches.
constexpr int MAPS_PER_LAUNCH = 16;
struct ScoreMaps {
    const float* p[MAPS_PER_LAUNCH];
};

// pooled[I][J] = (1/bs^2) sum_{i in I, j in J} sum_{t=-hk..hk} A[i+t][j+t]  (zero outside the map).
// Regrouped per source element A[p][q]: its weight is the number of shifts t that land in the block.
// fp64 accumulation in a fixed order, one rounding to fp32.
__global__ __launch_bounds__(POOL_THREADS) void conv_pool_kernel(ScoreMaps maps, float* __restrict__ pooled, int L,
                                                                 int bs, int nb, int hk) {
    __shared__ double red[POOL_THREADS];
    const int I = blockIdx.y, J = blockIdx.x, map = blockIdx.z;
    const float* Am = maps.p[map];
    const int p0 = max(0, I * bs - hk), p1 = min(L, I * bs + bs + hk);
    const int q0 = max(0, J * bs - hk), q1 = min(L, J * bs + bs + hk);
    const int w = q1 - q0, total = (p1 - p0) * w;
    double acc = 0.0;
    for (int e = threadIdx.x; e < total; e += POOL_THREADS) {
        const int p = p0 + e / w, q = q0 + e % w;
        const int dp = p - I * bs, dq = q - J * bs;  // t must satisfy dp-bs+1 <= t <= dp, same for dq
        const int lo = max(-hk, max(dp, dq) - bs + 1);
        const int hi = min(hk, min(dp, dq));
        if (hi >= lo) acc += (double)Am[(size_t)p * L + q] * (double)(hi - lo + 1);
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = POOL_THREADS / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) pooled[((size_t)map * nb + I) * nb + J] = (float)(red[0] / ((double)bs * (double)bs));
}

// The same sums for block sizes of at least twice the filter's reach (bs >= 2 hk, so a column feeds its own block
// and at most one neighbour): one work-group per (block row, group of adjacent blocks, map); thread (column, row
// group) walks its share of the bs + 2 hk rows of one column -- consecutive threads read consecutive floats -- and
// keeps two fp64 sums, for the column's own block and for the neighbour it reaches into; one wavefront per block
// then adds the block's partial sums in a fixed order.  Every element is read once per block row it touches
// ((bs + 2 hk) / bs times, the repeats from L2) instead of once per block, and in full rows.
// A column's filter shifts t form an interval [lo, hi]; element row dp (from the block's first row) counts for those
// of them in [dp - bs + 1, dp], a trapezoid in dp: min(dp + 1 - lo, hi - lo + 1, hi + bs - dp), not below zero.  Small
// whole numbers, so it is formed in fp32 (four instructions, the integer form took eight comparisons per element), and
// for one of the two sums only: the shifts of a column's own block and of its neighbour make up all of them, so the
// neighbour's weight is that of the full trapezoid, the same for every column and looked up per row, less the own one.
// The weights are subtracted, which is exact; the difference of the two sums would be rounding noise wherever a
// column's own sum is many orders above its neighbour's, as on maps that decay steeply away from the diagonal.
// A batch of loads is issued before any of them is used, with the row clamped instead of a remainder loop whose loads
// would each wait alone, and the next batch before one is used.
// The weights were half of the inner loop's instructions, so for the block sizes in use they come from a table, two LDS
// reads and four fp64 instructions an element; a thread per column instead of two halves what a work-group spends on its
// table and reduction, once there are enough work-groups (2048: 8 per CU) for the machine not to run dry.  us, weights
// formed / table, block 32: four maps of 2048^2 25.4 / 22.0, six of 4096^2 121 / 95 (two threads a column 106), two of 2048^2
// 14.6 / 13.7, one of 1024^2 6.2 / 6.1 (one thread 7.8); block 64: 21.5 / 20.5, 96.6 / 92.2 (fp64 table: 24).
// Left: without any load 18, without any sum 20 of the 22 us, i.e. latency of waves that live for 31 to 62 rows.  Several
// block rows per work-group, the next one's loads in flight during a reduction, need 94 registers and are slower (30.5); two
// one after the other with one table are slower too (calls of four maps of 2048^2 32.4 / 35.1, six of 4096^2 124 / 156), and
// the partial sums in the table's place, eight work-groups to a CU instead of seven, change nothing (1 % either way).
constexpr int CP_COLS = 256, CP_BATCH = 16;
// BS: 32 or 64 (filters of up to 33 taps), the own sum's weights in a table (fp64 for 32; for 64 that would leave room for two
// work-groups to a CU, so fp32, converted); 0, any block size, formed per element.  CP_RG: threads to a column, each every CP_RG-th row.
template <int BS, int CP_RG>
__global__ __launch_bounds__(CP_COLS* CP_RG) void conv_pool_cols_kernel(ScoreMaps maps, float* __restrict__ pooled, int L,
                                                                         int bs_, int nb, int hk, int gb) {
    __shared__ double part[CP_RG][2][CP_COLS];
    typedef typename std::conditional<BS == 32, double, float>::type weight_t;
    __shared__ weight_t full[BS ? 2 * BS : CP_COLS];  // full trapezoid of row dp at [dp + hk]
    __shared__ weight_t table[BS ? (BS + 32) * BS : 1];  // own weight of (row dp, column c of a block) at [(dp + hk) * BS + c]
    const int bs = BS ? BS : bs_;
    // consecutive items -- the groups of a block row, then the next block row of the same map, whose rows overlap --
    // run on one die, whose L2 then serves the bs + 2 hk rows' overlap
    const int groups = (nb + gb - 1) / gb;
    const int item = xcd_remap(blockIdx.x, gridDim.x);
    const int I = item / groups % nb, map = item / groups / nb;
    const int Jg = item % groups * gb;  // first block of this group
    const float* Am = maps.p[map];
    const int cc = threadIdx.x % CP_COLS;
    const int rg = __builtin_amdgcn_readfirstlane((int)threadIdx.x / CP_COLS);  // a wavefront's columns share their rows
    const int ncols = gb * bs + 2 * hk;
    const int q = Jg * bs - hk + cc;
    const int p0 = max(0, I * bs - hk), p1 = min(L, I * bs + bs + hk);
    const bool works = cc < ncols && q >= 0 && q < L;
    const float* col = Am + (works ? q : 0);
    const auto request = [&](int pb, float (&v)[CP_BATCH]) {
#pragma unroll
        for (int k = 0; k < CP_BATCH; ++k) v[k] = col[(size_t)min(pb + k * CP_RG, p1 - 1) * L];
    };
    float v[CP_BATCH];
    request(p0 + rg, v);
    const auto trapezoid = [&](float dp, float lo1, float n, float top) {
        return fmaxf(0.f, fminf(fminf(dp + lo1, n), top - dp));
    };
    const auto own_weight = [&](float dp, int c) {
        const int lo = max(-hk, c - bs + 1), hi = min(hk, c);
        return trapezoid(dp, (float)(1 - lo), (float)min(hi - lo + 1, bs), (float)(hi + bs));
    };
    if ((int)threadIdx.x < bs + 2 * hk)
        full[threadIdx.x] = trapezoid((float)((int)threadIdx.x - hk), (float)(1 + hk), (float)min(2 * hk + 1, bs),
                                      (float)(hk + bs));
    if constexpr (BS > 0)
        for (int e = threadIdx.x; e < (BS + 2 * hk) * BS; e += CP_COLS * CP_RG)
            table[e] = (weight_t)own_weight((float)(e / BS - hk), e % BS);
    __syncthreads();
    double a0 = 0.0, a1 = 0.0;
    const int c = (works ? q : 0) % bs;
    for (int pb = p0 + rg; pb < p1; pb += CP_RG * CP_BATCH) {
        float next[CP_BATCH];
        if (pb + CP_RG * CP_BATCH < p1) request(pb + CP_RG * CP_BATCH, next);
#pragma unroll
        for (int k = 0; k < CP_BATCH; ++k) {
            const int p = pb + k * CP_RG;
            if (p < p1) {
                const int dp = p - I * bs;
                const double x = (double)v[k];
                const weight_t own = BS ? table[(dp + hk) * BS + c] : (weight_t)own_weight((float)dp, c);
                a0 += x * (double)own;
                a1 += x * (double)(full[dp + hk] - own);
            }
        }
#pragma unroll
        for (int k = 0; k < CP_BATCH; ++k) v[k] = next[k];
    }
    if (!works) a0 = a1 = 0.0;
    part[rg][0][cc] = a0;
    part[rg][1][cc] = a1;
    __syncthreads();
    // a wavefront adds up a block: entries e = 0 .. CP_RG (bs + 2 hk) - 1, lane-strided, then a butterfly
    const int lane = threadIdx.x & 63;
    for (int b = threadIdx.x >> 6; b < gb && Jg + b < nb; b += CP_COLS * CP_RG / 64) {
        const int base = hk + b * bs, span = bs + 2 * hk;
        double s = 0.0;
        for (int e = lane; e < CP_RG * span; e += 64) {
            const int r = e >= span, k = e - r * span - hk;  // column base + k, k = -hk .. bs + hk - 1
            s += part[r][(k < 0 || k >= bs) ? 1 : 0][base + k];
        }
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane == 0) pooled[((size_t)map * nb + I) * nb + Jg + b] = (float)(s / ((double)bs * (double)bs));
    }
}

__device__ __forceinline__ uint32_t float_key(float f) {  // order-preserving map to unsigned
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_float(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Key of the element of ascending rank `rank` (0-based) among v[0..N): 8-bit radix select by the whole
// work-group.  hist: 256 ints of LDS, sh: 2 ints of LDS.
__device__ uint32_t block_select(const float* __restrict__ v, int N, int rank, int* hist, int* sh) {
    uint32_t prefix = 0, mask = 0;
    int rem = rank;
    for (int shift = 24; shift >= 0; shift -= 8) {
        for (int i = threadIdx.x; i < 256; i += blockDim.x) hist[i] = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < N; i += blockDim.x) {
            uint32_t k = float_key(v[i]);
            if ((k & mask) == prefix) atomicAdd(&hist[(k >> shift) & 255u], 1);
        }
        __syncthreads();
        if (threadIdx.x < 64) {
            // first wavefront: lane l owns bins 4l..4l+3; the bin whose cumulative count first exceeds rem
            const int l = threadIdx.x;
            const int h0 = hist[4 * l], h1 = hist[4 * l + 1], h2 = hist[4 * l + 2], h3 = hist[4 * l + 3];
            const int own = h0 + h1 + h2 + h3;
            int incl = own;
            for (int o = 1; o < 64; o <<= 1) {
                const int up = __shfl_up(incl, o, 64);
                if (l >= o) incl += up;
            }
            int c = incl - own;
            const bool last = (l == 63);
            if ((c <= rem && rem < incl) || (last && rem >= incl)) {
                int b = 4 * l;
                if (c + h0 <= rem) { c += h0; ++b;
                    if (c + h1 <= rem) { c += h1; ++b;
                        if (c + h2 <= rem) { c += h2; ++b; } } }
                sh[0] = b;
                sh[1] = rem - c;
            }
        }
        __syncthreads();
        prefix |= (uint32_t)sh[0] << shift;
        mask |= 255u << shift;
        rem = sh[1];
        __syncthreads();
    }
    return prefix;
}

// Wavefront reductions and sums over the lanes below, by DPP moves (a shuffle goes through the LDS and takes its latency
// at every one of the six steps).  The result of a reduction is in the last lane.
template <class Op>
__device__ __forceinline__ uint32_t dpp_scan(uint32_t v, uint32_t none, Op op) {
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x111, 0xf, 0xf, false));  // row_shr:1
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x112, 0xf, 0xf, false));  // row_shr:2
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x114, 0xf, 0xf, false));  // row_shr:4
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x118, 0xf, 0xf, false));  // row_shr:8
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31
    return v;
}
__device__ __forceinline__ uint32_t wave_min_last(uint32_t v) {
    return dpp_scan(v, 0xffffffffu, [](uint32_t a, uint32_t b) { return min(a, b); });
}
__device__ __forceinline__ uint32_t wave_max_last(uint32_t v) {
    return dpp_scan(v, 0u, [](uint32_t a, uint32_t b) { return max(a, b); });
}

// f(element, index) for every i < N, four of a thread's elements loaded before the first is used.
template <class F>
__device__ __forceinline__ void for_elements(const float* __restrict__ v, int N, F f) {
    for (int i0 = threadIdx.x; i0 < N; i0 += 4 * WALK_THREADS) {
        float x[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = v[min(i0 + k * WALK_THREADS, N - 1)];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (i0 + k * WALK_THREADS < N) f(x[k], i0 + k * WALK_THREADS);
    }
}

// Key of the element of ascending rank `rank` among v[0..N), and of rank + 1 (unspecified for the last).  The range of
// the keys is found first and cut into 2048 equal parts: one histogram (the keys of one map share their leading bits,
// so the digits of a plain radix pass put them all into a few bins and serialise the LDS atomics), then the elements
// of the part the rank falls into are collected and ranked against each other.  More than SEL_CAND of them:
// block_select over the whole map.
constexpr int SEL_BINS = 2 * WALK_THREADS, SEL_CAND = 512;
struct SelectSpace {
    int bins[SEL_BINS];
    uint32_t cand[SEL_CAND];
    int hist[256];
    int wave[WALK_THREADS / 64];
    uint32_t key_min, key_max, above, key, next;
    int part, rank, cnt, n_cand, sh[2];
};
struct Ranked {
    uint32_t key, next;
};
__device__ Ranked range_select(const float* __restrict__ v, int N, int rank, SelectSpace& S) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t mn = 0xffffffffu, mx = 0u;
    for_elements(v, N, [&](float x, int) {
        const uint32_t k = float_key(x);
        mn = min(mn, k);
        mx = max(mx, k);
    });
    mn = wave_min_last(mn);
    mx = wave_max_last(mx);
    if (threadIdx.x == 0) {
        S.key_min = S.above = 0xffffffffu;
        S.key_max = 0u;
        S.n_cand = 0;
    }
    reinterpret_cast<int2*>(S.bins)[threadIdx.x] = make_int2(0, 0);
    for (int i = threadIdx.x; i < SEL_CAND; i += WALK_THREADS) S.cand[i] = 0xffffffffu;
    __syncthreads();
    if (lane == 63) {
        atomicMin(&S.key_min, mn);
        atomicMax(&S.key_max, mx);
    }
    __syncthreads();
    const uint32_t kmin = S.key_min, span = S.key_max - kmin;
    const int shift = max(0, 32 - __builtin_clz(span | 1u) - 11);  // parts of 2^shift keys
    for_elements(v, N, [&](float x, int) { atomicAdd(&S.bins[(float_key(x) - kmin) >> shift], 1); });
    __syncthreads();
    const int2 b = reinterpret_cast<const int2*>(S.bins)[threadIdx.x];  // thread t owns parts 2t and 2t + 1
    const int own = b.x + b.y;
    const int incl = (int)dpp_scan((uint32_t)own, 0u, [](uint32_t p, uint32_t q) { return p + q; });
    if (lane == 63) S.wave[wave] = incl;
    __syncthreads();
    int before = incl - own;
    for (int w = 0; w < WALK_THREADS / 64; ++w) before += w < wave ? S.wave[w] : 0;
    if (before <= rank && rank < before + own) {
        const bool second = before + b.x <= rank;
        S.part = 2 * threadIdx.x + second;
        S.rank = rank - (second ? before + b.x : before);
        S.cnt = second ? b.y : b.x;
    }
    __syncthreads();
    const int part = S.part, r = S.rank, cnt = S.cnt;
    if (cnt > SEL_CAND && shift > 0) {
        const uint32_t key = block_select(v, N, rank, S.hist, S.sh);
        if (threadIdx.x == 0) S.cnt = 0;
        __syncthreads();
        int c = 0;
        mn = 0xffffffffu;
        for_elements(v, N, [&](float x, int) {
            const uint32_t k = float_key(x);
            if (k <= key) ++c;
            else mn = min(mn, k);
        });
        c = (int)dpp_scan((uint32_t)c, 0u, [](uint32_t p, uint32_t q) { return p + q; });
        mn = wave_min_last(mn);
        if (lane == 63) {
            atomicAdd(&S.cnt, c);
            atomicMin(&S.above, mn);
        }
        __syncthreads();
        return Ranked{key, rank + 1 < S.cnt ? key : S.above};
    }
    mn = 0xffffffffu;  // smallest key of the parts above
    for_elements(v, N, [&](float x, int) {
        const uint32_t k = float_key(x) - kmin;
        const int p = (int)(k >> shift);
        if (p == part && shift > 0) S.cand[atomicAdd(&S.n_cand, 1)] = k;
        if (p > part) mn = min(mn, k);
    });
    mn = wave_min_last(mn);
    if (lane == 63) atomicMin(&S.above, mn);
    __syncthreads();
    const uint32_t above = kmin + S.above;
    if (shift == 0) {  // a part is one key
        const uint32_t key = kmin + (uint32_t)part;
        return Ranked{key, r + 1 < cnt ? key : above};
    }
    for (int i = threadIdx.x; i < cnt; i += WALK_THREADS) {
        const uint32_t k = S.cand[i];
        uint32_t more = 0xffffffffu;
        int less = 0, same = 0;
#pragma unroll 4
        for (int j = 0; j < cnt; j += 4) {  // the rest of the last four is the largest key
            const uint4 o = *reinterpret_cast<const uint4*>(S.cand + j);
            const uint32_t e[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                less += e[q] < k;
                same += e[q] == k;
                more = min(more, e[q] > k ? e[q] : 0xffffffffu);
            }
        }
        if (less <= r && r < less + same) {  // several equal candidates write the same
            S.key = kmin + k;
            S.next = r + 1 < less + same ? kmin + k : more != 0xffffffffu ? kmin + more : above;
        }
    }
    __syncthreads();
    return Ranked{S.key, S.next};
}

// The move of the greedy walk at cell (x, y) (main_conv_ff.py:35-62), on the map with a row and a column of zeros
// beyond its end.
__device__ __forceinline__ void walk_move(const float* __restrict__ pooled, int nb, int& x, int& y) {
    auto at = [&](int xx, int yy) -> float { return (xx < nb && yy < nb) ? pooled[xx * nb + yy] : 0.f; };
    const float Dn = at(x + 1, y), Rt = at(x, y + 1), Dg = at(x + 1, y + 1);
    const bool down = Dn > Rt && Dn > Dg, right = !(Dn > Rt) && Rt > Dg;
    if (!right) ++x;
    if (!down) ++y;
}

// torch.quantile's rank arithmetic and lerp, every step rounded to fp32 (no fused multiply-add).
__device__ __forceinline__ float quantile_rank(float q, int N, int& lo, int& hi) {
#pragma clang fp contract(off)
    const float r = q * (float)(N - 1);
    lo = (int)floorf(r);
    hi = (int)ceilf(r);
    return r - (float)lo;
}
__device__ __forceinline__ float lerp_as_torch(float a, float b, float w) {
#pragma clang fp contract(off)
    const float diff = b - a;
    return w < 0.5f ? a + w * diff : b - diff * (1.0f - w);
}

// One work-group per map.  Block grids up to JUMP_NB x JUMP_NB: what a walker does at a cell depends on the cell alone,
// so every cell's move goes into a table in LDS, the table is squared twice, and four threads take a walker's path
// between them, each every fourth cell of it -- a quarter of up to 2 nb dependent look-ups of one word instead of that
// many of three, with their comparisons.  (Squaring until the whole path is covered was measured: every squaring is a
// pass over all cells, seven of them took longer than the walk they saved.)  Larger grids walk the map itself.
// Four maps, 64 x 64 blocks: 40.5 -> 12.1 us.
constexpr int JUMP_NB = 128;  // LDS at the limit: pooled 64 KB, two move tables 64 KB, marks 16 KB, selection 11 KB
constexpr int MOVE_MARKS = 0x8000;  // flag of a table entry: the cell's value passes the threshold (cells need 15 bits)
__global__ __launch_bounds__(WALK_THREADS) void threshold_walk_kernel(const float* __restrict__ pooled_all,
                                                                      float* __restrict__ mat_all,
                                                                      float* __restrict__ thresh_out, int nb, int mode,
                                                                      float q, int topk, int replicas,
                                                                      size_t replica_stride) {
    __shared__ int s_cnt;
    __shared__ uint32_t s_min;
    __shared__ __attribute__((aligned(16))) SelectSpace sel;
    extern __shared__ __attribute__((aligned(16))) float s_pooled[];  // N floats (N <= POOLED_LDS), then tables and marks
    const int map = blockIdx.x, N = nb * nb;
    const float* pooled = pooled_all + (size_t)map * N;
    float* mat = mat_all + (size_t)map * N;
    const bool jump = mode == SPION_PATTERN_FLOOD && nb <= JUMP_NB;
    unsigned short* move = reinterpret_cast<unsigned short*>(s_pooled + N);
    unsigned short* move2 = move + N + 1;
    unsigned char* marks = reinterpret_cast<unsigned char*>(move2 + N + 1);

    if (!jump)
        for (int i = threadIdx.x; i < N; i += blockDim.x) mat[i] = 0.f;
    if (N <= POOLED_LDS) {
        // the select passes and the walkers' dependent neighbour reads then stay in LDS
        for_elements(pooled, N, [&](float x, int i) { s_pooled[i] = x; });
        __syncthreads();
        pooled = s_pooled;
    }

    if (mode == SPION_PATTERN_FLOOD) {
        // torch.quantile, linear interpolation, every step in fp32 (main_conv_ff.py:268)
        int lo, hi;
        const float wgt = quantile_rank(q, N, lo, hi);
        const Ranked k = range_select(pooled, N, lo, sel);
        const float a = key_float(k.key);
        const float b = hi == lo ? a : key_float(k.next);  // sorted[hi]
        const float thresh = lerp_as_torch(a, b, wgt);
        if (threadIdx.x == 0 && thresh_out) thresh_out[map] = thresh;

        // walker k < nb starts at (0, k), walker nb + k at (k, 0)  (main_conv_ff.py:271-274); the cell moved to is
        // marked when its value exceeds the threshold, and binarised with ff_mat > 0
        if (jump) {
            const int dx = WALK_THREADS / nb, dy = WALK_THREADS % nb;
            int x = threadIdx.x / nb, y = threadIdx.x % nb;
            for (int i = threadIdx.x; i <= N; i += WALK_THREADS) {
                int nx = x, ny = y, e = N;  // N: beyond the grid, where a walker stays
                if (i < N) {
                    walk_move(pooled, nb, nx, ny);
                    if (nx < nb && ny < nb) e = nx * nb + ny;
                    if (pooled[i] > thresh && pooled[i] > 0.f) e |= MOVE_MARKS;
                }
                move[i] = (unsigned short)e;
                marks[i] = 0;
                x += dx;
                y += dy;
                if (y >= nb) {
                    y -= nb;
                    ++x;
                }
            }
            __syncthreads();
            auto square = [&](const unsigned short* from, unsigned short* to) {
                for (int i0 = threadIdx.x; i0 <= N; i0 += 4 * WALK_THREADS) {
                    int e[4], m[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c) e[c] = from[min(i0 + c * WALK_THREADS, N)];
#pragma unroll
                    for (int c = 0; c < 4; ++c) m[c] = from[e[c] & ~MOVE_MARKS];
#pragma unroll
                    for (int c = 0; c < 4; ++c)  // past the end: the last entry once more
                        to[min(i0 + c * WALK_THREADS, N)] = (unsigned short)((e[c] & MOVE_MARKS) | (m[c] & ~MOVE_MARKS));
                }
                __syncthreads();
            };
            square(move, move2);
            // threads 4w .. 4w + 3 share walker w: cells after 0, 1, 2 and 3 moves, then four moves at a time
            const int walker = threadIdx.x >> 2, phase = threadIdx.x & 3;  // 2 nb <= WALK_THREADS / 4
            const bool walks = walker < 2 * nb;
            int at = walker < nb ? walker : (walker - nb) * nb, arrived = phase != 0;
            if (!walks) at = N;
            if (phase & 1) at = move[at] & ~MOVE_MARKS;
            if (phase & 2) at = move2[at] & ~MOVE_MARKS;
            __syncthreads();  // the table of single moves makes room for that of four
            square(move2, move);
            while (at != N) {
                const int e = move[at];
                if (arrived && (e & MOVE_MARKS)) marks[at] = 1;
                arrived = 1;
                at = e & ~MOVE_MARKS;
            }
            __syncthreads();
            const bool fours = N % 4 == 0 && reinterpret_cast<size_t>(mat_all) % 16 == 0;
            for (int i0 = 4 * threadIdx.x; i0 < N; i0 += 4 * WALK_THREADS) {
                float o[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int i = min(i0 + c, N);
                    o[c] = (marks[i] || i % (nb + 1) == 0) ? 1.f : 0.f;  // the diagonal too (main_conv_ff.py:277-278)
                }
                for (int rep = 0; rep < replicas; ++rep) {
                    float* m = mat + rep * replica_stride + i0;
                    if (fours) {
                        *reinterpret_cast<float4*>(m) = make_float4(o[0], o[1], o[2], o[3]);
                    } else {
                        for (int c = 0; c < 4 && i0 + c < N; ++c) m[c] = o[c];
                    }
                }
            }
            return;
        }
        __syncthreads();  // mat is zeroed for everyone
        for (int wk = threadIdx.x; wk < 2 * nb; wk += blockDim.x) {
            int x = wk < nb ? 0 : wk - nb, y = wk < nb ? wk : 0;
            for (walk_move(pooled, nb, x, y); x < nb && y < nb; walk_move(pooled, nb, x, y)) {
                const float val = pooled[x * nb + y];
                if (val > thresh && val > 0.f) mat[x * nb + y] = 1.f;
            }
        }
    } else {
        // the topk largest pooled blocks (main_conv.py:246-249); ties at the boundary: lower index first
        if (threadIdx.x == 0 && thresh_out) thresh_out[map] = 0.f;
        if (topk > 0) {
            const int k = min(topk, N);
            const uint32_t kk = range_select(pooled, N, N - k, sel).key;  // k-th largest
            if (threadIdx.x == 0) s_cnt = 0;
            __syncthreads();
            if (threadIdx.x == 0) s_min = 0u;  // number of blocks equal to the k-th largest
            __syncthreads();
            int c = 0, ties = 0;
            for (int i = threadIdx.x; i < N; i += blockDim.x) {
                const uint32_t key = float_key(pooled[i]);
                if (key > kk) {
                    mat[i] = 1.f;
                    ++c;
                } else if (key == kk) {
                    ++ties;
                }
            }
            atomicAdd(&s_cnt, c);
            atomicAdd(&s_min, (uint32_t)ties);
            __syncthreads();
            const int need = k - s_cnt;
            if (need >= (int)s_min) {  // the usual case (one such block): every tie is selected
                for (int i = threadIdx.x; i < N; i += blockDim.x)
                    if (float_key(pooled[i]) == kk) mat[i] = 1.f;
            } else if (threadIdx.x == 0) {
                int left = need;
                for (int i = 0; i < N && left > 0; ++i)
                    if (float_key(pooled[i]) == kk) {
                        mat[i] = 1.f;
                        --left;
                    }
            }
            if (threadIdx.x == 0 && thresh_out) thresh_out[map] = key_float(kk);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nb; i += blockDim.x) mat[i * nb + i] = 1.f;  // main_conv_ff.py:277-278
    __syncthreads();
    for (int r = 1; r < replicas; ++r)
        for (int i = threadIdx.x; i < N; i += blockDim.x) mat[r * replica_stride + i] = mat[i];
}

static std::mutex g_ws_mutex;
static float* g_pool_ws = nullptr;
static size_t g_pool_ws_count = 0;

// Mean of the dense phase's probability maps over the batch, then over the heads
// (models/model_transformer.py:136-137: torch.mean(torch.mean(attn, dim=0), dim=0)), read once at HBM rate.
// A is [batch][heads][L][L]; KEY_MAJOR: the maps are stored keys x queries (what the dense kernels write, the
// reference's column-major map) and the mean is written queries x keys, transposed through LDS.
template <bool KEY_MAJOR>
__global__ __launch_bounds__(256) void score_map_mean_kernel(const float* __restrict__ A, int batch, int heads, int L,
                                                             float* __restrict__ Mean, float post) {
    __shared__ float tile[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
    const size_t map = (size_t)L * L;
    const float* a = A + (size_t)(r0 + ty) * L + c0 + tx;
    float hs[4] = {0.f, 0.f, 0.f, 0.f};
    for (int h = 0; h < heads; ++h) {
        float bs[4] = {0.f, 0.f, 0.f, 0.f};
        const float* ah = a + (size_t)h * map;
#pragma unroll 4
        for (int b = 0; b < batch; ++b) {  // 16 loads in flight per thread (measured: 32 are slower)
            const float* ab = ah + (size_t)b * heads * map;
#pragma unroll
            for (int j = 0; j < 4; ++j) bs[j] += __builtin_nontemporal_load(ab + (size_t)8 * j * L);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) hs[j] += bs[j] / (float)batch;
    }
    if (KEY_MAJOR) {
#pragma unroll
        for (int j = 0; j < 4; ++j) tile[ty + 8 * j][tx] = hs[j] / (float)heads * post;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 4; ++j) Mean[(size_t)(c0 + ty + 8 * j) * L + r0 + tx] = tile[tx][ty + 8 * j];
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) Mean[(size_t)(r0 + ty + 8 * j) * L + c0 + tx] = hs[j] / (float)heads * post;
    }
}

// The same sums, in the same order, on 16-byte aligned maps: a thread owns four neighbouring columns, MEAN_MAPS maps are requested
// together and the next ones before those are added, across the heads.  Memory bound; with 4-byte loads of four maps at a time a
// wavefront waited for every 64 bytes of a thread.  us, 4-byte loads / here: the eight partial maps that a forward of 32 and more heads
// of 1024 leaves 12.3 / 6.8, of 8 heads of 512 9.3 / 2.4, 32 maps of 1024^2 58.7 / 25.4 (d = 64, where the forward leaves the maps alone), eight of 2048^2
// 44.0 / 22.8 (5.9 TB/s).
constexpr int MEAN_MAPS = 8;
template <bool KEY_MAJOR>
__global__ __launch_bounds__(256) void score_map_mean_rows_kernel(const float* __restrict__ A, int batch, int heads, int L,
                                                                  float* __restrict__ Mean, float post) {
    __shared__ float tile[32][33];
    const int row = threadIdx.x >> 3, col = 4 * (threadIdx.x & 7);
    const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32, n = batch * heads;
    const size_t map = (size_t)L * L;
    const float* a = A + (size_t)(r0 + row) * L + c0 + col;
    int lb = 0, lh = 0;  // the map requested next: sample, head (the last one again past the end)
    auto request = [&](f32x4 (&v)[MEAN_MAPS]) {
#pragma unroll
        for (int u = 0; u < MEAN_MAPS; ++u) {
            v[u] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(a + ((size_t)lb * heads + lh) * map));
            if (lb + 1 < batch) {
                ++lb;
            } else if (lh + 1 < heads) {
                lb = 0;
                ++lh;
            }
        }
    };
    f32x4 v[MEAN_MAPS], w[MEAN_MAPS], hs = {0.f, 0.f, 0.f, 0.f}, bs = hs;
    request(v);
    int b = 0;
    for (int k = 0; k < n; k += MEAN_MAPS) {
        if (k + MEAN_MAPS < n) request(w);
#pragma unroll
        for (int u = 0; u < MEAN_MAPS; ++u) {
            if (k + u < n) {
                bs += v[u];
                if (++b == batch) {
                    hs += bs / (float)batch;
                    bs = (f32x4){0.f, 0.f, 0.f, 0.f};
                    b = 0;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < MEAN_MAPS; ++u) v[u] = w[u];
    }
    hs = hs / (float)heads * post;
    if (KEY_MAJOR) {
#pragma unroll
        for (int j = 0; j < 4; ++j) tile[row][col + j] = hs[j];
        __syncthreads();
        *reinterpret_cast<f32x4*>(Mean + (size_t)(c0 + row) * L + r0 + col) =
            (f32x4){tile[col][row], tile[col + 1][row], tile[col + 2][row], tile[col + 3][row]};
    } else {
        *reinterpret_cast<f32x4*>(Mean + (size_t)(r0 + row) * L + c0 + col) = hs;
    }
}

// post: factor applied to the result (1 for a plain mean; sums of several maps each are turned into the mean of all
// maps by batch / number of maps summed).
int score_map_mean(const float* Attn, int batch, int heads, int L, int key_major, float* Mean, hipStream_t stream,
                   float post) {
    if (!Attn || !Mean || batch <= 0 || heads <= 0 || L <= 0 || L % 32) {
        set_error("spion_score_map_mean: need Attn, Mean, batch > 0, heads > 0 and seq_len a positive multiple of 32 "
                  "(got %d, %d, %d)", batch, heads, L);
        return 1;
    }
    if (L / 32 > 65535) {
        set_error("spion_score_map_mean: seq_len %d too large", L);
        return 1;
    }
    const dim3 grid(L / 32, L / 32), block(256);
    if ((reinterpret_cast<uintptr_t>(Attn) | reinterpret_cast<uintptr_t>(Mean)) % 16 == 0 && (long long)batch * heads <= INT_MAX - MEAN_MAPS) {
        if (key_major)
            hipLaunchKernelGGL(score_map_mean_rows_kernel<true>, grid, block, 0, stream, Attn, batch, heads, L, Mean, post);
        else
            hipLaunchKernelGGL(score_map_mean_rows_kernel<false>, grid, block, 0, stream, Attn, batch, heads, L, Mean, post);
    } else if (key_major)
        hipLaunchKernelGGL(score_map_mean_kernel<true>, grid, block, 0, stream, Attn, batch, heads, L, Mean, post);
    else
        hipLaunchKernelGGL(score_map_mean_kernel<false>, grid, block, 0, stream, Attn, batch, heads, L, Mean, post);
    return SPION_HIP_OK(hipGetLastError()) ? 0 : 1;
}

// -------------------------------------------------------------------------------------------------
// Dense-to-sparse transition test on the device (main_conv_ff.py:211-242).  After every evaluation the averaged
// score map of each layer is compared with the map kept from an earlier evaluation; the Frobenius distance of the
// two is compared with the previous distance, and once it changed by less than `percent` per cent (after
// truncation to an integer) in every layer the pattern counts as settled.  All state lives in device memory:
//   Prev  [layers][n]  the kept maps;
//   State [2*layers+3] floats: before_distance per layer, change in per cent per layer, then stage
//         (0 = no map kept yet, 1 = a map but no distance yet, 2 = map and distance), the transition flag and a
//         scratch word (whether this call replaces the kept maps).
// The host reads State[2*layers+1] once per evaluation; nothing else comes back.
// -------------------------------------------------------------------------------------------------
constexpr int TRANS_BLOCK = 256;
__global__ __launch_bounds__(TRANS_BLOCK) void transition_partial_kernel(const float* __restrict__ Prev,
                                                                         const float* __restrict__ Cur, long long n,
                                                                         double* __restrict__ Partial) {
    __shared__ double red[TRANS_BLOCK];
    const int layer = blockIdx.y, nblk = gridDim.x;
    const float* a = Prev + (size_t)layer * n;
    const float* b = Cur + (size_t)layer * n;
    double s = 0.0;
    for (long long i = (long long)blockIdx.x * TRANS_BLOCK + threadIdx.x; i < n; i += (long long)nblk * TRANS_BLOCK) {
        const float dlt = a[i] - b[i];  // float difference, as torch computes it
        s += (double)dlt * (double)dlt;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = TRANS_BLOCK / 2; o > 0; o >>= 1) {  // fixed order: the result does not depend on timing
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) Partial[(size_t)layer * nblk + blockIdx.x] = red[0];
}

__global__ void transition_decide_kernel(const double* __restrict__ Partial, int nblk, int layers, int percent,
                                         float* __restrict__ State) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    float* before = State;
    float* diff = State + layers;
    float& stage = State[2 * layers];
    float& flag = State[2 * layers + 1];
    float& replace = State[2 * layers + 2];
    replace = 0.f;
    if (flag != 0.f) return;
    if (stage == 0.f) {  // first evaluation: keep the maps, nothing to compare with
        stage = 1.f;
        replace = 1.f;
        return;
    }
    int settled = 0;
    for (int l = 0; l < layers; ++l) {
        double s = 0.0;
        for (int k = 0; k < nblk; ++k) s += Partial[(size_t)l * nblk + k];
        const float dist = (float)sqrt(s);
        if (stage == 1.f) {  // second evaluation: the first distance; the kept maps stay
            before[l] = dist;
            diff[l] = 0.f;
        } else {
            // a previous distance of 0 (two identical maps in a row) gives inf or NaN here, where the
            // reference's int(diff) raises (main_conv_ff.py:228-233): such a layer counts as not settled
            const float dl = (fabsf(dist - before[l]) / before[l]) * 100.f;
            diff[l] = dl;
            before[l] = dist;
            if (isfinite(dl) && dl < 2.0e9f && (int)dl < percent) ++settled;
        }
    }
    if (stage == 1.f) {
        stage = 2.f;
        return;
    }
    if (settled == layers) flag = 1.f;
    else replace = 1.f;
}

__global__ __launch_bounds__(256) void transition_replace_kernel(float* __restrict__ Prev, const float* __restrict__ Cur,
                                                                 long long total, const float* __restrict__ State,
                                                                 int layers) {
    if (State[2 * layers + 2] == 0.f) return;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256)
        Prev[i] = Cur[i];
}

int transition_update(const float* Cur, float* Prev, int layers, long long n, float* State, double* Partial,
                      int partial_blocks, int percent, hipStream_t stream) {
    if (!Cur || !Prev || !State || !Partial || layers <= 0 || n <= 0 || partial_blocks <= 0 || layers > 65535) {
        set_error("spion_transition_update: bad arguments");
        return 1;
    }
    hipLaunchKernelGGL(transition_partial_kernel, dim3(partial_blocks, layers), dim3(TRANS_BLOCK), 0, stream, Prev, Cur,
                       n, Partial);
    hipLaunchKernelGGL(transition_decide_kernel, dim3(1), dim3(64), 0, stream, Partial, partial_blocks, layers, percent,
                       State);
    const long long total = n * layers;
    const int blocks = (int)std::min<long long>((total + 255) / 256, 2048);
    hipLaunchKernelGGL(transition_replace_kernel, dim3(blocks), dim3(256), 0, stream, Prev, Cur, total, State, layers);
    return SPION_HIP_OK(hipGetLastError()) ? 0 : 1;
}

int pattern_generate_maps(const float* const* Score, int n_maps, int L, int bs, int ksize, int mode, double param,
                          float* Mat, int replicas, float* Pooled, float* Thresh, hipStream_t stream) {
    if (!Score || !Mat) {
        set_error("spion_pattern_generate: null Score or Mat");
        return 1;
    }
    if (n_maps <= 0 || L <= 0 || bs <= 0 || L % bs || replicas <= 0) {
        set_error("spion_pattern_generate: need n_maps > 0, replicas > 0 and seq_len a positive multiple of block_size "
                  "(got %d, %d, %d, %d)", n_maps, replicas, L, bs);
        return 1;
    }
    for (int m = 0; m < n_maps; ++m)
        if (!Score[m]) {
            set_error("spion_pattern_generate: null Score or Mat");
            return 1;
        }
    if (ksize < 0 || (ksize && ksize % 2 == 0)) {
        set_error("spion_pattern_generate: conv_ksize must be 0 or odd (got %d)", ksize);
        return 1;
    }
    if (mode != SPION_PATTERN_FLOOD && mode != SPION_PATTERN_TOPK) {
        set_error("spion_pattern_generate: unknown mode %d", mode);
        return 1;
    }
    const int nb = L / bs;
    if (nb > 16384 || n_maps > 65535 || nb > 65535) {
        set_error("spion_pattern_generate: block grid %d or map count %d too large", nb, n_maps);
        return 1;
    }
    if (mode == SPION_PATTERN_FLOOD && !(param >= 0.0 && param <= 1.0)) {
        set_error("spion_pattern_generate: quantile %g outside [0, 1]", param);
        return 1;
    }
    // Without a caller's Pooled buffer the pooled maps go to one buffer the library owns: such calls are
    // serialised, and the buffer is reused by the next one as soon as this one has been enqueued -- callers that
    // work on several streams at once pass their own Pooled.
    float* pooled = Pooled;
    std::unique_lock<std::mutex> lock(g_ws_mutex, std::defer_lock);
    if (!pooled) {
        lock.lock();
        const size_t need = (size_t)n_maps * nb * nb;
        if (g_pool_ws_count < need) {
            if (g_pool_ws) (void)hipFree(g_pool_ws);
            g_pool_ws = nullptr;
            g_pool_ws_count = 0;
            if (!SPION_HIP_OK(hipMalloc((void**)&g_pool_ws, sizeof(float) * need))) return 1;
            g_pool_ws_count = need;
        }
        pooled = g_pool_ws;
    }
    const int hk = ksize / 2;
    // blocks per work-group of the streaming kernel (0: block size too small for it, or too wide)
    const int gb = bs >= 2 * hk && bs + 2 * hk <= CP_COLS ? (CP_COLS - 2 * hk) / bs : 0;
    for (int m0 = 0; m0 < n_maps; m0 += MAPS_PER_LAUNCH) {
        const int n = std::min(MAPS_PER_LAUNCH, n_maps - m0);
        ScoreMaps maps{};
        for (int m = 0; m < n; ++m) maps.p[m] = Score[m0 + m];
        float* out = pooled + (size_t)m0 * nb * nb;
        if (gb > 0) {
#define SPION_LAUNCH(BS, RG)                                                                                         \
    hipLaunchKernelGGL((conv_pool_cols_kernel<BS, RG>), dim3(groups), dim3(CP_COLS * RG), 0, stream, maps, out, L, bs, nb, hk, gb)
            const int groups = (nb + gb - 1) / gb * nb * n;
            if (bs == 32 && hk <= 16 && groups >= 8 * device_cus()) SPION_LAUNCH(32, 1);
            else if (bs == 32 && hk <= 16) SPION_LAUNCH(32, 2);
            else if (bs == 64 && hk <= 16) SPION_LAUNCH(64, 2);
            else SPION_LAUNCH(0, 2);
#undef SPION_LAUNCH
        } else
            hipLaunchKernelGGL(conv_pool_kernel, dim3(nb, nb, n), dim3(POOL_THREADS), 0, stream, maps, out, L, bs, nb,
                               hk);
    }
    if (!check_launch("conv_pool_kernel")) return 1;
    int topk = 0;
    if (mode == SPION_PATTERN_TOPK) topk = (int)((double)(nb * nb) * param - (double)nb);  // main_conv.py:247
    const size_t cells = (size_t)nb * nb;
    size_t walk_lds = cells <= (size_t)POOLED_LDS ? sizeof(float) * cells : 0;
    if (mode == SPION_PATTERN_FLOOD && nb <= JUMP_NB) walk_lds += 5 * (cells + 1);  // two 16-bit tables and the flags
    if (walk_lds > 32 * 1024) {  // beyond what a launch may ask for without saying so first
        static std::once_flag once;
        static hipError_t attr_err = hipSuccess;
        std::call_once(once, [] {
            constexpr size_t jump = sizeof(float) * JUMP_NB * JUMP_NB + 5 * (JUMP_NB * JUMP_NB + 1);
            attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(threshold_walk_kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)std::max(sizeof(float) * POOLED_LDS, jump));
        });
        if (!SPION_HIP_OK(attr_err)) return 1;
    }
    hipLaunchKernelGGL(threshold_walk_kernel, dim3(n_maps), dim3(WALK_THREADS), walk_lds, stream, pooled, Mat, Thresh, nb,
                       mode, (float)param, topk, replicas, (size_t)n_maps * cells);
    if (!check_launch("threshold_walk_kernel")) return 1;
    return 0;
}

// The same for maps that follow one another in memory.
int pattern_generate(const float* Score, int n_maps, int L, int bs, int ksize, int mode, double param, float* Mat,
                     float* Pooled, float* Thresh, hipStream_t stream) {
    if (!Score || n_maps <= 0 || L <= 0)
        return pattern_generate_maps(nullptr, n_maps, L, bs, ksize, mode, param, Mat, 1, Pooled, Thresh, stream);
    std::vector<const float*> maps(n_maps);
    for (int m = 0; m < n_maps; ++m) maps[m] = Score + (size_t)m * L * L;
    return pattern_generate_maps(maps.data(), n_maps, L, bs, ksize, mode, param, Mat, 1, Pooled, Thresh, stream);
}

}  // namespace spion
