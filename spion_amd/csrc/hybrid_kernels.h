// Hybrid kernels for element-sparse patterns (d = 32): the well-filled aligned 32 x 32 tiles of the pattern (the
// local window of a "window + random columns" pattern, say) run as dense MFMA tiles with a bit mask for the entries
// that are absent, the remaining entries by ranges of rows in LDS (remainder_kernels.h) or as per-row gathers; the softmax
// statistics are merged across the two parts, and P stays in CSR order exactly as the reference's kernels leave it (models/block_attn_mask.cu:88-140):
// a tile's entries of one row are consecutive in that row's CSR run, so `first position + number of present
// columns to the left` addresses them.
//
// Per pattern entry the gather path costs about as much machine time as 1/80 of a 32 x 32 MFMA tile, so a tile
// with more than ~10 % of its entries present is cheaper dense.
//
// The two parts run as separate launches, each at the occupancy that suits it: the tile kernels (one wavefront per
// strip of 32 rows or columns when strips hold few dense tiles, else a work-group of four wavefronts, wavefront w
// taking the strip's dense tiles w, w+4, ...) and the remainder's: work-groups of sixteen wavefronts that walk ranges
// of the sequence in LDS, or where that costs more (rem_by_ranges, sparse_attn.hip) gathers, one wavefront per row or column,
// sixteen per CU, because they are bound by the number of requests in flight.
// Forward: remainder logits and their row statistics (by ranges: the remainder's share of O as well), then the tiles (which
// merge the statistics, fix the row's maximum and denominator and rescale and add that share), then the remainder's
// probabilities (gathered: and its share of O).  Backward: tile part then remainder
// part of the row pass, the same for the column pass; the remainder kernels add to what the tile kernels wrote
// (each row or column has exactly one writer per launch).
#pragma once
#include <type_traits>
#include "gather_ops.h"
#include "remainder_kernels.h"

namespace spion {

// The analysed pattern as the kernels see it (device pointers, shared by all heads).
struct HybIndex {
    // dense tiles, by block row: tiles t_rp[I] .. t_rp[I+1]-1 of block row I; per tile its block column and, per
    // row of the tile, the position of the row's first entry inside a head's P and the 32-bit set of present columns
    const int* t_rp;
    const int* t_col;
    const int* t_pos;        // [tiles][32]
    const unsigned* t_bits;  // [tiles][32]
    // the same tiles by block column: tile ids t_ct[t_cp[J]] .. of block column J and their block rows t_ci
    const int* t_cp;
    const int* t_ct;
    const int* t_ci;
    // remainder entries in CSR form (r_off [L+1], columns, positions inside a head's P) and in CSC form (c_ptr
    // [L+1], rows ascending within a column, index of the entry in the CSR list); nr entries per head
    const int* r_off;
    const int* r_col;
    const int* r_pos;
    const int* c_ptr;
    const int* c_row;
    const int* c_src;
    int nr;
    int nt;  // dense tiles in all
};

// Tile kernels come in two shapes: one wavefront per strip (strips of up to HYB_MAXT1 dense tiles: the window
// patterns this path is for have about five; the wavefront walks them one after the other, nothing is shared and
// nothing waits at a barrier) and four wavefronts per strip (up to 4 * HYB_MAXT4 dense tiles).  With a handful of
// tiles per strip these launches live on latency, and a strip handled by one wavefront costs a quarter of the
// wavefront start-ups, index look-ups and final reductions.
constexpr int HYB_MAXT1 = 6;    // dense tiles whose logits a single wavefront keeps in registers (forward)
constexpr int HYB_MAXT4 = 4;    // the same per wavefront when four share a strip
constexpr int HYB_MAX_ROW_TILES = 4 * HYB_MAXT4;
constexpr int HYB_GWAVES = 4;    // wavefronts (rows / columns) per work-group of the gather kernels
// two wavefronts per SIMD, each with the next tile's operands in flight while it works on one
#define SPION_HYB_KERNEL(W) __global__ __launch_bounds__(64 * (W)) __attribute__((amdgpu_waves_per_eu(2, 2)))

// One value per tile row, held by lane li (and 32 + li) for row li, to the 16 rows acc_row(q, h), q = 0..15, a lane
// works on: through 32 words of the wavefront's own LDS space.
__device__ __forceinline__ void hyb_rows_from_lanes(int* xs, int l, int h, int v, int (&out)[16]) {
    xs[l] = v;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int4 p = *reinterpret_cast<const int4*>(xs + 8 * g + 4 * h);
        out[4 * g + 0] = p.x, out[4 * g + 1] = p.y, out[4 * g + 2] = p.z, out[4 * g + 3] = p.w;
    }
}
// The tile of P in the col-owner layout (lane li = column of the tile, register q = row acc_row(q, h)); absent
// entries read as 0 (their offset lies past the end of the buffer).  A tile row's entries are consecutive in memory:
// every instruction touches one run per half-wave.
__device__ __forceinline__ void hyb_load_p_cols(rsrc_t rP, const int (&pos)[16], const unsigned (&bits)[16], int li,
                                                float (&pc)[16]) {
    const unsigned below = (1u << li) - 1u;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const bool on = (bits[q] >> li) & 1u;
        pc[q] = ld1(rP, on ? 4 * (pos[q] + __popc(bits[q] & below)) : -1, 0);
    }
}
__device__ __forceinline__ void hyb_store_p_cols(float* __restrict__ Ph, const int (&pos)[16],
                                                 const int (&bits)[16], int li, const float (&pc)[16]) {
    const unsigned below = (1u << li) - 1u;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const unsigned b = (unsigned)bits[q];
        if ((b >> li) & 1u) Ph[pos[q] + __popc(b & below)] = pc[q];
    }
}

// Sum of the wavefronts' 32 x 32 accumulators (rows acc_row(r, h) of the strip, columns li) times `factor`, in a
// fixed order, to rows of stride ld.  `lds` (WAVES * 1024 floats, unused for one wavefront) may alias tile space no wavefront uses any
// more: the caller has a barrier between that use and this call.
// ADD: plus add[r] (the same in every wavefront); copy (optional): the result once more, rows of 32.
template <int WAVES, bool ADD = false>
__device__ __forceinline__ void hyb_reduce_store(const f32x16& acc, float factor, float* __restrict__ out, int ld,
                                                 int row0, int w, int li, int h, float* __restrict__ lds,
                                                 const float* add = nullptr, float* __restrict__ copy = nullptr) {
    const int l = h * 32 + li;
    if constexpr (WAVES > 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) lds[(w * 16 + r) * 64 + l] = acc[r];
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        if (WAVES > 1 && (r % WAVES) != w) continue;
        float s = acc[r];
        if constexpr (WAVES > 1) {
            s = 0.f;
#pragma unroll
            for (int ww = 0; ww < WAVES; ++ww) s += lds[(ww * 16 + r) * 64 + l];
        }
        s *= factor;
        if constexpr (ADD) s += add[r];
        out[(size_t)(row0 + acc_row(r, h)) * ld + li] = s;
        if constexpr (ADD)
            if (copy) copy[(size_t)(row0 + acc_row(r, h)) * 32 + li] = s;
    }
}

// acc += W . X of one tile, its 32 terms summed by themselves first: the sums over a strip's tiles are shorter chains.
__device__ __forceinline__ void hyb_mma_add(const float (&w)[16], const float (&x)[1][16], f32x16 (&acc)[1]) {
    f32x16 part[1] = {splat16(0.f)};
    mma_b<32>(w, x, part);
    acc[0] += part[0];
}

// A matrix product multiplies what a tile lacks by zero: an infinity or NaN of one row or column of an operand reaches all of the
// tile, while an entry of the pattern should take it to its own row and column only.  The kernels look at their sums at the end
// (sixteen instructions a strip) and form those that are not finite again, entry by entry.
__device__ __forceinline__ bool hyb_not_finite(const f32x16& acc) {
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) s = fmaf(acc[r], 0.f, s);
    return __any(s != s);
}
// What the wavefront itself (or an earlier kernel) stored: past the caches of the CU.
__device__ __forceinline__ float hyb_stored(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The sum over a half-wave, in all of its lanes.
__device__ __forceinline__ float hyb_half_sum(float x) {
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}
// Rows of a strip from the entries of n tiles: sums of weight(row of the strip, column, position in P) X[column], a half-wave to a
// row and a lane to a feature, back in the layout of the accumulators.  tile(u): the u-th tile; T: the wavefront's own LDS.
template <class Tile, class Weight>
__device__ __forceinline__ void hyb_rows_by_entries(float* T, int l, int n, const HybIndex& ix, rsrc_t X, int ld, Tile tile,
                                                    Weight weight, f32x16& acc) {
    l = second_walk(l);
    const int h = l >> 5, li = l & 31;
#pragma unroll 1
    for (int rr = 0; rr < 16; ++rr) {
        const int row = 2 * rr + h;
        const auto entry_weight = weight(row);
        float s = 0.f;
#pragma unroll 1
        for (int u = 0; u < n; ++u) {
            const int t = tile(u), col0 = ix.t_col[t] * 32;
            int pos = ix.t_pos[(size_t)t * 32 + row];
            unsigned bits = ix.t_bits[(size_t)t * 32 + row];
            while (bits) {
                const int col = col0 + __builtin_ctz(bits);
                bits &= bits - 1;
                s = fmaf(entry_weight(col, pos++), ld1(X, (col * ld + li) * 4, 0), s);
            }
        }
        T[row * TS + li] = s;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = T[acc_row(r, h) * TS + li];
}

// A tile's index: block column (or row), and position and present-column set of tile row li (lane li and lane 32 + li hold the
// same).
struct HybTile {
    int pos_l, blk;
    unsigned bits_l;
};
__device__ __forceinline__ void hyb_fetch_index(const HybIndex& ix, int t, int li, HybTile& x) {
    x.pos_l = ix.t_pos[(size_t)t * 32 + li];
    x.bits_l = ix.t_bits[(size_t)t * 32 + li];
}
// An element of the index that is the same for the wavefront, as a scalar load: the vector loads in flight are counted.
__device__ __forceinline__ int hyb_scalar(const int* p, int i) {
    return __builtin_amdgcn_readfirstlane(
        reinterpret_cast<const __attribute__((address_space(4))) int*>(reinterpret_cast<uintptr_t>(p))[i]);
}
// us per launch, operand tiles in two register sets and fp32 chains (row pass; in the column pass the product dO.V^T was split) /
// so, with all products split: 32 x 2 heads of 4096, 5 tiles a strip, 97 / 90 and 101 / 86; 2-norm errors against float64 of dQ
// 1.91e-7 / 1.57e-7, dK 1.76e-7 / 1.60e-7, dV 1.57e-7 / 1.41e-7.  (The index of a strip's first tile with its own rows: no
// difference; three wavefronts per SIMD spill 74 registers in the row pass.)
// The walk of the backward kernels over n > 0 tiles: while tile i is worked on, its operand tiles' places in LDS, read by then,
// take those of tile i + 1 (load: buffer loads into LDS), the registers of its P take the gathered entries of tile i + 1, and
// the index of tile i + 2 is on its way.  fetch(x, i): the index of tile i (two loads, past the end those of the last one);
// x: the first tile's.  work(p, next): reads tile i's operands out of LDS, calls next() and forms its products.
template <class Fetch, class Load, class Work>
__device__ __forceinline__ void hyb_walk(int n, HybTile x, int* X, int l, int h, int li, rsrc_t rP, Fetch fetch, Load load,
                                         Work work) {
    HybTile y;
    float p[16];
    auto request = [&](const HybTile& t) {
        int pos[16], bits[16];
        unsigned set[16];
        hyb_rows_from_lanes(X, l, h, t.pos_l, pos);
        hyb_rows_from_lanes(X + 64, l, h, (int)t.bits_l, bits);
#pragma unroll
        for (int q = 0; q < 16; ++q) set[q] = (unsigned)bits[q];
        load(__builtin_amdgcn_readfirstlane(t.blk));
        hyb_load_p_cols(rP, pos, set, li, p);
    };
    auto step = [&](int i, const HybTile& now, HybTile& then) {
        fetch(then, i + 2);
        wait_vm<2>();  // all but that index
        __builtin_amdgcn_sched_barrier(0);
        work(p, [&] {
            request(now);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    request(x);
    fetch(x, 1);
    int i = 0;
    for (; i + 1 < n; i += 2) {
        step(i, x, y);
        step(i + 1, y, x);
    }
    wait_vm<0>();
    if (i < n) work(p, [] {});
}

// =================================================================================================
// gather helpers (one wavefront per row / column of the remainder)
// =================================================================================================
// The gather primitives (gather_ops.h) with eight lanes to a 32-float row.
__device__ __forceinline__ int hyb_entry_of_lane(int lane) { return gather_entry_of_lane<8>(lane); }

// Start (in floats) and row stride of head bh in a tensor group: contiguous [NB][L][32] heads (ST = false, compile-time
// figures) or [B][H][L][32] views given by a layout.
template <bool ST>
__device__ __forceinline__ void hyb_head(const HeadLayout& y, int H, int bh, int L, size_t& base, int& ld) {
    size_t bytes;
    head_slice<ST, 32>(y, H, bh, L, base, ld, bytes);
}

__device__ __forceinline__ float hyb_gather_dot(const f32x4 a4, const float* __restrict__ X, int ld, int row_l,
                                                int nk, int lane) {
    return gather_dot<8>(a4, X, ld, row_l, nk, lane);
}
typedef GatherRowAcc<8> HybRowAcc;
#define SPION_HYB_GATHER_KERNEL __global__ __launch_bounds__(64 * HYB_GWAVES) __attribute__((amdgpu_waves_per_eu(6, 8)))

// -------------------------------------------------------------------------------------------------
// Forward, step 1: raw logits (log2 domain) of the remainder entries into P, and per row their maximum and the sum
// of their exponentials relative to it: Stats[bh][row] = {m, z} ({HYB_ABSENT, 0} for a row without remainder).
// -------------------------------------------------------------------------------------------------
template <bool MASK, bool ST>
SPION_HYB_GATHER_KERNEL void hyb_rem_logits_kernel(const float* __restrict__ Q, const float* __restrict__ K,
                                                   KeyTerms keys, float* __restrict__ Raw,
                                                   float2* __restrict__ Stats, HybIndex ix, int L, int NB,
                                                   float scale, Layouts ly) {
    const int lane = threadIdx.x & 63, ent = hyb_entry_of_lane(lane);
    const long long wrow = (long long)xcd_remap((int)blockIdx.x, (int)gridDim.x) * HYB_GWAVES + wave_index();
    if (wrow >= (long long)NB * L) return;
    const int bh = (int)(wrow / L), row = (int)(wrow % L);
    const int r0 = ix.r_off[row], rc = ix.r_off[row + 1] - r0;
    size_t ib;
    int ild;
    hyb_head<ST>(ly.in, ly.H, bh, L, ib, ild);
    float* raw = Raw + (size_t)bh * ix.nr + r0;  // this row's logits, in the order of the remainder's CSR list
    const float c2 = scale * LOG2E;
    f32x4 q4 = reinterpret_cast<const f32x4*>(Q + ib + (size_t)row * ild)[lane & 7];
    q4 *= c2;
    // the logits of the first chunks stay in registers; longer rows go back to what they stored in P
    constexpr int KEEP = 2;
    float vk[KEEP];
    float mx = HYB_ABSENT;
    for (int c0 = 0; c0 < rc; c0 += 64) {
        const int k = c0 + ent;
        const int col = k < rc ? ix.r_col[r0 + k] : 0;
        float v = hyb_gather_dot(q4, K + ib, ild, col, min(64, rc - c0), lane);
        if (k < rc) {
            if (MASK) v += fmaf(keys.row(bh, L)[col], keys.mul * LOG2E, keys.add * LOG2E);
            raw[k] = v;
            mx = fmaxf(mx, v);
        } else {
            v = HYB_ABSENT;
        }
#pragma unroll
        for (int c = 0; c < KEEP; ++c)
            if (c0 == 64 * c) vk[c] = v;
    }
    mx = wave_max(mx);
    float z = 0.f;
#pragma unroll
    for (int c = 0; c < KEEP; ++c)
        if (64 * c < rc) z += __builtin_amdgcn_exp2f(vk[c] - mx);
    for (int k = 64 * KEEP + lane; k < rc; k += 64) z += __builtin_amdgcn_exp2f(raw[k] - mx);
    z = wave_sum(z);
    if (lane == 0) Stats[(size_t)bh * L + row] = make_float2(mx, z);
}

// -------------------------------------------------------------------------------------------------
// Forward, step 2: the dense tiles of a strip.  Logits in the log2 domain as in tile_fwd_kernel; the row's
// maximum and denominator take in the remainder's statistics (Stats in: {m, z} of the remainder; out: {row
// maximum, 1 / denominator} for step 3).  Writes the tiles' probabilities to their CSR positions and O = P.V of the
// tile part (step 3 adds the remainder's share).
// -------------------------------------------------------------------------------------------------
// REM: the remainder went through rem_fwd_kernel: O holds its sums relative to its own maximum, which are rescaled and
// added (Oc, optional: second copy of O, contiguous heads).
template <bool MASK, int WAVES, int MAXT, bool ST, bool REM>
SPION_HYB_KERNEL(WAVES) void hyb_tile_fwd_kernel(const float* __restrict__ Q, const float* __restrict__ K,
                                          const float* __restrict__ V, KeyTerms keys,
                                          float* __restrict__ P, float* __restrict__ O, float* __restrict__ Oc,
                                          float2* __restrict__ Stats, const int* __restrict__ offs, HybIndex ix, int L,
                                          int nbr, int NB, int nnz, float scale, Layouts ly) {
    constexpr int D = 32, KH = 16;
    __shared__ float lds_m[WAVES][32], lds_z[WAVES][32];
    __shared__ __attribute__((aligned(16))) float lds_t[WAVES][64 * TS];  // two 32-row tiles per wavefront
    __shared__ __attribute__((aligned(16))) int lds_x[WAVES][128];
    float* lds = &lds_t[0][0];  // the final reduction reuses the tile space
    const int item = xcd_remap(blockIdx.x, nbr * NB);
    const int bh = item / nbr, I = item % nbr;
    const int w = wave_index(), l = threadIdx.x & 63, h = l >> 5, li = l & 31;
    size_t ib, ob, ibytes, obytes;
    int ild, old_;
    head_slice<ST, D>(ly.in, ly.H, bh, L, ib, ild, ibytes);
    head_slice<ST, D>(ly.out, ly.H, bh, L, ob, old_, obytes);
    const rsrc_t rQ = make_rsrc(Q + ib, ibytes), rK = make_rsrc(K + ib, ibytes), rV = make_rsrc(V + ib, ibytes);
    const rsrc_t rM = make_rsrc(MASK ? keys.row(bh, L) : nullptr, MASK ? (size_t)L * 4 : 0);
    const float kmul = keys.mul * LOG2E, kadd = keys.add * LOG2E;
    float* Ph = P + (size_t)bh * nnz;
    float* T = lds_t[w];
    float* Tx = T + 32 * TS;
    int* X = lds_x[w];
    const float c2 = scale * LOG2E;
    const int lin = lin_voff(l, ild), tile_bytes = 32 * ild * 4;

    auto load_q = [&](float (&q)[KH], int l) {
        ldr_rows<D>(rQ, ((l & 31) * ild + (l >> 5) * KH) * 4, I * tile_bytes, q);
#pragma unroll
        for (int s = 0; s < KH; ++s) q[s] *= c2;
    };
    float q[KH];
    load_q(q, l);
    const float2 rem = Stats[(size_t)bh * L + I * 32 + li];  // the remainder of row li

    // ---- index of this wavefront's tiles (positions past the end repeat the last one: valid, redundant) -----
    const int t0 = ix.t_rp[I], cnt = ix.t_rp[I + 1] - t0;
    const int nu = cnt > w ? (cnt - w + WAVES - 1) / WAVES : 0;
    int Js[MAXT], pos_l[MAXT];
    unsigned bits_l[MAXT];  // present columns / first position of tile row li
#pragma unroll
    for (int u = 0; u < MAXT; ++u) {
        const int t = min(t0 + w + min(u, max(nu, 1) - 1) * WAVES, ix.nt - 1);
        Js[u] = ix.t_col[t];
        pos_l[u] = ix.t_pos[(size_t)t * 32 + li];
        bits_l[u] = ix.t_bits[(size_t)t * 32 + li];
    }

    // ---- logits of the tiles, own maximum; the next tile of K is in flight while one is worked on --------
    float m, z;
    f32x16 S[MAXT];
    f32x4 raw[2][4];
    auto own_softmax = [&](const auto& qk, int l) {  // qk: the query operand, split or whole
    const int h = l >> 5, li = l & 31;
    const int lin = lin_voff(l, ild);
    m = MASK ? 0.f : -100.f * LOG2E;
    z = 0.f;
    float pj[2][16];
    ldr_tile_lin(rK, lin, Js[0] * tile_bytes, ild, raw[0]);
    if constexpr (MASK) ldr_4x4(rM, 16 * h, Js[0] * 128, pj[0]);
#pragma unroll
    for (int u = 0; u < MAXT; ++u) {
        if (u + 1 < MAXT) {
            ldr_tile_lin(rK, lin, Js[u + 1] * tile_bytes, ild, raw[(u + 1) & 1]);
            if constexpr (MASK) ldr_4x4(rM, 16 * h, Js[u + 1] * 128, pj[(u + 1) & 1]);
        } else {
            ldr_tile_lin(rV, lin, Js[0] * tile_bytes, ild, raw[(u + 1) & 1]);  // first tile of V for the last step
        }
        __builtin_amdgcn_sched_barrier(0);
        if (u < nu) {
            f32x16 init = splat16(0.f);
            if constexpr (MASK) {
#pragma unroll
                for (int r = 0; r < 16; ++r) init[r] = fmaf(pj[u & 1][r], kmul, kadd);
            }
            lds_put_lin(Tx, l, raw[u & 1]);
            float kf[KH];
            lds_get_feat32(Tx, li, h, kf);
            S[u] = mma_feat_init<D>(kf, qk, init);  // register = key acc_row(r, h), lane = query li
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (!((bits_l[u] >> acc_row(r, h)) & 1u)) S[u][r] = HYB_ABSENT;
            m = max16(S[u], m);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    m = fmaxf(m, __shfl_xor(m, 32, 64));
#pragma unroll
    for (int u = 0; u < MAXT; ++u) {
        if (u < nu) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float e = __builtin_amdgcn_exp2f(S[u][r] - m);
                S[u][r] = e;
                z += e;
            }
        }
    }
    };
    own_softmax(split3(q), l);
    if (split_failed(z)) {
        const int l2 = second_walk(l);
        load_q(q, l2);
        own_softmax(whole(q), l2);
    }
    const float m_own = m;
    z += __shfl_xor(z, 32, 64);

    // ---- merge: row maximum and denominator over the tiles of all wavefronts and the remainder ----
    float Mx = fmaxf(rem.x, m);
    float Z = rem.y * __builtin_amdgcn_exp2f(rem.x - Mx);
    if constexpr (WAVES > 1) {
        if (h == 0) {
            lds_m[w][li] = m;
            lds_z[w][li] = z;
        }
        __syncthreads();
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) Mx = fmaxf(Mx, lds_m[ww][li]);
        Z = rem.y * __builtin_amdgcn_exp2f(rem.x - Mx);
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) Z += lds_z[ww][li] * __builtin_amdgcn_exp2f(lds_m[ww][li] - Mx);
    } else {
        Z += z * __builtin_amdgcn_exp2f(m - Mx);
    }
    {
        const int row = I * 32 + li;
        const int n_i = offs[row + 1] - offs[row];
        Z += (float)(L - n_i) * __builtin_amdgcn_exp2f(-Mx);
    }
    const float zinv = 1.0f / Z;  // +inf denominator -> 0 -> P = 0, as in the reference
    const float rinv = __builtin_amdgcn_exp2f(m_own - Mx) * zinv;

    // ---- probabilities, O += P.V, P to its CSR positions; V of the next tile in flight ------------------
    f32x16 o[1] = {splat16(0.f)};
#pragma unroll
    for (int u = 0; u < MAXT; ++u) {
        constexpr int FIRST = MAXT & 1;  // the set the first tile of V went to
        if (u + 1 < MAXT) ldr_tile_lin(rV, lin, Js[u + 1] * tile_bytes, ild, raw[(FIRST + u + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        if (u < nu) {
            lds_put_lin(Tx, l, raw[(FIRST + u) & 1]);
            float p[16], vb[1][16], pc[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) p[r] = S[u][r] * rinv;
            lds_put_rows(T, li, h, p);
            lds_get_cols(Tx, li, h, vb[0]);
            lds_get_cols(T, li, h, pc);
            hyb_mma_add(p, vb, o);
            int pos[16], bits[16];
            hyb_rows_from_lanes(X, l, h, pos_l[u], pos);
            hyb_rows_from_lanes(X + 64, l, h, (int)bits_l[u], bits);
            hyb_store_p_cols(Ph, pos, bits, li, pc);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if (hyb_not_finite(o[0])) {
        __threadfence();  // P of these tiles, just stored
        hyb_rows_by_entries(
            T, l, nu, ix, rV, ild, [&](int u) { return t0 + w + u * WAVES; },
            [&](int) { return [&](int, int pos) { return hyb_stored(Ph + pos); }; }, o[0]);
    }
    float add[16];
    if constexpr (REM) {
        const float share = __builtin_amdgcn_exp2f(rem.x - Mx) * zinv;  // of the remainder's own sums
        int sh[16];
        hyb_rows_from_lanes(X, l, h, __float_as_int(share), sh);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if (WAVES > 1 && (r % WAVES) != w) continue;  // the registers this wavefront stores
            add[r] = O[ob + (size_t)(I * 32 + acc_row(r, h)) * old_ + li] * __int_as_float(sh[r]);
        }
    }
    if constexpr (WAVES > 1) __syncthreads();
    // every wavefront has consumed the remainder's statistics by now: replace them by the row's final ones
    if (w == 0 && h == 0) Stats[(size_t)bh * L + I * 32 + li] = make_float2(Mx, zinv);
    hyb_reduce_store<WAVES, REM>(o[0], 1.0f, O + ob, old_, I * 32, w, li, h, lds, add,
                                 REM && Oc ? Oc + (size_t)bh * L * D : nullptr);
}

// -------------------------------------------------------------------------------------------------
// Forward, step 3: probabilities of the remainder entries from their raw logits and the row's {maximum,
// 1 / denominator}; their share of O is added to what step 2 wrote.  Ocache (optional): second copy of O.
// -------------------------------------------------------------------------------------------------
template <bool ST>
SPION_HYB_GATHER_KERNEL void hyb_rem_pv_kernel(const float* __restrict__ V, const float* __restrict__ Raw,
                                               float* __restrict__ P, float* __restrict__ O,
                                               float* __restrict__ Ocache,
                                               const float2* __restrict__ Stats, HybIndex ix, int L, int NB, int nnz,
                                               Layouts ly) {
    const int lane = threadIdx.x & 63, ent = hyb_entry_of_lane(lane);
    const long long wrow = (long long)xcd_remap((int)blockIdx.x, (int)gridDim.x) * HYB_GWAVES + wave_index();
    if (wrow >= (long long)NB * L) return;
    const int bh = (int)(wrow / L), row = (int)(wrow % L);
    const int r0 = ix.r_off[row], rc = ix.r_off[row + 1] - r0;
    size_t ib, ob;
    int ild, old_;
    hyb_head<ST>(ly.in, ly.H, bh, L, ib, ild);
    hyb_head<ST>(ly.out, ly.H, bh, L, ob, old_);
    float* Ph = P + (size_t)bh * nnz;
    const float* raw = Raw + (size_t)bh * ix.nr + r0;
    const float2 st = Stats[(size_t)bh * L + row];
    HybRowAcc acc;
    acc.clear();
    for (int c0 = 0; c0 < rc; c0 += 64) {
        const int k = c0 + ent;
        float wgt = 0.f;
        int col = 0;
        if (k < rc) {
            const int pp = ix.r_pos[r0 + k];
            wgt = __builtin_amdgcn_exp2f(raw[k] - st.x) * st.y;
            col = ix.r_col[r0 + k];
            __builtin_nontemporal_store(wgt, Ph + pp);  // written once, not read again before the backward
        }
        acc.chunk(wgt, col, min(64, rc - c0), V + ib, ild, lane);
    }
    const f32x4 tot = acc.total();
    if (lane < 8) {
        f32x4* orow = reinterpret_cast<f32x4*>(O + ob + (size_t)row * old_) + lane;
        const f32x4 sum = *orow + tot;
        *orow = sum;
        if (Ocache) reinterpret_cast<f32x4*>(Ocache + ((size_t)bh * L + row) * 32)[lane] = sum;  // own copy: contiguous
    }
}

// -------------------------------------------------------------------------------------------------
// Backward, row pass, dense tiles: g_i = dO_i . O_i (G receives -g for the other kernels); dP^T - g = V_J.dO_I^T
// chain started from -g, dS' = (dP - g)*P, dQ = sum dS'.K_J / sqrt(d).
// -------------------------------------------------------------------------------------------------
template <int WAVES, bool ST>
SPION_HYB_KERNEL(WAVES) void hyb_tile_bwd_row_kernel(const float* __restrict__ K, const float* __restrict__ V,
                                              const float* __restrict__ P, const float* __restrict__ dO,
                                              const float* __restrict__ Out, float* __restrict__ G,
                                              float* __restrict__ dQ, HybIndex ix, int L, int nbr, int NB, int nnz,
                                              float scale, Layouts ly) {
    constexpr int D = 32, KH = 16;
    typedef DmaTileF32 DT;
    // per wavefront: the V and K tiles, a padded tile (layout change of P; the final reduction starts there) and the index
    constexpr int WB = 2 * DT::TILE + 32 * TS * 4 + 512;
    static_assert(WAVES == 1 || WAVES * WB >= WAVES * 4096, "the reduction fits in the tile space");
    __shared__ __attribute__((aligned(16))) char smem[WAVES * WB];
    float* lds = reinterpret_cast<float*>(smem);
    const int item = xcd_remap(blockIdx.x, nbr * NB);
    const int bh = item / nbr, I = item % nbr;
    const int w = wave_index(), l = threadIdx.x & 63, h = l >> 5, li = l & 31;
    size_t ib, ob, gb, ibytes, obytes, gbytes;
    int ild, old_, gld;
    head_slice<ST, D>(ly.in, ly.H, bh, L, ib, ild, ibytes);
    head_slice<ST, D>(ly.out, ly.H, bh, L, ob, old_, obytes);
    head_slice<ST, D>(ly.grad, ly.H, bh, L, gb, gld, gbytes);
    const rsrc_t rK = make_rsrc(K + ib, ibytes), rV = make_rsrc(V + ib, ibytes);
    const rsrc_t rdO = make_rsrc(dO + ob, obytes), rO = make_rsrc(Out + ob, obytes);
    const rsrc_t rP = make_rsrc(P + (size_t)bh * nnz, (size_t)nnz * 4);
    const u32x4 wV = rsrc_words(V + ib, ibytes), wK = rsrc_words(K + ib, ibytes);
    const char* Tv = smem + w * WB;
    const char* Tk = Tv + DT::TILE;
    float* T = reinterpret_cast<float*>(smem + w * WB + 2 * DT::TILE);
    int* X = reinterpret_cast<int*>(smem + w * WB + 2 * DT::TILE + 32 * TS * 4);
    const unsigned lv = lds_address(Tv), lk = lv + DT::TILE;
    const int tile_bytes = 32 * ild * 4;

    auto load_go = [&](float (&go)[KH], int l) {
        ldr_rows<D>(rdO, ((l & 31) * old_ + (l >> 5) * KH) * 4, I * 32 * old_ * 4, go);
    };
    const int t0 = hyb_scalar(ix.t_rp, I), cnt = hyb_scalar(ix.t_rp, I + 1) - t0;
    const int n = cnt > w ? (cnt - w + WAVES - 1) / WAVES : 0;
    auto fetch = [&](HybTile& x, int i, int li) {
        const int t = t0 + w + max(min(i, n - 1), 0) * WAVES;
        x.blk = hyb_scalar(ix.t_col, t);
        hyb_fetch_index(ix, t, li, x);
    };
    HybTile x0 = {};
    if (n > 0) fetch(x0, 0, li);  // on its way with the strip's own rows
    float go[KH], oo[KH];
    load_go(go, l);
    ldr_rows<D>(rO, (li * old_ + h * KH) * 4, I * 32 * old_ * 4, oo);
    float g = 0.f;
#pragma unroll
    for (int s = 0; s < KH; ++s) g = fmaf(go[s], oo[s], g);
    g += __shfl_xor(g, 32, 64);
    if (w == 0 && h == 0) G[(size_t)bh * L + I * 32 + li] = -g;
    const f32x16 gneg = splat16(-g);

    f32x16 acc[1];
    auto walk = [&](const auto& gk, int l) {  // gk: the dO operand, split or whole
        constexpr bool EXACT = is_whole<std::decay_t<decltype(gk)>>;
        const int h = l >> 5, li = l & 31;
        const int il = DT::voff(l, ild), ix_ = DT::extra_step(ild);
        const auto a_v = DT::own_addr(Tv, li, 4 * h, 1);
        const auto a_k = DT::cols_addr(Tk, li, h);
        settle(gk);
        acc[0] = splat16(0.f);
        if (n <= 0) return;
        hyb_walk(
            n, x0, X, l, h, li, rP, [&](HybTile& x, int i) { fetch(x, i, li); },
            [&](int blk) {
                DT::load(wV, lv, il, blk * tile_bytes, ix_);
                DT::load(wK, lk, il, blk * tile_bytes, ix_);
            },
            [&](const float (&p)[16], auto next) {
                float vt[KH], kb[1][16], pr[16];
                lds_put_cols(T, li, h, p);
                DT::get(a_v, vt);
                DT::get(a_k, kb[0]);
                lds_get_rows(T, li, h, pr);  // pr[r] = P[query li][key acc_row(r, h)]
                wait_lgkm0();
                next();
                const f32x16 dp = mma_feat_init<D>(vt, gk, gneg);  // dp[r] = dO_i . v_j - g_i
                float ds[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) ds[r] = dp[r] * pr[r];
                f32x16 part[1] = {splat16(0.f)};
                mma_b_split<D, EXACT>(ds, kb, part);
                acc[0] += part[0];
            });
    };
    walk(split3(go), l);
    if (split_failed(acc)) {
        const int l2 = second_walk(l);
        load_go(go, l2);
        walk(whole(go), l2);
    }
    if (hyb_not_finite(acc[0]))
        hyb_rows_by_entries(
            T, l, n, ix, rK, ild, [&](int u) { return t0 + w + u * WAVES; },
            [&](int row) {
                const int at = ((I * 32 + row) * old_ + li) * 4;
                const float go_i = ld1(rdO, at, 0), g_i = hyb_half_sum(go_i * ld1(rO, at, 0));
                return [=](int col, int pos) {
                    return (hyb_half_sum(go_i * ld1(rV, (col * ild + li) * 4, 0)) - g_i) * ld1(rP, pos * 4, 0);
                };
            },
            acc[0]);
    if constexpr (WAVES > 1) __syncthreads();
    hyb_reduce_store<WAVES>(acc[0], scale, dQ + gb, gld, I * 32, w, li, h, lds);
}

// -------------------------------------------------------------------------------------------------
// Backward, row pass, remainder: dS = (dO_i . v_j - g_i) * P / sqrt(d), dQ_i += sum dS . K[col].  The column pass
// walks the same entries column after column; looking P and dS up there inside a head's full P and dS (two arrays
// of nnz floats, more than the L2 cache holds per head) would fetch a memory sector for every four bytes, so this
// kernel leaves the pairs {dS, P} of the remainder alone in one compact list (Pairs [NB][nr], row order, inside the
// caller's dS scratch), small enough per head for the column pass to find in the L2 cache.
// -------------------------------------------------------------------------------------------------
template <bool ST>
SPION_HYB_GATHER_KERNEL void hyb_rem_bwd_row_kernel(const float* __restrict__ K, const float* __restrict__ V,
                                                    const float* __restrict__ P, const float* __restrict__ dO,
                                                    const float* __restrict__ G, float2* __restrict__ Pairs,
                                                    float* __restrict__ dQ, HybIndex ix, int L, int NB, int nnz,
                                                    float scale, Layouts ly) {
    const int lane = threadIdx.x & 63, ent = hyb_entry_of_lane(lane);
    const long long wrow = (long long)xcd_remap((int)blockIdx.x, (int)gridDim.x) * HYB_GWAVES + wave_index();
    if (wrow >= (long long)NB * L) return;
    const int bh = (int)(wrow / L), row = (int)(wrow % L);
    const int r0 = ix.r_off[row], rc = ix.r_off[row + 1] - r0;
    if (rc == 0) return;
    size_t ib, ob, gb;
    int ild, old_, gld;
    hyb_head<ST>(ly.in, ly.H, bh, L, ib, ild);
    hyb_head<ST>(ly.out, ly.H, bh, L, ob, old_);
    hyb_head<ST>(ly.grad, ly.H, bh, L, gb, gld);
    const f32x4 go4 = reinterpret_cast<const f32x4*>(dO + ob + (size_t)row * old_)[lane & 7];
    const float* Ph = P + (size_t)bh * nnz;
    float2* pairs = Pairs + (size_t)bh * ix.nr;
    const float gneg = G[(size_t)bh * L + row];
    HybRowAcc acc;
    acc.clear();
    for (int c0 = 0; c0 < rc; c0 += 64) {
        // Memory is accessed in the list's order, lane l entry c0 + l, and the gathers' order (entry c0 + ent, an exchange of
        // the two halves of the lane number, its own inverse) is made by lane moves: in the gathers' order neighbouring
        // lanes read and write eight entries apart.  64 heads of 4096 rows with 76 entries: 352 -> 338 us.
        const int k = c0 + lane, nk = min(64, rc - c0);
        const int col_l = k < rc ? ix.r_col[r0 + k] : 0;
        const int pp = k < rc ? ix.r_pos[r0 + k] : 0;
        const float pv = k < rc ? Ph[pp] : 0.f;
        const int col = __shfl(col_l, ent, 64);
        const float dp = __shfl(hyb_gather_dot(go4, V + ib, ild, col, nk, lane), ent, 64);
        float dsv = 0.f;
        if (k < rc) {
            dsv = (dp + gneg) * pv * scale;
            pairs[r0 + k] = make_float2(dsv, pv);
        }
        acc.chunk(__shfl(dsv, ent, 64), col, nk, K + ib, ild, lane);
    }
    const f32x4 tot = acc.total();
    if (lane < 8) {
        f32x4* qrow = reinterpret_cast<f32x4*>(dQ + gb + (size_t)row * gld) + lane;
        *qrow = *qrow + tot;
    }
}

// -------------------------------------------------------------------------------------------------
// Backward, column pass, dense tiles: dK_J = sum_I dS_IJ^T Q_I / sqrt(d), dV_J = sum_I P_IJ^T dO_I; dP - g is
// recomputed per tile by a chain started from the stored -g.
// -------------------------------------------------------------------------------------------------
template <int WAVES, bool ST>
SPION_HYB_KERNEL(WAVES) void hyb_tile_bwd_col_kernel(const float* __restrict__ Q, const float* __restrict__ V,
                                              const float* __restrict__ P, const float* __restrict__ dO,
                                              const float* __restrict__ G, float* __restrict__ dK,
                                              float* __restrict__ dV, HybIndex ix, int L, int nbr, int NB, int nnz,
                                              float scale, Layouts ly) {
    constexpr int D = 32, KH = 16;
    typedef DmaTileF32 DT;
    typedef DmaTile<32> Plane;
    // per wavefront: the Q and dO tiles, the parts of dO (its second product reads them transposed), -g and the index
    constexpr int WB = 2 * DT::TILE + 3 * Plane::TILE + 256 + 512;
    static_assert(2 * 32 * TS * 4 <= WB, "the sums by entries fit in the tile space");
    __shared__ __attribute__((aligned(16))) char smem[WAVES * WB];
    float* lds = reinterpret_cast<float*>(smem);
    const int item = xcd_remap(blockIdx.x, nbr * NB);
    const int bh = item / nbr, J = item % nbr;
    const int w = wave_index(), l = threadIdx.x & 63;
    const int h = l >> 5, li = l & 31;
    size_t ib, ob, gb, ibytes, obytes, gbytes;
    int ild, old_, gld;
    head_slice<ST, D>(ly.in, ly.H, bh, L, ib, ild, ibytes);
    head_slice<ST, D>(ly.out, ly.H, bh, L, ob, old_, obytes);
    head_slice<ST, D>(ly.grad, ly.H, bh, L, gb, gld, gbytes);
    const rsrc_t rQ = make_rsrc(Q + ib, ibytes), rV = make_rsrc(V + ib, ibytes);
    const rsrc_t rdO = make_rsrc(dO + ob, obytes);
    const rsrc_t rG = make_rsrc(G + (size_t)bh * L, (size_t)L * 4);
    const rsrc_t rP = make_rsrc(P + (size_t)bh * nnz, (size_t)nnz * 4);
    const u32x4 wQ = rsrc_words(Q + ib, ibytes), wO = rsrc_words(dO + ob, obytes), wG = rsrc_words(G + (size_t)bh * L, (size_t)L * 4);
    char* const Tq_ = smem + w * WB;
    char* const To_ = Tq_ + DT::TILE;
    char* const planes = Tq_ + 2 * DT::TILE;
    char* const Tg = planes + 3 * Plane::TILE;
    int* X = reinterpret_cast<int*>(Tg + 256);
    const unsigned lq = lds_address(Tq_), lo = lq + DT::TILE, lg = lds_address(Tg);

    auto load_vt = [&](float (&vt)[KH], int l) {
        ldr_rows<D>(rV, ((l & 31) * ild + (l >> 5) * KH) * 4, J * 32 * ild * 4, vt);
    };
    f32x16 ak[1], av[1];
    const int e0 = hyb_scalar(ix.t_cp, J), ecnt = hyb_scalar(ix.t_cp, J + 1) - e0;
    const int n = ecnt > w ? (ecnt - w + WAVES - 1) / WAVES : 0;
    auto fetch = [&](HybTile& x, int i, int li) {
        const int e = e0 + w + max(min(i, n - 1), 0) * WAVES;
        x.blk = hyb_scalar(ix.t_ci, e);
        hyb_fetch_index(ix, hyb_scalar(ix.t_ct, e), li, x);
    };
    HybTile x0 = {};
    if (n > 0) fetch(x0, 0, li);
    float vt[KH];
    load_vt(vt, l);

    auto walk = [&](const auto& vk, int l) {  // vk: the V operand, split or whole
        constexpr bool EXACT = is_whole<std::decay_t<decltype(vk)>>;
        const int h = l >> 5, li = l & 31;
        const int ql = DT::voff(l, ild), qx = DT::extra_step(ild), ol = DT::voff(l, old_), ox = DT::extra_step(old_);
        const auto a_q = DT::cols_addr(Tq_, li, h);  // the dO tile's are 4 KB on
        const auto a_go = DT::own_addr(To_, li, 4 * h, 1);
        const auto ra = Plane::row_addr(li, h);
        const auto ta = Plane::tr_addr(l);
        settle(vk);
        ak[0] = splat16(0.f);
        av[0] = splat16(0.f);
        if (n <= 0) return;
        hyb_walk(
            n, x0, X, l, h, li, rP, [&](HybTile& x, int i) { fetch(x, i, li); },
            [&](int blk) {
                DT::load(wQ, lq, ql, blk * 32 * ild * 4, qx);
                DT::load(wO, lo, ol, blk * 32 * old_ * 4, ox);
                dma_b32(wG, lg, l * 4, blk * 128);
            },
            [&](const float (&p)[16], auto next) {  // p[r] = P[query acc_row(r, h)][key li]
                float go[KH], qb[1][16], pc[16];
                f32x16 init;
                DT::get(a_go, go);
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x4 v = *reinterpret_cast<const f32x4*>(Tg + 16 * h + 32 * g);
                    init[4 * g + 0] = v.x;
                    init[4 * g + 1] = v.y;
                    init[4 * g + 2] = v.z;
                    init[4 * g + 3] = v.w;
                }
                DT::get(a_q, qb[0]);
#pragma unroll
                for (int r = 0; r < 16; ++r) pc[r] = p[r];
                f32x16 dp, part[1] = {splat16(0.f)};
                if constexpr (EXACT) {
                    float ot[1][16];
                    DT::get(a_q, ot[0], DT::TILE);
                    wait_lgkm0();
                    next();
                    dp = mma_feat_init<D>(go, vk, init);  // dO_i . v_j - g_i, i = acc_row(r, h), j = li
                    mma_b_f32<D>(pc, ot, part);
                } else {
                    wait_lgkm0();
                    next();
                    const Split3<16> gs = split3(go);
#pragma unroll
                    for (int k = 0; k < 3; ++k)
#pragma unroll
                        for (int t = 0; t < 2; ++t) *reinterpret_cast<bf16x8*>(planes + k * Plane::TILE + ra.a[t]) = gs.p[k][t];
                    dp = mma_split(gs, vk, init);
                    asm volatile("" ::: "memory");  // same-wave LDS accesses complete in order
                    Split3<16> ot;
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        bf16x8 x[1][2];
                        Plane::get_tile_t(planes + k * Plane::TILE, ta, x);
                        ot.p[k][0] = x[0][0];
                        ot.p[k][1] = x[0][1];
                    }
                    part[0] = mma_split(split3(pc), ot, part[0]);
                }
                av[0] += part[0];
                float ds[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) ds[r] = dp[r] * pc[r];
                part[0] = splat16(0.f);
                mma_b_split<D, EXACT>(ds, qb, part);
                ak[0] += part[0];
            });
    };
    walk(split3(vt), l);
    if (split_failed(ak) || split_failed(av)) {
        const int l2 = second_walk(l);
        load_vt(vt, l2);
        walk(whole(vt), l2);
    }
    float* Tq = reinterpret_cast<float*>(Tq_);
    float* To = Tq + 32 * TS;
    if (hyb_not_finite(ak[0]) || hyb_not_finite(av[0])) {
        const int l2 = second_walk(l), h = l2 >> 5, li = l2 & 31;
#pragma unroll 1
        for (int jj = 0; jj < 16; ++jj) {
            const int j = 2 * jj + h;
            const float v_j = ld1(rV, ((J * 32 + j) * ild + li) * 4, 0);
            float sk = 0.f, sv = 0.f;
#pragma unroll 1
            for (int u = 0; u < n; ++u) {
                const int e = e0 + w + u * WAVES, t = ix.t_ct[e], row0 = ix.t_ci[e] * 32;
#pragma unroll 1
                for (int i = 0; i < 32; ++i) {
                    const unsigned bits = ix.t_bits[(size_t)t * 32 + i];
                    if (!((bits >> j) & 1u)) continue;
                    const float p = ld1(rP, (ix.t_pos[(size_t)t * 32 + i] + __popc(bits & ((1u << j) - 1u))) * 4, 0);
                    const float go_i = ld1(rdO, ((row0 + i) * old_ + li) * 4, 0);
                    const float ds = (hyb_half_sum(go_i * v_j) + ld1(rG, (row0 + i) * 4, 0)) * p;
                    sk = fmaf(ds, ld1(rQ, ((row0 + i) * ild + li) * 4, 0), sk);
                    sv = fmaf(p, go_i, sv);
                }
            }
            Tq[j * TS + li] = sk;
            To[j * TS + li] = sv;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            ak[0][r] = Tq[acc_row(r, h) * TS + li];
            av[0][r] = To[acc_row(r, h) * TS + li];
        }
    }
    if constexpr (WAVES > 1) __syncthreads();
    hyb_reduce_store<WAVES>(ak[0], scale, dK + gb, gld, J * 32, w, li, h, lds);
    if constexpr (WAVES > 1) __syncthreads();
    hyb_reduce_store<WAVES>(av[0], 1.0f, dV + gb, gld, J * 32, w, li, h, lds);
}

// -------------------------------------------------------------------------------------------------
// Backward, column pass, remainder: dK_j += sum_i dS_ij Q_i, dV_j += sum_i P_ij dO_i over the remainder's
// transposed index, from the compact {dS, P} pairs of the row pass (dS already carries the 1/sqrt(d)).
// -------------------------------------------------------------------------------------------------
template <bool ST>
__global__ __launch_bounds__(64 * HYB_GWAVES) void hyb_rem_bwd_col_kernel(  // two gathers in flight per entry: four waves per SIMD
    const float* __restrict__ Q, const float* __restrict__ dO,
                                                    const float2* __restrict__ Pairs,
                                                    float* __restrict__ dK, float* __restrict__ dV, HybIndex ix, int L,
                                                    int NB, Layouts ly) {
    const int lane = threadIdx.x & 63, ent = hyb_entry_of_lane(lane);
    const long long wcol = (long long)xcd_remap((int)blockIdx.x, (int)gridDim.x) * HYB_GWAVES + wave_index();
    if (wcol >= (long long)NB * L) return;
    const int bh = (int)(wcol / L), colj = (int)(wcol % L);
    const int c0p = ix.c_ptr[colj], cnt = ix.c_ptr[colj + 1] - c0p;
    if (cnt == 0) return;
    size_t ib, ob, gb;
    int ild, old_, gld;
    hyb_head<ST>(ly.in, ly.H, bh, L, ib, ild);
    hyb_head<ST>(ly.out, ly.H, bh, L, ob, old_);
    hyb_head<ST>(ly.grad, ly.H, bh, L, gb, gld);
    const float2* pairs = Pairs + (size_t)bh * ix.nr;
    HybRowAcc ak, av;
    ak.clear();
    av.clear();
    for (int c0 = 0; c0 < cnt; c0 += 64) {
        const int e = c0 + ent;
        float wk = 0.f, wv = 0.f;
        int row = 0;
        if (e < cnt) {
            row = ix.c_row[c0p + e];
            const float2 pr = pairs[ix.c_src[c0p + e]];
            wk = pr.x;
            wv = pr.y;
        }
        const int nk = min(64, cnt - c0);
        ak.chunk(wk, row, nk, Q + ib, ild, lane);
        av.chunk(wv, row, nk, dO + ob, old_, lane);
    }
    const f32x4 tk = ak.total(), tv = av.total();
    if (lane < 8) {
        f32x4* kr = reinterpret_cast<f32x4*>(dK + gb + (size_t)colj * gld) + lane;
        f32x4* vr = reinterpret_cast<f32x4*>(dV + gb + (size_t)colj * gld) + lane;
        *kr = *kr + tk;
        *vr = *vr + tv;
    }
}

// -------------------------------------------------------------------------------------------------
// The element path's column pass (all entries of a pattern, d = 32) with the gathered operands in LDS instead of L2.  A
// work-group of sixteen wavefronts owns 128 * NC columns of a head and walks the sequence in ranges of HYB_CL_ROWS rows,
// whose Q and dO rows (128 KB) it loads once per range.  A group of eight lanes owns NC columns (lane s holds floats
// 4s .. 4s+3 of their dK and dV rows, 8 * NC accumulator registers that live across the ranges) and walks each column's
// entries -- rows ascending, so the entries of a range are the next ones of the column's list -- eight at a time: lane s
// fetches the s-th entry's row, dS and P, the eight are handed round the group, and every lane adds its 16-byte pieces of
// the Q and dO rows, read from LDS, to its sums.  Each lane's sums run in a fixed order along the column's list, so the
// result does not depend on the launch.
// -------------------------------------------------------------------------------------------------
constexpr int HYB_CL_ROWS = 512, HYB_CL_THREADS = 1024;  // a work-group owns NC * 128 columns: 1024 (NC = 8) or 512
// x of another lane of the same row of sixteen: quad_perm (CTRL = 0x55 * k: lane k of the own quad) or row_half_mirror
// (0x141: lane 7 - i of the own eight)
template <int CTRL>
__device__ __forceinline__ int hyb_dpp(int x) {
    return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, false);
}
// The list of a column: entries c_ptr[j] .. c_ptr[j+1]-1, their rows c_row (ascending) and c_src, the index of the
// entry's weights in the head's dS and P arrays ([NB][n] floats each).
template <bool ST, int NC>
__global__ __launch_bounds__(HYB_CL_THREADS) void elem_bwd_col_lds_kernel(
    const float* __restrict__ Q, const float* __restrict__ dO, const float* __restrict__ dSa,
    const float* __restrict__ Pa, float* __restrict__ dK, float* __restrict__ dV,
    const int* __restrict__ c_ptr, const int* __restrict__ c_row, const int* __restrict__ c_src, int n, int L, int NB,
    Layouts ly) {
    __shared__ f32x4 sq[HYB_CL_ROWS * 8], so[HYB_CL_ROWS * 8];
    constexpr int HYB_CL_COLS = NC * (HYB_CL_THREADS / 8);
    const int ncg = (L + HYB_CL_COLS - 1) / HYB_CL_COLS;  // the last one's columns past the end have no entries
    const int item = xcd_remap((int)blockIdx.x, (int)gridDim.x);  // the work-groups of a head share an XCD's L2
    const int bh = item / ncg, cg = item % ncg;
    const int t = threadIdx.x, grp = t >> 3, sub = t & 7, lane = t & 63;
    size_t ib, ob, gb;
    int ild, old_, gld;
    hyb_head<ST>(ly.in, ly.H, bh, L, ib, ild);
    hyb_head<ST>(ly.out, ly.H, bh, L, ob, old_);
    hyb_head<ST>(ly.grad, ly.H, bh, L, gb, gld);
    const float* dsh = dSa + (size_t)bh * n;
    const float* ph = Pa + (size_t)bh * n;
    f32x4 ak[NC], av[NC];
    int e[NC], eend[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int col = cg * HYB_CL_COLS + c * (HYB_CL_THREADS / 8) + grp;
        ak[c] = (f32x4){0.f, 0.f, 0.f, 0.f};
        av[c] = (f32x4){0.f, 0.f, 0.f, 0.f};
        e[c] = col < L ? c_ptr[col] : 0;
        eend[c] = col < L ? c_ptr[col + 1] : 0;
    }
    for (int r0 = 0; r0 < L; r0 += HYB_CL_ROWS) {
        __syncthreads();  // everybody has finished with the previous range
#pragma unroll
        for (int k = 0; k < HYB_CL_ROWS * 8 / HYB_CL_THREADS; ++k) {
            const int idx = t + k * HYB_CL_THREADS, row = min(r0 + (idx >> 3), L - 1), piece = idx & 7;
            sq[idx] = reinterpret_cast<const f32x4*>(Q + ib + (size_t)row * ild)[piece];
            so[idx] = reinterpret_cast<const f32x4*>(dO + ob + (size_t)row * old_)[piece];
        }
        __syncthreads();
        const int rend = r0 + HYB_CL_ROWS;
        auto fetch_idx = [&](int c, int& row, int& src) {
            const int my = e[c] + sub;
            const bool ok = my < eend[c];
            row = ok ? c_row[my] : 0x7fffffff;
            src = ok ? c_src[my] : 0;
        };
        // The eight entries go round the group by DPP moves: a quad broadcast hands entry k of a lane's own quad to
        // its four lanes, and the same on the values mirrored within the eight lanes hands over the other quad's
        // entries -- every lane sees all eight, each quad in an order of its own, which is fixed.
        auto add_batch = [&](int c, int lrow, float2 pr) {
            const int wx = __float_as_int(pr.x), wy = __float_as_int(pr.y);
            const int mrow = hyb_dpp<0x141>(lrow), mx = hyb_dpp<0x141>(wx), my_ = hyb_dpp<0x141>(wy);
#define SPION_HYB_ENTRY(CTRL, R, X, Y)                                           \
    {                                                                            \
        const int rk = hyb_dpp<CTRL>(R);                                         \
        const float wk = __int_as_float(hyb_dpp<CTRL>(X)), wv = __int_as_float(hyb_dpp<CTRL>(Y)); \
        ak[c] += sq[rk * 8 + sub] * wk;                                          \
        av[c] += so[rk * 8 + sub] * wv;                                          \
    }
            SPION_HYB_ENTRY(0x00, lrow, wx, wy)
            SPION_HYB_ENTRY(0x55, lrow, wx, wy)
            SPION_HYB_ENTRY(0xaa, lrow, wx, wy)
            SPION_HYB_ENTRY(0xff, lrow, wx, wy)
            SPION_HYB_ENTRY(0x00, mrow, mx, my_)
            SPION_HYB_ENTRY(0x55, mrow, mx, my_)
            SPION_HYB_ENTRY(0xaa, mrow, mx, my_)
            SPION_HYB_ENTRY(0xff, mrow, mx, my_)
#undef SPION_HYB_ENTRY
        };
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            int nn = 8;
            while (nn == 8) {
                int r1, s1;
                fetch_idx(c, r1, s1);
                const bool in = r1 < rend;
                nn = __popcll((__ballot(in) >> (lane & 56)) & 0xffull);
                if (nn == 0) break;
                add_batch(c, in ? r1 - r0 : 0, in ? (float2){dsh[s1], ph[s1]} : (float2){0.f, 0.f});
                e[c] += nn;
            }
        }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int col = cg * HYB_CL_COLS + c * (HYB_CL_THREADS / 8) + grp;
        if (col >= L) continue;
        f32x4* kr = reinterpret_cast<f32x4*>(dK + gb + (size_t)col * gld) + sub;
        f32x4* vr = reinterpret_cast<f32x4*>(dV + gb + (size_t)col * gld) + sub;
        *kr = ak[c];
        *vr = av[c];
    }
}

}  // namespace spion
