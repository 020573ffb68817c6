// Backward passes of the dense phase for row-major heads whose wavefronts walk the same tiles: a work-group owns G
// neighbouring strips of 32 queries (row pass) or keys (column pass) of one head, one to a wavefront, and every operand tile
// of the other dimension is loaded from global memory, split into its three bf16 parts (tile_ops.h) and laid out in LDS once
// for all of them.  (dense_attn.hip's other backward kernels give a strip to four wavefronts, each with tiles of its own.)
//
// Why: with every strip needing every tile, splitting is work that can be shared.  An operand tile costs a wavefront 22
// vector-ALU instructions (d = 32: 1024 elements over four wavefronts) instead of 88, and dO is split once for its two roles
// in the column pass: its feature-major view is read from the same parts with the transposing LDS reads of gfx950.  That
// pays for all products on the bf16 pipe, where the kernels without sharing need fp32 chains (1024 matrix cycles a product
// instead of 384, and no overlap with the vector ALU) in the d = 32 column pass and in both passes at d = 64.  There are no
// partial results to merge at the end either.
// Accuracy: a wavefront's sum over all tiles would round twelve times a tile at the size of the whole sum (2-norm errors of
// dQ, dK, dV against float64 5.0e-7 at 1024 queries), so a tile's product is summed by itself and added: 1.7e-7 to 1.9e-7, where
// four wavefronts with a quarter of the tiles each gave 2.9e-7 to 3.2e-7.
// Measured, us per launch in a training loop, without / with sharing, one machine: d = 32, 64 x 2 heads of 1024: row pass 157 /
// 123, column pass 208 / 169; 16 x 2 of 2048: 150 / 123, 204 / 173; d = 64, 64 x 2 of 1024: 260 / 208, 457 / 286.
// Bound (d = 32, 64 x 2 of 1024, counters): column pass, matrix pipe 59 % and vector ALU 57 % busy (36 and 281 instructions
// a tile) at 1.81 GHz, which is the power limit (the kernels without sharing run at 2.03); row pass, 4.9 TB/s of the map
// and operands, 5.5 being what a large copy reaches.
// Asking the compiler for alternating matrix and vector instructions (sched_group_barrier) makes the column pass 10 %
// slower; map tiles requested two steps ahead at two wavefronts per SIMD, instead of one step ahead at three, 3 to 5 %;
// the parts written after the last product instead of beside the second, 3 %.
#pragma once
#include "bf16_tile.h"
#include "tile_kernels.h"

namespace spion {

// 64 x 16 bytes to 1 KB of LDS
__device__ __forceinline__ void dma_b128(u32x4 r, unsigned lds, int voff, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(r),
                 "s"(soff)
                 : "memory");
}

// The two operand tiles (32 rows x D floats each) of a step.  Wavefront w of the G = D/8 loads 1 KB of each (rows RPW*w ..)
// into a place of its own, takes it back out, a lane 16 bytes, and writes the three parts into planes in the layout of
// DmaTile<D>.  The planes are double-buffered, so a step needs one barrier: parts of step i + 1 are written while step i's
// are read.
template <int D>
struct GroupTiles {
    typedef DmaTile<D> Plane;
    static constexpr int G = D / 8;  // wavefronts: 4 (d = 32) or 8 (d = 64)
    static constexpr int LPR = D / 4, RPW = 64 / LPR;
    static constexpr int RAW = 2 * G * 1024, SPLIT = 3 * Plane::TILE, BYTES = RAW + 4 * SPLIT;
    char* base;
    unsigned lraw;
    u32x4 r[2];
    int ld[2], voff[2], dst, w, l;
    __device__ __forceinline__ GroupTiles(char* smem, int w_, int l_, u32x4 r0, int ld0, u32x4 r1, int ld1)
        : base(smem), lraw(lds_address(smem) + w_ * 1024), r{r0, r1}, ld{ld0, ld1}, w(w_), l(l_) {
#pragma unroll
        for (int o = 0; o < 2; ++o) voff[o] = ((l / LPR) * ld[o] + 4 * (l % LPR)) * 4;
        const int row = w * RPW + l / LPR, c = l % LPR;
        dst = row * Plane::ROW + 16 * ((c >> 1) ^ Plane::swz(row)) + 8 * (c & 1);
    }
    __device__ __forceinline__ void issue(int tile) const {
#pragma unroll
        for (int o = 0; o < 2; ++o) dma_b128(r[o], lraw + o * G * 1024, voff[o], (tile * 32 + w * RPW) * ld[o] * 4);
    }
    __device__ __forceinline__ void take(f32x4 (&x)[2]) const {
#pragma unroll
        for (int o = 0; o < 2; ++o) x[o] = *reinterpret_cast<const f32x4*>(base + (w + G * o) * 1024 + l * 16);
    }
    __device__ __forceinline__ char* planes(int buf, int op) const { return base + RAW + (2 * buf + op) * SPLIT; }
    __device__ __forceinline__ void put(const f32x4 (&x)[2], int buf) const {
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            char* p = planes(buf, o) + dst;
            float a[4] = {x[o].x, x[o].y, x[o].z, x[o].w};
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                u32x2 v;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    v[j] = pack_bf16(a[2 * j], a[2 * j + 1]);
                    if (k < 2) {
                        a[2 * j] -= bf16_lo(v[j]);
                        a[2 * j + 1] -= bf16_hi(v[j]);
                    }
                }
                *reinterpret_cast<u32x2*>(p + k * Plane::TILE) = v;
            }
        }
    }
};
// acc = init + A.B over the head dimension, A from planes
template <int D>
__device__ __forceinline__ f32x16 mma_rows(const char* T, const typename DmaTile<D>::RowAddr& ra, const Split3<D / 2>& b,
                                           f32x16 acc) {
    typedef DmaTile<D> Plane;
    Split3<D / 2> a;
#pragma unroll
    for (int k = 0; k < 3; ++k) Plane::get_rows(T + k * Plane::TILE, ra, a.p[k]);
    return mma_split(a, b, acc);
}
// out[c] += A^T.B over the tile's 32 rows, A from planes
template <int D>
__device__ __forceinline__ void mma_cols(const char* T, const typename DmaTile<D>::TrAddr& ta, const Split3<16>& b,
                                         f32x16 (&out)[D / 32]) {
    typedef DmaTile<D> Plane;
    bf16x8 x[3][D / 32][2];
#pragma unroll
    for (int k = 0; k < 3; ++k) Plane::get_tile_t(T + k * Plane::TILE, ta, x[k]);
#pragma unroll
    for (int c = 0; c < D / 32; ++c) {
        Split3<16> a;
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int t = 0; t < 2; ++t) a.p[k][t] = x[k][c][t];
        out[c] += mma_split(a, b, splat16(0.f));
    }
}

// The sums of a strip of queries (dQ) or keys (dK, dV) once more with fp32 chains, straight from memory.  l2: the lane, hidden
// by second_walk; init(I, ..): -g of query tile I (register = query).
template <int D>
__device__ __forceinline__ void dense_row_again(const float* K, const float* V, const float* Attn, const float* dO, int L,
                                                int nbr, int I, int bh, int l2, const f32x16& gneg, size_t ib, int ild,
                                                size_t hbytes, size_t ob, int old_, size_t obytes, f32x16 (&acc)[D / 32]) {
    constexpr int KH = D / 2, NC = D / 32;
    const int h2 = l2 >> 5, li2 = l2 & 31;
    const rsrc_t rV = make_rsrc(V + ib, hbytes), rK = make_rsrc(K + ib, hbytes);
    const rsrc_t rP = make_rsrc(Attn + (size_t)bh * L * L, (size_t)L * L * 4);
    float go[KH];
    ldr_rows<D>(make_rsrc(dO + ob, obytes), (li2 * old_ + h2 * KH) * 4, I * 32 * old_ * 4, go);
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = splat16(0.f);
#pragma unroll 1
    for (int J = 0; J < nbr; ++J) {
        float vt[KH], p[16], kb[NC][16], ds[16];
        ldr_rows<D>(rV, (li2 * ild + h2 * KH) * 4, J * 32 * ild * 4, vt);
        ldr_tile_cols(rP, (4 * h2 * L + li2) * 4, (J * 32 * L + I * 32) * 4, L, p);
        ldr_tile_b<D>(rK, (4 * h2 * ild + li2) * 4, J * 32 * ild * 4, kb, ild);
        const f32x16 dp = mma_feat_f32<D>(vt, go, gneg);
#pragma unroll
        for (int r = 0; r < 16; ++r) ds[r] = dp[r] * p[r];
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] = mma_chain(kb[c], ds, acc[c]);
    }
}
template <int D, class Init>
__device__ __forceinline__ void dense_col_again(const float* Q, const float* V, const float* Attn, const float* dO, int L,
                                                int nbr, int J, int bh, int l, size_t ib, int ild, size_t hbytes, size_t ob,
                                                int old_, size_t obytes, f32x16 (&ak)[D / 32], f32x16 (&av)[D / 32],
                                                Init init) {
    constexpr int KH = D / 2, NC = D / 32;
    const int l2 = second_walk(l), h2 = l2 >> 5, li2 = l2 & 31;
    const rsrc_t rQ = make_rsrc(Q + ib, hbytes), rdO = make_rsrc(dO + ob, obytes);
    const rsrc_t rP = make_rsrc(Attn + (size_t)bh * L * L, (size_t)L * L * 4);
    float v[KH];
    ldr_rows<D>(make_rsrc(V + ib, hbytes), (li2 * ild + h2 * KH) * 4, J * 32 * ild * 4, v);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        ak[c] = splat16(0.f);
        av[c] = splat16(0.f);
    }
#pragma unroll 1
    for (int I = 0; I < nbr; ++I) {
        float go[KH], p[16], b[NC][16], ds[16];
        ldr_rows<D>(rdO, (li2 * old_ + h2 * KH) * 4, I * 32 * old_ * 4, go);
        ldr_4x4(rP, (li2 * L + 4 * h2) * 4, (J * 32 * L + I * 32) * 4, p);
        const f32x16 dp = mma_feat_f32<D>(go, v, init(I, li2, h2, rdO));
#pragma unroll
        for (int r = 0; r < 16; ++r) ds[r] = dp[r] * p[r];
        ldr_tile_b<D>(rdO, (4 * h2 * old_ + li2) * 4, I * 32 * old_ * 4, b, old_);
#pragma unroll
        for (int c = 0; c < NC; ++c) av[c] = mma_chain(b[c], p, av[c]);
        ldr_tile_b<D>(rQ, (4 * h2 * ild + li2) * 4, I * 32 * ild * 4, b, ild);
#pragma unroll
        for (int c = 0; c < NC; ++c) ak[c] = mma_chain(b[c], ds, ak[c]);
    }
}

// three work-groups of four wavefronts to a CU (d = 32: 50 KB of LDS each), one of eight (d = 64: 135 KB)
#define SPION_GROUP_KERNEL(D) \
    __global__ __launch_bounds__(8 * (D)) __attribute__((amdgpu_waves_per_eu((D) == 32 ? 3 : 2, (D) == 32 ? 3 : 2)))

// Row pass: dQ, and -g for the column pass.  A wavefront past the last strip (nbr not a multiple of G) repeats the last one,
// since the others need its share of the tiles, and stores nothing.
template <int D>
SPION_GROUP_KERNEL(D) void dense_group_row_kernel(
    const float* __restrict__ K, const float* __restrict__ V, const float* __restrict__ Attn,
    const float* __restrict__ dO, const float* __restrict__ Out, float* __restrict__ Gs, float* __restrict__ dQ, int L,
    int nbr, int NB, float scale, Layouts ly) {
    constexpr int KH = D / 2, NC = D / 32, G = D / 8;
    typedef GroupTiles<D> GT;
    typedef DmaTile<D> Plane;
    constexpr int PBUF = D == 32 ? 1 : 2;  // map tiles in LDS
    __shared__ __attribute__((aligned(16))) char smem[GT::BYTES + G * PBUF * DmaTileF32::TILE];
    const int ng = (nbr + G - 1) / G;
    const int item = xcd_remap(blockIdx.x, ng * NB);
    const int bh = NB - 1 - item / ng;
    const int w = wave_index(), l = threadIdx.x & 63, h = l >> 5, li = l & 31;
    const int Iw = (item % ng) * G + w, I = min(Iw, nbr - 1);
    size_t ib, ob, gb, hbytes, obytes, gbytes;
    int ild, old_, gld;
    head_slice<true, D>(ly.in, ly.H, bh, L, ib, ild, hbytes);
    head_slice<true, D>(ly.out, ly.H, bh, L, ob, old_, obytes);
    head_slice<true, D>(ly.grad, ly.H, bh, L, gb, gld, gbytes);
    const rsrc_t rdO = make_rsrc(dO + ob, obytes);
    const GT tiles(smem, w, l, rsrc_words(V + ib, hbytes), ild, rsrc_words(K + ib, hbytes), ild);
    const u32x4 wP = rsrc_words(Attn + (size_t)bh * L * L, (size_t)L * L * 4);
    const char* Tp = smem + GT::BYTES + w * PBUF * DmaTileF32::TILE;
    const unsigned lp = lds_address(Tp);
    const int pl = DmaTileF32::voff(l, L), px = DmaTileF32::extra_step(L);
    const auto a_p = DmaTileF32::cols_addr(Tp, li, h);
    auto issue_p = [&](int J) { DmaTileF32::load<true>(wP, lp + J % PBUF * DmaTileF32::TILE, pl, (J * 32 * L + I * 32) * 4, px); };
    const auto ra = Plane::row_addr(li, h);
    const auto ta = Plane::tr_addr(l);

    tiles.issue(0);
    Split3<KH> gk;
    float g = 0.f;
    {
        float go[KH], oo[KH];
        ldr_rows<D>(rdO, (li * old_ + h * KH) * 4, I * 32 * old_ * 4, go);
        ldr_rows<D>(make_rsrc(Out + ob, obytes), (li * old_ + h * KH) * 4, I * 32 * old_ * 4, oo);
#pragma unroll
        for (int s = 0; s < KH; ++s) g = fmaf(go[s], oo[s], g);
        gk = split3(go);
    }
    g += __shfl_xor(g, 32, 64);
    if (h == 0 && Iw < nbr) Gs[(size_t)bh * L + I * 32 + li] = -g;
    const f32x16 gneg = splat16(-g);
    f32x16 acc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = splat16(0.f);

    f32x4 raw[2];
    settle(gk);
    wait_vm<0>();
    tiles.take(raw);
    wait_lgkm0();
    issue_p(0);
    if (nbr > 1) {
        tiles.issue(1);
        if (PBUF > 1) issue_p(1);
    }
    tiles.put(raw, 0);
    group_barrier();
    auto step = [&](int J, auto par) {
        constexpr int PAR = decltype(par)::value;
        // this step's map tile and this wavefront's part of the next step's operands; a map tile after them may be on its way
        if (PBUF > 1 && J + 1 < nbr) wait_vm<4>();
        else wait_vm<0>();
        float p[16];
        DmaTileF32::get(a_p, p, PAR % PBUF * DmaTileF32::TILE);
        tiles.take(raw);
        wait_lgkm0();
        if (J + 2 < nbr) tiles.issue(J + 2);
        if (J + PBUF < nbr) issue_p(J + PBUF);
        __builtin_amdgcn_sched_barrier(0);
        f32x16 dp = mma_rows<D>(tiles.planes(PAR, 0), ra, gk, gneg);  // register = key, lane = query: dO_i . v_j - g_i
        tiles.put(raw, PAR ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        float ds[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) ds[r] = dp[r] * p[r];
        mma_cols<D>(tiles.planes(PAR, 1), ta, split3(ds), acc);
        group_barrier();
    };
    for (int J = 0; J < nbr; J += 2) {
        step(J, std::integral_constant<int, 0>());
        if (J + 1 < nbr) step(J + 1, std::integral_constant<int, 1>());
    }
    if (split_failed(acc)) dense_row_again<D>(K, V, Attn, dO, L, nbr, I, bh, second_walk(l), gneg, ib, ild, hbytes, ob, old_, obytes, acc);
    if (Iw < nbr) {
#pragma unroll
        for (int c = 0; c < NC; ++c) reduce_store_rows<1>(acc[c] * scale, dQ + gb + 32 * c, I * 32, w, li, h, nullptr, gld);
    }
}

// Column pass: dK and dV.
template <int D>
SPION_GROUP_KERNEL(D) void dense_group_col_kernel(
    const float* __restrict__ Q, const float* __restrict__ V, const float* __restrict__ Attn,
    const float* __restrict__ dO, const float* __restrict__ Gs, float* __restrict__ dK, float* __restrict__ dV, int L,
    int nbr, int NB, float scale, Layouts ly) {
    constexpr int KH = D / 2, NC = D / 32, G = D / 8;
    typedef GroupTiles<D> GT;
    typedef DmaTile<D> Plane;
    constexpr int PBUF = D == 32 ? 1 : 2, WP = PBUF * DmaTileF32::TILE + 2 * 256;  // map tiles and 32 values of -g, twice
    __shared__ __attribute__((aligned(16))) char smem[GT::BYTES + G * WP];
    const int ng = (nbr + G - 1) / G;
    const int item = xcd_remap(blockIdx.x, ng * NB);
    const int bh = item / ng;
    const int w = wave_index(), l = threadIdx.x & 63, h = l >> 5, li = l & 31;
    const int Jw = (item % ng) * G + w, J = min(Jw, nbr - 1);
    size_t ib, ob, gb, hbytes, obytes, gbytes;
    int ild, old_, gld;
    head_slice<true, D>(ly.in, ly.H, bh, L, ib, ild, hbytes);
    head_slice<true, D>(ly.out, ly.H, bh, L, ob, old_, obytes);
    head_slice<true, D>(ly.grad, ly.H, bh, L, gb, gld, gbytes);
    const rsrc_t rV = make_rsrc(V + ib, hbytes);
    const GT tiles(smem, w, l, rsrc_words(dO + ob, obytes), old_, rsrc_words(Q + ib, hbytes), ild);
    const u32x4 wP = rsrc_words(Attn + (size_t)bh * L * L, (size_t)L * L * 4), wG = rsrc_words(Gs + (size_t)bh * L, (size_t)L * 4);
    const char* Tp = smem + GT::BYTES + w * WP;
    const unsigned lp = lds_address(Tp);
    const int pl = DmaTileF32::voff(l, L), px = DmaTileF32::extra_step(L);
    const auto a_p = DmaTileF32::own_addr(Tp, li, h, 2);  // P[query acc_row(r, h)][key li]
    const char* a_g = Tp + PBUF * DmaTileF32::TILE + 16 * h;
    auto issue_p = [&](int I) { DmaTileF32::load<true>(wP, lp + I % PBUF * DmaTileF32::TILE, pl, (J * 32 * L + I * 32) * 4, px); };
    auto issue_g = [&](int I) { dma_b32(wG, lp + PBUF * DmaTileF32::TILE + (I & 1) * 256, l * 4, I * 128); };
    const auto ra = Plane::row_addr(li, h);
    const auto ta = Plane::tr_addr(l);

    tiles.issue(0);
    Split3<KH> vk;
    {
        float v[KH];
        ldr_rows<D>(rV, (li * ild + h * KH) * 4, J * 32 * ild * 4, v);
        vk = split3(v);
    }
    f32x16 ak[NC], av[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        ak[c] = splat16(0.f);
        av[c] = splat16(0.f);
    }
    f32x4 raw[2];
    settle(vk);
    wait_vm<0>();
    tiles.take(raw);
    wait_lgkm0();
    issue_g(0);
    issue_p(0);
    if (nbr > 1) {
        tiles.issue(1);
        if (PBUF > 1) issue_p(1);
    }
    tiles.put(raw, 0);
    group_barrier();
    auto step = [&](int I, auto par) {
        constexpr int PAR = decltype(par)::value;
        if (PBUF > 1 && I + 1 < nbr) wait_vm<4>();
        else wait_vm<0>();
        float p[16];
        DmaTileF32::get(a_p, p, PAR % PBUF * DmaTileF32::TILE);
        tiles.take(raw);
        wait_lgkm0();
        if (I + 2 < nbr) tiles.issue(I + 2);
        if (I + 1 < nbr) issue_g(I + 1);
        if (I + PBUF < nbr) issue_p(I + PBUF);
        __builtin_amdgcn_sched_barrier(0);
        mma_cols<D>(tiles.planes(PAR, 0), ta, split3(p), av);
        __builtin_amdgcn_sched_barrier(0);
        f32x16 init;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(a_g + PAR * 256 + 32 * g);
            init[4 * g + 0] = x.x;
            init[4 * g + 1] = x.y;
            init[4 * g + 2] = x.z;
            init[4 * g + 3] = x.w;
        }
        const f32x16 dp = mma_rows<D>(tiles.planes(PAR, 0), ra, vk, init);  // register = query, lane = key: dO_i . v_j - g_i
        tiles.put(raw, PAR ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        float ds[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) ds[r] = dp[r] * p[r];
        mma_cols<D>(tiles.planes(PAR, 1), ta, split3(ds), ak);
        group_barrier();
    };
    for (int I = 0; I < nbr; I += 2) {
        step(I, std::integral_constant<int, 0>());
        if (I + 1 < nbr) step(I + 1, std::integral_constant<int, 1>());
    }
    if (split_failed(ak) || split_failed(av)) {
        const rsrc_t rG = make_rsrc(Gs + (size_t)bh * L, (size_t)L * 4);
        dense_col_again<D>(Q, V, Attn, dO, L, nbr, J, bh, l, ib, ild, hbytes, ob, old_, obytes, ak, av,
                           [&](int I, int, int h2, const rsrc_t&) {
                               float gi[16];
                               ldr_4x4(rG, 16 * h2, I * 128, gi);
                               f32x16 init;
#pragma unroll
                               for (int r = 0; r < 16; ++r) init[r] = gi[r];
                               return init;
                           });
    }
    if (Jw < nbr) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            reduce_store_rows<1>(ak[c] * scale, dK + gb + 32 * c, J * 32, w, li, h, nullptr, gld);
            reduce_store_rows<1>(av[c], dV + gb + 32 * c, J * 32, w, li, h, nullptr, gld);
        }
    }
}

}  // namespace spion
