// Backward of the dense phase for row-major heads of 32 features in one walk over the map: a work-group owns G neighbouring
// strips of 32 keys of one head, one to a wavefront, as the column pass of dense_group_kernels.h does, and besides dK and dV
// leaves what its keys add to dQ; a second launch adds these parts.
//
// Why: the row pass and the column pass read the map, 4 L^2 bytes a head, once each and form dO.V^T twice; together they take
// three operand splits a tile (dS' twice, P).  Here a tile is read once, dS' is formed and split once -- its parts go through LDS
// to change sides for the product with K -- and the row sums g come from the operand tiles as they are split, so nothing is
// handed from launch to launch but the parts: ceil(L / 32 G) of [L][32] a head, a quarter (G = 4) or an eighth (G = 8) of the map's
// bytes, written once and read once.
// A step (one tile of 32 queries for all G strips) has two barriers: before the first one the products dO.V^T, P^T.dO and K^T.dS'^T,
// each wavefront by itself; between them the G partial tiles of dQ are added, the next operand tile is split, and the product
// dS'^T.Q, whose operands are in registers by then, keeps the matrix pipe busy meanwhile.
// Measured, us of a backward, row and column pass / G = 4 / G = 8, one machine: 128 heads of 1024 306 / 255 / 247, 32 of 2048 305 /
// 251 / 238, 256 of 512 159 / 136 / 132 (dense_attn.hip has more at the rule that picks one); the addition of the parts is 12 us of
// it at 128 heads of 1024 (G = 8; 22 with G = 4).
// Bound: two wavefronts to a SIMD (214 registers), each in one chain of LDS reads, products and splits: matrix pipe 47 %, issue of
// all kinds 63 % busy at 1.95 GHz, a sixth of the time at LDS waits.  Measured beside it: a quarter of the dQ tile to a wavefront
// over the keys of all four (16x16 products, dS' read by all) 430 against 424 us a step; the product with Q before the first barrier
// 434; the map tile in registers a step ahead +-0.
#pragma once
#include "dense_group_kernels.h"
#include "gather_ops.h"

namespace spion {

// dS' of a strip, transposed on its way through LDS: written as it is computed (lane = key, register = query), read back with
// lane = query.  Three planes of 32 keys x 32 queries in bf16, 64-byte rows; 8-byte piece (c, h) of row r lies at
// (c ^ r/4 % 4, h ^ r/16), which frees the writes (a column of pieces) and the transposing reads (four rows, all pieces) of
// bank conflicts.
struct DsTile {
    static constexpr int PLANE = 2048, TILE = 3 * PLANE;
    __device__ static __forceinline__ int put_addr(int li, int h, int c) {
        return li * 64 + 16 * (c ^ ((li >> 2) & 3)) + 8 * (h ^ (li >> 4));
    }
    struct Addr {
        int a[2][2];
    };
    __device__ static __forceinline__ Addr get_addr(int l) {  // as DmaTile::tr_addr, rows 16 t + 8 u + 4 h + j/4
        const int h = l >> 5, gm = (l >> 4) & 1, j = l & 15;
        Addr x;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int row = 16 * t + 8 * u + 4 * h + (j >> 2);
                x.a[t][u] = row * 64 + 16 * ((2 * gm + ((j & 3) >> 1)) ^ ((row >> 2) & 3)) + 8 * ((j & 1) ^ t);
            }
        return x;
    }
    __device__ static __forceinline__ bf16x8 get(const char* plane, const Addr& x, int t) {
        typedef s16x4 __attribute__((address_space(3))) * lds_ptr;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(plane + x.a[t][0]));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(plane + x.a[t][1]));
        return __builtin_shufflevector(__builtin_bit_cast(bf16x4, lo), __builtin_bit_cast(bf16x4, hi), 0, 1, 2, 3, 4, 5, 6, 7);
    }
};

// part: [ceil(nbr / G)][NB][L][32], what the work-groups of a head add to dQ (not yet scaled).
template <int G>
__global__ __launch_bounds__(64 * G) __attribute__((amdgpu_waves_per_eu(2, 2))) void dense_group_col_dq_kernel(
    const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V, const float* __restrict__ Attn,
    const float* __restrict__ dO, const float* __restrict__ Out, float* __restrict__ dK, float* __restrict__ dV,
    float* __restrict__ part, int L, int nbr, int NB, float scale, Layouts ly) {
    constexpr int D = 32, KH = D / 2;
    typedef DmaTile<D> Plane;
    static_assert(G == 4 || G == 8);
    constexpr int RAW = 4 * 4096, SPLIT = 3 * Plane::TILE, GN = 256;
    __shared__ __attribute__((aligned(16))) char smem[RAW + 2 * SPLIT + GN + G * (DmaTileF32::TILE + DsTile::TILE)];
    char* const planes0 = smem + RAW;           // dO
    char* const planes1 = planes0 + SPLIT;      // Q
    float* const gneg = reinterpret_cast<float*>(planes1 + SPLIT);
    char* const ptiles = planes1 + SPLIT + GN;  // the map tile of each wavefront
    char* const dstiles = ptiles + G * DmaTileF32::TILE;  // its dS', then what it adds to dQ

    const int ng = (nbr + G - 1) / G;
    const int item = xcd_remap(blockIdx.x, ng * NB);
    const int bh = item / ng, grp = item - bh * ng;
    const int w = wave_index(), l = threadIdx.x & 63, h = l >> 5, li = l & 31;
    const int Jw = grp * G + w, J = min(Jw, nbr - 1);
    size_t ib, ob, gb, hbytes, obytes, gbytes;
    int ild, old_, gld;
    head_slice<true, D>(ly.in, ly.H, bh, L, ib, ild, hbytes);
    head_slice<true, D>(ly.out, ly.H, bh, L, ob, old_, obytes);
    head_slice<true, D>(ly.grad, ly.H, bh, L, gb, gld, gbytes);

    // operand tiles, eight rows to a wavefront, a lane 16 bytes: dO (with Out, for -g) and Q (the second one's last load and sum
    // are of no use), both (G = 4) or one of them (G = 8: dO by the first four)
    constexpr int R = 8 / G;
    const int w4 = w & 3, row = w4 * 8 + (l >> 3), c = l & 7;
    const u32x4 wQ = rsrc_words(Q + ib, hbytes);
    u32x4 wX[R], wZ[R];
    int xld[R], vx[R];
    char* dst[R];
    float* gdst[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const bool first = R == 2 ? k == 0 : w < 4;
        xld[k] = first ? old_ : ild;
        wX[k] = first ? rsrc_words(dO + ob, obytes) : wQ;
        wZ[k] = first ? rsrc_words(Out + ob, obytes) : wQ;
        vx[k] = ((l >> 3) * xld[k] + 4 * c) * 4;
        dst[k] = (first ? planes0 : planes1) + row * Plane::ROW + 16 * ((c >> 1) ^ Plane::swz(row)) + 8 * (c & 1);
        gdst[k] = gneg + (first ? 0 : 32) + row;
    }
    char* const raw = smem + w * R * 2048;
    const unsigned lraw = lds_address(raw);
    auto issue = [&](int tile) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int so = (tile * 32 + w4 * 8) * xld[k] * 4;
            dma_b128(wX[k], lraw + k * 2048, vx[k], so);
            if (R == 1 || k == 0) dma_b128(wZ[k], lraw + k * 2048 + 1024, vx[k], so);
        }
    };
    auto take = [&](f32x4 (&x)[R], f32x4 (&z)[R]) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            x[k] = *reinterpret_cast<const f32x4*>(raw + k * 2048 + l * 16);
            if (R == 1 || k == 0) z[k] = *reinterpret_cast<const f32x4*>(raw + k * 2048 + 1024 + l * 16);
        }
    };
    auto put = [&](const f32x4 (&x)[R], const f32x4 (&z)[R]) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float a[4] = {x[r].x, x[r].y, x[r].z, x[r].w};
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
                *reinterpret_cast<u32x2*>(dst[r] + k * Plane::TILE) = v;
            }
            if (R == 2 && r == 1) continue;
            float g = x[r].x * z[r].x;
            g = fmaf(x[r].y, z[r].y, g);
            g = fmaf(x[r].z, z[r].z, g);
            g = fmaf(x[r].w, z[r].w, g);
            *gdst[r] = -gather_group_sum<8>(g);  // (the same value from all eight lanes of a row)
        }
    };
    const u32x4 wP = rsrc_words(Attn + (size_t)bh * L * L, (size_t)L * L * 4);
    const char* Tp = ptiles + w * DmaTileF32::TILE;
    const unsigned lp = lds_address(Tp);
    const int pl = DmaTileF32::voff(l, L), px = DmaTileF32::extra_step(L);
    const auto a_p = DmaTileF32::own_addr(Tp, li, h, 2);  // P[query acc_row(r, h)][key li]
    auto issue_p = [&](int I) { DmaTileF32::load<true>(wP, lp, pl, (J * 32 * L + I * 32) * 4, px); };
    const auto ra = Plane::row_addr(li, h);
    const auto ta = Plane::tr_addr(l);
    char* const Td = dstiles + w * DsTile::TILE;
    int pd[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) pd[g] = DsTile::put_addr(li, h, g);
    const auto da = DsTile::get_addr(l);
    const auto a_dq = DmaTileF32::own_addr(Td, li, h, 2);
    // this wavefront's share of a dQ tile: 32 / G rows, a lane G / 4 pieces of 4 G bytes .. 16 bytes (G = 4), 8 (G = 8)
    constexpr int LPR = 2 * G;  // lanes to a row
    const int srow = w * (32 / G) + l / LPR, sc = l % LPR;
    const char* const rd = dstiles + srow * 128 + (G == 4 ? 16 * (sc ^ (srow & 7)) : 16 * ((sc >> 1) ^ (srow & 7)) + 8 * (sc & 1));
    float* const dq = part + (((size_t)grp * NB + bh) * L + srow) * D + sc * (32 / LPR);

    issue(0);
    Split3<KH> vk;
    Split3<16> kt;
    {
        float v[KH], k[1][16];
        ldr_rows<D>(make_rsrc(V + ib, hbytes), (li * ild + h * KH) * 4, J * 32 * ild * 4, v);
        ldr_tile_b<D>(make_rsrc(K + ib, hbytes), (4 * h * ild + li) * 4, J * 32 * ild * 4, k, ild);
        if (Jw >= nbr) {  // no such strip: adds nothing to dQ
#pragma unroll
            for (int e = 0; e < 16; ++e) k[0][e] = 0.f;
        }
        vk = split3(v);
        kt = split3(k[0]);
    }
    settle(vk);
    settle(kt);
    f32x16 ak[1] = {splat16(0.f)}, av[1] = {splat16(0.f)};
    wait_vm<0>();
    issue_p(0);
    {
        f32x4 x[R], z[R];
        take(x, z);
        wait_lgkm0();
        issue(min(1, nbr - 1));
        put(x, z);
    }
    group_barrier();
    for (int I = 0; I < nbr; ++I) {
        wait_vm<2>();  // the map tile of this step; operands of the next one may be on their way
        float p[16];
        DmaTileF32::get(a_p, p);
        wait_lgkm0();
        issue_p(min(I + 1, nbr - 1));
        __builtin_amdgcn_sched_barrier(0);
        f32x16 init;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(gneg + 4 * h + 8 * g);
            init[4 * g + 0] = x.x;
            init[4 * g + 1] = x.y;
            init[4 * g + 2] = x.z;
            init[4 * g + 3] = x.w;
        }
        const f32x16 dp = mma_rows<D>(planes0, ra, vk, init);  // register = query, lane = key: dO_i . v_j - g_i
        const Split3<16> sp = split3(p);
        __builtin_amdgcn_sched_barrier(0);
        mma_cols<D>(planes0, ta, sp, av);
        float ds[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) ds[r] = dp[r] * p[r];
        const Split3<16> sd = split3(ds);
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const u32x4 x = __builtin_bit_cast(u32x4, sd.p[k][t]);
                *reinterpret_cast<u32x2*>(Td + pd[2 * t] + k * DsTile::PLANE) = (u32x2){x.x, x.y};
                *reinterpret_cast<u32x2*>(Td + pd[2 * t + 1] + k * DsTile::PLANE) = (u32x2){x.z, x.w};
            }
        __builtin_amdgcn_sched_barrier(0);
        Split3<16> qt, st;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            bf16x8 x[1][2];
            Plane::get_tile_t(planes1 + k * Plane::TILE, ta, x);
            qt.p[k][0] = x[0][0];
            qt.p[k][1] = x[0][1];
        }
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int t = 0; t < 2; ++t) st.p[k][t] = DsTile::get(Td + k * DsTile::PLANE, da, t);
        const f32x16 dqt = mma_split(kt, st, splat16(0.f));  // register = feature, lane = query
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<f32x4*>(const_cast<char*>(a_dq.a[g])) = (f32x4){dqt[4 * g], dqt[4 * g + 1], dqt[4 * g + 2], dqt[4 * g + 3]};
        group_barrier();  // all parts of the dQ tile are there, the operand planes are free
        wait_vm<4>();
        f32x4 x[R], z[R];
        take(x, z);
        typedef float part_t __attribute__((ext_vector_type(G == 4 ? 4 : 2)));
        part_t pp[G];
#pragma unroll
        for (int i = 0; i < G; ++i) pp[i] = *reinterpret_cast<const part_t*>(rd + i * DsTile::TILE);
        __builtin_amdgcn_sched_barrier(0);
        f32x16 t = mma_split(qt, sd, splat16(0.f));
        put(x, z);
        part_t s = pp[0];
#pragma unroll
        for (int i = 1; i < G; ++i) s += pp[i];
        ak[0] += t;
        wait_lgkm0();
        issue(min(I + 2, nbr - 1));
        *reinterpret_cast<part_t*>(dq + (size_t)I * 32 * D) = s;
        group_barrier();  // the next step's operands are there, the parts are free
    }
    wait_vm<0>();
    if (split_failed(ak) || split_failed(av)) {
        dense_col_again<D>(Q, V, Attn, dO, L, nbr, J, bh, l, ib, ild, hbytes, ob, old_, obytes, ak, av,
                           [&](int I, int li2, int h2, const rsrc_t& rdO) {
                               float go[KH], oo[KH], g = 0.f;
                               ldr_rows<D>(rdO, (li2 * old_ + h2 * KH) * 4, I * 32 * old_ * 4, go);
                               ldr_rows<D>(make_rsrc(Out + ob, obytes), (li2 * old_ + h2 * KH) * 4, I * 32 * old_ * 4, oo);
#pragma unroll
                               for (int s = 0; s < KH; ++s) g = fmaf(go[s], oo[s], g);
                               g += __shfl_xor(g, 32, 64);
                               f32x16 init;
#pragma unroll
                               for (int r = 0; r < 16; ++r) init[r] = -__shfl(g, acc_row(r, h2), 64);
                               return init;
                           });
    }
    if (Jw < nbr) {
        reduce_store_rows<1>(ak[0] * scale, dK + gb, J * 32, w, li, h, nullptr, gld);
        reduce_store_rows<1>(av[0], dV + gb, J * 32, w, li, h, nullptr, gld);
    }
}

// dQ: the sum of the C parts, a wavefront to 32 rows.
__global__ __launch_bounds__(256) void dense_group_row_sum_kernel(
    const float* __restrict__ K, const float* __restrict__ V, const float* __restrict__ Attn, const float* __restrict__ dO,
    const float* __restrict__ Out, const float* __restrict__ part, float* __restrict__ dQ, int C, int L, int nbr, int NB,
    float scale, Layouts ly) {
    constexpr int D = 32, KH = D / 2;
    const int l = threadIdx.x & 63;
    const int strip = blockIdx.x * 4 + wave_index();
    if (strip >= nbr * NB) return;
    const int bh = strip / nbr, I = strip - bh * nbr;
    size_t ib, ob, gb, hbytes, obytes, gbytes;
    int ild, old_, gld;
    head_slice<true, D>(ly.grad, ly.H, bh, L, gb, gld, gbytes);
    const f32x4* p = reinterpret_cast<const f32x4*>(part + (size_t)strip * 32 * D) + l;
    const size_t step = (size_t)NB * L * D / 4;
    f32x4 s[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) s[k] = p[64 * k];
    p += step;
    for (int i = 1; i < C; ++i, p += step) {
#pragma unroll
        for (int k = 0; k < 4; ++k) s[k] += p[64 * k];
    }
    f32x16 all[1];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) all[0][4 * k + j] = s[k][j];
    if (split_failed(all)) {
        head_slice<true, D>(ly.in, ly.H, bh, L, ib, ild, hbytes);
        head_slice<true, D>(ly.out, ly.H, bh, L, ob, old_, obytes);
        const int l2 = second_walk(l), h2 = l2 >> 5, li2 = l2 & 31;
        float go[KH], oo[KH], g = 0.f;
        ldr_rows<D>(make_rsrc(dO + ob, obytes), (li2 * old_ + h2 * KH) * 4, I * 32 * old_ * 4, go);
        ldr_rows<D>(make_rsrc(Out + ob, obytes), (li2 * old_ + h2 * KH) * 4, I * 32 * old_ * 4, oo);
#pragma unroll
        for (int s = 0; s < KH; ++s) g = fmaf(go[s], oo[s], g);
        g += __shfl_xor(g, 32, 64);
        dense_row_again<D>(K, V, Attn, dO, L, nbr, I, bh, l2, splat16(-g), ib, ild, hbytes, ob, old_, obytes, all);
        reduce_store_rows<1>(all[0] * scale, dQ + gb, I * 32, 0, li2, h2, nullptr, gld);
        return;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
        *reinterpret_cast<f32x4*>(dQ + gb + (size_t)(I * 32 + 8 * k + (l >> 3)) * gld + 4 * (l & 7)) = s[k] * scale;
}

}  // namespace spion
