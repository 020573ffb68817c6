// 32 x D bf16 tiles in LDS: their layout, the loads that fill them and the two kinds of operand reads.
#pragma once
#include "tile_ops.h"

namespace spion {

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// -------------------------------------------------------------------------------------------------
// Tiles that go from global memory straight into LDS (buffer loads with the LDS modifier): no registers hold a
// tile in flight and no ds_write is spent on it.  One instruction moves 64 x 16 bytes to 1 KB of consecutive LDS
// addresses starting at M0 (+ the instruction's immediate offset, which is added to the global address as well);
// which 16-byte piece of global memory a lane fetches is free, so the LDS image of a tile is unpadded rows with
// the pieces of a row permuted: piece c of tile row r lies at position c ^ swz(r).  With that permutation the
// transposing reads (four consecutive rows of two adjacent pieces, thirty-two lanes at a time) are free of bank
// conflicts; the 16-byte reads of an operand over the head dimension (sixteen consecutive rows of one piece at a
// time, 64 banks) meet rows r and r + 8 on the same banks and take 8 cycles instead of 4 -- measured, and measured
// not to matter: the LDS pipe is a third busy in these kernels.
// The loads are inline assembly, so the compiler neither tracks them in its s_waitcnt bookkeeping nor knows that
// they write LDS: the kernels wait for them with wait_vm<N> (N = loads issued after the ones waited for; loads
// return in order, and the compiler's own counts can only wait longer than needed) and order them against their
// LDS reads with wait_lgkm0; both carry a memory clobber, so no LDS access moves across them.
// -------------------------------------------------------------------------------------------------
template <int D>
struct DmaTile {
    static constexpr int ROW = D * 2;     // bytes per LDS row
    static constexpr int TILE = 32 * ROW;  // 2 KB (D = 32) or 4 KB (D = 64)
    static constexpr int CPR = D / 8;      // 16-byte pieces per row
    static constexpr int NI = D / 16;      // instructions per tile, 64 / CPR rows each
    __device__ static __forceinline__ int swz(int row) {
        if constexpr (D == 64) return ((row & 3) << 1) | ((row >> 2) & 1);
        else return (((row >> 1) & 1) << 1) | ((row >> 2) & 1);
    }
    // Lane offset into the head slice (bytes): lane l fills LDS piece l of every instruction's 1 KB, i.e. position
    // l % CPR of row l / CPR (+ 64 / CPR rows per instruction), with the global piece that belongs there.
    __device__ static __forceinline__ int voff(int l, int ld) {
        const int r = l / CPR, c = (l % CPR) ^ swz(r);
        return (r * ld + c * 8) * 2;
    }
    // what the scalar offset advances by from one instruction to the next, beyond the 1024 its immediate adds
    __device__ static __forceinline__ int extra_step(int ld) { return (64 / CPR) * ld * 2 - 1024; }
    __device__ static __forceinline__ void load(u32x4 r, unsigned lds, int lvoff, int soff, int xstep) {
        if constexpr (D == 64)
            asm volatile(
                "s_mov_b32 m0, %0\n\ts_nop 3\n\t"
                "buffer_load_dwordx4 %1, %2, %3 offen lds\n\t"
                "buffer_load_dwordx4 %1, %2, %4 offen offset:1024 lds\n\t"
                "buffer_load_dwordx4 %1, %2, %5 offen offset:2048 lds\n\t"
                "buffer_load_dwordx4 %1, %2, %6 offen offset:3072 lds" ::"s"(lds),
                "v"(lvoff), "s"(r), "s"(soff), "s"(soff + xstep), "s"(soff + 2 * xstep), "s"(soff + 3 * xstep)
                : "memory");
        else
            asm volatile(
                "s_mov_b32 m0, %0\n\ts_nop 3\n\t"
                "buffer_load_dwordx4 %1, %2, %3 offen lds\n\t"
                "buffer_load_dwordx4 %1, %2, %4 offen offset:1024 lds" ::"s"(lds),
                "v"(lvoff), "s"(r), "s"(soff), "s"(soff + xstep)
                : "memory");
    }
    // Byte offsets of lane (row li, half h) for its operand over the head dimension: features h*D/2 + 8t .. of row
    // li, t = 0 .. D/16-1 (piece h*CPR/2 + t).
    struct RowAddr {
        int a[D / 16];
    };
    __device__ static __forceinline__ RowAddr row_addr(int li, int h) {
        RowAddr x;
#pragma unroll
        for (int t = 0; t < D / 16; ++t) x.a[t] = li * ROW + 16 * ((h * (CPR / 2) + t) ^ swz(li));
        return x;
    }
    __device__ static __forceinline__ void get_rows(const char* T, const RowAddr& ra, bf16x8 (&x)[D / 16]) {
#pragma unroll
        for (int t = 0; t < D / 16; ++t) x[t] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(T + ra.a[t]));
    }
    // Transposing reads (see LdsTile::get_tile_t): lane j of a group of 16 points at features F + 4(j%4) .. +3 of
    // row R + j/4, R = 4h (+ 16t, + 8), F = 16*((l/16)%2) (+ 32c): 8 bytes inside piece 2*((l/16)%2) + (j%4)/2
    // (+ 4c).  Rows 8 apart share their permutation, so the row steps stay immediate offsets.
    struct TrAddr {
        int a[D / 32];
    };
    __device__ static __forceinline__ TrAddr tr_addr(int l) {
        const int h = l >> 5, gm = (l >> 4) & 1, j = l & 15, row = 4 * h + (j >> 2);
        TrAddr x;
#pragma unroll
        for (int c = 0; c < D / 32; ++c)
            x.a[c] = row * ROW + 16 * ((4 * c + 2 * gm + ((j & 3) >> 1)) ^ swz(row)) + 8 * (j & 1);
        return x;
    }
    __device__ static __forceinline__ void get_tile_t(const char* T, const TrAddr& ta, bf16x8 (&xt)[D / 32][2]) {
        typedef s16x4 __attribute__((address_space(3))) * lds_ptr;
#pragma unroll
        for (int c = 0; c < D / 32; ++c)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(T + ta.a[c] + (16 * t) * ROW));
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(T + ta.a[c] + (16 * t + 8) * ROW));
                xt[c][t] = __builtin_shufflevector(__builtin_bit_cast(bf16x4, lo), __builtin_bit_cast(bf16x4, hi), 0, 1,
                                                   2, 3, 4, 5, 6, 7);
            }
    }
    // LDS of one wavefront: two buffers of two tiles and 256 bytes of per-tile scalars (key penalties or row
    // statistics of the tile, 64 floats)
    static constexpr int BUF = 2 * TILE + 256;
    static constexpr int WAVE = 2 * BUF;
};

}  // namespace spion
