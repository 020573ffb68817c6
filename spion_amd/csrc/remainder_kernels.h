// The remainder of element-sparse patterns (hybrid_kernels.h; d = 32) with its gathered rows in LDS.
//
// What bounds it.  An entry costs two 128-byte rows (K and V of its column, or Q and dO of its row), 32 multiply-adds
// with each, and its index and weight.  The rows come from LDS: a work-group walks the sequence in ranges of REM_RANGE
// rows, of which it loads both operands (128 KB) straight into LDS, and owns NO x 256 rows (row-wise kernels) or columns
// (column pass) of the pattern, whose sums stay in registers across the ranges.  The four lanes of a quad take a row or
// column; lane i holds 8 of its 32 features (4 of either half) and i-th quarters of the index of its entries.
//
// Per entry and quad the wavefront spends 16 multiply-adds and 7 to 8 instructions that hand the entry round (DPP moves
// within the quad and the two or four LDS addresses, one exclusive-or each); the vector ALU is what is left as the bound
// (half of the slots of a visit are filled: the sixteen quads of a wavefront advance together, and of the ~10 entries a
// row has in a range the fullest of sixteen rows has ~15).  What kept the kernels from it:
//   * Latency.  The older kernels fetched an entry's index, then its weight, then worked, in one dependent chain
//     (SQ_WAIT_ANY 63 to 80 % of the resident cycles).  Here the index of the next visit and the weights it points to
//     are requested while the present visit is worked on, and a visit's index is one word per entry (rb_word, cb_word).
//   * Partly used lines.  The entries are ordered by range first (rb_: columns in ranges, then row, then column; cb_: rows
//     in ranges, then column, then row), so that neighbouring quads read and write neighbouring pieces of the compact lists
//     and the column pass finds the weights of a range, 39 KB, in the caches.
//   * Bank conflicts.  64 banks hold 256 bytes = four half rows, and the four quads that an instruction serves together
//     read one half row each.  Column pass: Q and dO of a row lie side by side (256 bytes), quad j takes its four half
//     rows in the order k ^ j: no conflicts whatever the rows.  Row-wise kernels, which need one operand before the other:
//     two rows of one operand side by side, quads take their halves in alternating order.
// Sums: a visit's entries are added by themselves and then to the row's sum (shorter chains: 2-norm errors against float64
// below those of the gather kernels).
#pragma once
#include "tile_kernels.h"

namespace spion {

constexpr int REM_RANGE = 512, REM_THREADS = 1024, REM_QUADS = REM_THREADS / 4;
constexpr int REM_BATCH = 16;  // entries of a quad in flight: four per lane
constexpr float HYB_ABSENT = -1.0e30f;  // logit of an entry that is not in the pattern: exp2 gives exactly 0

// The remainder's lists by ranges (device pointers, shared by all heads).  rb_off[k * L + i]: first entry of row i whose
// column lies in range k; rb_word: column in the range | (row % 32) << 9 | position in the CSR row << 14.  cb_off[k * L + j],
// cb_word: row in the range | (index in the rb list, less that of the first entry of the block of REM_RANGE x REM_RANGE) << 9.
// The word lists are readable REM_BATCH entries past their end.
struct RemIndex {
    const int* rb_off;
    const int* rb_word;
    const int* cb_off;
    const int* cb_word;
    int nr;  // entries per head
};

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef unsigned rem_u32x2 __attribute__((ext_vector_type(2)));

// x of lane CTRL / 0x55 of the own quad, or of a lane's partner (0xB1: lane ^ 1, 0x4E: lane ^ 2)
template <int CTRL>
__device__ __forceinline__ int quad_move(int x) {
    return __builtin_amdgcn_mov_dpp(x, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float quad_move(float x) {
    return __int_as_float(quad_move<CTRL>(__float_as_int(x)));
}
__device__ __forceinline__ float quad_sum(float x) {
    x += quad_move<0xB1>(x);
    return x + quad_move<0x4E>(x);
}

// LDS byte offset of row r of a range whose operands lie in pairs of rows: {A of 2m, A of 2m + 1, B of 2m, B of 2m + 1}
__device__ __forceinline__ int rem_pair_row(int r) { return (r >> 1) * 512 + (r & 1) * 128; }

// Rows [r0, r0 + REM_RANGE) of A and B, straight into LDS; rows past L repeat the last one (nothing reads them).  PAIRED: the
// layout of rem_pair_row; otherwise a row of A and the same row of B side by side.
template <bool PAIRED>
__device__ __forceinline__ void rem_load_range(const float* __restrict__ A, int lda, const float* __restrict__ B, int ldb,
                                               int r0, int L, f32x4* tile) {
    const int lane = threadIdx.x & 63, wave = wave_index(), piece = lane & 7;
#pragma unroll
    for (int k = 0; k < REM_RANGE * 16 / REM_THREADS; ++k) {  // 1 KB an instruction: four rows of both operands
        const int first = (wave * (REM_RANGE * 16 / REM_THREADS) + k) * 4;
        const int r = PAIRED ? ((lane >> 5) << 1) + ((lane >> 3) & 1) : lane >> 4;
        const bool second = (PAIRED ? lane >> 4 : lane >> 3) & 1;
        const int row = min(r0 + first + r, L - 1);
        const float* src = (second ? B + (size_t)row * ldb : A + (size_t)row * lda) + piece * 4;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)(tile + first * 16), 16, 0, 0);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
}

__device__ __forceinline__ f32x4 rem_lds(const f32x4* tile, int bytes) {
    return *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(tile) + bytes);
}
__device__ __forceinline__ i32x4 rem_words(rsrc_t r, int entry) {
    return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(r, entry * 4, 0, 0));
}
// {first entry, end} of element x (a row or column) of range k: nothing where x or the range does not exist
__device__ __forceinline__ i32x2 rem_span(rsrc_t r, int k, int x, int L) {
    const bool there = x < L && k * REM_RANGE < L;
    return __builtin_bit_cast(i32x2, __builtin_amdgcn_raw_buffer_load_b64(r, there ? (k * L + x) * 4 : -8, 0, 0));
}
__device__ __forceinline__ rsrc_t rem_span_rsrc(const int* off, int L) {
    return make_rsrc(off, ((size_t)((L + REM_RANGE - 1) / REM_RANGE) * L + 1) * 4);
}
__device__ __forceinline__ rsrc_t rem_word_rsrc(const int* w, int nr) { return make_rsrc(w, (size_t)(nr + REM_BATCH) * 4); }

// The kernels' loop: a quad visits its rows (columns) one after the other in every range, a visit taking REM_BATCH entries at
// a time (what the fullest quad of the wavefront needs).  While a batch is worked on (chunk i: the four entries of lane i),
// the words of the next one, of the same visit or of the next, are requested, half-way through turned into LDS addresses and
// the requests of their weights (convert), and at its end they become the present batch (take).

// -------------------------------------------------------------------------------------------------
// Forward: raw logits (log2 domain) of the remainder to Raw [NB][nr] in the order of the rb list, per row their maximum and
// the sum of their exponentials relative to it, Stats[bh][row] = {m, z} (z = 0 for a row without remainder), and sum e . V
// with the same exponentials into O.  The tile kernel that follows (hyb_tile_fwd_kernel) merges statistics and sums with its
// tiles'; rem_prob_kernel then makes the probabilities.
// A batch's maximum first, then its exponentials, each by the lane that owns the entry; the sums of the batches before are
// rescaled once a batch.  64 heads of 4096 rows with 76 entries: 139 us (logits) + 205 (P.V, probabilities) -> 174 + 75
// (rem_prob_kernel); vector ALU 79 % busy.
// -------------------------------------------------------------------------------------------------
template <bool MASK, bool ST, int NO>
__global__ __launch_bounds__(REM_THREADS) void rem_fwd_kernel(const float* __restrict__ Q, const float* __restrict__ K,
                                                              const float* __restrict__ V, KeyTerms keys,
                                                              float* __restrict__ Raw, float2* __restrict__ Stats,
                                                              float* __restrict__ O, RemIndex ix, int L, int NB, float scale,
                                                              Layouts ly) {
    __shared__ f32x4 tile[(REM_RANGE + 2) * 16];  // {K, K, V, V} per pair of rows; a pair of zeros for absent entries
    __shared__ float spen[MASK ? REM_RANGE + 1 : 1];
    constexpr int ROWS = NO * REM_QUADS;
    const int nrg = (L + ROWS - 1) / ROWS;
    const int item = xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int bh = item / nrg, row0 = item % nrg * ROWS + (threadIdx.x >> 2);
    const int qi = threadIdx.x & 3, j = (threadIdx.x >> 2) & 1;
    size_t ib, ob, bytes;
    int ild, old_;
    head_slice<ST, 32>(ly.in, ly.H, bh, L, ib, ild, bytes);
    head_slice<ST, 32>(ly.out, ly.H, bh, L, ob, old_, bytes);
    const rsrc_t rSpan = rem_span_rsrc(ix.rb_off, L), rWord = rem_word_rsrc(ix.rb_word, ix.nr);
    const rsrc_t rRaw = make_rsrc(Raw + (size_t)bh * ix.nr, (size_t)ix.nr * 4);
    if (threadIdx.x < 32) tile[REM_RANGE * 16 + threadIdx.x] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (MASK && threadIdx.x == 0) spen[REM_RANGE] = 0.f;
    const int off0 = 64 * j + 16 * qi, off1 = off0 ^ 64;
    const float c2 = scale * LOG2E;
    f32x4 acc[NO][2], q[NO][2];
    float m[NO], z[NO];
#pragma unroll
    for (int c = 0; c < NO; ++c) {
        const int row = min(row0 + c * REM_QUADS, L - 1);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            acc[c][k] = (f32x4){0.f, 0.f, 0.f, 0.f};
            q[c][k] = reinterpret_cast<const f32x4*>(Q + ib + (size_t)row * ild)[(k ^ j) * 4 + qi] * c2;
        }
        m[c] = HYB_ABSENT;
        z[c] = 0.f;
    }
    int addr[4], first = 0, left = 0, cnt = 0;
    float v[4], pn[4];
    i32x4 nw;
    auto take = [&](i32x2 sp) {
        first = sp.x + 4 * qi;
        cnt = sp.y - sp.x;
        left = cnt - 4 * qi;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int col = s < left ? nw[s] & (REM_RANGE - 1) : REM_RANGE;
            addr[s] = rem_pair_row(col);
            if constexpr (MASK) pn[s] = spen[col];
        }
    };
    auto logits = [&](auto I, int c) {
        constexpr int i = decltype(I)::value, CT = 0x55 * i;
        if (!__any(cnt > 4 * i)) return;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int base = quad_move<CT>(addr[s]);
            const f32x4 k0 = rem_lds(tile, base ^ off0), k1 = rem_lds(tile, base ^ off1);
            float d = k0[0] * q[c][0][0], d1 = k1[0] * q[c][1][0];
#pragma unroll
            for (int x = 1; x < 4; ++x) d = fmaf(k0[x], q[c][0][x], d), d1 = fmaf(k1[x], q[c][1][x], d1);
            d = quad_sum(d + d1);
            v[s] = qi == i ? d : v[s];
        }
    };
    f32x4 t0, t1;
    auto values = [&](auto I, int) {
        constexpr int i = decltype(I)::value, CT = 0x55 * i;
        if (!__any(cnt > 4 * i)) return;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int base = quad_move<CT>(addr[s]);
            const f32x4 v0 = rem_lds(tile, (base ^ off0) + 256), v1 = rem_lds(tile, (base ^ off1) + 256);
            const float w = quad_move<CT>(v[s]);
#pragma unroll
            for (int x = 0; x < 4; ++x) t0[x] = fmaf(w, v0[x], t0[x]), t1[x] = fmaf(w, v1[x], t1[x]);
        }
    };
    auto batch = [&](int c) {
        logits(std::integral_constant<int, 0>{}, c);
        logits(std::integral_constant<int, 1>{}, c);
        logits(std::integral_constant<int, 2>{}, c);
        logits(std::integral_constant<int, 3>{}, c);
        float bm = HYB_ABSENT;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if constexpr (MASK) v[s] -= pn[s];
            if (s < left) bm = fmaxf(bm, v[s]);
        }
        // four at a time where all are there; of two and one the rest
        store_b128((f32x4){v[0], v[1], v[2], v[3]}, rRaw, left >= 4 ? first * 4 : -16, 0);
        const rem_u32x2 two = {__float_as_uint(v[0]), __float_as_uint(v[1])};
        __builtin_amdgcn_raw_buffer_store_b64(two, rRaw, left == 2 || left == 3 ? first * 4 : -8, 0, 0);
        st1(rRaw, left == 3 ? (first + 2) * 4 : left == 1 ? first * 4 : -4, 0, left == 3 ? v[2] : v[0]);
        bm = fmaxf(bm, quad_move<0xB1>(bm));
        bm = fmaxf(bm, quad_move<0x4E>(bm));
        const float mnew = fmaxf(m[c], bm), f = __builtin_amdgcn_exp2f(m[c] - mnew);
        float ez = 0.f;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            v[s] = s < left ? __builtin_amdgcn_exp2f(v[s] - mnew) : 0.f;
            ez += v[s];
        }
        z[c] = fmaf(z[c], f, ez);
        m[c] = mnew;
        t0 = t1 = (f32x4){0.f, 0.f, 0.f, 0.f};
        values(std::integral_constant<int, 0>{}, c);
        values(std::integral_constant<int, 1>{}, c);
        values(std::integral_constant<int, 2>{}, c);
        values(std::integral_constant<int, 3>{}, c);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            acc[c][0][x] = fmaf(acc[c][0][x], f, t0[x]);
            acc[c][1][x] = fmaf(acc[c][1][x], f, t1[x]);
        }
    };

    i32x2 span = rem_span(rSpan, 0, row0, L), ahead = rem_span(rSpan, NO > 1 ? 0 : 1, row0 + (NO > 1 ? REM_QUADS : 0), L);
    nw = rem_words(rWord, span.x + 4 * qi);
    for (int k = 0; k * REM_RANGE < L; ++k) {
        __syncthreads();  // everybody has finished with the previous range
        if constexpr (MASK)
            if (threadIdx.x < REM_RANGE) spen[threadIdx.x] = fmaf(keys.row(bh, L)[min(k * REM_RANGE + (int)threadIdx.x, L - 1)], -keys.mul * LOG2E,
                                         -keys.add * LOG2E);
        rem_load_range<true>(K + ib, ild, V + ib, ild, k * REM_RANGE, L, tile);
        __syncthreads();
#pragma unroll
        for (int c = 0; c < NO; ++c) {
            bool more;
            do {
                take(span);
                more = __any(cnt > REM_BATCH);  // a row with more entries in the range: the rest of it is the next batch
                if (more) span.x += REM_BATCH;
                else span = ahead;
                nw = rem_words(rWord, span.x + 4 * qi);
                if (!more) ahead = rem_span(rSpan, k + (c + 2) / NO, row0 + (c + 2) % NO * REM_QUADS, L);
                batch(c);
            } while (more);
        }
    }
#pragma unroll
    for (int c = 0; c < NO; ++c) {
        const int row = row0 + c * REM_QUADS;
        const float zs = quad_sum(z[c]);
        if (row >= L) continue;
        if (qi == 0) Stats[(size_t)bh * L + row] = make_float2(m[c], zs);
#pragma unroll
        for (int k = 0; k < 2; ++k)
            reinterpret_cast<f32x4*>(O + ob + (size_t)row * old_)[(k ^ j) * 4 + qi] = acc[c][k];
    }
}

// -------------------------------------------------------------------------------------------------
// Forward, last step: probabilities of the remainder entries from their raw logits and their rows' {maximum, 1 / denominator},
// to their places in P.  A work-group per block row: the entries of 32 rows are one run of the rb list per range; the runs of
// REM_RUNS ranges are requested together.  Memory bound: 64 heads of 4096 with 76 entries a row, 80 MB in, 111 MB out, lines of
// P shared with the tiles': 75 us (45 where P lies in the memory-side cache).  At the end of the tile kernel, which writes the
// same rows of P, it took 70 to 84: that kernel's wavefronts hold more lines of P than the L2 caches, 334 MB were written
// instead of 213 + 111.
// -------------------------------------------------------------------------------------------------
constexpr int REM_RUNS = 4, REM_PROB_THREADS = 256;
__global__ __launch_bounds__(REM_PROB_THREADS) void rem_prob_kernel(const float* __restrict__ Raw, float* __restrict__ P,
                                                                    const float2* __restrict__ Stats,
                                                                    const int* __restrict__ offs, RemIndex ix, int L, int nbr,
                                                                    int NB, int nnz) {
    struct Row {
        float m, zinv;
        int first;  // its first entry in a head's P
    };
    __shared__ Row rows[32];
    const int item = xcd_remap((int)blockIdx.x, nbr * NB), bh = item / nbr, I = item % nbr, t = threadIdx.x;
    if (t < 32) {
        const float2 st = Stats[(size_t)bh * L + I * 32 + t];
        rows[t] = Row{st.x, st.y, offs[I * 32 + t]};
    }
    __syncthreads();
    constexpr int U = 2;  // U * REM_PROB_THREADS entries of a run at once
    const rsrc_t rWord = rem_word_rsrc(ix.rb_word, ix.nr), rRaw = make_rsrc(Raw + (size_t)bh * ix.nr, (size_t)ix.nr * 4);
    const rsrc_t rP = make_rsrc(P + (size_t)bh * nnz, (size_t)nnz * 4);
    const int* off = ix.rb_off + I * 32;
    auto put = [&](unsigned word, float raw, bool there) {
        const Row r = rows[(word >> 9) & 31];
        st1(rP, there ? (r.first + (int)(word >> 14)) * 4 : -4, 0, __builtin_amdgcn_exp2f(raw - r.m) * r.zinv);
    };
    auto at = [](int e, int end) { return e < end ? e * 4 : -4; };
    for (int k0 = 0; k0 * REM_RANGE < L; k0 += REM_RUNS) {
        int e[REM_RUNS], end[REM_RUNS];
        unsigned word[REM_RUNS][U];
        float raw[REM_RUNS][U];
#pragma unroll
        for (int g = 0; g < REM_RUNS; ++g) {
            const bool there = (k0 + g) * REM_RANGE < L;
            const size_t k = there ? (size_t)(k0 + g) * L : 0;
            e[g] = off[k] + t;
            end[g] = there ? off[k + 32] : 0;
        }
#pragma unroll
        for (int g = 0; g < REM_RUNS; ++g)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int a = at(e[g] + u * REM_PROB_THREADS, end[g]);
                word[g][u] = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(rWord, a, 0, 0);
                raw[g][u] = ld1(rRaw, a, 0);
            }
#pragma unroll
        for (int g = 0; g < REM_RUNS; ++g) {
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (__any(e[g] + u * REM_PROB_THREADS < end[g]))
                    put(word[g][u], raw[g][u], e[g] + u * REM_PROB_THREADS < end[g]);
            for (int x = e[g] + U * REM_PROB_THREADS; __any(x < end[g]); x += REM_PROB_THREADS)
                put((unsigned)__builtin_amdgcn_raw_buffer_load_b32(rWord, at(x, end[g]), 0, 0), ld1(rRaw, at(x, end[g]), 0), x < end[g]);
        }
    }
}

// -------------------------------------------------------------------------------------------------
// Backward, row pass: dS = (dO_i . v_j - g_i) * P / sqrt(d), dQ_i += sum dS . K[col]; {dS, P} of every entry to Pairs
// [NB][nr] in the order of the rb list, where the column pass reads them.
// 64 heads of 4096 rows with 76 remainder entries each: 337 us (gathering from L2) -> 180; vector ALU 65 % busy, 595 MB of
// traffic (P's lines come once per range).
// -------------------------------------------------------------------------------------------------
template <bool ST, int NO>
__global__ __launch_bounds__(REM_THREADS) void rem_bwd_row_kernel(
    const float* __restrict__ K, const float* __restrict__ V, const float* __restrict__ P, const float* __restrict__ dO,
    const float* __restrict__ G, float2* __restrict__ Pairs, float* __restrict__ dQ, const int* __restrict__ offs,
    RemIndex ix, int L, int NB, int nnz, float scale, Layouts ly) {
    __shared__ f32x4 tile[(REM_RANGE + 2) * 16];  // {V, V, K, K} per pair of rows; a pair of zeros for absent entries
    constexpr int ROWS = NO * REM_QUADS;
    const int nrg = (L + ROWS - 1) / ROWS;  // the last one's rows past the end have no entries
    const int item = xcd_remap((int)blockIdx.x, (int)gridDim.x);  // the work-groups of a head share an XCD's L2
    const int bh = item / nrg, row0 = item % nrg * ROWS + (threadIdx.x >> 2);
    const int qi = threadIdx.x & 3, j = (threadIdx.x >> 2) & 1;
    size_t ib, ob, gb, bytes;
    int ild, old_, gld;
    head_slice<ST, 32>(ly.in, ly.H, bh, L, ib, ild, bytes);
    head_slice<ST, 32>(ly.out, ly.H, bh, L, ob, old_, bytes);
    head_slice<ST, 32>(ly.grad, ly.H, bh, L, gb, gld, bytes);
    const rsrc_t rSpan = rem_span_rsrc(ix.rb_off, L), rWord = rem_word_rsrc(ix.rb_word, ix.nr);
    const rsrc_t rPair = make_rsrc(Pairs + (size_t)bh * ix.nr, (size_t)ix.nr * 8);
    const rsrc_t rP = make_rsrc(P + (size_t)bh * nnz, (size_t)nnz * 4);
    if (threadIdx.x < 32) tile[REM_RANGE * 16 + threadIdx.x] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int off0 = 64 * j + 16 * qi, off1 = off0 ^ 64;  // this lane's 16 bytes of its first and second half row
    f32x4 acc[NO][2], go[NO][2];
    float g0[NO];
    int pbase[NO];
    int entries[NO];  // 0: the row has none
#pragma unroll
    for (int c = 0; c < NO; ++c) {
        const int row = min(row0 + c * REM_QUADS, L - 1);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            acc[c][k] = (f32x4){0.f, 0.f, 0.f, 0.f};
            go[c][k] = reinterpret_cast<const f32x4*>(dO + ob + (size_t)row * old_)[(k ^ j) * 4 + qi];
        }
        g0[c] = qi == 0 ? G[(size_t)bh * L + row] : 0.f;  // one lane's sum starts from -g
        pbase[c] = offs[row];
        entries[c] = 0;
    }

    int addr[4], first = 0, left = 0, cnt = 0;  // the present batch: LDS rows, first entry of the lane, entries from it on
    float p[4], ds[4];
    i32x4 nw;  // the next batch
    int naddr[4], nfirst = 0, nleft = 0, ncnt = 0;
    float np[4];
    auto convert = [&](int pb, i32x2 sp) {
        nfirst = sp.x + 4 * qi;
        ncnt = sp.y - sp.x;
        nleft = ncnt - 4 * qi;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const bool in = s < nleft;
            naddr[s] = rem_pair_row(in ? nw[s] & (REM_RANGE - 1) : REM_RANGE);
            np[s] = ld1(rP, in ? (pb + (int)((unsigned)nw[s] >> 14)) * 4 : -4, 0);
        }
    };
    auto take = [&]() {
        first = nfirst, left = nleft, cnt = ncnt;
#pragma unroll
        for (int s = 0; s < 4; ++s) addr[s] = naddr[s], p[s] = np[s];
    };
    f32x4 t0, t1;
    auto chunk = [&](auto I, int c) {
        constexpr int i = decltype(I)::value, CT = 0x55 * i;
        if (!__any(cnt > 4 * i)) return;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int base = quad_move<CT>(addr[s]), b0 = base ^ off0, b1 = base ^ off1;
            const f32x4 v0 = rem_lds(tile, b0), v1 = rem_lds(tile, b1), k0 = rem_lds(tile, b0 + 256), k1 = rem_lds(tile, b1 + 256);
            float d = g0[c], d1 = v1[0] * go[c][1][0];
#pragma unroll
            for (int x = 0; x < 4; ++x) d = fmaf(v0[x], go[c][0][x], d);
#pragma unroll
            for (int x = 1; x < 4; ++x) d1 = fmaf(v1[x], go[c][1][x], d1);
            d = quad_sum(d + d1) * quad_move<CT>(p[s]);
            ds[s] = qi == i ? d : ds[s];
#pragma unroll
            for (int x = 0; x < 4; ++x) t0[x] = fmaf(d, k0[x], t0[x]), t1[x] = fmaf(d, k1[x], t1[x]);
        }
    };
    // {dS, P} of the lane's entries: two at a time where both are there, an odd last one by itself
    auto finish = [&]() {
#pragma unroll
        for (int s = 0; s < 4; s += 2) {
            const f32x4 two = {ds[s] * scale, p[s], ds[s + 1] * scale, p[s + 1]};
            store_b128<true>(two, rPair, left >= s + 2 ? (first + s) * 8 : -16, 0);
        }
        const bool third = left == 3;
        const rem_u32x2 one = {__float_as_uint((third ? ds[2] : ds[0]) * scale), __float_as_uint(third ? p[2] : p[0])};
        __builtin_amdgcn_raw_buffer_store_b64(one, rPair, third ? (first + 2) * 8 : left == 1 ? first * 8 : -8, 0, 2);
    };
#define SPION_REM_CHUNKS(A, B)                                  \
    chunk(std::integral_constant<int, A>{}, c);                 \
    chunk(std::integral_constant<int, B>{}, c)

    i32x2 span = rem_span(rSpan, 0, row0, L), ahead = rem_span(rSpan, NO > 1 ? 0 : 1, row0 + (NO > 1 ? REM_QUADS : 0), L);
    nw = rem_words(rWord, span.x + 4 * qi);
    convert(pbase[0], span);
    for (int k = 0; k * REM_RANGE < L; ++k) {
        __syncthreads();  // everybody has finished with the previous range
        rem_load_range<true>(V + ib, ild, K + ib, ild, k * REM_RANGE, L, tile);
        __syncthreads();
#pragma unroll
        for (int c = 0; c < NO; ++c) {
            t0 = t1 = (f32x4){0.f, 0.f, 0.f, 0.f};
            bool more;
            do {
                take();
                entries[c] = max(entries[c], cnt);
                more = __any(cnt > REM_BATCH);  // a row with more entries in the range: the rest of it is the next batch
                if (more) span.x += REM_BATCH;
                else span = ahead;
                nw = rem_words(rWord, span.x + 4 * qi);
                if (!more) ahead = rem_span(rSpan, k + (c + 2) / NO, row0 + (c + 2) % NO * REM_QUADS, L);
                SPION_REM_CHUNKS(0, 1);
                convert(more ? pbase[c] : pbase[(c + 1) % NO], span);
                SPION_REM_CHUNKS(2, 3);
                finish();
            } while (more);
            acc[c][0] += t0;
            acc[c][1] += t1;
        }
    }
#pragma unroll
    for (int c = 0; c < NO; ++c) {
        const int row = row0 + c * REM_QUADS;
        // Slots without an entry are walked with the row's dO and g: where these are not finite, a row of no entries at all has
        // NaN for a sum.  (Clearing the product of every such slot instead took 34 us of the launch at the shape above.)
        if (row >= L || !entries[c]) continue;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            f32x4* o = reinterpret_cast<f32x4*>(dQ + gb + (size_t)row * gld) + (k ^ j) * 4 + qi;
            *o = *o + acc[c][k] * scale;
        }
    }
}

// -------------------------------------------------------------------------------------------------
// Backward, column pass: dK_j += sum_i dS_ij Q_i, dV_j += sum_i P_ij dO_i from the {dS, P} pairs of the row pass (dS
// already carries the 1/sqrt(d)).  As above: 236 us (eight lanes to a column, weights looked up in row order) -> 171; vector ALU
// 70 % busy.  The look-ups in the pairs cost 30 of them: with the entries in plain row order, not by ranges, 55.
// -------------------------------------------------------------------------------------------------
template <bool ST, int NO>
__global__ __launch_bounds__(REM_THREADS) void rem_bwd_col_kernel(
    const float* __restrict__ Q, const float* __restrict__ dO, const float2* __restrict__ Pairs, float* __restrict__ dK,
    float* __restrict__ dV, RemIndex ix, int L, int NB, Layouts ly) {
    __shared__ f32x4 tile[(REM_RANGE + 1) * 16];  // {Q, dO} per row; a row of zeros for absent entries
    constexpr int COLS = NO * REM_QUADS;
    static_assert(REM_RANGE % COLS == 0, "the columns of a work-group lie in one range");
    const int ncg = (L + COLS - 1) / COLS;
    const int item = xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int bh = item / ncg, cg0 = item % ncg * COLS, col0 = cg0 + (threadIdx.x >> 2);
    const int qi = threadIdx.x & 3, j = (threadIdx.x >> 2) & 3;
    size_t ib, ob, gb, bytes;
    int ild, old_, gld;
    head_slice<ST, 32>(ly.in, ly.H, bh, L, ib, ild, bytes);
    head_slice<ST, 32>(ly.out, ly.H, bh, L, ob, old_, bytes);
    head_slice<ST, 32>(ly.grad, ly.H, bh, L, gb, gld, bytes);
    const rsrc_t rSpan = rem_span_rsrc(ix.cb_off, L), rWord = rem_word_rsrc(ix.cb_word, ix.nr);
    const rsrc_t rPair = make_rsrc(Pairs + (size_t)bh * ix.nr, (size_t)ix.nr * 8);
    // first entry in the rb list of the block (range k of the rows) x (range of these columns)
    const int* blocks = ix.rb_off + (size_t)(cg0 / REM_RANGE) * L;
    auto block = [&](int k) { return blocks[min(k * REM_RANGE, L - 1)]; };
    if (threadIdx.x < 16) tile[REM_RANGE * 16 + threadIdx.x] = (f32x4){0.f, 0.f, 0.f, 0.f};
    int off[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) off[k] = 64 * (k ^ j) + 16 * qi;
    f32x4 acc[NO][4];  // half row k ^ j of {dK, dV}
#pragma unroll
    for (int c = 0; c < NO; ++c)
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[c][k] = (f32x4){0.f, 0.f, 0.f, 0.f};

    int addr[4], cnt = 0;
    float wa[4], wb[4];  // weights of the lane's first two and last two half rows
    i32x4 nw;
    int naddr[4], ncnt = 0;
    float2 npair[4];
    auto convert = [&](i32x2 sp, int src0) {
        ncnt = sp.y - sp.x;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const bool in = s < ncnt - 4 * qi;
            naddr[s] = (in ? nw[s] & (REM_RANGE - 1) : REM_RANGE) * 256;
            const int src = in ? (src0 + (int)((unsigned)nw[s] >> 9)) * 8 : -8;
            npair[s] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(rPair, src, 0, 0));
        }
    };
    auto take = [&]() {
        cnt = ncnt;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            addr[s] = naddr[s];
            wa[s] = j < 2 ? npair[s].x : npair[s].y;
            wb[s] = j < 2 ? npair[s].y : npair[s].x;
        }
    };
    f32x4 t[4];
    auto chunk = [&](auto I, int) {
        constexpr int i = decltype(I)::value, CT = 0x55 * i;
        if (!__any(cnt > 4 * i)) return;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int base = quad_move<CT>(addr[s]);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const f32x4 x = rem_lds(tile, base ^ off[k]);
                const float w = quad_move<CT>(k < 2 ? wa[s] : wb[s]);
#pragma unroll
                for (int f = 0; f < 4; ++f) t[k][f] = fmaf(w, x[f], t[k][f]);
            }
        }
    };

    i32x2 span = rem_span(rSpan, 0, col0, L), ahead = rem_span(rSpan, NO > 1 ? 0 : 1, col0 + (NO > 1 ? REM_QUADS : 0), L);
    nw = rem_words(rWord, span.x + 4 * qi);
    int src0 = block(0), src1 = block(1);  // of the present and of the next range
    convert(span, src0);
    for (int k = 0; k * REM_RANGE < L; ++k) {
        __syncthreads();
        rem_load_range<false>(Q + ib, ild, dO + ob, old_, k * REM_RANGE, L, tile);
        __syncthreads();
#pragma unroll
        for (int c = 0; c < NO; ++c) {
#pragma unroll
            for (int x = 0; x < 4; ++x) t[x] = (f32x4){0.f, 0.f, 0.f, 0.f};
            bool more;
            do {
                take();
                more = __any(cnt > REM_BATCH);
                if (more) span.x += REM_BATCH;
                else span = ahead;
                nw = rem_words(rWord, span.x + 4 * qi);
                if (!more) ahead = rem_span(rSpan, k + (c + 2) / NO, col0 + (c + 2) % NO * REM_QUADS, L);
                SPION_REM_CHUNKS(0, 1);
                convert(span, more || c + 1 < NO ? src0 : src1);
                SPION_REM_CHUNKS(2, 3);
            } while (more);
#pragma unroll
            for (int x = 0; x < 4; ++x) acc[c][x] += t[x];
        }
        src0 = src1;
        src1 = block(k + 2);
    }
#pragma unroll
    for (int c = 0; c < NO; ++c) {
        const int col = col0 + c * REM_QUADS;
        if (col >= L) continue;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int half = k ^ j;
            f32x4* o = reinterpret_cast<f32x4*>((half & 2 ? dV : dK) + gb + (size_t)col * gld) + (half & 1) * 4 + qi;
            *o = *o + acc[c][k];
        }
    }
}

}  // namespace spion
