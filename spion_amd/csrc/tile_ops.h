// Device helpers shared by the sparse and dense attention kernels: wavefront reductions, the
// work-group -> XCD mapping and the register-level 32x32 MFMA tile operations.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

namespace spion {

// =================================================================================================
// wavefront helpers
// =================================================================================================
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Row of the 32x32 MFMA accumulator held in register r of a lane in half h (lane / 32); the column
// is lane % 32.
__device__ __forceinline__ int acc_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// Work-group id -> work item, so that consecutive work items (same head) run on the same XCD and
// share its L2: the hardware deals work-groups round-robin over the 8 XCDs.  (Numbers of items that eight does not divide were
// once left as they are, so that every XCD's L2 saw all heads at a time.  us, before / now: steps of 45 heads of 3296 231 / 209, of 202
// of 1056 161 / 142, with key mask of 75 of 1632 (d = 64) 259 / 243; discovery of two maps of 2720^2 49.4 / 41.6.)
__device__ __forceinline__ int xcd_remap(int pid, int total) {
    constexpr int XCDS = 8;
    const int xcd = pid % XCDS, share = total / XCDS, rest = total % XCDS;  // the first `rest` XCDs have one more
    return xcd * share + min(xcd, rest) + pid / XCDS;
}

// =================================================================================================
// MFMA tile operations
// =================================================================================================
// Operand conventions for v_mfma_f32_32x32x2_f32 (D = A.B + C, A 32x2, B 2x32):
//   lane l supplies A[l%32][l/32] and B[l/32][l%32]; register r of the 16-register accumulator of
//   lane l holds D[acc_row(r, l/32)][l%32].
// A contraction over the head dimension is a chain of D/2 such instructions; which feature index t a
// (step s, half h) slot stands for is free as long as A and B agree -- here t = h*(D/2) + s, so that a
// lane reads D/2 consecutive floats of a row-major row.
// A contraction over the 32 keys/queries of a tile is a chain of 16 instructions in which slot (s, h)
// stands for tile row acc_row(s, h): the accumulator of the first product is then already the A
// operand of the second one, register for register, and nothing goes through LDS.

// =================================================================================================
// fp32 products on the bf16 matrix pipe
// =================================================================================================
// A float is the exact sum of three bf16 numbers -- hi = bf16(x), mid = bf16(x - hi), lo = x - hi - mid, all rounded
// to nearest: 8 + 8 + 8 significant bits, the signs of mid and lo taking up what rounding up borrows -- and a product
// of two bf16 numbers is exact in fp32.  Of the nine partial products of a . b the six with hi.hi, hi.mid, mid.hi,
// mid.mid, hi.lo and lo.hi are formed; of the other three mid.lo and lo.mid reach 2^-25 of |a||b| each, so that all
// three together are at most 2^-24 (1 + 2^-9) of it, what one rounding of an fp32 product can be.  Sums are accumulated
// in fp32 by the MFMA as before.  Measured against float64 on MI355X (32x32x32 products of normal, positive, wide-range
// and one-signed operands, 1 to 128 of them accumulated): relative error 3.8e-8 against 1.0e-7 of the
// v_mfma_f32_32x32x2_f32 chain for one product, 1.02e-6 against 1.15e-6 for 128; all nine partial products give the same
// figures as six.
// Why: v_mfma_f32_32x32x16_bf16 does sixteen times the work of v_mfma_f32_32x32x2_f32 in half its time, so six of
// them per 16 terms take 384 cycles for a 32x32x32 product instead of 1024; they overlap with vector-ALU work, which
// the fp32 MFMA does not, so that the splitting (88 instructions per 16 floats and lane) is mostly hidden; and they
// draw less power: under sustained load the fp32 chain takes 435 to 755 ns per product and SIMD (the clock drops), the
// six-product chain 217 ns, 280 ns with one operand split on the way.
// Range: an infinite operand, or a finite one of 2^128 - 2^119 and more, whose hi rounds to infinity, gives parts that are
// not numbers and so a NaN in every sum it enters; below 2^-110 the lo part is subnormal or lost, an absolute error under
// 2^-133.  So a wavefront looks once a strip at what came out of its products (split_failed) and, where one of its sums is
// not finite, or so small that its operands may lie down there, walks its tiles again with fp32 chains: infinities, NaN and
// the ends of the range come out as those give them.  What is left: operands below 2^-110 whose products partners above 2^20
// lift above 2^-90, where the absolute error of 2^-133 of the operand remains; and sums that are zero because one operand of
// every product is below 2^-134, which the bf16 format does not hold (fp32 chains give up to 2^-134 times the partners).
// (The projections, project.hip, ask whether all sums of a wavefront are that small: they make 32 x 32 outputs and more of
// it, and an output of 2^-90 that a dying weight leaves among them would cost every call the second walk.)
template <int N>
struct Split3 {
    bf16x8 p[3][N / 8];  // hi, mid, lo of elements 8t .. 8t+7
};
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
    bf16x2 v;
    v[0] = (__bf16)a;
    v[1] = (__bf16)b;
    unsigned u = __builtin_bit_cast(unsigned, v);
    asm("" : "+v"(u));  // the compiler would otherwise convert a and b once more, one at a time, to widen them again
    return u;
}
__device__ __forceinline__ float bf16_lo(unsigned u) { return __builtin_bit_cast(float, u << 16); }
__device__ __forceinline__ float bf16_hi(unsigned u) { return __builtin_bit_cast(float, u & 0xffff0000u); }
template <int N>
__device__ __forceinline__ Split3<N> split3(const float (&x)[N]) {
    typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
    Split3<N> s;
#pragma unroll
    for (int t = 0; t < N / 8; ++t) {
        u32x4_t hi, mid, lo;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float a = x[8 * t + 2 * j], b = x[8 * t + 2 * j + 1];
            hi[j] = pack_bf16(a, b);
            a -= bf16_lo(hi[j]);
            b -= bf16_hi(hi[j]);
            mid[j] = pack_bf16(a, b);
            a -= bf16_lo(mid[j]);
            b -= bf16_hi(mid[j]);
            lo[j] = pack_bf16(a, b);
        }
        s.p[0][t] = __builtin_bit_cast(bf16x8, hi);
        s.p[1][t] = __builtin_bit_cast(bf16x8, mid);
        s.p[2][t] = __builtin_bit_cast(bf16x8, lo);
    }
    return s;
}
__device__ __forceinline__ f32x16 mfma_bf16(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// acc += A.B over the N slots of each half-wave (small partial products first)
template <int N>
__device__ __forceinline__ f32x16 mma_split(const Split3<N>& a, const Split3<N>& b, f32x16 acc) {
#pragma unroll
    for (int t = 0; t < N / 8; ++t) {
        acc = mfma_bf16(a.p[2][t], b.p[0][t], acc);
        acc = mfma_bf16(a.p[0][t], b.p[2][t], acc);
        acc = mfma_bf16(a.p[1][t], b.p[1][t], acc);
    }
#pragma unroll
    for (int t = 0; t < N / 8; ++t) {
        acc = mfma_bf16(a.p[1][t], b.p[0][t], acc);
        acc = mfma_bf16(a.p[0][t], b.p[1][t], acc);
    }
#pragma unroll
    for (int t = 0; t < N / 8; ++t) acc = mfma_bf16(a.p[0][t], b.p[0][t], acc);
    return acc;
}

// The same operand for fp32 chains.
template <int N>
struct Whole {
    float x[N];
};
template <int N>
__device__ __forceinline__ Whole<N> whole(const float (&x)[N]) {
    Whole<N> w;
#pragma unroll
    for (int s = 0; s < N; ++s) w.x[s] = x[s];
    return w;
}
template <class X>
constexpr bool is_whole = false;
template <int N>
constexpr bool is_whole<Whole<N>> = true;

// Whether sums of split products have to be formed again by fp32 chains (the same answer in every lane): one of them is not
// finite, or is not zero and below 2^-90.  Every sum by itself: a key or a query whose gradients are that small may lie among
// 31 ordinary ones (a key of probability 2^-118: relative error of its row of dV 1e-5, of 2^-124 1e-3, from split products).
// (Sums whose magnitudes overflow only together cost time and nothing else.)
template <int N>
__device__ __forceinline__ bool split_failed(const f32x16 (&acc)[N]) {
    float s = 0.f;
    unsigned least = ~0u;  // of twice the bits without the sign, less one: a zero is the largest
#pragma unroll
    for (int c = 0; c < N; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            s += fabsf(acc[c][r]);
            least = min(least, 2u * __float_as_uint(acc[c][r]) - 1u);
        }
    const bool finite = s < __builtin_inff();  // false for NaN
    return __builtin_expect(__any(!finite || least < 2u * __builtin_bit_cast(unsigned, 0x1p-90f) - 1u), 0);
}
// One of a wavefront's sums is not finite, or none of them reaches 2^-90 although not all are zero; s: the sum of a lane's
// magnitudes.
__device__ __forceinline__ bool split_failed_sum(float s) {
    const bool finite = s < __builtin_inff();
    return __builtin_expect(__any(!finite) || (!__any(s >= 0x1p-90f) && __any(s != 0.f)), 0);
}
// The same for the exponentials of logits: a NaN among them.  (Logits may be as small as they like.)
__device__ __forceinline__ bool split_failed(float z) { return __builtin_expect(__any(z != z), 0); }
// The lane for such a second walk, hidden from the compiler: addresses made from it are not shared with the first walk
// and so take no registers there.
__device__ __forceinline__ int second_walk(int l) {
    asm volatile("" : "+v"(l));
    return l;
}

// The lane once more, two instructions where it is asked for and no register in between.
__device__ __forceinline__ int lane_again() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(l));
    return l;
}

// acc += A.B over the 16 slots of each half-wave, an fp32 chain
__device__ __forceinline__ f32x16 mma_chain(const float (&a)[16], const float (&b)[16], f32x16 acc) {
#pragma unroll
    for (int s = 0; s < 16; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], b[s], acc, 0, 0, 0);
    return acc;
}

template <int D>
__device__ __forceinline__ void load_rows(const float* __restrict__ X, int row0, int li, int h, float (&x)[D / 2]) {
    const float4* p = reinterpret_cast<const float4*>(X + (size_t)(row0 + li) * D + h * (D / 2));
#pragma unroll
    for (int q = 0; q < D / 8; ++q) {
        float4 v = p[q];
        x[4 * q + 0] = v.x;
        x[4 * q + 1] = v.y;
        x[4 * q + 2] = v.z;
        x[4 * q + 3] = v.w;
    }
}

template <int D>
__device__ __forceinline__ void load_cols(const float* __restrict__ Xt, int L, int col0, int li, int h,
                                          float (&x)[D / 2]) {
    const float* p = Xt + (size_t)(h * (D / 2)) * L + col0 + li;
#pragma unroll
    for (int s = 0; s < D / 2; ++s) x[s] = p[(size_t)s * L];
}

template <int D>
__device__ __forceinline__ f32x16 mma_feat(const float (&a)[D / 2], const float (&b)[D / 2]) {
    f32x16 acc = {0};
#pragma unroll
    for (int s = 0; s < D / 2; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], b[s], acc, 0, 0, 0);
    return acc;
}

// out[c] += W(32x32, as accumulator-layout registers w[16]) . X[row0 .. row0+32)[c*32 .. c*32+32)
template <int D>
__device__ __forceinline__ void mma_tile(const float (&w)[16], const float* __restrict__ X, int row0, int li,
                                         int h, f32x16 (&out)[D / 32]) {
#pragma unroll
    for (int c = 0; c < D / 32; ++c) {
        float x[16];
#pragma unroll
        for (int s = 0; s < 16; ++s) x[s] = X[(size_t)(row0 + acc_row(s, h)) * D + c * 32 + li];
#pragma unroll
        for (int s = 0; s < 16; ++s) out[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[s], x[s], out[c], 0, 0, 0);
    }
}

// out[c] (+)= X^T-tile . W for operands stored feature-major (Xt [D][ld], the dense-phase layout):
// result row = feature c*32 + (lane%32 as A row), column = the accumulator column of W.  W enters as
// the B operand (slot (s, h) = tile row acc_row(s, h)), Xt as the A operand read with float4 loads.
template <int D>
__device__ __forceinline__ void mma_tile_t(const float (&w)[16], const float* __restrict__ Xt, size_t ld, int col0,
                                           int li, int h, f32x16 (&out)[D / 32]) {
#pragma unroll
    for (int c = 0; c < D / 32; ++c) {
        float x[16];
        const float* p = Xt + (size_t)(c * 32 + li) * ld + col0 + 4 * h;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float4 v = *reinterpret_cast<const float4*>(p + 8 * g);
            x[4 * g + 0] = v.x;
            x[4 * g + 1] = v.y;
            x[4 * g + 2] = v.z;
            x[4 * g + 3] = v.w;
        }
#pragma unroll
        for (int s = 0; s < 16; ++s) out[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[s], w[s], out[c], 0, 0, 0);
    }
}

// Sum the per-wave accumulators of a work-group and store the result tile(s).
//   TRANS == false: accumulator c holds rows row0+acc_row of a row-major [.][D] array, columns c*32+lane%32.
//   TRANS == true : accumulator c holds rows c*32+acc_row of a feature-major [D][ld] array, columns row0+lane%32.
template <int D, int WAVES, bool TRANS = false>
__device__ __forceinline__ void reduce_store(f32x16 (&acc)[D / 32], float* __restrict__ out, int row0, int w,
                                             int li, int h, float* __restrict__ lds, size_t ld = D) {
    constexpr int NC = D / 32;
    auto addr = [&](int c, int r) -> size_t {
        return TRANS ? (size_t)(c * 32 + acc_row(r, h)) * ld + row0 + li
                     : (size_t)(row0 + acc_row(r, h)) * ld + c * 32 + li;
    };
    if (WAVES == 1) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r) out[addr(c, r)] = acc[c][r];
        return;
    }
    const int l = h * 32 + li;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) lds[((w * NC + c) * 16 + r) * 64 + l] = acc[c][r];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if ((r % WAVES) != w) continue;
            float s = 0.f;
#pragma unroll
            for (int ww = 0; ww < WAVES; ++ww) s += lds[((ww * NC + c) * 16 + r) * 64 + l];
            out[addr(c, r)] = s;
        }
}

// A transposed 32-feature accumulator (register = feature acc_row(r, h), lane = row li of the strip) summed over
// the waves and written row-major, rows `ld` floats apart: register group g = r/4 is four consecutive features,
// one 16-byte store per lane; wave g % WAVES writes group g.
template <int WAVES>
__device__ __forceinline__ void reduce_store_rows(const f32x16& acc, float* __restrict__ out, int row0, int w, int li,
                                                  int h, float* __restrict__ lds, size_t ld) {
    const int l = h * 32 + li;
    if (WAVES > 1) {
#pragma unroll
        for (int r = 0; r < 16; ++r) lds[(w * 16 + r) * 64 + l] = acc[r];
        __syncthreads();
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        if (WAVES > 1 && (g % WAVES) != w) continue;
        float s[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = 4 * g + j;
            s[j] = acc[r];
            if (WAVES > 1) {
                s[j] = 0.f;
#pragma unroll
                for (int ww = 0; ww < WAVES; ++ww) s[j] += lds[(ww * 16 + r) * 64 + l];
            }
        }
        *reinterpret_cast<f32x4*>(out + (size_t)(row0 + li) * ld + 8 * g + 4 * h) = (f32x4){s[0], s[1], s[2], s[3]};
    }
}

// Like reduce_store (row-major form), but the reduced tile goes to two arrays.
template <int D, int WAVES>
__device__ __forceinline__ void reduce_store2(f32x16 (&acc)[D / 32], float* __restrict__ out, float* __restrict__ out2,
                                              int row0, int w, int li, int h, float* __restrict__ lds) {
    constexpr int NC = D / 32;
    const int l = h * 32 + li;
    if (WAVES > 1) {
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int r = 0; r < 16; ++r) lds[((w * NC + c) * 16 + r) * 64 + l] = acc[c][r];
        __syncthreads();
    }
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if (WAVES > 1 && (r % WAVES) != w) continue;
            float s = acc[c][r];
            if (WAVES > 1) {
                s = 0.f;
#pragma unroll
                for (int ww = 0; ww < WAVES; ++ww) s += lds[((ww * NC + c) * 16 + r) * 64 + l];
            }
            const size_t a = (size_t)(row0 + acc_row(r, h)) * D + c * 32 + li;
            out[a] = s;
            out2[a] = s;
        }
}

}  // namespace spion
