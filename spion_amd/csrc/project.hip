// The projections around the attention core (models/attention.py:84-103: W_q, W_k, W_v and ff): y = x.W^T + b, and in the
// backward dx = dy.W, dW = dy^T.x, db = column sums of dy.  fp32 in and out.
//
// The shapes are lopsided -- some 10^4 to 10^5 rows against 32 to a few hundred features -- and a product of 192 x 64
// outputs summed over 65536 rows leaves a library's GEMM with a handful of work-groups: 198 us for a weight gradient
// whose operands are 67 MB.  Here the sum over the rows is cut into as many pieces as fill the chip, each piece leaves
// its fp32 result in a workspace and a second launch adds them in a fixed order; db falls out of the same pass over
// dy.  The three projections take their weights from three matrices, so nothing is concatenated.  Measured, rows x dim ->
// outputs, in us, torch (rocBLAS) and here: 65536 x 64 -> 192: forward 27 / 22, dx 22 / 21, dW and db 200 + 23 / 24;
// 32768 x 256 -> 768: 104 / 93, 94 / 79, 400 + 31 / 104; 2048 x 64 -> 192: 20 / 6.5, 20 / 8, 21 + 11 / 9.  The smallest are
// bound by the launch, the first by memory (67 MB), the second by the matrix pipe and the splitting.
//
// Products run on the bf16 matrix pipe with operands split into three bf16 parts each (Split3 in tile_ops.h: fp32
// accuracy).  A work-group stages both operands through LDS already split: every element is split once by the thread
// that loads it and then read by every wavefront whose tiles it belongs to.
#include "bf16_kernels.h"
#include "common.h"
#include "../../include/spion_hip.h"

#include <algorithm>
#include <climits>

namespace spion {

// Most rows a call may have, and what a matrix stored in one piece has for `seg`: no row index reaches it, and twice as
// much is still an int.
constexpr int MAX_ROWS = INT_MAX / 2, ONE_PIECE = INT_MAX / 2;
static_assert(MAX_ROWS - 1 < ONE_PIECE && ONE_PIECE <= INT_MAX - ONE_PIECE, "every row lies in the first piece");

// Rows of a matrix that is stored as up to three matrices of `seg` rows each.
struct SegRows {
    const float* p[3];
    int seg;
    int ld;
    __device__ __forceinline__ const float* row(int r) const {
        const int s = r >= seg ? (r >= 2 * seg ? 2 : 1) : 0;
        const float* b = s == 0 ? p[0] : s == 1 ? p[1] : p[2];
        return b + (size_t)(r - s * seg) * ld;
    }
};
struct SegBias {
    const float* p[3];
    int seg;
};

// The two LDS images of an operand chunk of 32 reduction indices, one per bf16 part, in 8-byte pieces of four elements:
//   along (reduction index along the rows in memory): rows x 32, 64-byte rows, piece c of row r at c ^ (r/4 % 8);
//   across (reduction index across the rows): 32 x 64 columns, the tile image of DmaTile<64>.
// Both spread the writes (eight or sixteen consecutive threads to a row) and the operand reads over all banks.  Slot e
// of instruction t in half h is reduction index 16t + 8(e/4) + 4h + e%4 in both, which is what the transposing LDS
// read delivers.
template <bool ACROSS, int BLOCKS>  // BLOCKS: of 64 rows (along) or columns (across)
struct OperandLds {
    static constexpr int PART = BLOCKS * 64 * 32 * 2;  // bytes of one part
    static constexpr int BYTES = 3 * PART;
    static constexpr int F4 = BLOCKS * 2;  // float4 a thread loads per chunk (256 threads)
    typedef DmaTile<64> DT;
    // element (row, column) of thread t's float4 number i, relative to the chunk
    __device__ static __forceinline__ void place(int t, int i, int& row, int& col) {
        if constexpr (ACROSS) {
            row = (t >> 4) + 16 * (i & 1);
            col = 4 * (t & 15) + 64 * (i >> 1);
        } else {
            row = (t >> 3) + 32 * i;
            col = 4 * (t & 7);
        }
    }
    __device__ static __forceinline__ int addr(int row, int col) {
        if constexpr (ACROSS) {
            const int b = col >> 6, c4 = (col & 63) >> 2;
            return b * (64 * 32 * 2) + row * DT::ROW + 16 * ((c4 >> 1) ^ DT::swz(row)) + 8 * (c4 & 1);
        } else {
            return row * 64 + 8 * ((col >> 2) ^ ((row >> 2) & 7));
        }
    }
    __device__ static __forceinline__ void put(char* S, int t, int i, f32x4 v) {
        int row, col;
        place(t, i, row, col);
        const float x[4] = {v.x, v.y, v.z, v.w};
        u32x2 part[3];
        split4(x, part);
        const int a = addr(row, col);
#pragma unroll
        for (int k = 0; k < 3; ++k) *reinterpret_cast<u32x2*>(S + k * PART + a) = part[k];
    }
    __device__ static __forceinline__ void split4(const float (&x)[4], u32x2 (&part)[3]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            float a = x[2 * j], b = x[2 * j + 1];
            const unsigned hi = pack_bf16(a, b);
            a -= bf16_lo(hi);
            b -= bf16_hi(hi);
            const unsigned mid = pack_bf16(a, b);
            a -= bf16_lo(mid);
            b -= bf16_hi(mid);
            part[0][j] = hi;
            part[1][j] = mid;
            part[2][j] = pack_bf16(a, b);
        }
    }
    // the wavefront's operand: 32 rows / columns from `first` on (a multiple of 32)
    __device__ static __forceinline__ void get(const char* S, int first, int l, bf16x8 (&x)[3][2]) {
        const int h = l >> 5, li = l & 31;
        if constexpr (ACROSS) {
            typedef s16x4 __attribute__((address_space(3))) * lds_ptr;
            const int gm = (l >> 4) & 1, j = l & 15, row = 4 * h + (j >> 2), c = (first >> 5) & 1;
            const int a = (first >> 6) * (64 * 32 * 2) + row * DT::ROW +
                          16 * ((4 * c + 2 * gm + ((j & 3) >> 1)) ^ DT::swz(row)) + 8 * (j & 1);
#pragma unroll
            for (int k = 0; k < 3; ++k)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const char* p = S + k * PART + a + 16 * t * DT::ROW;
                    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)p);
                    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p + 8 * DT::ROW));
                    x[k][t] = __builtin_shufflevector(__builtin_bit_cast(bf16x4, lo), __builtin_bit_cast(bf16x4, hi), 0, 1,
                                                      2, 3, 4, 5, 6, 7);
                }
        } else {
            const int row = first + li, s = (row >> 2) & 7;
#pragma unroll
            for (int k = 0; k < 3; ++k)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const char* p = S + k * PART + row * 64;
                    const u32x2 lo = *reinterpret_cast<const u32x2*>(p + 8 * ((4 * t + h) ^ s));
                    const u32x2 hi = *reinterpret_cast<const u32x2*>(p + 8 * ((4 * t + 2 + h) ^ s));
                    const u32x4 v = {lo.x, lo.y, hi.x, hi.y};
                    x[k][t] = __builtin_bit_cast(bf16x8, v);
                }
        }
    }
};

// C[m][n] = sum_r A.B over reduction indices [32 z chunks, 32 (z + 1) chunks) of work-group z (+ bias[n]); z > 0 only
// for partial sums, which lie M * N floats apart.  A is [m][r] (A_ACROSS: [r][m]), B is [n][r] (B_ACROSS: [r][n]).
// Four wavefronts, 2 x 2, of WM x WN 32 x 32 tiles each.  One LDS buffer and two barriers a chunk: with a second buffer
// (one barrier) fewer work-groups fit on a CU, 33 us instead of 26 for 65536 x 64 -> 192 in 128 x 128 tiles.
// COLSUM (the sums over many rows): the hi.hi products and the small ones have accumulators of their own -- adding the
// small ones one by one to a sum that has grown a hundredfold would lose their last bits when they share a sign -- and
// the work-groups of the first column of tiles also leave sum_r A[r][m] in Csum[z][m].
// A wavefront whose sums are not finite, or all too small for split operands (Split3, tile_ops.h), forms them again from
// the operands in memory, one fp32 term after the other: some 30 us at 256 terms, and rare.
struct Product {
    SegRows A, B;
    SegBias bias;
    float* C;
    float* Csum;
    int ldc, M, N, R, chunks, mtiles, ntiles;
};
template <bool A_ACROSS, bool B_ACROSS, int WM, int WN, bool COLSUM>
__device__ __forceinline__ void project_item(const Product& y, int item, char* smem) {
    const SegRows A = y.A, B = y.B;
    const SegBias bias = y.bias;
    float *__restrict__ C = y.C, *__restrict__ Csum = y.Csum;
    const int ldc = y.ldc, M = y.M, N = y.N, R = y.R, chunks = y.chunks, mtiles = y.mtiles, ntiles = y.ntiles;
    typedef OperandLds<A_ACROSS, WM> LA;
    typedef OperandLds<B_ACROSS, WN> LB;
    const int t = threadIdx.x, w = t >> 6, l = t & 63, h = l >> 5, li = l & 31;
    const int nt = item % ntiles, mt = item / ntiles % mtiles, z = item / ntiles / mtiles;
    const int m0 = mt * 64 * WM, n0 = nt * 64 * WN;
    const int r0 = z * chunks * 32, nchunks = min(chunks, R / 32 - z * chunks);
    const int wm = (w >> 1) * 32 * WM, wn = (w & 1) * 32 * WN;

    f32x4 ra[LA::F4], rb[LB::F4];
    // rows and columns past the end are read from the last valid ones; their results are not stored
    auto fetch = [&](int r) {
#pragma unroll
        for (int i = 0; i < LA::F4; ++i) {
            int row, col;
            LA::place(t, i, row, col);
            ra[i] = *reinterpret_cast<const f32x4*>(A_ACROSS ? A.row(r + row) + min(m0 + col, M - 4)
                                                             : A.row(min(m0 + row, M - 1)) + r + col);
        }
#pragma unroll
        for (int i = 0; i < LB::F4; ++i) {
            int row, col;
            LB::place(t, i, row, col);
            rb[i] = *reinterpret_cast<const f32x4*>(B_ACROSS ? B.row(r + row) + min(n0 + col, N - 4)
                                                             : B.row(min(n0 + row, N - 1)) + r + col);
        }
    };
    f32x16 hi[WM][WN], lo[COLSUM ? WM : 1][COLSUM ? WN : 1];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            hi[i][j] = splat16(0.f);
            if constexpr (COLSUM) lo[i][j] = splat16(0.f);
        }
    f32x4 csum[LA::F4 / 2];
#pragma unroll
    for (int i = 0; i < LA::F4 / 2; ++i) csum[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const bool sums = COLSUM && nt == 0;

    fetch(r0);
    for (int c = 0; c < nchunks; ++c) {
        char* S = smem;
        if (c) __syncthreads();  // every wavefront has read the chunk before
#pragma unroll
        for (int i = 0; i < LA::F4; ++i) LA::put(S, t, i, ra[i]);
#pragma unroll
        for (int i = 0; i < LB::F4; ++i) LB::put(S + LA::BYTES, t, i, rb[i]);
        if constexpr (COLSUM) {
            if (sums) {
#pragma unroll
                for (int i = 0; i < LA::F4; ++i) csum[i >> 1] += ra[i];
            }
        }
        __syncthreads();
        if (c + 1 < nchunks) fetch(r0 + (c + 1) * 32);  // (two chunks ahead: measured, no gain)
        bf16x8 b[WN][3][2];
#pragma unroll
        for (int j = 0; j < WN; ++j) LB::get(S + LA::BYTES, wn + 32 * j, l, b[j]);
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            bf16x8 a[3][2];
            LA::get(S, wm + 32 * i, l, a);
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                f32x16& small = [&]() -> f32x16& {
                    if constexpr (COLSUM) return lo[i][j];
                    else return hi[i][j];
                }();
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    small = mfma_bf16(a[2][k], b[j][0][k], small);
                    small = mfma_bf16(a[0][k], b[j][2][k], small);
                    small = mfma_bf16(a[1][k], b[j][1][k], small);
                }
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    small = mfma_bf16(a[1][k], b[j][0][k], small);
                    small = mfma_bf16(a[0][k], b[j][1][k], small);
                }
#pragma unroll
                for (int k = 0; k < 2; ++k) hi[i][j] = mfma_bf16(a[0][k], b[j][0][k], hi[i][j]);
            }
        }
    }
    float mag = 0.f;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                mag += fabsf(hi[i][j][q]);
                if constexpr (COLSUM) mag += fabsf(lo[i][j][q]);
            }
    if (split_failed_sum(mag)) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                hi[i][j] = splat16(0.f);
                if constexpr (COLSUM) lo[i][j] = splat16(0.f);
            }
#pragma unroll 1
        for (int r = r0; r < r0 + nchunks * 32; ++r) {
            float b[WN];
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                const int n = min(n0 + wn + 32 * j + li, N - 1);
                b[j] = B_ACROSS ? B.row(r)[n] : B.row(n)[r];
            }
#pragma unroll
            for (int i = 0; i < WM; ++i)
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const int m = min(m0 + wm + 32 * i + acc_row(q, h), M - 1);
                    const float a = A_ACROSS ? A.row(r)[m] : A.row(m)[r];
#pragma unroll
                    for (int j = 0; j < WN; ++j) hi[i][j][q] = fmaf(a, b[j], hi[i][j][q]);
                }
        }
    }
    float* Cz = C + (size_t)z * M * N;
#pragma unroll
    for (int j = 0; j < WN; ++j) {
        const int n = n0 + wn + 32 * j + li;
        if (n - li >= N) continue;
        float bn = 0.f;
        if (bias.p[0]) {
            const int s = n >= bias.seg ? (n >= 2 * bias.seg ? 2 : 1) : 0;
            bn = (s == 0 ? bias.p[0] : s == 1 ? bias.p[1] : bias.p[2])[n - s * bias.seg];
        }
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            const int m = m0 + wm + 32 * i;
            if (m >= M) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float v = hi[i][j][r];
                if constexpr (COLSUM) v += lo[i][j][r];
                Cz[(size_t)(m + acc_row(r, h)) * ldc + n] = v + bn;
            }
        }
    }
    if constexpr (COLSUM) {
        if (!sums) return;
        static_assert(A_ACROSS, "column sums of the operand that is read across its rows");
        __syncthreads();
        f32x4* red = reinterpret_cast<f32x4*>(smem);  // [16 threads of a column][WM * 16 columns of four]
#pragma unroll
        for (int i = 0; i < WM; ++i) red[(t >> 4) * (WM * 16) + i * 16 + (t & 15)] = csum[i];
        __syncthreads();
        if (t < WM * 16) {
            f32x4 s = red[t];
            for (int k = 1; k < 16; ++k) s += red[k * (WM * 16) + t];
            const int m = m0 + 4 * t;
            if (m < M) *reinterpret_cast<f32x4*>(Csum + (size_t)z * M + m) = s;
        }
    }
}
// consecutive items share the rows of A (the larger operand) and run on one die
template <bool A_ACROSS, bool B_ACROSS, int WM, int WN, bool COLSUM>
__global__ __launch_bounds__(256, 2) void project_kernel(Product y) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    project_item<A_ACROSS, B_ACROSS, WM, WN, COLSUM>(y, xcd_remap(blockIdx.x, gridDim.x), smem);
}
// Both products of a backward, which read the same dY, in one launch: the pieces of dW (and db) first, whose work-groups live
// longest, then the tiles of dX, which fill what those leave idle.  By themselves both wait for memory most of their time (3.3
// TB/s of operands) and, at a few thousand rows, for a launch.  us, dX, then dW and db / in one launch, each with the launch
// that adds the pieces: 65536 x 64 -> 192 37.1 / 34.3, 65536 x 64 -> 64 22.9 / 16.9, 16384 x 64 -> 192 20.9 / 16.0, 2048 x 64 -> 192 16.5 /
// 10.7, 8192 x 128 -> 384 31.2 / 22.8, 524288 x 64 -> 192 254 / 243.  (As many registers as the larger of the two needs: with dX in
// 128 x 128 tiles 242, so that two work-groups to a CU are left where dW had four: 32768 x 256 -> 768 183 / 208.)
__global__ __launch_bounds__(256, 2) void project_backward_kernel(Product weight, Product input, int pieces) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    if ((int)blockIdx.x < pieces) project_item<true, true, 1, 1, true>(weight, xcd_remap(blockIdx.x, pieces), smem);
    else project_item<false, true, 1, 1, false>(input, xcd_remap(blockIdx.x - pieces, gridDim.x - pieces), smem);
}

// out[i] = sum_z part[z][i] for the weight gradient and, behind it, the bias gradient; eight threads share a float4.
__global__ __launch_bounds__(256) void project_reduce_kernel(const float* __restrict__ part, float* __restrict__ out,
                                                             int n, const float* __restrict__ part2,
                                                             float* __restrict__ out2, int n2, int pieces) {
    __shared__ f32x4 red[8][32];
    const int c = threadIdx.x & 31, g = threadIdx.x >> 5;
    int i = 4 * (blockIdx.x * 32 + c);
    const bool second = i >= n;
    if (second) i -= n;
    const float* p = second ? part2 : part;
    const int size = second ? n2 : n;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    if (i < size) {
#pragma unroll 8
        for (int z = g; z < pieces; z += 8) s += *reinterpret_cast<const f32x4*>(p + (size_t)z * size + i);
    }
    red[g][c] = s;
    __syncthreads();
    if (g == 0 && i < size) {
        for (int k = 1; k < 8; ++k) s += red[k][c];
        *reinterpret_cast<f32x4*>((second ? out2 : out) + i) = s;
    }
}

template <int WM, int WN>
static Product product(const SegRows& A, const SegRows& B, const SegBias& bias, float* C, int ldc, float* Csum, int M, int N,
                       int R, int chunks) {
    return Product{A, B, bias, C, Csum, ldc, M, N, R, chunks, (M + 64 * WM - 1) / (64 * WM), (N + 64 * WN - 1) / (64 * WN)};
}
template <bool AA, bool BA, int WM, int WN, bool CS>
static bool launch_project(const SegRows& A, const SegRows& B, const SegBias& bias, float* C, int ldc, float* Csum, int M,
                           int N, int R, int pieces, int chunks, hipStream_t stream) {
    constexpr int lds = OperandLds<AA, WM>::BYTES + OperandLds<BA, WN>::BYTES;
    if (lds > 64 * 1024) {  // beyond what a launch may ask for without saying so first
        static const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(project_kernel<AA, BA, WM, WN, CS>),
                                                          hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (!SPION_HIP_OK(err)) return false;
    }
    const Product y = product<WM, WN>(A, B, bias, C, ldc, Csum, M, N, R, chunks);
    hipLaunchKernelGGL((project_kernel<AA, BA, WM, WN, CS>), dim3((unsigned)y.mtiles * y.ntiles * pieces), dim3(256), lds, stream,
                       y);
    return check_launch("project_kernel");
}

// 128 x 128 tiles (half the operand traffic and splitting per product) once they give every CU two work-groups and waste
// little of their width; else 64 x 64.  Forward at 32768 x 256 -> 768: 93.5 us wide, 129 narrow; at 65536 x 64 -> 192, where
// a third of the second tile would be empty: 25.6 and 21.2; at 4096 x 512 -> 1536, 384 wide tiles: 57.4 and 56.1.
static bool wide_tiles(long long M, long long N) {
    return (M / 128) * (N / 128) >= 2 * device_cus() && (N + 127) / 128 * 128 * 5 <= N * 6;
}

static bool project_args(const char* who, long long M, int n, int segs, int K, std::initializer_list<const void*> ptrs) {
    bool ok = M > 0 && M % 32 == 0 && n > 0 && n % 32 == 0 && K > 0 && K % 32 == 0 && segs >= 1 && segs <= 3 &&
              M <= MAX_ROWS && (long long)segs * n <= 1 << 20 && (long long)segs * n * K <= 1 << 30;
    for (const void* p : ptrs) ok = ok && p && reinterpret_cast<uintptr_t>(p) % 16 == 0;
    if (!ok) set_error("%s: rows, features and outputs must be positive multiples of 32 (at most 2^30 rows, 2^20 outputs, 2^30 weights), pointers 16-byte aligned (got %lld, %d, %d x %d)",
                       who, M, K, segs, n);
    return ok;
}
static SegRows plain_rows(const float* p, int ld) { return SegRows{{p, p, p}, ONE_PIECE, ld}; }
static SegRows weight_rows(const float* const* W, int segs, int n, int K) {
    return SegRows{{W[0], W[segs > 1 ? 1 : 0], W[segs > 2 ? 2 : 0]}, segs > 1 ? n : ONE_PIECE, K};
}

int project_forward(const float* X, const float* const* W, const float* const* b, float* Y, long long M, int n, int segs,
                    int K, hipStream_t stream) {
    if (!W || !b || !project_args("spion_project_forward", M, n, segs, K, {X, Y})) {
        if (!W || !b) set_error("spion_project_forward: null weights");
        return 1;
    }
    for (int s = 0; s < segs; ++s)
        if (!project_args("spion_project_forward", M, n, segs, K, {W[s], b[s]})) return 1;
    const SegBias bias{{b[0], b[segs > 1 ? 1 : 0], b[segs > 2 ? 2 : 0]}, segs > 1 ? n : ONE_PIECE};
    const int N = segs * n;
    const bool ok = wide_tiles(M, N)
        ? launch_project<false, false, 2, 2, false>(plain_rows(X, K), weight_rows(W, segs, n, K), bias, Y, N, nullptr, (int)M, N, K, 1, K / 32, stream)
        : launch_project<false, false, 1, 1, false>(plain_rows(X, K), weight_rows(W, segs, n, K), bias, Y, N, nullptr, (int)M, N, K, 1, K / 32, stream);
    return ok ? 0 : 1;
}

int project_backward_input(const float* dY, const float* const* W, float* dX, long long M, int n, int segs, int K,
                           hipStream_t stream) {
    if (!W || !project_args("spion_project_backward_input", M, n, segs, K, {dY, dX})) {
        if (!W) set_error("spion_project_backward_input: null weights");
        return 1;
    }
    for (int s = 0; s < segs; ++s)
        if (!project_args("spion_project_backward_input", M, n, segs, K, {W[s]})) return 1;
    const int N = segs * n;
    const SegBias none{{nullptr, nullptr, nullptr}, ONE_PIECE};
    const bool ok = wide_tiles(M, K)
        ? launch_project<false, true, 2, 2, false>(plain_rows(dY, N), weight_rows(W, segs, n, K), none, dX, K, nullptr, (int)M, K, N, 1, N / 32, stream)
        : launch_project<false, true, 1, 1, false>(plain_rows(dY, N), weight_rows(W, segs, n, K), none, dX, K, nullptr, (int)M, K, N, 1, N / 32, stream);
    return ok ? 0 : 1;
}

// Pieces the sum over the rows is cut into: enough 64 x 64 tiles for three work-groups per CU, no piece under 128 rows,
// no more than 256 of them (what a piece leaves is written and read back once).
static int weight_pieces(long long M, int N, int K) {
    const long long tiles = (long long)((N + 63) / 64) * ((K + 63) / 64);
    long long p = (3 * device_cus() + tiles - 1) / tiles;
    p = std::min<long long>(std::min<long long>(p, 256), M / 128);
    return (int)std::max<long long>(p, 1);
}
long long project_workspace(long long M, int N, int K) {
    return (long long)weight_pieces(M, N, K) * ((long long)N * K + N);
}
// The pieces' results, `pieces` of [N][K] and of [N] behind them, to dW and db.
static bool add_pieces(const float* ws, float* dW, float* db, int N, int K, int pieces, hipStream_t stream) {
    const int n = N * K;
    hipLaunchKernelGGL(project_reduce_kernel, dim3((n + N + 127) / 128), dim3(256), 0, stream, ws, dW, n,
                       ws + (size_t)pieces * n, db, N, pieces);
    return check_launch("project_reduce_kernel");
}
static void weight_split(long long M, int N, int K, int& pieces, int& chunks) {
    const int want = weight_pieces(M, N, K), rows = (int)(M / 32);
    chunks = (rows + want - 1) / want;
    pieces = (rows + chunks - 1) / chunks;
}
int project_backward_weight(const float* dY, const float* X, float* dW, float* db, float* ws, long long M, int N, int K,
                            hipStream_t stream) {
    if (!project_args("spion_project_backward_weight", M, N, 1, K, {dY, X, dW, db, ws})) return 1;
    int pieces, chunks;
    weight_split(M, N, K, pieces, chunks);
    const SegBias none{{nullptr, nullptr, nullptr}, ONE_PIECE};
    return launch_project<true, true, 1, 1, true>(plain_rows(dY, N), plain_rows(X, K), none, ws, K, ws + (size_t)pieces * N * K, N,
                                                  K, (int)M, pieces, chunks, stream) &&
                   add_pieces(ws, dW, db, N, K, pieces, stream)
               ? 0
               : 1;
}

// dX, dW and db in one launch, and the one that adds the pieces; by the calls above where dX takes 128 x 128 tiles.
int project_backward(const float* dY, const float* const* W, const float* X, float* dX, float* dW, float* db, float* ws,
                     long long M, int n, int segs, int K, hipStream_t stream) {
    if (!W || !project_args("spion_project_backward", M, n, segs, K, {dY, X, dX, dW, db, ws})) {
        if (!W) set_error("spion_project_backward: null weights");
        return 1;
    }
    for (int s = 0; s < segs; ++s)
        if (!project_args("spion_project_backward", M, n, segs, K, {W[s]})) return 1;
    const int N = segs * n;
    if (wide_tiles(M, K)) {
        const int err = project_backward_input(dY, W, dX, M, n, segs, K, stream);
        return err ? err : project_backward_weight(dY, X, dW, db, ws, M, N, K, stream);
    }
    int pieces, chunks;
    weight_split(M, N, K, pieces, chunks);
    const SegBias none{{nullptr, nullptr, nullptr}, ONE_PIECE};
    const Product weight = product<1, 1>(plain_rows(dY, N), plain_rows(X, K), none, ws, K, ws + (size_t)pieces * N * K, N, K, (int)M,
                                         chunks),
                  input = product<1, 1>(plain_rows(dY, N), weight_rows(W, segs, n, K), none, dX, K, nullptr, (int)M, K, N, N / 32);
    const int wi = weight.mtiles * weight.ntiles * pieces;
    constexpr int lds = OperandLds<true, 1>::BYTES + std::max(OperandLds<true, 1>::BYTES, OperandLds<false, 1>::BYTES);
    hipLaunchKernelGGL(project_backward_kernel, dim3((unsigned)wi + (unsigned)input.mtiles * input.ntiles), dim3(256), lds, stream,
                       weight, input, wi);
    return check_launch("project_backward_kernel") && add_pieces(ws, dW, db, N, K, pieces, stream) ? 0 : 1;
}

// [B][L] key mask (1 valid, 0 padded) -> [B*H][L] additive penalties 1e6 (1 - mask), one copy per head
// (models/attention_blockcuda_mask.py:42-43).
__global__ __launch_bounds__(256) void key_penalty_kernel(const float* __restrict__ mask, float* __restrict__ pen, long long total,
                                                          long long L, int H) {
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256) {
        const long long bh = i / L;
        pen[i] = 1e6f * (1.0f - mask[bh / H * L + (i - bh * L)]);
    }
}
static bool key_mask_args(const char* who, const float* mask, const float* pen, int B, int H, int L) {
    if (mask && pen && B > 0 && H > 0 && L > 0) return true;
    set_error("%s: bad arguments", who);
    return false;
}
int key_penalty(const float* mask, float* pen, int B, int H, int L, hipStream_t stream) {
    if (!key_mask_args("spion_key_penalty", mask, pen, B, H, L)) return 1;
    const long long total = (long long)B * H * L;
    hipLaunchKernelGGL(key_penalty_kernel, dim3((unsigned)std::min<long long>((total + 255) / 256, 2048)), dim3(256), 0, stream, mask,
                       pen, total, (long long)L, H);
    return check_launch("key_penalty_kernel") ? 0 : 1;
}
int project_forward_keys(const float* X, const float* const* W, const float* const* b, float* Y, long long M, int n, int segs, int K,
                         const float* mask, float* pen, int B, int H, int L, hipStream_t stream) {
    if (!key_mask_args("spion_project_forward_keys", mask, pen, B, H, L)) return 1;
    return project_forward(X, W, b, Y, M, n, segs, K, stream) || key_penalty(mask, pen, B, H, L, stream) ? 1 : 0;
}

}  // namespace spion
