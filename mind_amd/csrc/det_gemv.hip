// det_gemv.hip -- exact Q16.16 and int16 GEMV, HBM-streaming.
//
//   y[b][i] = (int32) sum_k ( (int64)W[i,k] * (int64)x[b][k]  >>arith 16 )
// Semantics of __mind_blas_gemv_q16_mt / __mind_blas_matmul_rmajor_q16_v
// (reference src/mlir/lowering.rs:9822-9997 emit_gemv_q16_row_band and
// :6675-7035; oracle benches/det_gemv_q16_mt.rs:186-197 and the per-row
// runtime-support/mind_intrinsics.c:1459-1471 dot).
//
// floor(p / 2^16) = (p - (p mod 2^16)) / 2^16 and p mod 2^16 is the product
// of the operands' low halves mod 2^16, so with S = sum of the 64-bit products
// and R = sum of those residues the result is bits [16, 48) of S - R, both mod
// 2^64: one v_mad_i64_i32 per term and half a v_pk_mul_lo_u16 and half a
// v_dot2_u32_u16 (20 issue cycles per wave and term against 40 for
// mul_lo + mul_hi + alignbit + add, which is what bounds more than two
// vectors at the rate W streams).
//   int16: y[r] = (int32) sum_i (int64)W[r,i] * (int64)x[i]
// (__mind_blas_matmul_rmajor_i16_v; reference src/mlir/lowering.rs:
// 10723-11150, oracle benches/det_matmul_i16.rs:218-230): sums mod 2^32 of the
// exact products (v_dot2_i32_i16).
// Integer addition is associative, so the split of a row over lanes and waves
// and the order of the reduction do not change the bits.
//
// W is read exactly once in 16-byte vectors, at whatever element alignment a
// row starts (gfx950 global loads need none; a wave still reads one
// contiguous run of each row), with the K remainder by element.  LPR lanes
// share a row (16 for short rows, so that a lane has several vectors), a lane
// owns ROWS rows and all NB vectors, and KS waves of a block split K, joined
// in LDS; the rules are at the launches.
#include <type_traits>

#include "det_common.h"
#include "det_kernels.h"

namespace det {
namespace gemv {

constexpr int THREADS = 256, WAVES = THREADS / 64;

// 16-byte loads at element alignment
typedef int v4i32_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef int v4i32_a2 __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ v4i32 load16(const int32_t *p) { return *(const v4i32_a4 *)p; }
__device__ __forceinline__ v4i32 load16(const int16_t *p) { return *(const v4i32_a2 *)p; }
// read once: non-temporal
__device__ __forceinline__ v4i32 stream16(const int32_t *p) { return __builtin_nontemporal_load((const v4i32_a4 *)p); }
__device__ __forceinline__ v4i32 stream16(const int16_t *p) { return __builtin_nontemporal_load((const v4i32_a2 *)p); }

struct Q16 {
    typedef int32_t T;
    static constexpr int PER = 4;   // elements per vector
    struct Op { v4i32 v; v2u16 lo[2]; };
    struct Acc { unsigned long long s; uint32_t r; };   // s mod 2^64
    static __device__ __forceinline__ Acc zero() { return {0, 0}; }
    static __device__ __forceinline__ Op op(v4i32 v) {
        Op o;
        o.v = v;
        o.lo[0] = __builtin_bit_cast(v2u16, __builtin_amdgcn_perm((uint32_t)v.y, (uint32_t)v.x, 0x05040100u));
        o.lo[1] = __builtin_bit_cast(v2u16, __builtin_amdgcn_perm((uint32_t)v.w, (uint32_t)v.z, 0x05040100u));
        return o;
    }
    // two products of the type's lowest value already reach 2^63: unsigned sums
    static __device__ __forceinline__ unsigned long long prod(T w, T x) {
        return (unsigned long long)((long long)w * x);
    }
    static __device__ __forceinline__ void add(Acc &a, const Op &w, const Op &x) {
        const v2u16 one = {1, 1};
        a.s += prod(w.v.x, x.v.x);
        a.s += prod(w.v.y, x.v.y);
        a.s += prod(w.v.z, x.v.z);
        a.s += prod(w.v.w, x.v.w);
        a.r = __builtin_amdgcn_udot2(w.lo[0] * x.lo[0], one, a.r, false);
        a.r = __builtin_amdgcn_udot2(w.lo[1] * x.lo[1], one, a.r, false);
    }
    static __device__ __forceinline__ void add1(Acc &a, T w, T x) {
        a.s += prod(w, x);
        a.r += ((uint32_t)w * (uint32_t)x) & 0xffffu;
    }
    // residue sums stay below 2^32 for 2^14 vectors (2^16 terms below 2^16)
    static constexpr int FOLD = 1 << 14;
    static __device__ __forceinline__ void fold(Acc &a) { a.s -= a.r, a.r = 0; }
    typedef unsigned long long Sum;
    static __device__ __forceinline__ Sum sum(const Acc &a) { return a.s - a.r; }
    static __device__ __forceinline__ int32_t out(Sum v) { return (int32_t)(uint32_t)(v >> 16); }
};

struct I16 {
    typedef int16_t T;
    static constexpr int PER = 8;
    struct Op { v4i32 v; };
    typedef int Acc;
    static __device__ __forceinline__ Acc zero() { return 0; }
    static __device__ __forceinline__ Op op(v4i32 v) { return {v}; }
    static __device__ __forceinline__ void add(Acc &a, const Op &w, const Op &x) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int we = w.v[e], xe = x.v[e];
            a = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2i16, we), __builtin_bit_cast(v2i16, xe), a, false);
        }
    }
    static __device__ __forceinline__ void add1(Acc &a, T w, T x) {
        a = (int)((uint32_t)a + (uint32_t)((int)w * (int)x));
    }
    static constexpr int FOLD = 1 << 30;
    static __device__ __forceinline__ void fold(Acc &) {}
    typedef uint32_t Sum;
    static __device__ __forceinline__ Sum sum(const Acc &a) { return (Sum)a; }
    static __device__ __forceinline__ int32_t out(Sum v) { return (int32_t)v; }
};

__device__ __forceinline__ uint32_t shx(uint32_t v, int m) { return (uint32_t)__shfl_xor((int)v, m); }
__device__ __forceinline__ unsigned long long shx(unsigned long long v, int m) {
    return ((unsigned long long)shx((uint32_t)(v >> 32), m) << 32) | shx((uint32_t)v, m);
}

// Sums v[0..N) over the lanes that differ in the bits below 2 M.  While N > 1
// each step halves the values: the lanes with bit M set go on with the upper
// half.  Returns the index of the value left in v[0] of this lane.
template <int N, int M, typename S, int TOT>
__device__ __forceinline__ int lane_sums(S (&v)[TOT], int lane) {
    if constexpr (M == 0) {
        return 0;
    } else if constexpr (N > 1) {
        const bool up = lane & M;
#pragma unroll
        for (int i = 0; i < N / 2; ++i) {
            const S send = up ? v[i] : v[i + N / 2], keep = up ? v[i + N / 2] : v[i];
            v[i] = keep + shx(send, M);
        }
        return (up ? N / 2 : 0) + lane_sums<N / 2, M / 2>(v, lane);
    } else {
        v[0] += shx(v[0], M);
        return lane_sums<1, M / 2>(v, lane);
    }
}

// X: [nb][K], Y: [nb][M], nb <= NB.  ROWS NB values must be a power of two not above LPR.
template <class O, int NB, int ROWS, int LPR, int KS, int U>
__global__ __launch_bounds__(THREADS) void gemv_kernel(const typename O::T *__restrict__ W,
                                                       const typename O::T *__restrict__ X, int32_t *__restrict__ Y,
                                                       int M, int K, int nb) {
    typedef typename O::T T;
    typedef typename O::Sum S;
    constexpr int V = ROWS * NB, RPW = ROWS * (64 / LPR);   // values per lane, rows per wave
    static_assert((V & (V - 1)) == 0 && V <= LPR && WAVES % KS == 0, "lane_sums shape");
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cl = lane % LPR, ks = wave % KS;
    const int row0 = (blockIdx.x * (WAVES / KS) + wave / KS) * RPW + lane / LPR * ROWS;
    const T *wr[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) wr[r] = W + (size_t)min(row0 + r, M - 1) * K;
    const T *xr[NB];   // vectors past nb repeat the last one and are not stored
#pragma unroll
    for (int b = 0; b < NB; ++b) xr[b] = X + (size_t)min(b, nb - 1) * K;
    typename O::Acc acc[ROWS][NB];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[r][b] = O::zero();

    constexpr int STEP = LPR * KS;
    const int KV = K / O::PER;
    auto trip = [&](int c, auto un) {
        constexpr int UU = decltype(un)::value;
        v4i32 wv[UU][ROWS];
#pragma unroll
        for (int u = 0; u < UU; ++u)
#pragma unroll
            for (int r = 0; r < ROWS; ++r)
                wv[u][r] = stream16(wr[r] + (size_t)(c + STEP * u) * O::PER);
#pragma unroll
        for (int u = 0; u < UU; ++u) {
            typename O::Op x[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b)
                x[b] = O::op(load16(xr[b] + (size_t)(c + STEP * u) * O::PER));
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const typename O::Op w = O::op(wv[u][r]);
#pragma unroll
                for (int b = 0; b < NB; ++b) O::add(acc[r][b], w, x[b]);
            }
        }
    };
    int c = cl + LPR * ks;
    while (true) {
        // at most FOLD vectors per lane, then the residues go into the sums
        const long long stop = (long long)c + (long long)STEP * O::FOLD;
        const int end = stop < KV ? (int)stop : KV;
        for (; c + STEP * (U - 1) < end; c += STEP * U) trip(c, std::integral_constant<int, U>());
        for (; c < end; c += STEP) trip(c, std::integral_constant<int, 1>());
        if (end == KV) break;
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
#pragma unroll
            for (int b = 0; b < NB; ++b) O::fold(acc[r][b]);
    }
    const int k = KV * O::PER + cl;   // the K remainder
    if (ks == 0 && k < K) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const T xv = xr[b][k];
#pragma unroll
            for (int r = 0; r < ROWS; ++r) O::add1(acc[r][b], wr[r][k], xv);
        }
    }

    S v[V];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int b = 0; b < NB; ++b) v[r * NB + b] = O::sum(acc[r][b]);
    const int i = lane_sums<V, LPR / 2>(v, lane);
    // lanes that share the low bits hold the same value: one of them writes
    bool mine = cl % (LPR / V) == 0;
    if constexpr (KS > 1) {
        __shared__ S part[WAVES][64];
        part[wave][lane] = v[0];
        __syncthreads();
        mine = mine && ks == 0;
        if (mine) {
#pragma unroll
            for (int s = 1; s < KS; ++s) v[0] += part[wave + s][lane];
        }
    }
    const int row = row0 + i / NB;
    if (mine && row < M && i % NB < nb) Y[(size_t)(i % NB) * M + row] = O::out(v[0]);
}

template <class O, int NB, int ROWS, int LPR, int KS, int U>
static void launch(const typename O::T *W, const typename O::T *X, int32_t *Y, int M, int K, int nb,
                   hipStream_t s) {
    constexpr int RPB = WAVES / KS * ROWS * (64 / LPR);
    hipLaunchKernelGGL((gemv_kernel<O, NB, ROWS, LPR, KS, U>), dim3((unsigned)((M + RPB - 1) / RPB)), dim3(THREADS), 0,
                       s, W, X, Y, M, K, nb);
}

// Rows of up to 256 vectors take 16 lanes where there are enough of them, rows
// of up to 64 always (x is then read once for 4 rows: a host call of 64 x 64
// 16.3 us against 18.0 with a wave per row);
// longer ones a wave, or 2 or 4 waves where one per 4 rows would leave the
// chip short of loads in flight.  Device time per call, before (one wave per 2
// or 4 rows, by element off the 16-byte grid, groups of 8, 4, 2, 1 vectors, or
// the MFMA kernel of det_gemv_mfma.hip) -> now:
//   16 lanes:  11922 x 384 8 vectors 18.5 -> 10.3 us, 3 vectors 13.7 -> 8.7;
//   1 wave:    16384^2 164.2 -> 163.9 (6.6 TB/s), 16384 x 16383 200 -> 172,
//              16384 x 8192 2 vectors 142.7 -> 98, 8192^2 4 vectors 87 -> 64;
//              int16 16384^2 95.3 -> 92.0 (5.8 TB/s), 16384 x 16383 150 -> 90,
//              8192 x 8190 64.0 -> 23.4 (5.7 TB/s);
//   2 waves:   4096^2 16.1 -> 11.9, 8 vectors 39.5 -> 27.2;
//   4 waves:   300 x 8191 41 -> 7.2, 1024 x 16384 27 -> 14.2 (4.7 TB/s),
//              320 x 6882 3 vectors 74 -> 7 (calls of about 7 us are host
//              submission); int16 300 x 16384 21 -> 6.8.
// One vector is bound by the stream of W, 8 by the products (8192^2 81 us at
// 71 us of issue).  4 rows per wave against 2 for 8 vectors: 8192^2 81 against
// 86 us although 225 registers leave 2 waves per SIMD instead of 3; int16 one
// column per trip against two: 16384^2 92 against 102 us.
template <class O, int NB>
static void launch_rows(const typename O::T *W, const typename O::T *X, int32_t *Y, int M, int K, int nb,
                        hipStream_t s) {
    constexpr int R = NB >= 8 ? 2 : 4;
    if (K / O::PER <= 256 && M >= 4096) launch<O, NB, R, 16, 1, 2>(W, X, Y, M, K, nb, s);
    else if (K / O::PER <= 64) launch<O, NB, (NB >= 4 ? 2 : 1), 16, 1, 2>(W, X, Y, M, K, nb, s);
    else if (M >= 8192) launch<O, NB, 4, 64, 1, (O::PER == 8 ? 1 : 2)>(W, X, Y, M, K, nb, s);
    else if (M >= 2048) launch<O, NB, R, 64, 2, 2>(W, X, Y, M, K, nb, s);
    else launch<O, NB, (NB >= 4 ? 2 : 1), 64, 4, (NB >= 4 ? 2 : 4)>(W, X, Y, M, K, nb, s);
}

}  // namespace gemv

// X: [nb][K], Y: [nb][M]: up to 8 vectors at a time, W streamed once per group.
hipError_t launch_gemv_q16(const int32_t *W, const int32_t *X, int32_t *Y, int M, int K, int nb, hipStream_t s) {
    using namespace gemv;
    for (int b = 0; b < nb; b += 8) {
        const int g = nb - b < 8 ? nb - b : 8;
        const int32_t *Xb = X + (size_t)b * K;
        int32_t *Yb = Y + (size_t)b * M;
        if (g > 4) launch_rows<Q16, 8>(W, Xb, Yb, M, K, g, s);
        else if (g > 2) launch_rows<Q16, 4>(W, Xb, Yb, M, K, g, s);
        else if (g == 2) launch_rows<Q16, 2>(W, Xb, Yb, M, K, g, s);
        else launch_rows<Q16, 1>(W, Xb, Yb, M, K, g, s);
    }
    return hipGetLastError();
}

hipError_t launch_gemv_i16(const int16_t *W, const int16_t *x, int32_t *y, int M, int K, hipStream_t s) {
    gemv::launch_rows<gemv::I16, 1>(W, x, y, M, K, 1, s);
    return hipGetLastError();
}

}  // namespace det
