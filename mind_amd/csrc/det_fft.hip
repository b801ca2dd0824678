// det_fft.hip -- deterministic Q16.16 radix-2 DIT FFT, batched, in place.
//
// Semantics (examples/fft_q16.mind:15-120, the fft256(re, im, tw, logn, n)
// symbol that benches/fft_q16.rs:66-168 and bench/fft/harness.c dlopen):
// re / im are n = 2^logn int64 Q16.16 samples; tw[2k], tw[2k+1] (k < n/2) the
// twiddle (wr, wi).  After the bit-reversal permutation, the span-2 stage is
// a plain add / subtract (the kernel peels it: no twiddle), and every span
// s >= 4 stage runs, for each block base and j < s/2, with k = j * (n / s):
//     t = (qmul(wr, x_b) - qmul(wi, y_b),  qmul(wr, y_b) + qmul(wi, x_b))
//     a' = a + t,  b' = a - t,        qmul(w, v) = low64(w * v) >>arith 16
// All adds, subtracts and products wrap in int64, like MIND's i64 ops.
//
// GPU mapping.  Butterflies of one stage are independent, and the stage
// order is all that the result depends on, so any data layout that performs
// the same butterflies stage by stage gives the same bits.  The position
// (after bit reversal) of a point is a logn-bit number; stage b pairs points
// that differ in bit b.  A pass keeps 16 points per lane whose positions
// differ exactly in a 4-bit window [s, s + 4) (register index r = those
// bits, lane index t = the other bits) and runs the stages of that window in
// registers:
//   * n <= 16        : one FFT per thread (fft_small_kernel);
//   * 32 <= n <= 2048: whole transforms in one workgroup, n / 16 lanes each,
//                      windows separated by an LDS transpose, one HBM read
//                      and one write per point (fft_rows_kernel up to 512
//                      points, fft_block_kernel above; fft_few_kernel for a
//                      few transforms of up to 1024 points);
//   * n >= 4096      : the same up to 8192 points, else passes of 6 to 9
//                      stages over columns of 16 points (fft_cols_kernel).
// A window runs in int32 when a bound on its inputs proves that every
// intermediate fits (same integers, cheaper products), else in int64.
#include "det_common.h"
#include "det_kernels.h"

namespace det {
namespace fft {

// Value arithmetic.  int64_t: the general path, wrapping like MIND's i64.
// int32_t: the bounded path, only taken when every intermediate value is
// known to fit in int32 (then 32-bit arithmetic gives the same integers):
// one signed 32 x 32 -> 64 product per qmul, and the shifted product fits in
// int32 because |qmul(w, x)| <= |x| for |w| <= 2^16.
__device__ __forceinline__ int64_t vadd(int64_t a, int64_t b) { return (int64_t)((uint64_t)a + (uint64_t)b); }
__device__ __forceinline__ int64_t vsub(int64_t a, int64_t b) { return (int64_t)((uint64_t)a - (uint64_t)b); }
__device__ __forceinline__ int32_t vadd(int32_t a, int32_t b) { return (int32_t)((uint32_t)a + (uint32_t)b); }
__device__ __forceinline__ int32_t vsub(int32_t a, int32_t b) { return (int32_t)((uint32_t)a - (uint32_t)b); }
__device__ __forceinline__ int64_t qm(int64_t w, int64_t v) { return ((int64_t)((uint64_t)w * (uint64_t)v)) >> 16; }
__device__ __forceinline__ int32_t qm(int64_t w, int32_t v) {
    const int64_t p = (int64_t)(int32_t)w * (int64_t)v;
    return (int32_t)(p >> 16);
}

// One butterfly (peeled: the span-2 stage, no twiddle) on (a, b).
template <typename V>
__device__ __forceinline__ void butterfly(V &ar, V &ai, V &br, V &bi, int64_t wr, int64_t wi, bool peeled) {
    V tr, ti;
    if (peeled) {
        tr = br, ti = bi;
    } else {
        tr = vsub(qm(wr, br), qm(wi, bi));
        ti = vadd(qm(wr, bi), qm(wi, br));
    }
    const V ur = ar, ui = ai;
    ar = vadd(ur, tr), ai = vadd(ui, ti);
    br = vsub(ur, tr), bi = vsub(ui, ti);
}

// Largest input component for which `stages` stages (the first of them peeled
// if `peeled`) stay in int32 when every twiddle component is within
// [-2^16, 2^16].  A twiddle then has complex magnitude at most sqrt 2, and the
// floors of the two products of a component add an error of at most (1, 2), so
// a butterfly takes the largest magnitude M to at most
// (1 + sqrt 2) M + 2.24 (a peeled one to 2 M): components stay below 2^31, and
// so do the products, |qmul(w, x)| <= |x| + 1.  A component-wise bound (each
// stage triples the largest component) would send n >= 1024 with Q16 inputs in
// [-1, 1) to int64.
__host__ __device__ constexpr int32_t i32_bound(int stages, bool peeled) {
    double g = peeled ? 2.0 : 1.0;
    for (int i = peeled ? 1 : 0; i < stages; ++i) g *= 2.4143;   // > 1 + sqrt 2
    return (int32_t)((2147483647.0 / g - 4.0) / 1.41422);        // > sqrt 2: component -> magnitude
}
constexpr int64_t TW_SMALL = 65536;
// (any int64: no sum that could overflow)
__device__ __forceinline__ bool in_range(int64_t v, int64_t bound) { return v >= -bound && v <= bound; }

__device__ __forceinline__ uint32_t bitrev(uint32_t v, int bits) { return bits ? __brev(v) >> (32 - bits) : 0u; }

// Position of register r of lane-group index t for the window [s, s + 4).
__device__ __forceinline__ uint32_t win_pos(uint32_t t, int r, int s) {
    return ((t >> s) << (s + 4)) | ((uint32_t)r << s) | (t & ((1u << s) - 1u));
}

// A window's twiddles on the int32 path (valid when every component is
// within [-2^16, 2^16]).  Slot (2^rb - 1) + j of a window's table holds
// the twiddle of stage s + rb for butterflies whose register index has low
// bits j (the position bits below the stage bit are those low bits and the
// lane's own bits, so 1 + 2 + 4 + 8 slots cover a window).
struct WinTw {
    int32_t r[15], i[15];
};

// ---------------------------------------------------------------- n <= 16
// One thread per FFT; registers indexed by position.
template <int LOGN>
__global__ __launch_bounds__(256) void fft_small_kernel(const int64_t *__restrict__ sre,
                                                        const int64_t *__restrict__ sim, int64_t *__restrict__ dre,
                                                        int64_t *__restrict__ dim, const int64_t *__restrict__ tw,
                                                        int64_t batch) {
    constexpr int N = 1 << LOGN;
    const int64_t f = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (f >= batch) return;
    const int64_t *R = sre + f * N, *I = sim + f * N;
    int64_t xr[N], xi[N];
#pragma unroll
    for (int p = 0; p < N; ++p) {
        const uint32_t src = bitrev((uint32_t)p, LOGN);
        xr[p] = R[src], xi[p] = I[src];
    }
#pragma unroll
    for (int b = 0; b < LOGN; ++b)
#pragma unroll
        for (int p = 0; p < N; ++p) {
            if (p & (1 << b)) continue;
            int64_t wr = 0, wi = 0;
            if (b > 0) {
                const int k = (p & ((1 << b) - 1)) << (LOGN - 1 - b);
                wr = tw[2 * k], wi = tw[2 * k + 1];
            }
            butterfly(xr[p], xi[p], xr[p | (1 << b)], xi[p | (1 << b)], wr, wi, b == 0);
        }
#pragma unroll
    for (int p = 0; p < N; ++p) dre[f * N + p] = xr[p], dim[f * N + p] = xi[p];
}

// ---------------------------------------------------------------- n >= 32
// The stages are cut into windows of 4 position bits as above, and the
// windows into pieces of work that live in one workgroup's LDS:
//   * short transforms (fft_rows_kernel, n <= 512): 4096 consecutive points
//     per workgroup;
//   * whole transforms (fft_block_kernel, n = 1024 .. 8192): one workgroup per
//     transform;
//   * column passes (fft_cols_kernel<NB>): a pass runs NB = 6..9 stages
//     [s, s + NB).  A workgroup holds the 2^NB positions l << s of 16
//     neighbouring columns, so every load and store moves runs of 16
//     consecutive points (128 bytes) or longer, also the first pass's loads
//     through the bit reversal: 16 neighbouring source points are 16 columns.
//     logn / 9 passes, rounded up (10 stages would need 1024 threads of 128
//     registers, which spill: 2 x 2^20 points 131 us in two passes, 58 in
//     three); a pass writes the positions it reads, so every pass after the
//     first may run in place.
// What bounds them: a pass streams 32 bytes per point and spends about
// 300 cycles per wave and butterfly in int64 (12 quarter-rate multiplies) or
// 104 in int32, so the arithmetic matters as much as the stream.  A window
// therefore runs in int32 whenever its inputs and twiddles allow it
// (i32_bound).  The test is repeated at each window, so only the window's own
// growth has to be allowed for; when a test fails the block goes on in int64
// from that window (RESUME: the kernels that hold whole transforms), or starts
// again from the source (column passes, where going on costs 5% of the int32
// path: 16 x 2^16 points 27.8 -> 29.2 us; nothing is stored before the last
// window).  Same butterflies, same stage order, same integers on either path.
// Device time per call, out of place, inputs within 2^16 (before: windows of
// the short transforms in one kernel with an all-or-nothing int32 test that
// left n >= 1024 in int64; one global-memory pass per 4 stages beyond, whose
// first pass gathered single 8-byte points):
//   65536 x 256 points 102 -> 95 us (5.6 TB/s; a large copy reaches 5.2),
//   32768 x 512 146 -> 99, 13594 x 1024 231 -> 90, 8192 x 2048 302 -> 115,
//   100000 x 64 87 -> 34, 100000 x 128 104 -> 66, 300000 x 32 355 -> 48,
//   8192 x 128 10.0 -> 9.2, 5000 x 128 8.2 -> 8.3, 1000 x 256 7.5 -> 7.5;
//   16 x 2^16 points 86.1 -> 25.5 (34 MB read and written once: 6.6 us at the
//   copy rate; the two passes wait for memory, then compute, with one workgroup
//   per compute unit), 32 x 2^16 128 -> 36.4, 8 x 2^18 148 -> 44.2, 1 x 2^16
//   61 -> 17.1, 512 x 4096 91 -> 20.6, 256 x 8192 94 -> 25.7.
// Inputs within 2^40 (int64): 65536 x 256 113 -> 115, 8192 x 256 16.3 -> 16.3,
//   32768 x 512 191 -> 136, 13594 x 1024 231 -> 135, 8192 x 2048 301 -> 172,
//   100000 x 64 81 -> 46, 100000 x 128 105 -> 87, 5000 x 128 10.3 -> 10.2, 16 x
//   2^16 86 -> 36.
// Inputs up to 2^25, where a later window's test fails (before: int64
// throughout; restarting; going on): 65536 x 256 113, 161, 108 us, 8192 x 256
// 16.3, 20.6, 14.9, 600 x 512 12.5, 14.8, 10.9, 300 x 1024 10.8, 12.2, 9.5,
// 16 x 2048 11.6, 13.2, 10.2 (2^22: 11.6, 15.0, 9.0).
// Window P of NB bits: first bit of its 4 registers, and the stages it runs.
template <int NB, int P>
struct Win {
    static constexpr int S = 4 * P < NB - 4 ? 4 * P : NB - 4, B0 = 4 * P, B1 = 4 * P + 4 < NB ? 4 * P + 4 : NB;
};

// LDS layouts.  label(): the position bits of thread t outside a window;
// col(): its column; idx(): the 8-byte LDS element of position l, column c,
// swizzled so that 32 consecutive lanes touch 32 different elements mod 32.
template <int NB>
struct BlockLay {   // a whole transform, one column
    static constexpr int THREADS = 1 << (NB - 4), ELEMS = 1 << NB;
    static constexpr bool FIRST = true, STAGED = false, KEEP = false, RESUME = true;
    using Wide = BlockLay;
    // window 0 takes its labels bit-reversed: neighbouring threads then load
    // neighbouring source points
    template <int P>
    static __device__ __forceinline__ uint32_t label(uint32_t t) { return P == 0 ? bitrev(t, NB - 4) : t; }
    template <int P>
    static __device__ __forceinline__ uint32_t col(uint32_t) { return 0; }
    static __device__ __forceinline__ uint32_t idx(uint32_t l, uint32_t) {
        // window 0 writes with lanes on the top 5 position bits, window 1 reads
        // on bits 0..3 and 8, later windows on bits 0..4
        uint32_t f = ((l >> 9) & 15u) ^ (((l >> 8) & 1u) << 4);
        if (NB == 10) f ^= ((l >> 5) & 7u) << 1;
        if (NB == 11) f ^= ((l >> 6) & 3u) << 2;
        if (NB == 12) f ^= ((l >> 7) & 1u) << 3;
        return l ^ f;
    }
};
template <int NB, bool STAGED_>
struct RowsLay {   // 4096 consecutive points: 2^(12 - NB) whole short transforms
    static constexpr int THREADS = 256, ELEMS = 4096;
    static constexpr bool FIRST = true;
    // STAGED: loads and stores are linear and go through LDS (below 256 points
    // a window's lanes cover less than a 128-byte line of each transform).
    // The int64 path, 16 bytes a point, is staged below 128 points only.
    // KEEP: inputs that fail window 0's test stay in registers.  Staged ones are
    // read again, which leaves a third wave per SIMD (300000 x 32 points 54 us
    // kept, 48 read again, 100000 x 64 38, 34; in +-2^40 65, 62 and 49, 46).
    static constexpr bool STAGED = STAGED_, KEEP = !STAGED, RESUME = true;
    using Wide = RowsLay<NB, STAGED_ && (NB < 7)>;
    template <int P>
    static __device__ __forceinline__ uint32_t label(uint32_t t) {
        const uint32_t j = t & ((1u << (NB - 4)) - 1u);
        return P == 0 && !STAGED ? bitrev(j, NB - 4) : j;
    }
    template <int P>
    static __device__ __forceinline__ uint32_t col(uint32_t t) { return t >> (NB - 4); }
    static __device__ __forceinline__ uint32_t idx(uint32_t l, uint32_t c) {
        // 32 lanes cover, in turn: the top 5 position bits (linear loads), the
        // label bits 4.. and columns (window 0), the label's low bits and
        // columns (last window), the low 5 position bits (linear stores)
        uint32_t f = 0;
        if (NB == 5) f = (c & 15u) ^ ((c & 1u) << 4);
        if (NB == 6) f = ((l >> 5) & 1u) ^ ((c & 3u) << 2) ^ (((c >> 2) & 1u) * 0x12u);
        if (NB == 7) f = ((l >> 5) & 3u) ^ ((c & 3u) << 2) ^ ((c & 1u) << 4);
        if (NB == 8) f = ((l >> 5) & 7u) ^ ((c & 1u) * 0x18u);
        if (NB == 9) f = ((l >> 5) & 15u) ^ (((l >> 8) & 1u) << 4);
        return ((c << NB) | l) ^ f;
    }
};
template <int NB, bool FIRST_>
struct ColsLay {   // 2^NB positions of 16 columns
    static constexpr int THREADS = 1 << NB, ELEMS = 16 << NB, NP = (NB + 3) / 4;
    static constexpr bool FIRST = FIRST_, STAGED = false, KEEP = false, RESUME = false;
    using Wide = ColsLay;
    // the first pass stores runs of consecutive positions of one column, so
    // its last window has lanes along the positions; else lanes run along
    // the 16 columns
    template <int P>
    static __device__ __forceinline__ uint32_t label(uint32_t t) {
        return FIRST && P == NP - 1 ? t & ((1u << (NB - 4)) - 1u) : t >> 4;
    }
    template <int P>
    static __device__ __forceinline__ uint32_t col(uint32_t t) {
        return FIRST && P == NP - 1 ? t >> (NB - 4) : t & 15u;
    }
    static __device__ __forceinline__ uint32_t idx(uint32_t l, uint32_t c) {
        return ((l << 4) | (c ^ (l & 15u))) ^ (l & 16u);
    }
};

// Twiddles of window P for a thread: `low` holds the position bits below the
// window's registers, shifted by s, and the column.  Stage bit b of the
// transform uses table entry (position mod 2^b) << (logn - 1 - b).
template <class L, int NB, int P, typename F>
__device__ __forceinline__ void each_twiddle(uint32_t low, int s, int logn, F &&f) {
    using W = Win<NB, P>;
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
        const int bb = W::S + rb;
        if (bb < W::B0 || bb >= W::B1) continue;
        if (L::FIRST && bb == 0) continue;   // the peeled stage
#pragma unroll
        for (int q = 0; q < (1 << rb); ++q)
            f(rb, q, (low << (logn - 1 - s - bb)) + ((uint32_t)q << (logn - 1 - rb)));
    }
}

// int32 twiddles of window P; returns whether every component is within
// [-2^16, 2^16].
template <class L, int NB, int P>
__device__ __forceinline__ bool load_tw32(WinTw &w, const int64_t *__restrict__ tw, uint32_t low, int s, int logn) {
    bool ok = true;
    each_twiddle<L, NB, P>(low, s, logn, [&](int rb, int q, uint32_t k) {
        const int64_t wr = tw[2 * (size_t)k], wi = tw[2 * (size_t)k + 1];
        ok = ok && in_range(wr, TW_SMALL) && in_range(wi, TW_SMALL);
        w.r[(1 << rb) - 1 + q] = (int32_t)wr, w.i[(1 << rb) - 1 + q] = (int32_t)wi;
    });
    return ok;
}

template <class L, int NB, int P>
__device__ __forceinline__ void run_win32(int32_t (&xr)[16], int32_t (&xi)[16], const WinTw &w) {
    using W = Win<NB, P>;
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
        const int bb = W::S + rb;
        if (bb < W::B0 || bb >= W::B1) continue;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if (r & (1 << rb)) continue;
            const int slot = (1 << rb) - 1 + (r & ((1 << rb) - 1)), q = r | (1 << rb);
            const bool peeled = L::FIRST && bb == 0;
            butterfly(xr[r], xi[r], xr[q], xi[q], peeled ? 0 : (int64_t)w.r[slot], peeled ? 0 : (int64_t)w.i[slot],
                      peeled);
        }
    }
}

template <class L, int NB, int P>
__device__ __forceinline__ void run_win64(int64_t (&xr)[16], int64_t (&xi)[16], const int64_t *__restrict__ tw,
                                          uint32_t low, int s, int logn) {
    using W = Win<NB, P>;
    // loads of its own: sharing the int32 path's would keep their 64-bit
    // values in registers across it
    asm volatile("" : "+s"(tw));
    if (L::FIRST && W::B0 == 0) {   // the peeled stage
#pragma unroll
        for (int r = 0; r < 16; r += 2) butterfly(xr[r], xi[r], xr[r + 1], xi[r + 1], 0, 0, true);
    }
    each_twiddle<L, NB, P>(low, s, logn, [&](int rb, int q, uint32_t k) {
        const int64_t wr = tw[2 * (size_t)k], wi = tw[2 * (size_t)k + 1];
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if (!(r & (1 << rb)) && (r & ((1 << rb) - 1)) == q)
                butterfly(xr[r], xi[r], xr[r | (1 << rb)], xi[r | (1 << rb)], wr, wi, false);
    });
}

// Block-wide AND, known to the compiler as uniform.
__device__ __forceinline__ bool block_all(bool v) { return __builtin_amdgcn_readfirstlane(__syncthreads_and(v)); }

// LDS element of register r of thread t in window P; P = -1 and NP: the
// linear order of staged loads (element r * THREADS + t of the sources) and
// stores.
template <class L, int NB, int P>
__device__ __forceinline__ uint32_t elem(uint32_t t, int r) {
    if constexpr (P < 0 || P == (NB + 3) / 4) {
        const uint32_t i = (uint32_t)r * L::THREADS + t, p = i & ((1u << NB) - 1u);
        return L::idx(P < 0 ? bitrev(p, NB) : p, i >> NB);
    } else {
        return L::idx(win_pos(L::template label<P>(t), r, Win<NB, P>::S), L::template col<P>(t));
    }
}

// Re-layout from window P - 1 to window P.
template <class L, int NB, int P, typename T>
__device__ __forceinline__ void exchange(T (&x)[16], uint32_t t, T *sm) {
#pragma unroll
    for (int r = 0; r < 16; ++r) sm[elem<L, NB, P - 1>(t, r)] = x[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = sm[elem<L, NB, P>(t, r)];
    __syncthreads();
}

// The same for int32 pairs, in two halves: to LDS as window P - 1 has them, and
// back (widened if V is int64_t) as window P wants them.
template <class L, int NB, int P>
__device__ __forceinline__ void put32(const int32_t (&yr)[16], const int32_t (&yi)[16], uint32_t t, uint64_t *sm) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
        sm[elem<L, NB, P - 1>(t, r)] = (uint64_t)(uint32_t)yr[r] | ((uint64_t)(uint32_t)yi[r] << 32);
    __syncthreads();
}
template <class L, int NB, int P, typename V>
__device__ __forceinline__ void get32(V (&yr)[16], V (&yi)[16], uint32_t t, const uint64_t *sm) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const uint64_t z = sm[elem<L, NB, P>(t, r)];
        yr[r] = (int32_t)(uint32_t)z, yi[r] = (int32_t)(uint32_t)(z >> 32);
    }
    __syncthreads();
}
template <class L, int NB, int P>
__device__ __forceinline__ void exchange32(int32_t (&yr)[16], int32_t (&yi)[16], uint32_t t, uint64_t *sm) {
    put32<L, NB, P>(yr, yi, t, sm);
    get32<L, NB, P>(yr, yi, t, sm);
}

template <class L, int NB, int P>
__device__ __forceinline__ uint32_t low_bits(uint32_t t, int s, uint32_t c0) {
    const uint32_t jl = L::template label<P>(t) & ((1u << Win<NB, P>::S) - 1u);
    return L::FIRST ? jl : (jl << s) | (c0 + L::template col<P>(t));
}

// Windows P.. of the int32 path.  Where window 0's twiddles are uniform
// (L::FIRST) w holds window P's (w_ok: all small), loaded one window ahead;
// in later passes that would cost the second wave per SIMD (16 transforms of
// 2^16 25.8 us instead of 27, 32 of them 41.9 instead of 38.6), so they are
// loaded here.  Returns the window whose test failed (L::RESUME: its inputs
// are then in LDS), or NP when all have run.
template <class L, int NB, int P>
__device__ __forceinline__ int narrow_from(int32_t (&yr)[16], int32_t (&yi)[16], const int64_t *__restrict__ tw,
                                           uint32_t t, int s, uint32_t c0, int logn, uint64_t *sm, WinTw &w, bool w_ok) {
    if constexpr (P < (NB + 3) / 4) {
        constexpr int32_t B = i32_bound(Win<NB, P>::B1 - Win<NB, P>::B0, false);
        WinTw wn;
        bool wn_ok = true;
        if constexpr (!L::FIRST) w_ok = load_tw32<L, NB, P>(w, tw, low_bits<L, NB, P>(t, s, c0), s, logn);
        else if constexpr (P + 1 < (NB + 3) / 4)
            wn_ok = load_tw32<L, NB, P + 1>(wn, tw, low_bits<L, NB, P + 1>(t, s, c0), s, logn);
        int32_t hi = yr[0], lo = yr[0];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            hi = max(max(hi, yr[r]), yi[r]);
            lo = min(min(lo, yr[r]), yi[r]);
        }
        const bool fits = block_all(w_ok && hi <= B && lo >= -B);
        if (!L::RESUME && !fits) return P;
        put32<L, NB, P>(yr, yi, t, sm);
        if (!fits) return P;
        get32<L, NB, P>(yr, yi, t, sm);
        run_win32<L, NB, P>(yr, yi, w);
        return narrow_from<L, NB, P + 1>(yr, yi, tw, t, s, c0, logn, sm, wn, wn_ok);
    }
    return P;
}

template <class L, int NB, int P>
__device__ __forceinline__ void exchange64(int64_t (&xr)[16], int64_t (&xi)[16], uint32_t t, uint64_t *sm) {
    exchange<L, NB, P>(xr, t, (int64_t *)sm);
    exchange<L, NB, P>(xi, t, (int64_t *)sm);
}

// Windows P.. of the int64 path, or those from `from` on (uniform): x holds
// window P's inputs if P >= from, later inputs are where the int32 path left them
// in LDS.  (W's labels are L's from window 1 on.)
template <class L, class W, int NB, int P>
__device__ __forceinline__ void wide_from(int64_t (&xr)[16], int64_t (&xi)[16], const int64_t *__restrict__ tw,
                                          uint32_t t, int s, uint32_t c0, int logn, uint64_t *sm, int from) {
    constexpr int NP = (NB + 3) / 4;
    if constexpr (P < NP) {
        if (from <= P) {
            run_win64<W, NB, P>(xr, xi, tw, low_bits<W, NB, P>(t, s, c0), s, logn);
            if constexpr (P + 1 < NP || W::STAGED) exchange64<W, NB, P + 1>(xr, xi, t, sm);
        } else if (P + 1 < NP && from == P + 1) {
            get32<L, NB, P + 1>(xr, xi, t, sm);
        }
        wide_from<L, W, NB, P + 1>(xr, xi, tw, t, s, c0, logn, sm, from);
    }
}

// All NB stages [s, s + NB): load(layout, t, r, re, im) gives window 0's
// points (twice if need be), store(layout, t, r, re, im) takes the last
// window's (linear order on both sides where staged).
template <class L, int NB, typename LD, typename ST>
__device__ __forceinline__ void run_pass(const int64_t *__restrict__ tw, uint32_t t, int s, uint32_t c0, int logn,
                                         uint64_t *sm, LD &&load, ST &&store) {
    constexpr int NP = (NB + 3) / 4;
    int64_t xr[16], xi[16];
    int from = 0;   // the window at which the int64 path takes over
    {
        constexpr int64_t B = i32_bound(Win<NB, 0>::B1, L::FIRST);
#pragma unroll
        for (int r = 0; r < 16; ++r) load(L(), t, r, xr[r], xi[r]);
        WinTw w, w1;
        bool ok = load_tw32<L, NB, 0>(w, tw, low_bits<L, NB, 0>(t, s, c0), s, logn);
        bool ok1 = true;
        if constexpr (L::FIRST) ok1 = load_tw32<L, NB, 1>(w1, tw, low_bits<L, NB, 1>(t, s, c0), s, logn);
#pragma unroll
        for (int r = 0; r < 16; ++r)
            ok = ok && in_range(xr[r], B) && in_range(xi[r], B);
        if (block_all(ok)) {
            int32_t yr[16], yi[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) yr[r] = (int32_t)xr[r], yi[r] = (int32_t)xi[r];
            if constexpr (L::STAGED) exchange32<L, NB, 0>(yr, yi, t, sm);
            run_win32<L, NB, 0>(yr, yi, w);
            from = narrow_from<L, NB, 1>(yr, yi, tw, t, s, c0, logn, sm, w1, ok1);
            if (from == NP) {
                if constexpr (L::STAGED) exchange32<L, NB, NP>(yr, yi, t, sm);
#pragma unroll
                for (int r = 0; r < 16; ++r) store(L(), t, r, (int64_t)yr[r], (int64_t)yi[r]);
                return;
            }
        }
    }
    using W = typename L::Wide;
    // One copy of each int64 window, entered with inputs from LDS: values held
    // across the branch cost 128 points the third wave per SIMD (100000 in +-2^40
    // 87 -> 95 us).
    if constexpr (L::RESUME) {
        // LDS positions and addresses of its own: sharing the int32 path's
        // would hold them in registers across it
        asm volatile("" : "+v"(t));
    } else {
        from = 0;   // again from the source
    }
    if (from == 0) {
        if (!L::KEEP) {
            // the twiddles of a test that failed have come: or each load would
            // wait for the one before (100000 x 128 in +-2^40 87 -> 128 us)
            __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
            asm volatile("" ::: "memory");
#pragma unroll
            for (int r = 0; r < 16; ++r) load(W(), t, r, xr[r], xi[r]);
        }
        if constexpr (W::STAGED) exchange64<W, NB, 0>(xr, xi, t, sm);
        run_win64<W, NB, 0>(xr, xi, tw, low_bits<W, NB, 0>(t, s, c0), s, logn);
        exchange64<W, NB, 1>(xr, xi, t, sm);
    } else if (from == 1) {
        get32<L, NB, 1>(xr, xi, t, sm);
    }
    wide_from<L, W, NB, 1>(xr, xi, tw, t, s, c0, logn, sm, from);
#pragma unroll
    for (int r = 0; r < 16; ++r) store(W(), t, r, xr[r], xi[r]);
}

// 4096 consecutive points per workgroup: 16 transforms of 256 points and so
// on.  Points past the batch load as zero and are not stored.  Staging adds
// two LDS exchanges to save partial-line requests: below 256 points, whose 16
// lanes cover whole lines as they are (8000 x 32 points 7.0 us against 10.5
// without, 8000 x 64 7.4 against 9.7; 5000 x 128 8.0 against 8.8, 16000 12.5
// against 16.1; inputs past 2^26, read again in the other order, 5000 10.4
// against 10.2, 16000 17.0 against 19.9).
template <int LOGN>
__global__ __launch_bounds__(256) void fft_rows_kernel(const int64_t *sre, const int64_t *sim, int64_t *dre,
                                                       int64_t *dim, const int64_t *__restrict__ tw, int64_t points) {
    using L = RowsLay<LOGN, (LOGN < 8)>;
    constexpr int NP = (LOGN + 3) / 4;
    __shared__ uint64_t sm[L::ELEMS];
    const int64_t off = (int64_t)blockIdx.x << 12;
    const uint32_t left = (uint32_t)(points - off < 4096 ? points - off : 4096);   // whole transforms
    auto load = [&](auto lay, uint32_t t, int r, int64_t &re, int64_t &im) {
        using Y = decltype(lay);
        const uint32_t tr = L::template col<0>(t) << LOGN, j = t & ((1u << (LOGN - 4)) - 1u);
        const uint32_t i = Y::STAGED ? (uint32_t)r * 256u + t : tr | (bitrev((uint32_t)r, 4) << (LOGN - 4)) | j;
        if constexpr (L::KEEP && !L::STAGED) {   // each point is read once
            re = i < left ? __builtin_nontemporal_load(sre + off + i) : 0;
            im = i < left ? __builtin_nontemporal_load(sim + off + i) : 0;
        } else {
            re = i < left ? sre[off + i] : 0;
            im = i < left ? sim[off + i] : 0;
        }
    };
    run_pass<L, LOGN>(tw, threadIdx.x, 0, 0, LOGN, sm, load, [&](auto lay, uint32_t t, int r, int64_t re, int64_t im) {
        using Y = decltype(lay);
        const uint32_t tr = L::template col<0>(t) << LOGN;
        const uint32_t i = Y::STAGED ? (uint32_t)r * 256u + t
                                     : tr | win_pos(L::template label<NP - 1>(t), r, Win<LOGN, NP - 1>::S);
        if (i < left) {
            __builtin_nontemporal_store(re, dre + off + i);   // streamed: read by no one here
            __builtin_nontemporal_store(im, dim + off + i);
        }
    });
}

// One workgroup per transform (in place allowed: a workgroup holds its whole
// transform before it stores).
template <int LOGN>
__global__ __launch_bounds__(1 << (LOGN - 4)) void fft_block_kernel(const int64_t *sre, const int64_t *sim,
                                                                    int64_t *dre, int64_t *dim,
                                                                    const int64_t *__restrict__ tw) {
    using L = BlockLay<LOGN>;
    constexpr int NP = (LOGN + 3) / 4;
    __shared__ uint64_t sm[L::ELEMS];
    const int64_t off = (int64_t)blockIdx.x << LOGN;
    auto load = [&](auto, uint32_t t, int r, int64_t &re, int64_t &im) {
        const uint32_t src = (bitrev((uint32_t)r, 4) << (LOGN - 4)) | t;
        re = sre[off + src], im = sim[off + src];
    };
    run_pass<L, LOGN>(tw, threadIdx.x, 0, 0, LOGN, sm, load, [&](auto, uint32_t t, int r, int64_t re, int64_t im) {
        const uint32_t pos = win_pos(L::template label<NP - 1>(t), r, Win<LOGN, NP - 1>::S);
        dre[off + pos] = re, dim[off + pos] = im;
    });
}

// Stages [s, s + NB) of 16 columns; grid: 2^lgb workgroups per transform.
// The first pass (s = 0) reads through the bit reversal: its columns are the
// low logn - NB bits of the source index (the high position bits, reversed),
// and its source must not overlap its destination.
template <int NB, bool FIRST>
__global__ __launch_bounds__(1 << NB) void fft_cols_kernel(const int64_t *sre, const int64_t *sim, int64_t *dre,
                                                           int64_t *dim, const int64_t *__restrict__ tw, int logn,
                                                           int s, int lgb) {
    using L = ColsLay<NB, FIRST>;
    constexpr int NP = (NB + 3) / 4;
    __shared__ uint64_t sm[L::ELEMS];
    const uint32_t blk = blockIdx.x & ((1u << lgb) - 1u);
    const int64_t off = (int64_t)(blockIdx.x >> lgb) << logn;
    const uint32_t c0 = (FIRST ? blk : blk & ((1u << (s - 4)) - 1u)) << 4;
    const uint32_t high = FIRST ? 0u : (blk >> (s - 4)) << (s + NB);
    auto load = [&](auto, uint32_t t, int r, int64_t &re, int64_t &im) {
        const uint32_t j = t >> 4, c = c0 + (t & 15u);
        const uint32_t base = FIRST ? (bitrev(j, NB - 4) << (logn - NB)) | c : high | (j << (s + 4)) | c;
        const uint32_t src = base + (FIRST ? bitrev((uint32_t)r, 4) << (logn - 4) : (uint32_t)r << s);
        re = sre[off + src], im = sim[off + src];
    };
    run_pass<L, NB>(tw, threadIdx.x, s, c0, logn, sm, load, [&](auto, uint32_t t, int r, int64_t re, int64_t im) {
        const uint32_t l = win_pos(L::template label<NP - 1>(t), r, Win<NB, NP - 1>::S);
        const uint32_t cc = c0 + L::template col<NP - 1>(t);
        const uint32_t pos = FIRST ? (bitrev(cc, logn - NB) << NB) | l : high | (l << s) | cc;
        dre[off + pos] = re, dim[off + pos] = im;
    });
}

template <int NB>
static void launch_cols(const int64_t *sre, const int64_t *sim, int64_t *dre, int64_t *dim, const int64_t *tw,
                        int logn, int s, int64_t batch, hipStream_t st) {
    const int lgb = logn - NB - 4;
    const dim3 grid((unsigned)(batch << lgb)), block(1u << NB);
    if (s == 0)
        hipLaunchKernelGGL((fft_cols_kernel<NB, true>), grid, block, 0, st, sre, sim, dre, dim, tw, logn, s, lgb);
    else
        hipLaunchKernelGGL((fft_cols_kernel<NB, false>), grid, block, 0, st, sre, sim, dre, dim, tw, logn, s, lgb);
}

// A few transforms (batch <= few_batch(logn), 32 <= n <= 1024): one workgroup
// per transform, its points and the twiddle table in LDS, and one butterfly
// per thread and stage, so the latency of a lone call is logn
// barrier-separated stages instead of a lane walking its 16 points through
// every stage.  Same butterflies, same stage order: same bits.  Loads and
// stores touch each point once (an in-place call reads all of its transform
// before writing, at the first barrier).  LDS is sized by n: at 24 KiB for every
// n six workgroups fit a compute unit (4096 x 32 points 8.3 us, now 5.0; 3000 x
// 128 8.3, now 6.2).
// Device time per call, this against the window kernels, inputs within 2^16
// (2^40): 256 points x100 4.2 against 6.9 us (9.2), x768 5.6 against 7.2 (9.4),
// x1536 7.7 against 7.5 (9.8); 32 x8192 7.1 against 7.3 (9.3), x12288 9.2
// against 7.5; 64 x6144 7.2 against 7.7 (10.0), x8192 8.6 against 8.1; 128 x4096
// 7.4 against 7.6 (9.4), x6144 9.9 against 8.7; 512 x512 7.1 against 8.7 (10.8),
// x1024 10.4 against 9.2; 1024 x256 7.7 against 6.6 (9.6), x300 10.6 against
// 7.2 (10.8).
constexpr int few_batch(int logn) {
    constexpr int most[] = {8192, 6144, 4096, 768, 512, 256};
    return logn >= 5 && logn <= 10 ? most[logn - 5] : 0;
}

template <int LOGN>
__global__ __launch_bounds__((1 << LOGN) / 2) void fft_few_kernel(const int64_t *__restrict__ sre,
                                                                  const int64_t *__restrict__ sim, int64_t *dre,
                                                                  int64_t *dim, const int64_t *__restrict__ tw) {
    constexpr int logn = LOGN, n = 1 << logn, half_n = n >> 1;
    __shared__ int64_t lre[n], lim[n], ltw[n];
    const int t = threadIdx.x;
    const size_t base = (size_t)blockIdx.x * n;
    for (int i = t; i < n; i += blockDim.x) {   // bit reversal on the way in
        const uint32_t p = bitrev((uint32_t)i, logn);
        lre[p] = sre[base + i];
        lim[p] = sim[base + i];
        ltw[i] = tw[i];                          // the table is read once, then from LDS
    }
    __syncthreads();
    for (int b = 0; b < logn; ++b) {   // stage b pairs positions that differ in bit b
        const int h = 1 << b;
        for (int q = t; q < half_n; q += blockDim.x) {
            const int j = q & (h - 1), ia = ((q >> b) << (b + 1)) | j, ib = ia + h;
            int64_t wr = 0, wi = 0;
            if (b > 0) {
                const int k = j << (logn - 1 - b);
                wr = ltw[2 * k], wi = ltw[2 * k + 1];
            }
            int64_t ar = lre[ia], ai = lim[ia], br = lre[ib], bi = lim[ib];
            butterfly(ar, ai, br, bi, wr, wi, b == 0);
            lre[ia] = ar, lim[ia] = ai, lre[ib] = br, lim[ib] = bi;
        }
        __syncthreads();
    }
    for (int i = t; i < n; i += blockDim.x) {
        dre[base + i] = lre[i];
        dim[base + i] = lim[i];
    }
}

}  // namespace fft

// The largest scratch any call of this size takes (a call whose first pass may
// write its destination directly takes none: fft_scratch_bytes).
size_t fft_workspace_bytes(int logn, int64_t batch) {
    if (logn <= 11) return 0;
    return 2 * (size_t)batch * ((size_t)1 << logn) * sizeof(int64_t);
}

namespace fft {
static bool overlap(const int64_t *a, const int64_t *b, int64_t count) { return a < b + count && b < a + count; }

// Whole transforms per workgroup: 4096 points always (1 transform 9.5 us
// against 10.9 in two passes, 64 10.2 against 13.2), 8192 once there are 128
// of them (21.8 us against 24.5; 64 21.5 against 16.1).  In place (or
// disjoint) only: a workgroup reads its own transform alone.
static bool whole(const int64_t *sre, const int64_t *sim, const int64_t *dre, const int64_t *dim, int logn,
                  int64_t batch) {
    if (logn > 13 || batch < (logn == 12 ? 1 : 128)) return false;
    const int64_t cnt = batch << logn;
    return !overlap(sre, dim, cnt) && !overlap(sim, dre, cnt) && (sre == dre || !overlap(sre, dre, cnt)) &&
           (sim == dim || !overlap(sim, dim, cnt));
}
}  // namespace fft

// Scratch a call takes: the first column pass permutes points across
// workgroups, so it goes through scratch when a source range overlaps a
// destination range.
size_t fft_scratch_bytes(const int64_t *sre, const int64_t *sim, const int64_t *dre, const int64_t *dim, int logn,
                         int64_t batch) {
    using namespace fft;
    if (logn <= 11 || whole(sre, sim, dre, dim, logn, batch)) return 0;
    const int64_t cnt = batch << logn;
    const bool any = overlap(sre, dre, cnt) || overlap(sre, dim, cnt) || overlap(sim, dre, cnt) ||
                     overlap(sim, dim, cnt);
    return any ? fft_workspace_bytes(logn, batch) : 0;
}

// batch transforms of n = 2^logn points: transform f read from sre / sim
// + f n and written to dre / dim + f n (the same pointers for in place).
// logn in [0, 30]; ws: fft_scratch_bytes() bytes.
hipError_t launch_fft_q16(const int64_t *sre, const int64_t *sim, int64_t *dre, int64_t *dim, const int64_t *tw,
                          int logn, int64_t batch, void *ws, hipStream_t s) {
    using namespace fft;
    if (batch <= 0) return hipSuccess;
    if (logn < 0 || logn > 30) return hipErrorInvalidValue;
    const int64_t n = (int64_t)1 << logn;
    switch (logn) {
#define SMALL(LG)                                                                                              \
    case LG:                                                                                                   \
        hipLaunchKernelGGL(fft_small_kernel<LG>, dim3((unsigned)((batch + 255) / 256)), dim3(256), 0, s, sre, sim, \
                           dre, dim, tw, batch);                                                               \
        break;
    SMALL(0) SMALL(1) SMALL(2) SMALL(3) SMALL(4)
#undef SMALL
#define LDS(LG)                                                                                                \
    case LG: {                                                                                                 \
        if (batch <= few_batch(LG)) {                                                                          \
            hipLaunchKernelGGL(fft_few_kernel<(LG < 10 ? LG : 10)>, dim3((unsigned)batch), dim3((1u << LG) / 2), 0, s, \
                               sre, sim, dre, dim, tw);                                                        \
            break;                                                                                             \
        }                                                                                                      \
        if constexpr (LG >= 10) {                                                                              \
            hipLaunchKernelGGL(fft_block_kernel<LG>, dim3((unsigned)batch), dim3(1u << (LG - 4)), 0, s, sre, sim,  \
                               dre, dim, tw);                                                                  \
        } else {                                                                                               \
            const int64_t points = batch << LG;                                                                \
            const dim3 grid((unsigned)((points + 4095) / 4096));                                               \
            hipLaunchKernelGGL(fft_rows_kernel<LG>, grid, dim3(256), 0, s, sre, sim, dre, dim, tw, points);    \
        }                                                                                                      \
        break;                                                                                                 \
    }
    LDS(5) LDS(6) LDS(7) LDS(8) LDS(9) LDS(10) LDS(11)
#undef LDS
    default: {
        if (whole(sre, sim, dre, dim, logn, batch)) {
            const dim3 grid((unsigned)batch), block(1u << (logn - 4));
            if (logn == 12) hipLaunchKernelGGL(fft_block_kernel<12>, grid, block, 0, s, sre, sim, dre, dim, tw);
            else hipLaunchKernelGGL(fft_block_kernel<13>, grid, block, 0, s, sre, sim, dre, dim, tw);
            break;
        }
        const bool scratch = fft_scratch_bytes(sre, sim, dre, dim, logn, batch) != 0;
        if (scratch && !ws) return hipErrorInvalidValue;
        const int np = (logn + 8) / 9;
        const int64_t *from_re = sre, *from_im = sim;
        for (int p = 0, b = 0; p < np; ++p) {
            const int nb = (logn - b + np - p - 1) / (np - p);   // the rest, split evenly
            int64_t *to_re = scratch && p == 0 ? (int64_t *)ws : dre;
            int64_t *to_im = scratch && p == 0 ? (int64_t *)ws + batch * n : dim;
            switch (nb) {
            case 6: launch_cols<6>(from_re, from_im, to_re, to_im, tw, logn, b, batch, s); break;
            case 7: launch_cols<7>(from_re, from_im, to_re, to_im, tw, logn, b, batch, s); break;
            case 8: launch_cols<8>(from_re, from_im, to_re, to_im, tw, logn, b, batch, s); break;
            default: launch_cols<9>(from_re, from_im, to_re, to_im, tw, logn, b, batch, s); break;
            }
            b += nb;
            from_re = to_re, from_im = to_im;
        }
        break;
    }
    }
    return hipGetLastError();
}

}  // namespace det
