// det_gemm_rows.hip -- int8 GEMM with few rows of A: C = A . B streamed over B.
//
// C[i,j] = (int32) sum_k A[i,k] B[k,j], i32 accumulation wrapping mod 2^32
// (benches/det_matmul_i8.rs:232-245), for at most ROWS_MAX rows: a weight
// matrix against a few activation rows.  The 128- and 256-row tiles of
// det_gemm_i8.hip give such a shape one tile row, i.e. N / 256 workgroups, each
// streaming its columns alone (16 x 4096 x 11008: 43 of 256 CUs, 39 us).
//
// Bound: reading B once (K N bytes).  A workgroup owns 64 columns and all rows;
// its WAVES waves take the 64-k steps in turn, so the whole workgroup has
// about WAVES x 8 KiB of B in flight.  No LDS staging: a lane loads a dword (4
// columns) of 16 consecutive k rows and transposes them in registers (4 byte
// transposes of 4 x 4, 32 v_perm per 64 x 64 bytes) into the K-contiguous
// 16-byte operands of v_mfma_i32_16x16x64_i8; A rows are K-contiguous as they
// are.  Lane (g = lane / 16, c = lane % 16): operand j of the step is column
// 4 c + j, k = 16 g .. 16 g + 15, so a lane ends with 4 consecutive columns of
// each of its rows.  The waves' sums are added in LDS (integer atomics: any
// order gives the same bits).
//
// Any size and alignment (gfx950 loads need none): the last column tile starts
// at N - 64, overlapping its neighbour, which stores the same values; rows past
// M repeat the last; the K remainder is one step whose B rows are clamped and
// whose A bytes past K are zero.
#include "det_common.h"
#include "det_kernels.h"

namespace det {
namespace rows8 {

constexpr int TN = 64, KSTEP = 64, ROWS_MAX = 64;
typedef uint32_t u32_a1 __attribute__((aligned(1)));
typedef int v4i32_a1 __attribute__((ext_vector_type(4), aligned(1)));
typedef int v4i32_a4 __attribute__((ext_vector_type(4), aligned(4)));

template <int MR>
struct Step {
    uint32_t b[16];   // B rows 16 g + 0 .. 15, columns 4 c .. 4 c + 3
    v4i32 a[MR];      // A rows c + 16 i, k = 16 g .. 16 g + 15
};

template <int MR>
__device__ __forceinline__ void mac(v4i32 (&acc)[MR][4], const Step<MR> &s) {
    uint32_t t[4][4];   // [k group of 4][column]
#pragma unroll
    for (int q = 0; q < 4; ++q)
        transpose4x4(s.b[4 * q], s.b[4 * q + 1], s.b[4 * q + 2], s.b[4 * q + 3], t[q][0], t[q][1], t[q][2], t[q][3]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const v4i32 bj = {(int)t[0][j], (int)t[1][j], (int)t[2][j], (int)t[3][j]};
#pragma unroll
        for (int i = 0; i < MR; ++i)
            acc[i][j] = mfma16x16x64(__builtin_bit_cast(v2i64, s.a[i]), __builtin_bit_cast(v2i64, bj), acc[i][j]);
    }
}

// D steps per wave are in flight: a register ring whose slots are reloaded
// as they are consumed.
template <int MR, int WAVES, int D>
__global__ __launch_bounds__(WAVES * 64) void gemm_i8_rows_kernel(const int8_t *__restrict__ A,
                                                                  const int8_t *__restrict__ B,
                                                                  int32_t *__restrict__ C, int M, int N, int K,
                                                                  int units, int gy, int split) {
    __shared__ int32_t sum[MR * 16 * TN];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, g = lane >> 4;
    // a unit is one column tile of one group of 16 MR rows; the row groups of a
    // tile, and neighbouring tiles, which share 128-byte lines of B, on one XCD
    const int per = (units + 7) / 8, un = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (un >= units) return;   // block-uniform
    const int ks = un % split, unit = un / split;   // this workgroup's part of K
    const int n0 = min(unit / gy * TN, N - TN), m0 = unit % gy * (MR * 16);
    for (int i = tid; i < MR * 16 * TN; i += WAVES * 64) sum[i] = 0;
    const int8_t *ar[MR];
#pragma unroll
    for (int i = 0; i < MR; ++i) ar[i] = A + (size_t)min(m0 + i * 16 + c, M - 1) * K + 16 * g;
    const uint32_t boff = (uint32_t)(16 * g) * (uint32_t)N + 4u * c;   // per lane; the rest of a B address is uniform
    v4i32 acc[MR][4];
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = (v4i32){0, 0, 0, 0};
    // full steps: this workgroup's are [sbeg, send), this wave's every WAVES-th
    const int full = K / KSTEP;
    const int sbeg = (int)((long long)full * ks / split), send = (int)((long long)full * (ks + 1) / split);
    const int mine = send - sbeg > wave ? (send - sbeg - wave - 1) / WAVES + 1 : 0;
    auto load = [&](Step<MR> &s, int i) {   // the wave's step i
        const size_t k0 = (size_t)(sbeg + wave + i * WAVES) * KSTEP;
        const int8_t *bp = B + k0 * N + n0;
#pragma unroll
        for (int kk = 0; kk < 16; ++kk)
            s.b[kk] = *(const u32_a1 *)(bp + (size_t)kk * N + boff);
#pragma unroll
        for (int m = 0; m < MR; ++m) s.a[m] = *(const v4i32_a1 *)(ar[m] + k0);
    };
    if (mine >= D) {
        Step<MR> ring[D];
#pragma unroll
        for (int d = 0; d < D; ++d) load(ring[d], d);
        int i = 0;
        for (; i + 2 * D <= mine; i += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                mac(acc, ring[d]);
                load(ring[d], i + D + d);
            }
        }
        const int more = mine - i - D;   // 0 .. D - 1 steps not loaded yet
#pragma unroll
        for (int d = 0; d < D; ++d) {
            mac(acc, ring[d]);
            if (d < more) load(ring[d], i + D + d);
        }
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (d < more) mac(acc, ring[d]);
    } else {
        for (int i = 0; i < mine; ++i) {
            Step<MR> s;
            load(s, i);
            mac(acc, s);
        }
    }
    if (ks == split - 1 && (send - sbeg) % WAVES == wave && K % KSTEP) {   // the K remainder
        Step<MR> s;
        const int k0 = full * KSTEP + 16 * g;
#pragma unroll
        for (int kk = 0; kk < 16; ++kk)
            s.b[kk] = *(const u32_a1 *)(B + (size_t)min(k0 + kk, K - 1) * N + n0 + 4 * c);
#pragma unroll
        for (int i = 0; i < MR; ++i) {
            const int8_t *p = ar[i] - 16 * g;
            uint8_t v[16];   // every load in range: one round trip for all of them
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = (uint8_t)p[min(k0 + e, K - 1)];
            uint32_t d[4] = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 16; ++e) d[e >> 2] |= (k0 + e < K ? (uint32_t)v[e] : 0u) << (8 * (e & 3));
            s.a[i] = (v4i32){(int)d[0], (int)d[1], (int)d[2], (int)d[3]};
        }
        mac(acc, s);
    }
    __syncthreads();   // the sums are zero
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < 4; ++j)   // row 16 i + 4 g + r, column 4 c + j; [j][c]: 16 lanes on 16 banks
                atomicAdd(&sum[(i * 16 + 4 * g + r) * TN + j * 16 + c], acc[i][j][r]);
    __syncthreads();
    for (int o = tid; o < MR * 16 * 16; o += WAVES * 64) {
        const int row = o >> 4, cc = o & 15;
        if (m0 + row < M) {
            const int32_t *sp = sum + row * TN + cc;
            int32_t *cp = C + (size_t)(m0 + row) * N + n0 + 4 * cc;
            if (split == 1) {
                *(v4i32_a4 *)cp = (v4i32){sp[0], sp[16], sp[32], sp[48]};
            } else {   // C was zeroed; columns an earlier tile also covers are that tile's
                const int skip = unit / gy * TN - n0;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (4 * cc + j >= skip) atomicAdd(cp + j, sp[16 * j]);
            }
        }
    }
}

__global__ __launch_bounds__(256) void zero_kernel(int32_t *__restrict__ C, int n) {
    const int i = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (i + 4 <= n) *(v4i32_a4 *)(C + i) = (v4i32){0, 0, 0, 0};
    else
        for (int j = i; j < n; ++j) C[j] = 0;
}

template <int MR, int WAVES, int D>
static void launch(const int8_t *A, const int8_t *B, int32_t *C, int M, int N, int K, int split, hipStream_t s) {
    const int gy = (M + MR * 16 - 1) / (MR * 16), units = (N + TN - 1) / TN * gy * split, per = (units + 7) / 8;
    if (split > 1) {
        const int n = M * N;
        hipLaunchKernelGGL(zero_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, s, C, n);
    }
    hipLaunchKernelGGL((gemm_i8_rows_kernel<MR, WAVES, D>), dim3((unsigned)(per * 8)), dim3(WAVES * 64), 0, s, A, B, C,
                       M, N, K, units, gy, split);
}

// 16-row groups per workgroup: 1 while that leaves compute units free (B then
// comes from L2 for all groups but one), else as many as there are, up to 4.
static int group_rows(int M, int N) {
    const int tiles = (N + TN - 1) / TN, mr = (M + 15) / 16, cus = cu_count();
    return mr == 1 || tiles * mr <= cus ? 1 : mr == 2 || tiles * 2 <= cus ? 2 : mr;
}

}  // namespace rows8

// Up to 64 rows and 64 columns or more; N < 2^26 keeps a lane's B offset in 32
// bits.  Up to K = 512 the tiny-shape kernel is as fast where it applies
// (64 x 256 x 256: both at the launch floor).
bool i8_rows(int M, int N, int K) {
    return M <= rows8::ROWS_MAX && N >= rows8::TN && N < (1 << 26) && K >= 1 &&
           !(K <= I8_SMALL_K && i8_small(M, N, K));
}

// Workgroups that share a unit's K range: each adds its sums to a zeroed C with
// integer atomics, which only this device's memory is sure to take.
int i8_rows_split(int M, int N, int K) {
    using namespace rows8;
    const int mr = group_rows(M, N), units = (N + TN - 1) / TN * ((M + mr * 16 - 1) / (mr * 16));
    const int cus = cu_count(), steps = K / KSTEP;
    if (steps < 48 || units * 2 > cus) return 1;
    return max(1, min(cus / units, steps / 16));
}

// Memory of the current device, as opposed to mapped host or managed memory or
// another device's (an atomic there depends on the bus) and to addresses the
// runtime does not know.
static bool device_memory(const void *p) {
    hipPointerAttribute_t at;
    int d = -1;
    if (hipPointerGetAttributes(&at, p) != hipSuccess || hipGetDevice(&d) != hipSuccess) {
        (void)hipGetLastError();   // handled: clear it
        return false;
    }
    return at.type == hipMemoryTypeDevice && at.device == d;
}

hipError_t launch_gemm_i8_rows(const int8_t *A, const int8_t *B, int32_t *C, int M, int N, int K, hipStream_t s) {
    using namespace rows8;
    int split = i8_rows_split(M, N, K);
    if (split > 1 && !device_memory(C)) split = 1;   // plain stores
    switch (group_rows(M, N)) {
    case 1: launch<1, 16, 3>(A, B, C, M, N, K, split, s); break;
    case 2: launch<2, 8, 4>(A, B, C, M, N, K, split, s); break;
    case 3: launch<3, 8, 3>(A, B, C, M, N, K, split, s); break;
    default: launch<4, 8, 3>(A, B, C, M, N, K, split, s); break;
    }
    return hipGetLastError();
}

}  // namespace det
