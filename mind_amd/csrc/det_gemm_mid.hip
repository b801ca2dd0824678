// det_gemm_mid.hip -- int8 and int16 GEMM in one launch, any size and
// alignment: 64-column tiles staged through LDS by registers.
//
//   int8 : C[i,j] = (int32) sum_k A[i,k] B[k,j]           (wrapped)
//   int16: C[i,j] = (int32) sum_k (int64)A[i,k] B[k,j]    (mod 2^32)
// int16 uses the limb identity of det_gemm_i16x.hip: a = T(a) + 128, T(a) =
// t0 + 2^8 t1 with signed bytes t0 = low ^ 0x80, t1 = high, so
//   sum a b = sum_{x,y} 2^(8(x+y)) sum t_x(a) t_y(b)
//             + 128 (sum T(a) + sum T(b)) + 2^14 K        (mod 2^32).
//
// The kernels of det_gemm_i8.hip move operands straight from memory into LDS,
// which wants rows on the 16-byte grid and (int16) bytes already split into
// limbs, i.e. a launch that rewrites both operands first, and tiles of 128 or
// 256 rows and columns, which leave most compute units idle on mid sizes.
// Here 4 waves compute 64 x 64 outputs (16 rows per wave) over steps of 64 k:
// the next steps' operands are loaded into registers (16-byte loads of A and
// 4-column loads of 4 k rows of B, at element alignment) while the MFMAs of the
// current one run, then split into limbs and (B) transposed by v_perm on their
// way into one of two LDS stages, rows of 64 k at a stride of 80 bytes (16 rows
// on 64 banks).  Column n of a tile is LDS row (n % 4) 16 + n / 4, so the 16
// threads of a k group write 16 consecutive rows, and a lane ends with 4
// consecutive columns of each of its rows.
//
// What bounds it: a lone workgroup the chain of a step (about 0.35 us: wait for
// the loads, split, LDS write, barrier, LDS read, MFMA), full grids the LDS
// traffic (int16: 40 KiB read and 16 KiB written per step against 256 cycles of
// MFMA per wave).  128- and 256-row tiles (fewer B reads) measured slower at
// every size here (1500^3 int16 39 against 34 us, 1300^3 int8 14.5 against
// 13.2), as did K split over workgroups with atomics on a zeroed C (1024^3
// int16, 2 parts: 29.5 against 12.7).
//
// Edges: the last column tile starts at N - 64 and stores its neighbour's
// columns again (the same values); rows past M repeat row M - 1 and are not
// stored; the K remainder is a step whose A bytes (and, for the limb sums, B
// bytes) past K are zero.
#include <type_traits>

#include "det_common.h"
#include "det_kernels.h"

namespace det {
namespace mid {

constexpr int TM = 64, TN = 64, KSTEP = 64, LDR = 80;
typedef uint32_t u32_a1 __attribute__((aligned(1)));
typedef uint32_t v2u32_a2 __attribute__((ext_vector_type(2), aligned(2)));
typedef int v4i32_a1 __attribute__((ext_vector_type(4), aligned(1)));
typedef int v4i32_a4 __attribute__((ext_vector_type(4), aligned(4)));

template <typename T>
struct Regs {
    v4i32 a[sizeof(T)];             // 16 elements of a row
    uint32_t b[4][sizeof(T)];       // 4 columns of 4 k rows
};

template <typename T, int KG>
__global__ __launch_bounds__(256 * KG, KG == 1 ? 3 : KG) void gemm_mid_kernel(const T *__restrict__ A,
                                                                              const T *__restrict__ B,
                                                                              int32_t *__restrict__ C, int M, int N,
                                                                              int K, int tm, int tiles) {
    constexpr int ES = sizeof(T), STAGE = ES * TM * LDR;
    // per group of 4 waves: two stages of A, two of B
    __shared__ __attribute__((aligned(16))) uint8_t smem[KG * 4 * STAGE];
    __shared__ uint32_t sRow[ES == 2 ? TM : 1], sCol[ES == 2 ? TN : 1];
    const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), tid = threadIdx.x & 255;
    const int lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
    uint8_t *sA = smem + grp * 4 * STAGE, *sB = sA + 2 * STAGE;   // [stage][limb][row]
    // contiguous runs of tiles per XCD, down the column panels
    const int per = (tiles + 7) / 8, tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (tile >= tiles) return;   // block-uniform
    const int m0 = tile % tm * TM, n0 = min(tile / tm * TN, N - TN);
    const int full = K / KSTEP;
    // staging roles: A row ar, elements 16 ac ..; B columns 4 bc .., k rows 4 bk ..
    const int ar = tid >> 2, ac = tid & 3, bc = tid & 15, bk = tid >> 4;
    const T *pa = A + (size_t)min(m0 + ar, M - 1) * K + 16 * ac;
    uint32_t rsum[2] = {0, 0}, csum[4][2];
#pragma unroll
    for (int j = 0; j < 4; ++j) csum[j][0] = csum[j][1] = 0;

    auto load_b = [&](Regs<T> &st, int e, const T *bp) {
        if constexpr (ES == 1) {
            st.b[e][0] = *(const u32_a1 *)bp;
        } else {
            const v2u32_a2 v = *(const v2u32_a2 *)bp;
            st.b[e][0] = v.x, st.b[e][ES - 1] = v.y;
        }
    };
    auto load = [&](Regs<T> &st, int s) {   // a full step
        const int k0 = s * KSTEP;
#pragma unroll
        for (int h = 0; h < ES; ++h) st.a[h] = *(const v4i32_a1 *)(pa + k0 + 16 / ES * h);
        const T *bp = B + (size_t)(k0 + 4 * bk) * N + n0 + 4 * bc;
#pragma unroll
        for (int e = 0; e < 4; ++e) load_b(st, e, bp + (size_t)e * N);
    };
    auto load_rest = [&](Regs<T> &st) {   // the K remainder: clamped addresses, one round trip for all of them
        const int k0 = full * KSTEP, nv = min(max(K - k0 - 16 * ac, 0), 16), kb = k0 + 4 * bk;
        uint32_t v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e)
            v[e] = (uint32_t)(std::conditional_t<ES == 1, uint8_t, uint16_t>)pa[min(k0 + e, K - 1 - 16 * ac)];
#pragma unroll
        for (int h = 0; h < ES; ++h)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                uint32_t d = 0;
#pragma unroll
                for (int e = 0; e < 4 / ES; ++e) {
                    const int x = 16 / ES * h + 4 / ES * q + e;
                    d |= (x < nv ? v[x] : 0u) << (8 * ES * e);
                }
                st.a[h][q] = (int)d;
            }
#pragma unroll
        for (int e = 0; e < 4; ++e) load_b(st, e, B + (size_t)min(kb + e, K - 1) * N + n0 + 4 * bc);
    };
    auto store = [&](const Regs<T> &st, auto rest, int buf) {
        const uint32_t ones = 0x01010101u;
        // the biases of bytes past K: none
        uint32_t xa[4] = {0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u}, mb = 0xffffffffu;
        if constexpr (ES == 2 && decltype(rest)::value) {
            const int nv = K - full * KSTEP - 16 * ac, nb = K - full * KSTEP - 4 * bk;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = nv - 4 * q;
                xa[q] = r >= 4 ? 0x80808080u : r <= 0 ? 0u : 0x80808080u & ((1u << (8 * r)) - 1u);
            }
            mb = nb >= 4 ? 0xffffffffu : nb <= 0 ? 0u : (1u << (8 * nb)) - 1u;
        }
        uint8_t *d = sA + buf * STAGE + ar * LDR + 16 * ac;
        if constexpr (ES == 1) {
            *(v4i32 *)d = st.a[0];
        } else {
            v4i32 lo, hi;
#pragma unroll
            for (int q = 0; q < 4; ++q) {   // 4 elements: dwords 2 q, 2 q + 1 of the 8
                const v4i32 v = st.a[q >> 1];
                const uint32_t d0 = (uint32_t)(q & 1 ? v.z : v.x), d1 = (uint32_t)(q & 1 ? v.w : v.y);
                const uint32_t l = perm(d1, d0, 0x06040200u) ^ xa[q], h = perm(d1, d0, 0x07050301u);
                lo[q] = (int)l, hi[q] = (int)h;
                rsum[0] = (uint32_t)__builtin_amdgcn_sdot4((int)l, (int)ones, (int)rsum[0], false);
                rsum[1] = (uint32_t)__builtin_amdgcn_sdot4((int)h, (int)ones, (int)rsum[1], false);
            }
            *(v4i32 *)d = lo;
            *(v4i32 *)(d + TM * LDR) = hi;
        }
        uint8_t *e0 = sB + buf * STAGE + bc * LDR + 4 * bk;
#pragma unroll
        for (int h = 0; h < ES; ++h) {
            uint32_t t[4];
            transpose4x4(st.b[0][h], st.b[1][h], st.b[2][h], st.b[3][h], t[0], t[1], t[2], t[3]);
            if constexpr (ES == 1) {
#pragma unroll
                for (int j = 0; j < 4; ++j) *(uint32_t *)(e0 + 16 * j * LDR) = t[j];
            } else {   // t = low, high byte of column 2 h, then of column 2 h + 1
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int col = 2 * h + (j >> 1), pl = j & 1;
                    const uint32_t v = (pl ? t[j] : t[j] ^ 0x80808080u) & mb;
                    csum[col][pl] = (uint32_t)__builtin_amdgcn_sdot4((int)v, (int)ones, (int)csum[col][pl], false);
                    *(uint32_t *)(e0 + (pl * TN + 16 * col) * LDR) = v;
                }
            }
        }
    };

    constexpr int NACC = ES == 1 ? 1 : 3;   // shift 0 (and 8, 16)
    v4i32 acc[NACC][4];
#pragma unroll
    for (int p = 0; p < NACC; ++p)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[p][j] = (v4i32){0, 0, 0, 0};
    auto compute = [&](int buf) {
        const uint8_t *ap = sA + buf * STAGE + (wave * 16 + c) * LDR + 16 * g, *bp = sB + buf * STAGE + c * LDR + 16 * g;
        v2i64 a[ES], b[ES][4];
#pragma unroll
        for (int p = 0; p < ES; ++p) {
            a[p] = *(const v2i64 *)(ap + p * TM * LDR);
#pragma unroll
            for (int j = 0; j < 4; ++j) b[p][j] = *(const v2i64 *)(bp + (p * TN + 16 * j) * LDR);
        }
#pragma unroll
        for (int x = 0; x < ES; ++x)
#pragma unroll
            for (int y = 0; y < ES; ++y)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[x + y][j] = mfma16x16x64(a[x], b[y][j], acc[x + y][j]);
    };
    if (ES == 2 && threadIdx.x < TM) sRow[threadIdx.x] = sCol[threadIdx.x] = 0;
    // Group grp runs the full steps [grp nf, grp nf + nf), then one of the rest:
    // the full steps left over, and the K remainder.  The next steps' operands
    // (int8: two steps; int16: one, or the registers cost a workgroup per
    // compute unit: 1500^3 40 us against 33) are in flight in loops without
    // branches: a loop that tests for its end waits for all loads at every
    // step.  Past the end they load the last step again, which nothing uses.
    const int nf = full / KG, fbeg = grp * nf, last = fbeg + nf - 1;
    Regs<T> st0;
    if (nf > 0) {
        load(st0, fbeg);
        if constexpr (ES == 1) {
            Regs<T> st1;
            load(st1, min(fbeg + 1, last));
            for (int i = 0; i + 2 <= nf; i += 2) {
                store(st0, std::false_type(), 0);
                load(st0, min(fbeg + i + 2, last));
                __syncthreads();
                compute(0);
                store(st1, std::false_type(), 1);
                load(st1, min(fbeg + i + 3, last));
                __syncthreads();
                compute(1);
            }
            if (nf & 1) {
                store(st0, std::false_type(), 0);
                __syncthreads();
                compute(0);
            }
        } else {
            for (int i = 0; i < nf; ++i) {
                store(st0, std::false_type(), i & 1);
                load(st0, min(fbeg + i + 1, last));
                __syncthreads();
                compute(i & 1);
            }
        }
    }
    const int rest = full - KG * nf;   // below KG
    const bool tail = K % KSTEP != 0;
    if (rest || tail) {   // into the stage the last step did not use
        if (grp < rest) {
            load(st0, KG * nf + grp);
            store(st0, std::false_type(), nf & 1);
        } else if (grp == rest && tail) {
            load_rest(st0);
            store(st0, std::true_type(), nf & 1);
        }
        __syncthreads();
        if (grp < rest || (grp == rest && tail)) compute(nf & 1);
    }
    __syncthreads();   // the stages are free
    // the groups' sums, joined in group 0: [row][column] of int32 per group
    v4i32 sum[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        sum[j] = acc[0][j];
        if constexpr (ES == 2)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                sum[j][r] = (int)((uint32_t)sum[j][r] + ((uint32_t)acc[NACC / 2][j][r] << 8) +
                                  ((uint32_t)acc[NACC - 1][j][r] << 16));
    }
    if constexpr (KG > 1) {
        v4i32 *part = (v4i32 *)smem;
        if (grp > 0)
#pragma unroll
            for (int j = 0; j < 4; ++j) part[((grp - 1) * 4 + j) * 256 + tid] = sum[j];
    }
    if constexpr (ES == 2) {   // the limb sums times 128
        uint32_t v = rsum[0] + (rsum[1] << 8);
        v += (uint32_t)__shfl_xor((int)v, 1);
        v += (uint32_t)__shfl_xor((int)v, 2);
        if (ac == 0) atomicAdd(&sRow[ar], v << 7);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t w = csum[j][0] + (csum[j][1] << 8);
            w += (uint32_t)__shfl_xor((int)w, 16);
            w += (uint32_t)__shfl_xor((int)w, 32);
            if (lane < 16) atomicAdd(&sCol[4 * bc + j], w << 7);
        }
    }
    if constexpr (KG > 1 || ES == 2) __syncthreads();
    if (grp > 0) return;
    if constexpr (KG > 1) {
        const v4i32 *part = (const v4i32 *)smem;
#pragma unroll
        for (int h = 0; h < KG - 1; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j) sum[j] += part[(h * 4 + j) * 256 + tid];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int lr = wave * 16 + 4 * g + r, row = m0 + lr;
        v4i32 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t v = (uint32_t)sum[j][r];
            if constexpr (ES == 2) v += sRow[lr] + sCol[4 * c + j] + ((uint32_t)K << 14);
            o[j] = (int)v;
        }
        if (row < M) *(v4i32_a4 *)(C + (size_t)row * N + n0 + 4 * c) = o;
    }
}

template <typename T, int KG>
static hipError_t launch(const T *A, const T *B, int32_t *C, int M, int N, int K, hipStream_t s) {
    const int tm = (M + TM - 1) / TM, tiles = tm * ((N + TN - 1) / TN), per = (tiles + 7) / 8;
    hipLaunchKernelGGL((gemm_mid_kernel<T, KG>), dim3((unsigned)(per * 8)), dim3(256 * KG), 0, s, A, B, C, M, N, K, tm,
                       tiles);
    return hipGetLastError();
}

}  // namespace mid

// 64 x 64 tiles times 64-k steps: what the kernel's time goes by on full grids.
static long long mid_tiles(int M, int N) {
    return ((long long)M + mid::TM - 1) / mid::TM * (((long long)N + mid::TN - 1) / mid::TN);
}
static long long mid_work(int M, int N, int K) {
    return mid_tiles(M, N) * ((K + mid::KSTEP - 1) / mid::KSTEP);
}
// A launch holds below 2^32 threads: 2^24 workgroups of 256, rounded up to a
// multiple of 8 (few rows of 2^30 columns are past that).
static bool mid_fits(int M, int N) { return N >= mid::TN && mid_tiles(M, N) <= (1LL << 24) - 8; }

// int8, against repacked panels (or the 256 x 256 edge kernel, on the 16-byte
// grid) on shapes that the full-tile kernels do not take as they are; device
// time per call, there -> here:
//   up to one tile per compute unit: 384 x 2735 x 338 21.1 -> 14.2 us,
//     1024 x 1920 x 822 (208 tiles) 16.4 -> 9.3, 1001^3 12.6 -> 8.1, 1500 x
//     4000 x 500 25.8 -> 18.2, 463 x 256 x 1792 11.2 -> 7.4;
//   beyond: 1300^3 (9261 tile steps) 17.8 -> 13.4, 2000 x 300 x 2000 13.5 -> 11.8,
//     3000 x 300 x 3000 (11045) 26.6 -> 23.5.
// Past that, 256 x 256 tiles there read each operand from L2 a fourth as often,
// so a step costs them less.  With a K remainder, a step of its own in every round
// of tiles here, the crossover therefore lies at fewer steps the more rounds there
// are (a last one here, a first one there):
//   on the grid, against one round of 256 x 256 tiles: 4 rounds 2000 x 624 x 2000
//     (10 steps) 15.8 -> 15.4, 2000 x 752 14.6 -> 17.4; 5 rounds 3008 x 240 x 1408
//     12.4 -> 11.9, 15008 x 368 x 304 13.4 -> 15.6; 6 rounds 2304 x 112 x 2304 11.3 ->
//     9.8, 2304 x 304 13.1 -> 15.8; 9 rounds 3008 x 48 x 3008 11.1 -> 10.2, 3008 x
//     176 13.1 -> 17.6; but against two rounds 3392 x 96 x 4704 21.9 -> 17.9;
//   off it, against one round of little padded 128 x 128 tiles: 3 rounds 2609 x 559
//     x 1009 14 -> 13, 1505 x 687 x 1505 13 -> 14; 4 rounds 2001 x 303 x 2001 14 ->
//     13, 2001 x 495 13.5 -> 15.5; of 128 x 256 tiles: 5 rounds 977 x 367 x 5009 17
//     -> 16, 3009 x 431 x 1409 17 -> 18; 7 rounds 2513 x 111 x 2513 18 -> 12, 2513 x
//     367 18 -> 21.  Rows on the 4-byte grid load faster here: 1500 x 900 x 1500 14.2
//     -> 13.2, 2000 x 500 x 2000 13.5 -> 13.1, but 2000 x 600 14.2 -> 15.0; 3159 x 521
//     x 1376 (5 rounds) 19.4 -> 15.4, 2677 x 257 x 2352 (7) 18.0 -> 15.4, but 2500 x
//     380 x 2500 18.4 -> 20.3.
// Of 230 drawn shapes near these lines the taken kernel is the slower one by more
// than 4% for 7, by 14% at most where it is this one, 25% where not.
// Without a remainder all of these stay faster here: 2000 x 640 x 2000 16.0 -> 11.5,
//   4688 x 576 x 896 15.2 -> 11.7, 3008 x 192 x 3008 13 -> 10, 2513 x 512 x 2512 18 ->
//   17, 4000 x 192 x 4000 16 -> 16.
// Without a workspace the alternative for operands off the 16-byte grid is the
// byte-load kernel (4095^3 829 us; here 280): any size.
bool i8_mid(int M, int N, int K, bool panels, bool on_grid) {
    if (!mid_fits(M, N)) return false;
    if (!panels) return true;
    const long long cus = cu_count(), tiles = mid_tiles(M, N), rounds = (tiles + cus - 1) / cus;
    const long long steps = ((long long)K + mid::KSTEP - 1) / mid::KSTEP;
    if (rounds == 1 && K <= 8192) return true;
    if (tiles * steps > 11100) return false;
    if (rounds <= 2 || K % mid::KSTEP == 0) return true;
    const long long m256 = ((long long)M + 255) / 256, n256 = ((long long)N + 255) / 256;
    if (on_grid) return m256 * n256 > cus || rounds <= 4 || steps <= (rounds == 5 ? 4 : rounds <= 7 ? 2 : 1);
    const bool one_round = m256 * n256 * 2 <= cus;   // of 128 x 256 tiles
    const bool little_padded = min(M, N) >= 512 && 4 * 65536 * m256 * n256 <= 5LL * M * N;
    if (!one_round || !little_padded) return true;
    if (m256 * n256 * 4 <= cus)   // 128 x 128 tiles
        return K % 4 == 0 && N % 4 == 0 ? rounds == 3 || rounds * steps <= 34 : rounds * steps <= 27;
    return rounds * steps <= (N % 4 ? (rounds <= 4 ? 40 : 30) : rounds <= 5 ? 50 : 36);
}

// int16, against the operand prep plus the interleaved limb GEMM, whose prep
// reads by element off the 16-byte grid:
//   up to one tile per compute unit: 1024^3 17.9 -> 10.6, 1403 x 791 x 640
//     21.1 -> 11.7, 300 x 2000 x 300 36.2 -> 18.6, 1024 x 2048 x 1024 26.5 -> 17.5;
//   beyond, off the grid: 1200^3 27.9 -> 20.3, 1500^3 (13824 tile steps) 37.4 ->
//     32.7, 3009 x 527 x 1409 39 -> 33, 3009 x 367 x 3009 47 -> 41, 4001 x 175 x 4001
//     48 -> 44; on it: 1280^3 (8000) 25.0 -> 18.9, 2048 x 512 x 2048 19.8 -> 17.7,
//     2304 x 176 x 2304 22 -> 17, but 2048^3 (32768) 39 -> 58.
// The crossover in tile steps varies from family to family, so the limits lie
// where no family loses much: at 2000^2, where the limbs fill exactly one round of
// 256 x 256 tiles, it is 10000 off the grid (2000 x 601 x 2000 24.0 -> 25.4, the
// largest loss) and 7500 on it; on 1300^2 and 800 x 1700 it is past 30000, and
// 1550^3 (15625) and 1700^3 (19683), past the limit, would gain as well (41.0 -> 33.4,
// 43.6 -> 37.8).
bool i16_mid(int M, int N, int K, bool on_grid) {
    if (!mid_fits(M, N)) return false;
    return (mid_tiles(M, N) <= cu_count() && K <= 4096) || mid_work(M, N, K) <= (on_grid ? 8000 : 14000);
}

// Two groups of waves per tile (each half of K, joined in LDS) where a tile
// has a compute unit of its own: int16 1024^3 12.5 -> 10.6 us, int8 256 x 4096 x
// 256 16.5 -> 12.4, 1024 x 1920 x 822 9.7 -> 9.3; beyond one tile per compute
// unit the groups only compete (int16 1500^3 34 -> 45).  Four groups measured
// slower than two.
hipError_t launch_gemm_mid(const int8_t *A, const int8_t *B, int32_t *C, int M, int N, int K, hipStream_t s) {
    return mid_tiles(M, N) <= cu_count() && K >= 1024 ? mid::launch<int8_t, 2>(A, B, C, M, N, K, s)
                                                      : mid::launch<int8_t, 1>(A, B, C, M, N, K, s);
}
hipError_t launch_gemm_mid(const int16_t *A, const int16_t *B, int32_t *C, int M, int N, int K, hipStream_t s) {
    return mid_tiles(M, N) <= cu_count() ? mid::launch<int16_t, 2>(A, B, C, M, N, K, s)
                                         : mid::launch<int16_t, 1>(A, B, C, M, N, K, s);
}

}  // namespace det
