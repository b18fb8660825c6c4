// The projections either side of the GatedDeltaNet / attention core at decode and verify time, for gfx950: y = W . f(x) for a
// handful of rows (M <= a few hundred), W [N, K] bf16 row-major.  Replaces the reference's fused_gemv (qwen35/kernels.py:80-319)
// and its stand-alone prologue rms_rows (qwen35/batch.py:249-301); the gated-norm prologue is the existing gated RMSNorm kernel.
//     prologue  rms:    x' = BF(nw * (x * inv)),  inv = rsqrt(mean(x^2) + eps)                       (kernels.py:106-131)
//     product           s[m][n] = sum_k W[n][k] x'[m][k]                      fp32 accumulation       (kernels.py:249-262)
//     epilogue  none:   y = bf16(s)                                                                     (kernels.py:153-160)
//               add:    y = bf16(BF(s) + res)                                                           (kernels.py:161-169)
//               swiglu: y[m][p] = bf16(silu_bf16(BF(s[m][2p])) * BF(s[m][2p+1]))   interleaved rows     (kernels.py:170-182)
// The batch is small, so the product is bound by what ONE CU has to pull in (its share of W and of x) and by the launch itself.
// Four kernels by shape:
//   rows_gemm_kernel  the wide projections of a decode / verify batch (K = 1024, N >= 4096): the rows live in LDS, the rms
//                     prologue is applied on the way there, a workgroup owns 32 or 64 output features (and up to four more)
//   quad_gemm_kernel  narrow outputs: small tiles (4 x 4 .. 16 x 16 outputs) so that every CU has one
//   tile_gemm_kernel  narrow outputs where one tile of 16 x 16 per CU does: operands through LDS
//   skinny_gemm_kernel  everything else: 16 features x up to 64 rows per workgroup
// What decides the first two is how a load maps to lanes.  An MFMA operand wants 16 different rows in 16 neighbouring lanes; a
// load shaped like that asks for 16 bytes of 16 different rows per quarter-wavefront, and a CU then takes in 16 bytes per clock
// (512 threads a CU that read rows 2 KiB apart from the L2: 38 GB/s per CU).  Where four neighbouring lanes read 64 contiguous bytes it
// is 63 GB/s, and 78 with 256 bytes per 16 lanes.  The two kernels load in the second shape and put the lanes right afterwards,
// each in its own way.
// Arithmetic contract of rms_rows: sum of squares exact, rounded to float once; inv = correctly rounded 1/sqrt(ss / K + eps);
// t = x * inv and w * t rounded to float separately, then to bf16.
#include "qt_common.h"
#include <type_traits>

using namespace qt;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// one wavefront per row, four rows per workgroup: lane l owns elements 8 (l + 64 c) .. + 8 of chunk c
__global__ __launch_bounds__(256) void rms_rows_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ nw,
                                                       bf16_t* __restrict__ y, int M, int K, float eps) {
    const int m = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (m >= M) return;
    const u32x4* xr = reinterpret_cast<const u32x4*>(x + (size_t)m * K);
    const u32x4* wr = reinterpret_cast<const u32x4*>(nw);
    u32x4* yr = reinterpret_cast<u32x4*>(y + (size_t)m * K);
    const int nvec = K / 8;
    double ss = 0.0;
    for (int i = lane; i < nvec; i += 64) {
        const u32x4 v = xr[i];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const double lo = (double)__uint_as_float(v[j] << 16), hi = (double)__uint_as_float(v[j] & 0xffff0000u);
            ss += lo * lo + hi * hi;
        }
    }
    ss = wave_sum_d(ss);
    const float inv = rsqrt_rn((float)ss / (float)K + eps);
    for (int i = lane; i < nvec; i += 64) {
        const u32x4 v = xr[i], wv = wr[i];
        u32x4 o;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float lo = __fmul_rn(__uint_as_float(wv[j] << 16), __fmul_rn(__uint_as_float(v[j] << 16), inv));
            const float hi = __fmul_rn(__uint_as_float(wv[j] & 0xffff0000u), __fmul_rn(__uint_as_float(v[j] & 0xffff0000u), inv));
            o[j] = pack_bf(lo, hi);
        }
        yr[i] = o;
    }
}

constexpr int EPI_NONE = 0, EPI_ADD = 1, EPI_SWIGLU = 2;
constexpr int MT = 64;                 // most rows a workgroup takes
constexpr int G = 2;                   // k chunks (of 32) per register batch

// One workgroup = 16 output features x 16 MS rows; its NWV wavefronts split K.  grid = (ceil(N / 16), ceil(M / 16 MS)).
// K / 32 is a multiple of G NWV: every wavefront gets a whole number of batches of G chunks.  At most 128 registers, so that
// four workgroups of four wavefronts (or one of sixteen) share a CU: 514 workgroups of the widest projection (N = 8224) are
// resident at once, and the narrow ones (N = 1024: 64 workgroups) get short K chains from sixteen wavefronts each.
// MS = 16-row blocks per workgroup (1, 2 or 4; rows past M repeat the last row and are dropped): a compile-time count keeps
// the MFMA sequence free of branches, and a small one spreads a narrow output over more workgroups.
template <int NWV, int MS, int EPI>
__global__ __launch_bounds__(64 * NWV, 16 / NWV) void skinny_gemm_kernel(const bf16_t* __restrict__ W, const bf16_t* __restrict__ x,
                                                                         const bf16_t* __restrict__ res, bf16_t* __restrict__ y, int M, int N,
                                                                         int K) {
    __shared__ float red[NWV][16][16 * MS + 1];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16, m0 = blockIdx.y * (16 * MS);
    const int kc_w = K / 32 / NWV;                                // chunks of this wavefront
    const int k_base = w * kc_w * 32 + 8 * g;
    // lane (n, g) loads feature n0 + n and row m0 + 16 ms + n, elements k + 8 g .. + 8; rows past the end repeat the last
    const bf16_t* wp = W + (size_t)min(n0 + n, N - 1) * K + k_base;
    const bf16_t* xp[MS];
#pragma unroll
    for (int ms = 0; ms < MS; ms++) xp[ms] = x + (size_t)min(m0 + 16 * ms + n, M - 1) * K + k_base;

    f32x4 acc[MS];
#pragma unroll
    for (int ms = 0; ms < MS; ms++) acc[ms] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 a[2][G], b[2][G][MS];
    auto load = [&](int buf, int c0) {
#pragma unroll
        for (int c = 0; c < G; c++) {
            a[buf][c] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp + (c0 + c) * 32));   // W is read once
#pragma unroll
            for (int ms = 0; ms < MS; ms++) b[buf][c][ms] = *reinterpret_cast<const u32x4*>(xp[ms] + (c0 + c) * 32);
        }
    };
    auto mma = [&](int buf) {
#pragma unroll
        for (int c = 0; c < G; c++)
#pragma unroll
            for (int ms = 0; ms < MS; ms++)
                acc[ms] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[buf][c]),
                                                                 __builtin_bit_cast(bf16x8, b[buf][c][ms]), acc[ms], 0, 0, 0);
    };
    load(0, 0);
    for (int c0 = 0; c0 < kc_w; c0 += 2 * G) {                    // two batches per trip: the next one loads while this one multiplies
        if (c0 + G < kc_w) load(1, c0 + G);
        mma(0);
        if (c0 + G < kc_w) {
            if (c0 + 2 * G < kc_w) load(0, c0 + 2 * G);
            mma(1);
        }
    }
    // accumulator element i of lane (n, g) is feature 4 g + i, row 16 ms + n
#pragma unroll
    for (int ms = 0; ms < MS; ms++)
#pragma unroll
        for (int i = 0; i < 4; i++) red[w][4 * g + i][16 * ms + n] = acc[ms][i];
    __syncthreads();
    auto total = [&](int f, int m) {                              // fixed order: pairs, then pairs of pairs, ...
        float t[NWV];
#pragma unroll
        for (int i = 0; i < NWV; i++) t[i] = red[i][f][m];
#pragma unroll
        for (int st = 1; st < NWV; st *= 2)
#pragma unroll
            for (int i = 0; i < NWV; i += 2 * st) t[i] += t[i + st];
        return t[0];
    };
    if (EPI == EPI_SWIGLU) {
        for (int idx = threadIdx.x; idx < 8 * 16 * MS; idx += 64 * NWV) {
            const int p = idx % 8, m = idx / 8;
            if (m0 + m < M && n0 + 2 * p + 1 < N) {
                const float gt = BF(total(2 * p, m)), up = BF(total(2 * p + 1, m));
                y[(size_t)(m0 + m) * (N / 2) + n0 / 2 + p] = f2bf(silu_bf16(gt) * up);
            }
        }
    } else {
        for (int idx = threadIdx.x; idx < 16 * 16 * MS; idx += 64 * NWV) {
            const int f = idx % 16, m = idx / 16;
            if (m0 + m < M && n0 + f < N) {
                const size_t o = (size_t)(m0 + m) * N + n0 + f;
                const float s = total(f, m);
                y[o] = EPI == EPI_ADD ? f2bf(BF(s) + bf2f(res[o])) : f2bf(s);
            }
        }
    }
}

// barrier for data that goes through LDS only: global loads stay in flight across it (__syncthreads() would drain them)
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// a + b over lane pairs (l, l + 32) / (l, l + 16): one v_permlane swap per dword serves two values at once, so that two rows'
// sums are folded together and land in different lanes
__device__ __forceinline__ double swap_add32(double a, double b) {
    const auto l = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
}
__device__ __forceinline__ double swap_add16(double a, double b) {
    const auto l = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
}
constexpr int XK = 1024;
// inv[r] = 1 / sqrt(sum / 1024 + eps) of NR = 2, 4 or 6 rows whose exact (double) sums of squares lie spread over the 64 lanes of
// ss[r].  The first two folding steps halve the number of values (row r ends in 16-lane row (r & 1) * 2 + (r >> 1 & 1) of value
// r / 4), so the reduction costs about a third of NR separate ones, and the root is taken once.
template <int NR>
__device__ __forceinline__ void rows_inv(const double (&ss)[NR], float eps, int lane, float (&inv)[NR]) {
    constexpr int NT = NR / 2, NU = (NT + 1) / 2;
    double t[NT], u[NU];
#pragma unroll
    for (int i = 0; i < NT; i++) t[i] = swap_add32(ss[2 * i], ss[2 * i + 1]);
#pragma unroll
    for (int i = 0; i < NU; i++) u[i] = row16_sum_d(swap_add16(t[2 * i], t[2 * i + 1 < NT ? 2 * i + 1 : 2 * i]));
    const float mine = NU > 1 && (lane & 1) ? (float)u[NU - 1] : (float)u[0];
    const float rv = rsqrt_rn(mine / (float)XK + eps);
#pragma unroll
    for (int r = 0; r < NR; r++)
        inv[r] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(rv), (r & 1) * 32 + (r & 2) * 8 + r / 4));
}

// 4 x 4 transpose of 16-byte items between four registers and the four lanes of a quad: 48 vector instructions
__device__ __forceinline__ void quad_transpose(u32x4 (&v)[4], bool odd, bool high) {
    auto swz = [](unsigned v, auto ctrl) { return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, ctrl.value, 0xF, 0xF, true); };
    constexpr std::integral_constant<int, 0xB1> by1{};            // quad_perm [1,0,3,2]
    constexpr std::integral_constant<int, 0x4E> by2{};            // quad_perm [2,3,0,1]
#pragma unroll
    for (int i = 0; i < 4; i++) {
        unsigned x0 = v[0][i], x1 = v[1][i], x2 = v[2][i], x3 = v[3][i];
        unsigned t = swz(odd ? x0 : x1, by1), u = swz(odd ? x2 : x3, by1);
        x0 = odd ? t : x0, x1 = odd ? x1 : t, x2 = odd ? u : x2, x3 = odd ? x3 : u;
        t = swz(high ? x0 : x2, by2), u = swz(high ? x1 : x3, by2);
        v[0][i] = high ? t : x0, v[2][i] = high ? x2 : t, v[1][i] = high ? u : x1, v[3][i] = high ? x3 : u;
    }
}

// K = 1024, wide outputs.  A workgroup of eight wavefronts owns NB = 2 FB blocks of 16 features and 16 RB rows; wavefront (half,
// q) multiplies FB of the blocks over the quarter q of K (two of the eight 128-wide steps of a row), and the quarters meet in
// LDS in a fixed order.
// Rows: every wavefront brings in 2 RB of them, a row per two loads of 1 KiB, asks for the W of its first block right after, and applies the
// rms prologue (RMS) while that is on its way from HBM; the rows then go to LDS, their 16-byte chunks XOR-swizzled by the row number
// so that the 16 rows of one k group fall on distinct banks.  (Not yet those of a whole read: 16 bytes a lane are read for lanes 0 - 3, 12 - 15 and 20 - 27
// together, then 4 - 11, 16 - 19 and 28 - 31, which are rows of two k groups, and the XOR puts the one on the other's banks.  Such a read takes eight
// cycles instead of four: the conflicts in half of the LDS's active cycles that the counters show here and in tile_gemm_kernel.)
// Every workgroup normalises its rows itself: 0.1 us (16 rows) to 0.7 us (32 rows x 64 features) instead of a launch of its own at 2.6 us.
// W: a load takes 256 contiguous bytes of four features, 64 of them in each quad of lanes (register j of lane (g, h, c): feature
// 4 h + j, elements 32 g + 8 c ..), and quad_transpose turns four such loads into the MFMA layout: feature n in lane (n, g),
// elements 32 g + 8 r .. in register r.  The x fragments are read from LDS in the same enumeration of k.  Which wavefront takes
// which quarter differs from workgroup to workgroup, so that they do not all ask the same memory channels first; a quarter's
// product and the sum of the four do not depend on it, so a row has the same bits in every place of a batch of any size.  (Letting
// half of the workgroups begin with their quarter's second step would take another 3 % off 16 rows at N = 5120 and 7168, but the order of
// summation would follow; with the order kept by exchanging registers, in a branch, or by summing the steps apart it costs as much or more.)
// N need not divide: with `extra` > 0 the first `extra` tiles take four features more each, from the end of N (N = 8224 is 256 tiles of 32
// and eight times four; a 257th workgroup would take a CU twice as long as the others).  They come in MFMA layout, four lanes to an
// address, and need no transpose; with a whole block of 16 more for two workgroups those two ended the launch 0.5 us late.
// A workgroup's time (in-kernel time stamps).  At one row: rows in LDS after 1.9 us, W there after 3.0, product 0.65, the quarters' sum and
// the store 0.6.  With 32 rows x 64 features: a CU takes a load of 1 KiB every 16 clocks and a wavefront waits at a load that is not taken yet, so
// that 26 loads a wavefront ahead of the prologue held it up for 2.1 - 2.9 us, with the rows long there.  Hence the order: the rows' loads
// ahead of all W (0.2 us from 16 rows on); of W what 8 loads a wavefront bring before the prologue, and the second block's behind the rows'
// barrier (0.7 us at 64 rows; 4 or 6 loads ahead 0.2 - 0.4 more, all ahead as before; interleaved with the prologue 0.1 - 0.5 more); the row
// fragments read before W is waited for and each block multiplied as it comes (0.3 us at 32 - 48 rows); the partial sums beside the rows in
// LDS, without a barrier between (0.4 us).
// Transposing through LDS (4 KiB a wavefront, 8 accesses instead of 64 vector instructions) takes as long: what follows the arrival
// of W is serial either way.
// Tile sizes (us in a HIP graph, rms prologue included, N = 8224 / 7168 swiglu / 5120; in brackets the build before this order): 1 row 5.4 / 5.15 /
// 4.5 (5.45 / 5.2 / 4.6), 16 rows 5.45 / 5.1 / 4.5 (5.5 / 5.2 / 4.6), 32 rows 6.1 / 5.95 / 5.4 (6.6 / 6.2 / 5.7), 48 and 64 rows 7.1 / 6.7 / 6.2 (8.0 - 8.2 / 7.4 - 7.9 / 7.0 -
// 7.4), 80 rows 8.2 / 8.0 / 6.2 (9.8 / 9.4 / 7.4).  An empty kernel takes 1.8 us there; one that only loads takes 4.05 for the 16.8 MB, 5.2
// with the loads of 32 rows x 64 features: what is left is the prologue and what follows the last of W.
template <int RB, int FB, bool RMS, int EPI, bool ALONE>
__global__ __launch_bounds__(512, RB == 1 ? 4 : 2) void rows_gemm_kernel(const bf16_t* __restrict__ W, const bf16_t* __restrict__ x,
                                                                         const bf16_t* __restrict__ nw, float eps,
                                                                         const bf16_t* __restrict__ res, bf16_t* __restrict__ y, int M, int N,
                                                                         int tiles, int extra) {
    constexpr int NB = 2 * FB, R = 16 * RB, RW = R / 8;
    // row fragments in registers before W is there, partial sums beside the rows: not where the registers (64 rows) or the LDS (two workgroups
    // of 32 rows x 32 features on a CU) do not hold them
    constexpr bool PRE = RB == 1 || (RB <= 3 && ALONE);
    __shared__ __align__(1024) bf16_t x_s[R * XK];
    __shared__ __align__(16) float red_s[PRE ? (NB + 1) * 4 * R * 16 : 4];     // the partial sums [NB + 1][4 quarters][R][16 features], or in the rows' place
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    // the row groups of a tile sit on one XCD (workgroups are dealt to the eight XCDs in turn) and share its W through the L2, also though
    // it is loaded nontemporally (N = 8224, two groups: 18.1 MB fetched, W is 16.8 and the rows on eight XCDs 1.0)
    const int grp = blockIdx.y, tile = blockIdx.z * 8 + blockIdx.x;
    if (tile >= tiles) return;
    const int q = (w + grp + blockIdx.z) & 3, half = w >> 2, m0 = grp * R, nb0 = tile * 16 * NB, nx = 16 * NB * tiles + 4 * tile;
    const bool has_x = tile < extra && half == 0;
    u32x4 xr[RW][2], wn[2];
#pragma unroll
    for (int i = 0; i < RW; i++) {
        const bf16_t* src = x + (size_t)min(m0 + w + 8 * i, M - 1) * XK + 8 * lane;      // (rows past M repeat the last one)
        xr[i][0] = *reinterpret_cast<const u32x4*>(src);
        xr[i][1] = *reinterpret_cast<const u32x4*>(src + 512);
    }
    if (RMS) {
        wn[0] = *reinterpret_cast<const u32x4*>(nw + 8 * lane);
        wn[1] = *reinterpret_cast<const u32x4*>(nw + 512 + 8 * lane);
    }
    // a CU's loads return in the order in which they were issued, whichever wavefront asked: no W before the last row has been requested
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    u32x4 a[FB][2][4], ax[8];
    auto load_w = [&](int f, int i) {
        a[f][i >> 2][i & 3] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(
            W + (size_t)min(nb0 + 16 * (half * FB + f) + (n & 12) + (i & 3), N - 1) * XK + 128 * (2 * q + (i >> 2)) + 32 * g + 8 * (n & 3)));
    };
    auto load_extra = [&] {
        if (has_x)
#pragma unroll
            for (int i = 0; i < 8; i++)
                ax[i] = *reinterpret_cast<const u32x4*>(W + (size_t)(nx + (n & 3)) * XK + 128 * (2 * q + (i >> 2)) + 32 * g + 8 * (i & 3));
    };
#pragma unroll
    for (int i = 0; i < 8; i++) load_w(0, i);
    if (FB == 1) load_extra();
    __builtin_amdgcn_sched_barrier(0);                            // all this is in flight before the first row is looked at
    if (RMS) {
        double ss[RW];
#pragma unroll
        for (int i = 0; i < RW; i++) {
            ss[i] = 0.0;
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const double lo = (double)lo_bf(xr[i][c][j]), hi = (double)hi_bf(xr[i][c][j]);
                    ss[i] = fma(hi, hi, fma(lo, lo, ss[i]));
                }
        }
        float inv[RW];
        rows_inv<RW>(ss, eps, lane, inv);
#pragma unroll
        for (int i = 0; i < RW; i++)
#pragma unroll
            for (int c = 0; c < 2; c++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    xr[i][c][j] = pack2_bf(lo_bf(wn[c][j]) * (lo_bf(xr[i][c][j]) * inv[i]), hi_bf(wn[c][j]) * (hi_bf(xr[i][c][j]) * inv[i]));
    }
#pragma unroll
    for (int i = 0; i < RW; i++) {
        const int r = w + 8 * i;
#pragma unroll
        for (int c = 0; c < 2; c++) *reinterpret_cast<u32x4*>(x_s + r * XK + 8 * ((lane + 64 * c) ^ (r & 15))) = xr[i][c];
    }
    lds_barrier();
    if (FB == 2) {
#pragma unroll
        for (int i = 0; i < 8; i++) load_w(1, i);
        load_extra();
    }
    f32x4 acc[FB][RB], acc_x[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) acc_x[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int f = 0; f < FB; f++)
#pragma unroll
        for (int rb = 0; rb < RB; rb++) acc[f][rb] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bool odd = n & 1, high = n & 2;
    auto x_frag = [&](int i, int rb) {
        return *reinterpret_cast<const u32x4*>(x_s + (16 * rb + n) * XK + 8 * ((16 * (2 * q + (i >> 2)) + 4 * g + (i & 3)) ^ n));
    };
    auto mma = [](const u32x4& av, const u32x4& bv, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av), __builtin_bit_cast(bf16x8, bv), c, 0, 0, 0);
    };
    u32x4 xf[PRE ? 8 : 1][PRE ? RB : 1];                          // (read while W is still on its way)
    if constexpr (PRE) {
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int rb = 0; rb < RB; rb++) xf[i][rb] = x_frag(i, rb);
        __builtin_amdgcn_sched_barrier(0);
    }
    auto x_at = [&](int i, int rb) { return PRE ? xf[PRE ? i : 0][PRE ? rb : 0] : x_frag(i, rb); };
    // block by block, so that one is multiplied while the next one's W arrives; where the fragments are read for each use, all blocks at once
#pragma unroll
    for (int f = 0; f < FB; f++) {
#pragma unroll
        for (int t = 0; t < 2; t++) quad_transpose(a[f][t], odd, high);
        if (PRE)
#pragma unroll
            for (int i = 0; i < 8; i++)
#pragma unroll
                for (int rb = 0; rb < RB; rb++) acc[f][rb] = mma(a[f][i >> 2][i & 3], x_at(i, rb), acc[f][rb]);
    }
    if (!PRE)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            u32x4 b[RB];
#pragma unroll
            for (int rb = 0; rb < RB; rb++) b[rb] = x_frag(i, rb);
#pragma unroll
            for (int f = 0; f < FB; f++)
#pragma unroll
                for (int rb = 0; rb < RB; rb++) acc[f][rb] = mma(a[f][i >> 2][i & 3], b[rb], acc[f][rb]);
        }
    if (has_x) {
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int rb = 0; rb < RB; rb++) acc_x[rb] = mma(ax[i], x_at(i, rb), acc_x[rb]);
    }
    if (!PRE) lds_barrier();                                      // the rows have been read: their memory takes the partial sums
    // accumulator element i of lane (n, g) is feature 4 g + i of row 16 rb + n
    float* red = PRE ? red_s : reinterpret_cast<float*>(x_s);
    auto put = [&](int blk, const f32x4 (&v)[RB]) {
#pragma unroll
        for (int rb = 0; rb < RB; rb++) *reinterpret_cast<f32x4*>(red + ((blk * 4 + q) * R + 16 * rb + n) * 16 + 4 * g) = v[rb];
    };
#pragma unroll
    for (int f = 0; f < FB; f++) put(half * FB + f, acc[f]);
    if (has_x && g == 0) put(NB, acc_x);
    lds_barrier();
    const int items = NB * R * 4 + (tile < extra ? R : 0);
    for (int idx = threadIdx.x; idx < items; idx += 512) {        // four adjacent features of a row each (N is a multiple of 4)
        const bool own = idx < NB * R * 4;
        const int blk = idx / (R * 4), r = own ? (idx / 4) % R : idx - NB * R * 4, f4 = own ? idx & 3 : 0;
        const int m = m0 + r, f0 = own ? nb0 + 16 * blk + 4 * f4 : nx;
        if (m >= M || f0 >= N) continue;
        f32x4 t[4];
#pragma unroll
        for (int k = 0; k < 4; k++) t[k] = *reinterpret_cast<const f32x4*>(red + ((blk * 4 + k) * R + r) * 16 + 4 * f4);
        f32x4 v = (t[0] + t[1]) + (t[2] + t[3]);
        if (EPI == EPI_SWIGLU) {
            *reinterpret_cast<uint32_t*>(y + (size_t)m * (N / 2) + f0 / 2) = pack_bf(silu_bf16(BF(v[0])) * BF(v[1]), silu_bf16(BF(v[2])) * BF(v[3]));
        } else {
            const size_t o = (size_t)m * N + f0;
            if (EPI == EPI_ADD) {
                const uint2 rr = *reinterpret_cast<const uint2*>(res + o);
                v = f32x4{BF(v[0]) + lo_bf(rr.x), BF(v[1]) + hi_bf(rr.x), BF(v[2]) + lo_bf(rr.y), BF(v[3]) + hi_bf(rr.y)};
            }
            *reinterpret_cast<uint2*>(y + o) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
        }
    }
}

// Narrow outputs (N = 1024: out_proj, o_proj, down_proj): a workgroup owns 4 FG features x 4 MG rows, its NWV wavefronts deal the
// 128-wide steps of K among themselves, KS at a time with all their loads in flight, and meet in LDS in a fixed order.  The
// point of the small tile is that every CU has one: at 1 to 16 rows a 16-feature tile leaves 192 of 256 CUs idle, and one CU
// takes its 115 KiB of W in at 38 - 63 GB/s at best.
// Operand layout: lane (n, g) of a load holds elements 32 g + 8 (n & 3) .. of row 4 i + (n >> 2), so a quad of lanes reads 64 and the
// wavefront 256 contiguous bytes of four rows; W and x alike.  Taken as it is by a 16 x 16 x 32 MFMA, "row" n of the operand is
// (row n >> 2, k slice n & 3), and of the 16 x 16 results those whose k slices agree are partial sums: element i of lane (n, g)
// belongs to feature g and row n >> 2 if i = n & 3.  Three of four MFMA results are thrown away; the matrix cores have nothing
// else to do here (8 x 8 tile, K = 3584: 28 steps x 4 MFMAs per CU).
// ONE: K of up to 128 NWV KS, a single trip for every wavefront (one past the end loads the last step and multiplies nothing): the residual behind the
// operands, as with PEEL (4 rows, K = 1024, N = 1024 / 2048 / 3072
// 2.8 / 3.0 / 3.6 us; in a loop and with the residual ahead of the operands 3.25 / 3.75 / 4.05).
// PEEL: the first trip is taken out of the loop (by the residual's load, which only that trip makes): 0.2 - 0.6 us less, for a tenth more
// registers, which costs where several workgroups share a CU (80 rows 7.2 / 10.8 us against 6.4 / 10.3).
// Measured in a HIP graph with the residual epilogue, K = 2048 / 3584 (before: residual loaded behind the last barrier, no trip peeled): 1 row
// 3.0 / 3.5 us (3.3 / 3.8), 16 rows 3.4 / 4.4 (3.7 / 4.8), 32 rows 3.8 / 5.2 (4.2 / 5.6), 64 rows - / 6.2 (5.4 / 6.9).
template <int NWV, int KS, int FG, int MG, int EPI, bool PEEL, bool ONE>
__global__ __launch_bounds__(64 * NWV) void quad_gemm_kernel(const bf16_t* __restrict__ W, const bf16_t* __restrict__ x,
                                                             const bf16_t* __restrict__ res, bf16_t* __restrict__ y, int M, int N, int K,
                                                             int groups) {
    constexpr int F = 4 * FG, R = 4 * MG;
    __shared__ __align__(16) float red[NWV][R][F];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int s = blockIdx.x >> 3, grp = s % groups, tile = (s / groups) * 8 + (blockIdx.x & 7);      // row groups of a tile: one XCD
    const int n0 = tile * F, m0 = grp * R, steps = K / 128;
    if (n0 >= N) return;
    const bf16_t *wp[FG], *xp[MG];
#pragma unroll
    for (int f = 0; f < FG; f++) wp[f] = W + (size_t)min(n0 + 4 * f + (n >> 2), N - 1) * K + 32 * g + 8 * (n & 3);
#pragma unroll
    for (int m = 0; m < MG; m++) xp[m] = x + (size_t)min(m0 + 4 * m + (n >> 2), M - 1) * K + 32 * g + 8 * (n & 3);
    // the thread's output in the epilogue; its residual is requested with the operands, not behind their last barrier
    const int er = threadIdx.x / F, ef = threadIdx.x % F;
    const bool e_mine = er < R && m0 + er < M && n0 + ef < N;
    const size_t eo = (size_t)(m0 + er) * N + n0 + ef;
    unsigned res_raw = 0;
    if (EPI == EPI_ADD && !PEEL && !ONE && e_mine) res_raw = res[eo];
    f32x4 acc[FG][MG];
#pragma unroll
    for (int f = 0; f < FG; f++)
#pragma unroll
        for (int m = 0; m < MG; m++) acc[f][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int base = w; ONE ? base == w : base < steps; base += NWV * KS) {
        u32x4 a[KS][FG], b[KS][MG];
#pragma unroll
        for (int c = 0; c < KS; c++) {
            const int k0 = min(base + c * NWV, steps - 1) * 128;  // (a step past the end loads the last one and is not multiplied)
#pragma unroll
            for (int f = 0; f < FG; f++) a[c][f] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp[f] + k0));
#pragma unroll
            for (int m = 0; m < MG; m++) b[c][m] = *reinterpret_cast<const u32x4*>(xp[m] + k0);
        }
        // (what only the first trip does makes the compiler take that trip out of the loop)
        if (EPI == EPI_ADD && (PEEL || ONE) && base == w && e_mine) res_raw = res[eo];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < KS; c++)
            if (base + c * NWV < steps)
#pragma unroll
                for (int f = 0; f < FG; f++)
#pragma unroll
                    for (int m = 0; m < MG; m++)
                        acc[f][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[c][f]),
                                                                           __builtin_bit_cast(bf16x8, b[c][m]), acc[f][m], 0, 0, 0);
    }
    const int c = n & 3;                                          // of the quad's four sums lane c keeps the one of row block c
#pragma unroll
    for (int f = 0; f < FG; f++) {
        float keep = 0.f;
#pragma unroll
        for (int m = 0; m < MG; m++) {
            float v = c == 0 ? acc[f][m][0] : c == 1 ? acc[f][m][1] : c == 2 ? acc[f][m][2] : acc[f][m][3];
            v += dpp_mov<0xB1>(v);
            v += dpp_mov<0x4E>(v);
            keep = (m == 0 || c == m) ? v : keep;
        }
        if (c < MG) red[w][4 * c + (n >> 2)][4 * f + g] = keep;
    }
    lds_barrier();
    auto total = [&](int r, int f) {                              // fixed order: pairs, then pairs of pairs, ...
        float t[NWV];
#pragma unroll
        for (int k = 0; k < NWV; k++) t[k] = red[k][r][f];
#pragma unroll
        for (int st = 1; st < NWV; st *= 2)
#pragma unroll
            for (int k = 0; k < NWV; k += 2 * st) t[k] += t[k + st];
        return t[0];
    };
    if (EPI == EPI_SWIGLU) {
        const int r = threadIdx.x / (F / 2), p = threadIdx.x % (F / 2), m = m0 + r;
        if (r < R && m < M && n0 + 2 * p + 1 < N)
            y[(size_t)m * (N / 2) + n0 / 2 + p] = f2bf(silu_bf16(BF(total(r, 2 * p))) * BF(total(r, 2 * p + 1)));
    } else {
        if (e_mine) {
            const float v = total(er, ef);
            y[eo] = EPI == EPI_ADD ? f2bf(BF(v) + bf2f((bf16_t)res_raw)) : f2bf(v);
        }
    }
}

// Narrow outputs of 1024 < K <= 2048 whose 16 x 16 tiles leave at most one workgroup per CU and whose 8 x 16 tiles do not.  A CU takes a load of
// 1 KiB every 16 clocks, so what counts is the bytes of its tiles: 128 KiB for one of 16 x 16 at K = 2048, 192 for two of 8 x 16.  The wavefronts
// deal the 128-wide steps of K among themselves as quad_gemm_kernel's do; the operands go straight to LDS, into 16 KiB that belong to the
// wavefront (no barrier, no registers: a wavefront waits for its own loads), the 16-byte chunks of a row XOR-swizzled by the row number, so
// that an MFMA takes 16 rows of each and none of its results is thrown away (16 MFMAs a step there, 4 here).
// MFMA j of a step takes k slice j (elements 32 g + 8 j ..), each slice has an accumulator of its own and the four are added as there: the
// same bits.
// us in a graph with the residual, quad_gemm_kernel / here: N = 1024, K = 2048 at 33 / 48 / 64 rows 4.8 / 5.05 / 5.1 -> 3.8 / 4.2 / 4.25, N = 2048 at 24 / 32
// rows 5.2 / 5.4 -> 4.2 / 4.6, N = 4096 at 16 rows 6.0 -> 5.3, N = 520 at 96 rows 4.7 -> 4.2, K = 1280 0.5 less.  A kernel that only loads these
// bytes takes 3.6 (N = 1024, 64 rows).  Longer K (224 KiB at K = 3584) with the steps beyond 128 KiB held in registers: 6.4, 6.1 there.  Through a ring in LDS it is
// 5.9 alone, but slower inside a step of eight layers (64 x 1 rows 415.3 us against 408.3), or no faster with nontemporal W (407.3 against 407.5).
// W is loaded plainly here: nontemporal, that step takes 415 us against 410.8.
template <int EPI>
__global__ __launch_bounds__(512) void tile_gemm_kernel(const bf16_t* __restrict__ W, const bf16_t* __restrict__ x, const bf16_t* __restrict__ res,
                                                        bf16_t* __restrict__ y, int M, int N, int K, int groups) {
    __shared__ __align__(1024) char own_s[8 * 16384];
    __shared__ __align__(16) float red[8][16][16];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int s = blockIdx.x >> 3, grp = s % groups, tile = (s / groups) * 8 + (blockIdx.x & 7);      // row groups of a tile: one XCD
    const int n0 = tile * 16, m0 = grp * 16, steps = K / 128;
    if (n0 >= N) return;
    const char *wsrc[4], *xsrc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int r = 4 * i + g, off = (n ^ r) * 16;
        wsrc[i] = reinterpret_cast<const char*>(W + (size_t)min(n0 + r, N - 1) * K) + off;
        xsrc[i] = reinterpret_cast<const char*>(x + (size_t)min(m0 + r, M - 1) * K) + off;
    }
    const char* own = own_s + w * 16384;
    const unsigned own_a = (unsigned)(size_t)(__attribute__((address_space(3))) const void*)own_s + w * 16384;
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int k0 = min(w + 8 * c, steps - 1) * 256;           // (a step past the end loads the last one and is not multiplied)
#pragma unroll
        for (int i = 0; i < 4; i++) lds_dma16_from(wsrc[i] + k0, own_a + c * 8192 + i * 1024);
#pragma unroll
        for (int i = 0; i < 4; i++) lds_dma16_from(xsrc[i] + k0, own_a + c * 8192 + 4096 + i * 1024);
    }
    // the thread's output in the epilogue; its residual is requested behind the operands
    const int er = threadIdx.x >> 4, ef = threadIdx.x & 15;
    const bool e_mine = er < 16 && m0 + er < M && n0 + ef < N;
    const size_t eo = (size_t)(m0 + er) * N + n0 + ef;
    unsigned res_raw = 0;
    if (EPI == EPI_ADD && e_mine) res_raw = res[eo];
    __builtin_amdgcn_sched_barrier(0);
    f32x4 acc[4];
#pragma unroll
    for (int c = 0; c < 4; c++) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int c) {
        u32x4 a[4], b[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const char* q = own + c * 8192 + n * 256 + ((4 * g + j) ^ n) * 16;
            a[j] = *reinterpret_cast<const u32x4*>(q);
            b[j] = *reinterpret_cast<const u32x4*>(q + 4096);
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[j]), __builtin_bit_cast(bf16x8, b[j]), acc[j], 0, 0, 0);
    };
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");              // (the second step's loads; the residual's may be one more)
    multiply(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (w + 8 < steps) multiply(1);
    *reinterpret_cast<f32x4*>(&red[w][n][4 * g]) = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    lds_barrier();
    auto total = [&](int r, int f) {                              // fixed order: pairs, then pairs of pairs, ...
        float t[8];
#pragma unroll
        for (int k = 0; k < 8; k++) t[k] = red[k][r][f];
#pragma unroll
        for (int st = 1; st < 8; st *= 2)
#pragma unroll
            for (int k = 0; k < 8; k += 2 * st) t[k] += t[k + st];
        return t[0];
    };
    if (EPI == EPI_SWIGLU) {
        const int r = threadIdx.x / 8, p = threadIdx.x % 8, m = m0 + r;
        if (r < 16 && m < M && n0 + 2 * p + 1 < N)
            y[(size_t)m * (N / 2) + n0 / 2 + p] = f2bf(silu_bf16(BF(total(r, 2 * p))) * BF(total(r, 2 * p + 1)));
    } else if (e_mine) {
        const float v = total(er, ef);
        y[eo] = EPI == EPI_ADD ? f2bf(BF(v) + bf2f((bf16_t)res_raw)) : f2bf(v);
    }
}

struct gemv_args {
    const bf16_t *W, *x, *nw, *res;
    bf16_t* y;
    int M, N, K, epi;
    float eps;
    hipStream_t stream;
};

// the workgroups of a launch: `tiles` of 32 FB features, of which the first `extra` take four features more, times `groups` of 16 RB rows
struct RowsGrid {
    int groups, tiles, extra;
    RowsGrid(const gemv_args& p, int cus, int RB, int FB) {
        groups = (p.M + 16 * RB - 1) / (16 * RB), extra = 0;
        const int blocks = (p.N + 15) / 16, per_cu = cus / groups > 0 ? cus / groups : 1;
        tiles = (blocks + 2 * FB - 1) / (2 * FB);
        // a few features more than a whole tile per CU: the first tiles take four each instead of a workgroup of their own
        if (blocks > per_cu * 2 * FB && blocks - per_cu * 2 * FB <= per_cu / 16) tiles = per_cu, extra = (p.N - per_cu * 32 * FB) / 4;
    }
    bool one_round(int cus) const { return (long)tiles * groups <= cus; }        // a workgroup per CU at most
};
constexpr int MAX_GROUPS = 65535;      // of a launch (second dimension of a grid)
template <int RB, int FB, bool RMS, bool ALONE = true>
void launch_rows(const gemv_args& p, int cus) {
    const RowsGrid r(p, cus, RB, FB);
    const dim3 block(512);
    for (int g0 = 0; g0 < r.groups; g0 += MAX_GROUPS) {          // (one launch up to 65535 row groups)
        const size_t row0 = (size_t)g0 * 16 * RB;
        const dim3 grid(8, r.groups - g0 < MAX_GROUPS ? r.groups - g0 : MAX_GROUPS, (r.tiles + 7) / 8);
        const bf16_t *x = p.x + row0 * p.K, *res = p.res ? p.res + row0 * p.N : nullptr;
        bf16_t* y = p.y + row0 * (p.epi == EPI_SWIGLU ? p.N / 2 : p.N);
        const int M = p.M - (int)row0;
        if (p.epi == EPI_NONE)
            hipLaunchKernelGGL((rows_gemm_kernel<RB, FB, RMS, EPI_NONE, ALONE>), grid, block, 0, p.stream, p.W, x, p.nw, p.eps, res, y, M, p.N, r.tiles, r.extra);
        else if (p.epi == EPI_ADD)
            hipLaunchKernelGGL((rows_gemm_kernel<RB, FB, RMS, EPI_ADD, ALONE>), grid, block, 0, p.stream, p.W, x, p.nw, p.eps, res, y, M, p.N, r.tiles, r.extra);
        else
            hipLaunchKernelGGL((rows_gemm_kernel<RB, FB, RMS, EPI_SWIGLU, ALONE>), grid, block, 0, p.stream, p.W, x, p.nw, p.eps, res, y, M, p.N, r.tiles, r.extra);
    }
}
// the shapes rows_gemm_kernel takes (its 8-byte stores and residual loads want y and res aligned to 8 bytes)
inline bool rows_shape(const gemv_args& p) {
    return p.K == XK && p.N >= 4096 && (p.N & 3) == 0 && ((reinterpret_cast<uintptr_t>(p.y) | reinterpret_cast<uintptr_t>(p.res)) & 7u) == 0;
}
constexpr int RMS_ROWS_MAX = 96;       // most rows with the prologue fused in: beyond, the rows are normalised too often
// Tile by rows.  Up to 96 rows: the smallest tile that leaves at most one workgroup per CU (32 features as long as one row
// group holds the batch, then 64; at 33 - 48 rows with the prologue 32 rows x 64 features, which normalise fewer rows each: 7.1 / 6.7 / 6.2 us against
// 7.3 / 7.0 / 6.5 with 48 x 32, without it 6.5 against 6.0; where 64 features leave no room for the extra fours, N = 8324 .. 8448, 48 x 32 takes 7.9 and
// 8.1 with swiglu, 48 x 64 8.05 and 8.4).  Where none does, W is what costs, and one row group is better than two that read it twice:
// 64 features x 48 or 64 rows (N = 9216 / 32768 / 151936 at 48 rows 6.6 / 15.9 / 70 us; with an earlier build 8.5 / 19.2 / 82, 11.3 / 24.4 / 102 with 32
// features, at 64 rows 9.1 / 20.8 / 88, 11.9 / 25.7 / 108 with two groups of 32 rows); up to 32 rows 32 features again, whose two workgroups per CU overlap (N =
// 32768 / 151936 16 / 61 us at 17 rows, 17.3 / 68 with 64).  Beyond 96 rows 64 x 64 up to 128 rows, then 32 x 32 (N = 8224 / 7168 / 5120 at
// 128 rows 13.1 / 12.5 / 11.6 us with the rms launch, 256 23 / 21.4 / 16.8, 4096 351 / 301 / 221; 23.7 / 22.6 / 14.7, 33.8 / 31.5 / 24.7 and 429 / 325 / 274
// with the 64-row tiles of general loads before).
// The rms prologue: false (nothing launched) where more than one workgroup per CU would normalise the same rows, which then cost
// more than the launch they save (from 17 rows on; N = 32768 / 151936 at 64 rows 29 / 124 us fused, 24 / 91 in two launches).
template <bool RMS>
bool launch_rows_any(const gemv_args& p, int cus) {
    auto one_round = [&](int RB, int FB) { return RowsGrid(p, cus, RB, FB).one_round(cus); };
    if (p.M <= 16) {
        launch_rows<1, 1, RMS>(p, cus);
        return true;
    }
    if (p.M <= 32) {
        if (!one_round(2, 1) && one_round(2, 2))
            launch_rows<2, 2, RMS>(p, cus);
        else if (one_round(2, 1))
            launch_rows<2, 1, RMS>(p, cus);
        else if constexpr (!RMS)
            launch_rows<2, 1, false, false>(p, cus);
        else
            return false;
        return true;
    }
    if (p.M <= 96 && (RMS || p.M > 48) && one_round(2, 2)) {
        launch_rows<2, 2, RMS>(p, cus);
        return true;
    }
    if (p.M <= 48 && one_round(3, 1)) {
        launch_rows<3, 1, RMS>(p, cus);
        return true;
    }
    if ((p.M <= 48 || (p.M > 64 && p.M <= 96)) && (!RMS || one_round(3, 2))) {
        launch_rows<3, 2, RMS>(p, cus);
        return true;
    }
    if constexpr (!RMS) {
        if (p.M <= 128)
            launch_rows<4, 2, false>(p, cus);
        else
            launch_rows<2, 1, false, false>(p, cus);
        return true;
    }
    return false;
}

template <int NWV, int KS, int FG, int MG, bool PEEL, bool ONE = false>
void launch_quad_tile(const gemv_args& p) {
    const int groups = (p.M + 4 * MG - 1) / (4 * MG), tiles = (p.N + 4 * FG - 1) / (4 * FG);
    const dim3 grid((tiles + 7) / 8 * 8 * groups), block(64 * NWV);
    if (p.epi == EPI_NONE)
        hipLaunchKernelGGL((quad_gemm_kernel<NWV, KS, FG, MG, EPI_NONE, PEEL, ONE>), grid, block, 0, p.stream, p.W, p.x, p.res, p.y, p.M, p.N, p.K, groups);
    else if (p.epi == EPI_ADD)
        hipLaunchKernelGGL((quad_gemm_kernel<NWV, KS, FG, MG, EPI_ADD, PEEL, ONE>), grid, block, 0, p.stream, p.W, p.x, p.res, p.y, p.M, p.N, p.K, groups);
    else
        hipLaunchKernelGGL((quad_gemm_kernel<NWV, KS, FG, MG, EPI_SWIGLU, PEEL, ONE>), grid, block, 0, p.stream, p.W, p.x, p.res, p.y, p.M, p.N, p.K, groups);
}
// wavefronts and steps at a time by K: all of K in flight at once up to 4096.  PEEL_: the first trip taken out of the loop
template <int FG, int MG, bool PEEL_ = true>
void launch_quad(const gemv_args& p) {
    if (p.K <= 1024)
        launch_quad_tile<4, 2, FG, MG, false, true>(p);
    else if (p.K <= 2048)
        launch_quad_tile<8, 2, FG, MG, PEEL_>(p);
    else
        launch_quad_tile<8, 4, FG, MG, PEEL_>(p);
}
void launch_tile(const gemv_args& p) {
    const int groups = (p.M + 15) / 16, tiles = (p.N + 15) / 16;
    const dim3 grid((tiles + 7) / 8 * 8 * groups), block(512);
    if (p.epi == EPI_NONE)
        hipLaunchKernelGGL(tile_gemm_kernel<EPI_NONE>, grid, block, 0, p.stream, p.W, p.x, p.res, p.y, p.M, p.N, p.K, groups);
    else if (p.epi == EPI_ADD)
        hipLaunchKernelGGL(tile_gemm_kernel<EPI_ADD>, grid, block, 0, p.stream, p.W, p.x, p.res, p.y, p.M, p.N, p.K, groups);
    else
        hipLaunchKernelGGL(tile_gemm_kernel<EPI_SWIGLU>, grid, block, 0, p.stream, p.W, p.x, p.res, p.y, p.M, p.N, p.K, groups);
}
// The smallest tile that leaves at most one workgroup per CU; beyond, small tiles still win with several workgroups per CU (measured
// against skinny_gemm_kernel over N = 264 .. 3072, K = 512 .. 4096, 16 .. 192 rows, us: three workgroups of 8 x 16 per CU N = 1024, K = 2048 / 3584 at 80
// rows 6.4 / 10.3 against 9.5 / 16.1, N = 3072, K = 2048 at 32 rows 7.3 against 10.1; N = 8192, K = 2048, 8 rows, four of 8 x 8 8.3 against 9.4; two
// of 16 x 16 N = 1024, K = 2048 at 128 rows 7.3 against 7.9, but K = 3584 12.2 against 11.9, K = 1024 and N = 2048 at 64 rows 5.4 against 5.2; four of 8 x
// 16 at 128 rows 8.3 / 12.6 against 7.9 / 11.9).  Returns false where the skinny kernel is the better one.
inline bool launch_quad_any(const gemv_args& p, int cus) {
    auto wgs = [&](int f, int r) { return (long)((p.N + f - 1) / f) * ((p.M + r - 1) / r); };
    if (wgs(4, 4) <= cus || (p.M <= 4 && wgs(4, 4) <= 2 * cus))
        launch_quad<1, 1>(p);
    else if (wgs(8, 8) <= cus || (p.M <= 8 && wgs(8, 8) <= 4 * cus))
        launch_quad<2, 2>(p);
    else if (wgs(8, 16) <= cus)
        launch_quad<2, 4>(p);
    else if (p.K > 1024 && p.K <= 2048 && wgs(16, 16) <= cus)
        launch_tile(p);
    else if (p.K > 2048 && wgs(16, 16) <= cus)
        launch_quad<4, 4>(p);
    else if (wgs(8, 16) <= 3 * cus)
        launch_quad<2, 4, false>(p);
    else if (p.K > 1024 && p.K <= 2048 && wgs(16, 16) <= 2 * cus)
        launch_quad<4, 4>(p);
    else
        return false;
    return true;
}

// row blocks per pass: 1, 2 or 4 (3 rounds up)
inline int row_blocks(int M) { return M <= 16 ? 1 : M <= 32 ? 2 : 4; }

template <int NWV, int MS>
void launch_gemm_ms(int epi, const bf16_t* W, const bf16_t* x, const bf16_t* res, bf16_t* y, int M, int N, int K, hipStream_t stream) {
    const dim3 grid((N + 15) / 16, (M + 16 * MS - 1) / (16 * MS)), block(64 * NWV);
    if (epi == EPI_NONE)
        hipLaunchKernelGGL((skinny_gemm_kernel<NWV, MS, EPI_NONE>), grid, block, 0, stream, W, x, res, y, M, N, K);
    else if (epi == EPI_ADD)
        hipLaunchKernelGGL((skinny_gemm_kernel<NWV, MS, EPI_ADD>), grid, block, 0, stream, W, x, res, y, M, N, K);
    else
        hipLaunchKernelGGL((skinny_gemm_kernel<NWV, MS, EPI_SWIGLU>), grid, block, 0, stream, W, x, res, y, M, N, K);
}
// narrow: the output has few feature blocks, so fewer rows per workgroup (more workgroups) pay for re-reading W from L2
template <int NWV>
void launch_gemm(int epi, const bf16_t* W, const bf16_t* x, const bf16_t* res, bf16_t* y, int M, int N, int K, hipStream_t stream,
                 bool narrow) {
    int ms = row_blocks(M);
    while (narrow && ms > 1 && (long)((N + 15) / 16) * ((M + 16 * ms - 1) / (16 * ms)) < 256) ms /= 2;
    switch (ms) {
        case 1: launch_gemm_ms<NWV, 1>(epi, W, x, res, y, M, N, K, stream); break;
        case 2: launch_gemm_ms<NWV, 2>(epi, W, x, res, y, M, N, K, stream); break;
        default: launch_gemm_ms<NWV, 4>(epi, W, x, res, y, M, N, K, stream);
    }
}


}  // namespace

extern "C" {

// y [M, K] bf16 = rms prologue of x [M, K] bf16 with weight nw [K] bf16.  K a multiple of 8.
int qt_rms_rows(const void* x, const void* nw, void* y, int M, int K, float eps, hipStream_t stream) {
    if (M < 0 || K < 8 || (K & 7)) return QT_ERR_DIM;
    if (M == 0) return QT_OK;                                     // nothing to do: empty buffers may be null
    if (!x || !nw || !y) return QT_ERR_NULL;
    for (const void* p : {x, nw, (const void*)y})
        if (reinterpret_cast<uintptr_t>(p) & 15u) return QT_ERR_ALIGN;
    hipLaunchKernelGGL(rms_rows_kernel, dim3((M + 3) / 4), dim3(256), 0, stream, (const bf16_t*)x, (const bf16_t*)nw, (bf16_t*)y, M, K, eps);
    QT_CHECK_LAUNCH();
    return QT_OK;
}

static int check_gemv(const gemv_args& p) {
    if (p.epi < 0 || p.epi > 2) return QT_ERR_UNSUPPORTED;
    if (p.M < 0 || p.N < 1 || p.K < 256 || (p.K % 256) || (p.epi == EPI_SWIGLU && (p.N & 1))) return QT_ERR_DIM;
    if (p.M == 0) return QT_OK;                                   // nothing to do: empty buffers may be null
    if (!p.W || !p.x || !p.y || (p.epi == EPI_ADD && !p.res)) return QT_ERR_NULL;
    for (const void* v : {p.W, p.x, p.nw})
        if (reinterpret_cast<uintptr_t>(v) & 15u) return QT_ERR_ALIGN;
    return QT_OK;
}

// y = epilogue(W [N, K] . x [M, K]^T): epilogue 0 none (y [M, N]), 1 add (res [M, N], y [M, N]), 2 swiglu (y [M, N / 2], N even).
// K a multiple of 256.
int qt_fused_gemv(const void* W, const void* x, const void* res, void* y, int M, int N, int K, int epilogue, hipStream_t stream) {
    const gemv_args p{(const bf16_t*)W, (const bf16_t*)x, nullptr, (const bf16_t*)res, (bf16_t*)y, M, N, K, epilogue, 0.f, stream};
    const int rc = check_gemv(p);
    if (rc != QT_OK || M == 0) return rc;
    const int cus = cu_count();
    if (rows_shape(p)) {
        launch_rows_any<false>(p, cus);
        QT_CHECK_LAUNCH();
        return QT_OK;
    }
    if (launch_quad_any(p, cus)) {
        QT_CHECK_LAUNCH();
        return QT_OK;
    }
    // wavefronts per workgroup: 4 when the output is wide enough to fill the chip with workgroups; 16 or 8 (as K divides) for
    // the narrow outputs, whose few workgroups would otherwise walk long K chains
    const int kc = K / 32;
    const bool wide = (long)((N + 15) / 16) * ((M + MT - 1) / MT) >= 512;
    if (!wide && kc % (2 * 16) == 0)
        launch_gemm<16>(epilogue, p.W, p.x, p.res, p.y, M, N, K, stream, true);
    else if (!wide && kc % (2 * 8) == 0)
        launch_gemm<8>(epilogue, p.W, p.x, p.res, p.y, M, N, K, stream, true);
    else
        launch_gemm<4>(epilogue, p.W, p.x, p.res, p.y, M, N, K, stream, !wide);
    QT_CHECK_LAUNCH();
    return QT_OK;
}

// qt_rms_rows and qt_fused_gemv in one launch, for the shapes where that is the faster form; -4 for the others (nothing launched).
int qt_fused_gemv_rms(const void* W, const void* x, const void* nw, float eps, const void* res, void* y, int M, int N, int K, int epilogue,
                      hipStream_t stream) {
    const gemv_args p{(const bf16_t*)W, (const bf16_t*)x, (const bf16_t*)nw, (const bf16_t*)res, (bf16_t*)y, M, N, K, epilogue, eps, stream};
    const int rc = check_gemv(p);
    if (rc != QT_OK || M == 0) return rc;
    if (!nw) return QT_ERR_NULL;
    if (!rows_shape(p) || M > RMS_ROWS_MAX) return QT_ERR_UNSUPPORTED;
    if (!launch_rows_any<true>(p, cu_count())) return QT_ERR_UNSUPPORTED;
    QT_CHECK_LAUNCH();
    return QT_OK;
}

}  // extern "C"
