// Causal prefill attention, 8 query heads on 2 KV heads, head dim 256, for gfx950 (flash-attention forward on bf16 MFMA).
// Replaces the call mx.fast.scaled_dot_product_attention(q, K[:, :, :kv_len], V[:, :, :kv_len], scale=256**-0.5,
// mask="causal") of the reference's full-attention layers (qwen35/model.py:160-167, qwen35/prefill.py:468).
//
// attn_prefill_kernel<NH>: one workgroup = 16 NH query rows x the 4 query heads that share a KV head, on eight wavefronts in
// two roles; NH = heads per pair of wavefronts:
//   NH = 2   32 rows; every K or V fragment read from LDS feeds two MFMAs (one per head): launches of about 1500 rows and more, fewer behind
//            a long prefix
//   NH = 1   16 rows: twice the workgroups (and twice the LDS traffic per MFMA), for launches that would leave CUs idle
// The arithmetic, per 64-key tile and 16 rows of a head:
//     S^T[keys x rows] = K_tile . Q^T     A = K rows from LDS, B = Q^T resident in registers (16x16x32 bf16 MFMA)
//     online softmax in the accumulator layout: lane (row n, group g) holds keys 4g..4g+3 of each 16-key sub-tile
//     O^T[256 x rows] += V^T . P^T        A = V^T through the transposing LDS load (4 consecutive keys of one column),
//                                         B = two exponentiated S^T accumulators packed to bf16 (they ARE the B operand
//                                         when a 32-key block is enumerated as 16 (j >> 2) + 4 g + (j & 3));
//                                         the row sums are one more product, 1 . P^T: every element is the row's sum.
//                                         A lane then holds one row, eight adjacent columns in two blocks: 16-byte stores
// K / V tiles travel HBM -> LDS directly (global_load_lds_dwordx4: 64 lanes x 16 bytes land as one contiguous KiB, no
// registers in between) into double-buffered tiles.  The LDS rows are unpadded (a direct load cannot pad); instead the
// 16-byte chunks of row r are stored XOR-swizzled by r & 15 (the loading lane picks the matching global chunk), which keeps
// the fragment reads of 16 rows on distinct banks.  The tile loop runs around one workgroup barrier per tile: the score MFMAs
// of tile t + 1 follow the exponentials of tile t, which are taken against the running reference points before the tile's
// row maxima are known; the bet is checked afterwards (see `publish` below).
#include "qt_common.h"

#include <algorithm>
#include <type_traits>

using namespace qt;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr float SCALE_LOG2E = 0.0625f * 1.4426950408889634f;   // 256^-0.5 log2 e: scores are exponentiated in base 2
constexpr float NEG = -3.0e38f;
constexpr float LAZY = 8.0f;            // log2 of the growth of a row maximum that is tolerated before the row is rescaled
constexpr int KT = 64;                 // keys per tile
constexpr int FRAG_AHEAD = 5;          // steps between the LDS read of a K fragment and its MFMAs in the tile loop
constexpr int V_FRAG_AHEAD = 2;        // 16-column blocks between the LDS reads of V fragments and their MFMAs
constexpr int TILE = KT * AD;          // elements of one K or V tile in LDS (32 KiB), rows unpadded, chunks swizzled

// PHASE_FENCE(): the phases of an iteration are scheduled separately
#define PHASE_FENCE() __builtin_amdgcn_sched_barrier(0)

// One direct-to-LDS load of 16 bytes per lane (global_load_lds_dwordx4): lane l fetches base + voff + IMM and the 64 pieces land
// at lds + IMM + 16 l.  Issued as inline assembly, not through the builtin: while a direct-to-LDS load that the compiler knows
// of is outstanding, it closes every wait for an LDS read with lgkmcnt(0) (the load counts as an access of both memories), and
// the tile loop below always has such loads in flight, so each of its fragment reads would be waited for in full.  These loads
// are waited for by hand (vmcnt(0) before the workgroup barrier of a tile).  base and lds are wavefront-uniform.
// LDS byte address of a __shared__ array, taken of the array itself: a constant.  (Taken of a pointer that has been moved, the
// cast from a generic pointer costs a null test and two scalar registers per use.)
__device__ __forceinline__ unsigned lds_address(const bf16_t* shared_array) {
    return (unsigned)(size_t)(__attribute__((address_space(3))) const void*)shared_array;
}
template <int IMM>
__device__ __forceinline__ void lds_dma16(const char* base, unsigned voff, unsigned lds) {
    const unsigned la = __builtin_amdgcn_readfirstlane(lds);
    unsigned keep;                                                // M0 belongs to the compiler: put back what it held
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%4\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(voff), "s"(base), "s"(la), "n"(IMM)
                 : "memory");
}
// four such loads, KiB 0 .. 3 behind lds, under one setting of M0 (a wavefront issues one instruction every four clocks, and
// the tile loop is bound by exactly that, so the five scalar instructions around a single load count)
__device__ __forceinline__ void lds_dma16x4(const char* base, unsigned v0, unsigned v1, unsigned v2, unsigned v3, unsigned lds) {
    const unsigned la = __builtin_amdgcn_readfirstlane(lds);
    unsigned keep;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %6\n\ts_nop 0\n\t"
                 "global_load_lds_dwordx4 %1, %5\n\tglobal_load_lds_dwordx4 %2, %5 offset:1024\n\t"
                 "global_load_lds_dwordx4 %3, %5 offset:2048\n\tglobal_load_lds_dwordx4 %4, %5 offset:3072\n\ts_mov_b32 m0, %0"
                 : "=&s"(keep)
                 : "v"(v0), "v"(v1), "v"(v2), "v"(v3), "s"(base), "s"(la)
                 : "memory");
}

// max over the four lanes n, n + 16, n + 32, n + 48 with the VALU lane swaps of gfx950 (v_permlane32_swap exchanges the upper half
// of one register with the lower half of the other, v_permlane16_swap the odd 16-lane rows of one with the even rows of the
// other), which keeps the softmax free of LDS traffic
__device__ __forceinline__ float max_over_groups(float x) {
    const unsigned xi = __float_as_uint(x);
    const auto a = __builtin_amdgcn_permlane32_swap(xi, xi, false, false);
    const unsigned mi = __float_as_uint(fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
    const auto b = __builtin_amdgcn_permlane16_swap(mi, mi, false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// max(|a|, |b|, c), a NaN among them left out (as one instruction: fmaxf first makes a copy of everything that may be a signalling NaN).
// The compiler counts no wait states between an MFMA and inline assembly that reads its result: mfma_results_settle() comes before.
__device__ __forceinline__ void mfma_results_settle() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }
__device__ __forceinline__ float max3_abs(float a, float b, float c) {
    asm volatile("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(c) : "v"(a), "v"(b));
    return c;
}

// Key split.  A causal launch with few workgroups is as slow as its longest row block, twice the average.  With tmax > 0 the
// tiles of a row block (RB = 16 or 32 rows) are cut into parts of tmax tiles, one workgroup per part; a block with more than
// one part leaves unnormalised partial results (O, reference point m, row sums l) in the workspace and
// attn_prefill_merge_kernel combines them.  Block i counts ceil((p + i + 1) / c) parts, p = ceil(q_pos0 / RB),
// c = (64 / RB) tmax (RB rows advance the visible keys by RB / 64 of a tile), which is never fewer than its tiles need (a part
// may be empty); the parts of blocks 0 .. r-1 are then parts_upto(p + r, c) - parts_upto(p, c), and a workgroup inverts that
// sum to find its part.
__host__ __device__ inline long parts_upto(long n, long c) {      // sum over j = 1 .. n of ceil(j / c)
    const long k = n / c;
    return c * (k * (k + 1) / 2) + (n - k * c) * (k + 1);
}
// elements of one part's O, [4 heads][RB rows][256] in single (`wide`) or half precision, and floats of its m, l, [4 heads][m | l][RB
// rows] (RB = rows of a block: 16 or 32).  Half precision: so that a V of any size survives, each row of O is stored times the power of two that brings its largest value
// to 2^13 .. 2^14.  The exponent of that power takes the place of the low eight bits of m (tagged_m); what this adds to m is taken out
// of O and l again.  Where m is 2^14 or more its low bits count: there O is stored divided by l instead, weighted means of V.
// (333 rows on 1500 keys 18.8 us, 2048 rows 33.9; without the scaling 18.6 and 33.8; the exponent in an array of its own 19.5 and 34.4; O in
// single precision 22.8 and 36.3.)
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
constexpr int part_o_size(int RB) { return 4 * RB * AD; }
constexpr int part_ml_floats(int RB) { return 4 * 2 * RB; }
constexpr long part_bytes(int RB, bool wide) { return (long)part_o_size(RB) * (wide ? 4 : 2) + (long)part_ml_floats(RB) * 4; }
constexpr float TAG_BELOW = 16384.f;
__device__ __forceinline__ float tagged_m(float m, int e) { return __uint_as_float((__float_as_uint(m) & ~255u) | (unsigned)e); }
// what a part's O is multiplied by in the merge, besides its factor 2^(m - reference)
template <class PT>
__device__ __forceinline__ float part_unit(float m, float l) {
    if (sizeof(PT) == 4) return 1.f;
    return fabsf(m) < TAG_BELOW ? __uint_as_float((254 - (__float_as_uint(m) & 255u)) << 23) : l;
}

// a word of LDS as a volatile object in the LDS address space (through a generic pointer, a volatile access is a flat
// instruction, which is also counted, and waited for, as an access of global memory)
__device__ __forceinline__ volatile __attribute__((address_space(3))) int* lds_word(int* shared_word) {
    return (volatile __attribute__((address_space(3))) int*)shared_word;
}

// The tile loop, with the two halves of a tile's work on different wavefronts.  The eight wavefronts of a workgroup, two per
// SIMD, form four pairs: wavefront pr (0 .. 3, the "score" wavefront of pair pr) computes the scores and the softmax of the
// pair's 16 rows x NH heads (NH = 2: rows 16 (pr >> 1) .. + 16 of the block, heads 2 (pr & 1), + 1; NH = 1: the block's 16 rows,
// head pr), and wavefront 4 + pr (the pair's "output" wavefront) multiplies the resulting P by V, one tile behind.  A
// wavefront's instructions issue one after the other (an MFMA holds its wavefront for about as long as it holds the matrix
// unit, and every LDS read, exponential or wait comes on top), while two wavefronts of a SIMD do overlap: one feeds the unit
// Q K^T while the other reads V fragments, and the softmax arithmetic of the one runs beside the P V MFMAs of the other.
// (The whole loop on one wavefront per SIMD, four per workgroup, measured 5 - 12 % slower on the same rows and heads; the
// compiler's order within the score wavefront, the softmax arithmetic as one block and then the MFMA steps back to back,
// measures better than the same arithmetic tied into the steps.)  With eight wavefronts the 512 registers of a SIMD lane are
// split in two, 256 per wavefront and no separate accumulation half: for NH = 2 the score side holds Q^T (64 registers) and
// two tiles of scores (64), the output side O (128).
//     iteration t (after barrier X(t): K(t + 1) and V(t - 1) are in LDS):
//         score wavefront:  softmax of tile t (its scores are in registers since iteration t - 1) and the score MFMAs of
//                           tile t + 1; then P(t), as packed B operands, and the rows' rescale factors go to LDS
//         output wavefront: takes P(t - 1) and the factors from LDS, rescales O and the row sums if any row's reference
//                           moved, O += P(t - 1) V(t - 1)
//         all eight:        direct-to-LDS loads of K(t + 2) into K(t)'s buffer and of V(t) into V(t - 2)'s
// P has one buffer per pair: the output wavefront reads it into registers first thing in an iteration and says so
// (taken_s[pr] = t), and the score wavefront, which writes the next P a few thousand clocks later, looks at that word first.
// grid = (row blocks, or parts when tmax > 0) x KV heads in one dimension, the KV head varying fastest: workgroups are
// dispatched in the order of their index, so both heads' long row blocks come first.
// PT: what O of a part is kept in, _Float16 or float.
template <int NH, class PT>
__global__ __launch_bounds__(512) void attn_prefill_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ K,
                                                              const bf16_t* __restrict__ V, bf16_t* __restrict__ out, int S, int L,
                                                              int q_pos0, long q_head_stride, int q_row_stride, long kv_head_stride, int tmax,
                                                              PT* __restrict__ part_o, float* __restrict__ part_ml) {
    __shared__ __align__(1024) bf16_t kv_s[4 * TILE];            // K tiles of even / odd iterations, then the V tiles
    __shared__ __align__(16) u32x4 p_s[4][NH][2][64];             // [pair][head][32-key half][lane]: P as the lanes hold it
    __shared__ __align__(16) float c_s[4][NH][16];               // [pair][head][row]: factor of a row whose reference moved
    __shared__ float m_s[4][NH][16];                             // final reference points (only the parts' epilogue needs them)
    __shared__ int moved_s[4];                                   // pair: did any reference move in the tile whose P lies in p_s
    __shared__ int taken_s[4];                                   // pair: the iteration in which p_s / c_s / moved_s were last read
    constexpr int RB = 16 * NH;
    const int nitems = gridDim.x / AKV, item = blockIdx.x / AKV;
    int rb = nitems - 1 - item;                                  // long rows first
    int part = 0, nparts = 1;
    if (tmax > 0) {                                              // items are parts, again from the long end
        const int c = (KT / RB) * tmax, p = (q_pos0 + RB - 1) / RB;
        const long y = (long)rb + parts_upto(p, c);              // parts_upto(nn) <= y < parts_upto(nn + 1), nn = p + row block
        int k = 0;
        while ((long)c * ((k + 1) * (k + 2) / 2) <= y) k++;
        const int nn = k * c + (int)((y - (long)c * (k * (k + 1) / 2)) / (k + 1));
        part = (int)(y - parts_upto(nn, c));
        nparts = k + 1;
        rb = nn - p;
    }
    const int kvh = blockIdx.x % AKV;
    const size_t slot = (size_t)kvh * nitems + (nitems - 1 - item);     // parts of a block: consecutive slots
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int pr = w & 3;                                        // pair; w >> 2: 0 = score, 1 = output wavefront
    const int hq0 = NH == 2 ? 2 * (pr & 1) : pr;                  // this pair's first head within the KV group
    const int h0 = kvh * (AH / AKV) + hq0;
    const int r0 = rb * RB + (NH == 2 ? 16 * (pr >> 1) : 0), row = r0 + n;
    const bool row_ok = row < S;
    const int my_last = q_pos0 + row;                            // last key this query row may see
    const int kend = min(L, q_pos0 + min(rb * RB + RB - 1, S - 1) + 1);        // keys any row of the workgroup sees
    const int ntiles = (kend + KT - 1) / KT;
    const int kend_w = r0 < S ? min(L, q_pos0 + min(r0 + 15, S - 1) + 1) : 0;  // keys any row of this pair sees
    const int ntiles_w = (kend_w + KT - 1) / KT;
    // this workgroup's tiles [ta, tb); tw: where this pair's rows end (the upper rows of a block may see one tile more)
    const int ta = part * tmax, tb = tmax > 0 ? min(ntiles, ta + tmax) : ntiles;
    const int tw = min(ntiles_w, tb);

    // tile loader: wavefront w issues four direct-to-LDS loads of K and four of V per tile; load i fills rows 8 w + 2 i, + 1
    // (one KiB): lane l lands at chunk position l & 31 of row 8 w + 2 i + (l >> 5) and fetches chunk (l & 31) ^ (row & 15).  The
    // per-lane byte offsets within a tile do not change from tile to tile: load i differs from load 0 by 2 i rows, which go into
    // the instruction's immediate offset (it moves the global address and the LDS destination alike), and by an XOR of the
    // chunk with 2 i.  A tile that would run past the end of the sequence is shifted back to end at L (tile_row0): its first
    // rows repeat keys of the tile before and are masked.  Only a sequence shorter than one tile repeats its last key instead.
    const char* kg = reinterpret_cast<const char*>(K + (size_t)kvh * kv_head_stride);
    const char* vg = reinterpret_cast<const char*>(V + (size_t)kvh * kv_head_stride);
    const unsigned ld_row0 = 8u * w + (lane >> 5);
    const unsigned ld_off0 = ld_row0 * (AD * 2) + ((unsigned)((lane & 31) ^ (ld_row0 & 15u)) << 4);
    auto tile_row0 = [&](int t) { return max(0, min(t * KT, L - KT)); };
    // a copy of ld_off0 the compiler cannot see through: the offsets of the four loads are then recomputed where they are
    // used (one XOR each) instead of living in registers through the loop
    auto opaque_off0 = [&]() {
        unsigned off0 = ld_off0;
        asm volatile("" : "+v"(off0));
        return off0;
    };
    const unsigned w_lds = 4096u * w;                            // this wavefront's 4 KiB of a tile buffer
    auto load_four = [&](const char* src, unsigned dst, int t, unsigned off0) {
        if (L >= KT) {
            const char* base = src + (size_t)tile_row0(t) * (AD * 2);
            lds_dma16x4(base, off0, off0 ^ 32u, off0 ^ 64u, off0 ^ 96u, dst + w_lds);
        } else {                                                 // t = 0: rows past the end repeat the last key; they are masked
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const unsigned o = (ld_off0 ^ (32u * i)) + 1024u * i;
                lds_dma16<0>(src, (unsigned)min((int)(o >> 9), L - 1) * (AD * 2) + (o & 511u), dst + w_lds + 1024u * i);
            }
        }
    };
    // A operand of the scores: row 16 kt + n of the tile, chunk (4 kb + g) ^ n
    const int ka_row = n * AD;
    // transposing load: within 16 lanes, lane 4q + i receives element i of the 8-byte chunks addressed by lanes q, q+4,
    // q+8, q+12; lane n of group g points at key 4g + n/4, columns 4 (n%4).. of the block and receives keys 4g..4g+3 of column n
    // Blocks j and j + 1 (j even) share 32 columns: the four lanes of a key take a 16-byte chunk each, and block j the lower half of it in the
    // even and the upper half in the odd lanes, block j + 1 the other halves.  Afterwards lane group g holds eight adjacent columns in its
    // two blocks (16-byte stores), and a fragment read still touches every bank twice.
    const int vrow = 4 * g + (n >> 2);                           // row within a 16-key block = its swizzle
    const int vq = n & 3;
    // byte offsets of the lane's reads of blocks j and j + 8 in a tile: one value each, which the compiler would form again in every tile, two
    // adds and a shift ahead of the first read (0.5 % of a pass over 8192 rows)
    int va_off[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        va_off[j] = 2 * (vrow * AD + (((4 * (j >> 1) + vq) ^ vrow) << 3) + 4 * ((vq ^ j) & 1));
        asm("" : "+v"(va_off[j]));
    }
    // K fragment kb of sub-tile kt: chunk (4 kb + g) ^ n; n < 16 leaves bit 4 alone, so fragments kb and kb + 4 share an
    // address register
    auto k_frag = [&](const bf16_t* ka, int kt, int kb) {
        return *reinterpret_cast<const bf16x8*>(ka + 16 * kt * AD + (((4 * (kb & 3) + g) ^ n) << 3) + 128 * (kb >> 2));
    };

    if (tid < 4) taken_s[tid] = -1, moved_s[tid] = 0;
    if (tid < 4 * NH * 16) (&m_s[0][0][0])[tid] = NEG;
    bf16_t* const q_s = kv_s + 2 * TILE;                         // Q waits in the V buffers, [pair][head][16 rows][256], swizzled as the tiles
    if (ta < tb) {                                               // (a part past the block's last tile is empty)
        load_four(kg, lds_address(kv_s), ta, ld_off0);
        // Q goes through LDS as well, whole rows per load: as the score wavefronts' operand it would be asked for 16 bytes of 16 rows at a
        // time, which a CU takes in at a quarter of the rate (1.2 us of a workgroup with 32 rows).  Rows past the end repeat the last one.
#pragma unroll
        for (int i = 0; i < 4 * NH; i++) {
            const int piece = 4 * NH * w + i, qp = piece / (8 * NH), qh = piece / 8 % NH, rr = 2 * (piece & 7) + (lane >> 5);
            const int qrow = min(rb * RB + (NH == 2 ? 16 * (qp >> 1) : 0) + rr, S - 1), head = kvh * (AH / AKV) + (NH == 2 ? 2 * (qp & 1) + qh : qp);
            lds_dma16_from(reinterpret_cast<const char*>(q + (size_t)head * q_head_stride + (size_t)qrow * q_row_stride + 8 * ((lane & 31) ^ rr)),
                           lds_address(kv_s) + 4 * TILE + 1024 * piece);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tb - ta > 1) load_four(kg, lds_address(kv_s) + 2 * TILE, ta + 1, ld_off0);
    }

    if (w < 4) {
        // ------------------------------------------------------------------------------------------ score wavefront
        if (ta >= tb) return;
        // Q^T as the B operand of the score MFMA: lane (row n, group g) holds q[row][32 kb + 8 g .. + 8] of each head
        bf16x8 bq[NH][8];
#pragma unroll
        for (int hh = 0; hh < NH; hh++)
#pragma unroll
            for (int kb = 0; kb < 8; kb++) bq[hh][kb] = k_frag(q_s + (pr * NH + hh) * 16 * AD + ka_row, 0, kb);
        float m_run[NH];
#pragma unroll
        for (int hh = 0; hh < NH; hh++) m_run[hh] = NEG;
        // scores of the first tile, S^T = K_tile . Q^T: each K fragment multiplies the Q^T of every head of the pair; the fragments
        // of the next 16-key sub-tile are read while the MFMAs of the current one run
        auto first_scores = [&](f32x4 (&acc0)[NH][4]) {
            const bf16_t* ka = kv_s + ka_row;
            bf16x8 Af[2][8];
#pragma unroll
            for (int kb = 0; kb < 8; kb++) Af[0][kb] = k_frag(ka, 0, kb);
#pragma unroll
            for (int kt = 0; kt < 4; kt++) {
                __builtin_amdgcn_sched_barrier(0);
                if (kt < 3) {
#pragma unroll
                    for (int kb = 0; kb < 8; kb++) Af[(kt + 1) & 1][kb] = k_frag(ka, kt + 1, kb);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int hh = 0; hh < NH; hh++) acc0[hh][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kb = 0; kb < 8; kb++)
#pragma unroll
                    for (int hh = 0; hh < NH; hh++)
                        acc0[hh][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Af[kt & 1][kb], bq[hh][kb], acc0[hh][kt], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // the scores of tile t live in accs[(t - ta) & 1]: two iterations in the source, so that both sets are registers
        f32x4 accs[2][NH][4] = {};
        if (tw > ta) first_scores(accs[0]);
        auto s_iter = [&](const int t, f32x4 (&acc)[NH][4], f32x4 (&acc_next)[NH][4]) {
            const unsigned par = (unsigned)(t - ta) & 1u;
            const unsigned k_cur = lds_address(kv_s) + par * (2 * TILE);           // K(t): consumed, refilled with K(t + 2)
            const bf16_t* const k_nxt = kv_s + (par ^ 1u) * TILE;                  // K(t + 1)
            const unsigned v_new = lds_address(kv_s) + 4 * TILE + par * (2 * TILE);   // takes V(t)
            PHASE_FENCE();
            // this wavefront's loads of K(t + 1), V(t - 1) have landed, and its writes of P(t - 1) (the wait for those is
            // spelled out: at a loop header the compiler does not always see the LDS stores that arrive over the back edge)
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            PHASE_FENCE();
            __syncthreads();                                         // X(t)
            // While scores of a further tile are due (then L > KT), this wavefront's loads of K(t + 2) and V(t) ride on the steps
            // below: a burst would stall on the memory pipeline's queue.  There a tile index past the end loads the last tile
            // again, harmlessly: nothing reads that buffer any more.
            const bool more = t + 1 < tw;                            // wavefront-uniform
            const int tk = min(t + 2, tb - 1);
            if (!more) {
                if (t + 2 < tb) load_four(kg, k_cur, t + 2, opaque_off0());
                if (t < tb) load_four(vg, v_new, t, opaque_off0());
            }
            PHASE_FENCE();
            if (t >= tw) return;
            // only tiles that touch the diagonal or the end of the sequence need the mask (wavefront-uniform)
            if (t * KT + KT - 1 > q_pos0 + r0 || t * KT + KT > L) {
#pragma unroll
                for (int hh = 0; hh < NH; hh++)
#pragma unroll
                    for (int kt = 0; kt < 4; kt++)
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const int key = tile_row0(t) + 16 * kt + 4 * g + i;     // a shifted tile repeats keys below t * KT
                            if (!(key >= t * KT && key <= my_last && key < L)) acc[hh][kt][i] = NEG;
                        }
            }
            const bf16_t* ka = k_nxt + ka_row;
            // Online softmax in base 2 on the raw products: p = 2^(c s - m), c = 256^-0.5 log2 e; every row sees key 0, so its
            // maximum is finite from the first tile on and masked entries come out as 2^-huge = 0.  The exponentials are taken
            // against the running reference point of each row at once, on the bet that no row's maximum grows by more than
            // 2^LAZY in this tile (true for all but the first few tiles of a row block); the maxima are folded in beside them
            // and the bet is checked here.  A reference point only moves when the row's maximum has grown by more than 2^LAZY:
            // until then p stays below 2^LAZY, which bf16 and the f32 sums hold as well as values below 1.
            auto publish = [&](s16x8 (&P)[NH][2], float (&mx)[NH], int taken_early) {
                bool grow = false;
#pragma unroll
                for (int hh = 0; hh < NH; hh++) {
                    mx[hh] = max_over_groups(mx[hh]) * SCALE_LOG2E;
                    grow |= mx[hh] > m_run[hh] + LAZY;
                }
                const bool any_grow = __any(grow);
                float corr[NH];
#pragma unroll
                for (int hh = 0; hh < NH; hh++) corr[hh] = 1.f;
                if (any_grow) {                                      // wavefront-uniform and rare
#pragma unroll
                    for (int hh = 0; hh < NH; hh++) {
                        const float m_new = mx[hh] > m_run[hh] + LAZY ? mx[hh] : m_run[hh];
                        corr[hh] = __builtin_amdgcn_exp2f(m_run[hh] - m_new);    // m_run = NEG initially: 2^-huge = 0
                        m_run[hh] = m_new;
                        // this tile's p again, against the new reference points (rows that did not move get the same bits)
#pragma unroll
                        for (int kt2 = 0; kt2 < 4; kt2++)
#pragma unroll
                            for (int i = 0; i < 4; i += 2) {
                                const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(acc[hh][kt2][i], SCALE_LOG2E, -m_new));
                                const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(acc[hh][kt2][i + 1], SCALE_LOG2E, -m_new));
                                const uint32_t pk = pack_bf(p0, p1);
                                P[hh][kt2 >> 1][(kt2 & 1) * 4 + i] = (short)(pk & 0xffff);
                                P[hh][kt2 >> 1][(kt2 & 1) * 4 + i + 1] = (short)(pk >> 16);
                            }
                    }
                }
                // the pair's buffers are free once the output wavefront has read tile t - 1 out of them (it does so first
                // thing in this iteration; the word was read some steps ago, so that its LDS latency is not waited for here).
                // The wait is bounded (the word is always written, and a bound costs nothing); a wait that does run out must not
                // pass in silence: the pair's rows are then rescaled by NaN, which every later stage carries to the output.
                bool gave_up = false;
                if (t > ta && __builtin_amdgcn_readfirstlane(taken_early) != t) {
                    gave_up = true;
                    for (int spin = 0; spin < (1 << 20); spin++) {
                        if (__builtin_amdgcn_readfirstlane(*lds_word(&taken_s[pr])) == t) {
                            gave_up = false;
                            break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                    }
                }
                asm volatile("" ::: "memory");
                if (any_grow || gave_up) {
#pragma unroll
                    for (int hh = 0; hh < NH; hh++)              // all four groups store the same value
                        c_s[pr][hh][n] = gave_up ? __builtin_nanf("") : corr[hh];
                }
                moved_s[pr] = any_grow || gave_up ? 1 : 0;
#pragma unroll
                for (int hh = 0; hh < NH; hh++)
#pragma unroll
                    for (int pp = 0; pp < 2; pp++) p_s[pr][hh][pp][lane] = __builtin_bit_cast(u32x4, P[hh][pp]);
                if (t == tw - 1) {
#pragma unroll
                    for (int hh = 0; hh < NH; hh++) m_s[pr][hh][n] = m_run[hh];
                }
            };
            auto body = [&](auto with_scores) {
                constexpr bool SC = decltype(with_scores)::value;
                s16x8 P[NH][2];
                float mx[NH];
#pragma unroll
                for (int hh = 0; hh < NH; hh++) mx[hh] = NEG;
                bf16x8 Af[FRAG_AHEAD + 1];
                if (SC) {
#pragma unroll
                    for (int f = 0; f < FRAG_AHEAD; f++) Af[f] = k_frag(ka, f >> 3, f & 7);
                }
                // softmax elements 2 e, 2 e + 1 of tile t
                auto softmax_pair = [&](int e) {
                    const int hh = e >> 3, kt2 = (e >> 1) & 3, i = 2 * (e & 1);
                    const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(acc[hh][kt2][i], SCALE_LOG2E, -m_run[hh]));
                    const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(acc[hh][kt2][i + 1], SCALE_LOG2E, -m_run[hh]));
                    mx[hh] = fmaxf(mx[hh], fmaxf(acc[hh][kt2][i], acc[hh][kt2][i + 1]));
                    const uint32_t pk = pack_bf(p0, p1);
                    P[hh][kt2 >> 1][(kt2 & 1) * 4 + i] = (short)(pk & 0xffff);
                    P[hh][kt2 >> 1][(kt2 & 1) * 4 + i + 1] = (short)(pk >> 16);
                };
                PHASE_FENCE();
                const unsigned step_off0 = SC ? opaque_off0() : 0u;
                int taken_early = -1;
                // 32 steps: one K fragment read (FRAG_AHEAD steps ahead, a ring) and its MFMAs, one per head.  The softmax
                // pairs are written beside them, but nothing ties them to their step: the compiler gathers the arithmetic
                // into one block beside the steps, which measures better than the same arithmetic held between the MFMAs.
#pragma unroll
                for (int st = 0; st < 32; st++) {
                    const int kt = st >> 3, kb = st & 7;
                    __builtin_amdgcn_sched_barrier(0);
                    if (SC && st == 0) load_four(kg, k_cur, tk, step_off0);
                    if (SC && st == 20) load_four(vg, v_new, t, step_off0);
                    if (SC) {
                        if (st + FRAG_AHEAD < 32)
                            Af[(st + FRAG_AHEAD) % (FRAG_AHEAD + 1)] = k_frag(ka, (st + FRAG_AHEAD) >> 3, (st + FRAG_AHEAD) & 7);
#pragma unroll
                        for (int hh = 0; hh < NH; hh++)
                            acc_next[hh][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                Af[st % (FRAG_AHEAD + 1)], bq[hh][kb], kb == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc_next[hh][kt], 0, 0, 0);
                    }
                    if (st % (4 / NH) == 0) softmax_pair(st / (4 / NH));       // 8 NH pairs over the 32 steps
                    if (st == 20) taken_early = *lds_word(&taken_s[pr]);   // (read early: its LDS latency passes under the steps)
                }
                __builtin_amdgcn_sched_barrier(0);
                publish(P, mx, taken_early);
            };
            if (more)
                body(std::true_type{});
            else
                body(std::false_type{});
            PHASE_FENCE();
        };
        for (int t = ta; t <= tb; t += 2) {
            s_iter(t, accs[0], accs[1]);
            if (t + 1 <= tb) s_iter(t + 1, accs[1], accs[0]);
        }
        return;
    }
    // ---------------------------------------------------------------------------------------------- output wavefront
    // O^T: lane (n, g) holds row n of the pair's rows, columns 32 jj + 8 g .. + 7 in blocks 2 jj and 2 jj + 1 (odd g: the halves change places);
    // every element of Lsum is row n's sum
    f32x4 O[NH][16];
    f32x4 Lsum[NH];                                                  // row sums of P, accumulated by MFMA against a block of ones
#pragma unroll
    for (int hh = 0; hh < NH; hh++) {
        Lsum[hh] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 16; j++) O[hh][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // iterations in which this wavefront only loads: the first one (no P yet), and those after its rows' last tile
    auto idle_iter = [&](int t) {
        const unsigned par = (unsigned)(t - ta) & 1u;
        PHASE_FENCE();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        PHASE_FENCE();
        __syncthreads();                                             // X(t)
        if (t + 2 < tb) load_four(kg, lds_address(kv_s) + par * (2 * TILE), t + 2, opaque_off0());
        if (t < tb) load_four(vg, lds_address(kv_s) + 4 * TILE + par * (2 * TILE), t, opaque_off0());
    };
    if (ta < tb) idle_iter(ta);
    for (int t = ta + 1; t <= tw; t++) {                             // (tw <= tb; nothing if tw <= ta)
        const unsigned par = (unsigned)(t - ta) & 1u;
        const unsigned k_cur = lds_address(kv_s) + par * (2 * TILE);               // takes K(t + 2)
        const unsigned v_new = lds_address(kv_s) + 4 * TILE + par * (2 * TILE);    // takes V(t)
        const bf16_t* const v_cur = kv_s + 2 * TILE + (par ^ 1u) * TILE;           // V(t - 1)
        PHASE_FENCE();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        PHASE_FENCE();
        __syncthreads();                                             // X(t)
        const int mv = __builtin_amdgcn_readfirstlane(moved_s[pr]);
        s16x8 P[NH][2];
#pragma unroll
        for (int hh = 0; hh < NH; hh++)
#pragma unroll
            for (int pp = 0; pp < 2; pp++) P[hh][pp] = __builtin_bit_cast(s16x8, p_s[pr][hh][pp][lane]);
        float cr[NH];
#pragma unroll
        for (int hh = 0; hh < NH; hh++) cr[hh] = mv ? c_s[pr][hh][n] : 1.f;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        *lds_word(&taken_s[pr]) = t;
        asm volatile("" ::: "memory");
        auto v_frag = [&](int j, int q4) {
            const char* at = reinterpret_cast<const char*>(v_cur) + va_off[j & 7] + 2 * ((16 * q4) * AD + 128 * (j >> 3));
            return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)const_cast<char*>(at));
        };
        s16x4 Bf[V_FRAG_AHEAD + 1][4];
#pragma unroll
        for (int j = 0; j < V_FRAG_AHEAD; j++)
#pragma unroll
            for (int q4 = 0; q4 < 4; q4++) Bf[j][q4] = v_frag(j, q4);
        if (mv) {                                                    // a reference moved: rescale what is accumulated
#pragma unroll
            for (int hh = 0; hh < NH; hh++) {
#pragma unroll
                for (int j = 0; j < 16; j++) O[hh][j] *= cr[hh];
                Lsum[hh] *= cr[hh];
            }
        }
        PHASE_FENCE();
        {                                                            // the row sums: 1 . P^T, the sum of exactly the rounded values
            s16x8 ones;
#pragma unroll
            for (int e = 0; e < 8; e++) ones[e] = (short)0x3f80;
#pragma unroll
            for (int pp = 0; pp < 2; pp++)
#pragma unroll
                for (int hh = 0; hh < NH; hh++)
                    Lsum[hh] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ones),
                                                                      __builtin_bit_cast(bf16x8, P[hh][pp]), Lsum[hh], 0, 0, 0);
        }
        const unsigned step_off0 = opaque_off0();
#pragma unroll
        for (int j = 0; j < 16; j++) {
            __builtin_amdgcn_sched_barrier(0);
            if (j == 0 && t + 2 < tb) load_four(kg, k_cur, t + 2, step_off0);
            if (j == 8 && t < tb) load_four(vg, v_new, t, step_off0);
            if (j + V_FRAG_AHEAD < 16) {
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) Bf[(j + V_FRAG_AHEAD) % (V_FRAG_AHEAD + 1)][q4] = v_frag(j + V_FRAG_AHEAD, q4);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int pp = 0; pp < 2; pp++) {
                const s16x8 B = __builtin_shufflevector(Bf[j % (V_FRAG_AHEAD + 1)][2 * pp], Bf[j % (V_FRAG_AHEAD + 1)][2 * pp + 1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int hh = 0; hh < NH; hh++)
                    O[hh][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, B),
                                                                      __builtin_bit_cast(bf16x8, P[hh][pp]), O[hh][j], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        PHASE_FENCE();
    }
    if (ta < tb)
        for (int t = max(tw, ta) + 1; t <= tb; t++) idle_iter(t);
    // ---- normalise and store: lane (n, g) holds row n, columns 32 jj + 8 g .. + 7 in blocks 2 jj and 2 jj + 1 (odd g: the other way round)
    auto columns = [&](const f32x4 (&o)[16], int jj, float scale, f32x4& lo, f32x4& hi) {
        const bool odd = g & 1;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float a = o[2 * jj][i] * scale, b = o[2 * jj + 1][i] * scale;
            lo[i] = odd ? b : a, hi[i] = odd ? a : b;
        }
    };
    if (nparts > 1) {
        // One part of several: leave the scaled O, m, l of this pair's heads.  A row that sees no key of this part (its
        // last key lies before the part's first) has exponentiated masked scores against a masked maximum: it is written as
        // the neutral element (m = NEG, l = 0, O = 0).
        constexpr bool HALF = sizeof(PT) == 2;
        const int lr = r0 - rb * RB + n;
        const bool seen = my_last >= ta * KT;
        if (HALF) mfma_results_settle();
#pragma unroll
        for (int hh = 0; hh < NH; hh++) {
            const int hq = hq0 + hh;
            PT* po = part_o + (slot * 4 + hq) * (RB * AD) + lr * AD + 8 * g;
            float* pml = part_ml + (slot * 4 + hq) * (2 * RB);
            const float m = m_s[pr][hh][n], l = Lsum[hh][0];
            float m_part = m, back = 1.f, up = 1.f;
            if constexpr (HALF) {
                // the row's largest finite |O|, over this lane's 64 columns and the three lanes with the others
                constexpr float FINITE = 3.4028234e38f;
                float tops[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 16; j += 2)
#pragma unroll
                    for (int i = 0; i < 4; i++) tops[i] = max3_abs(O[hh][j][i], O[hh][j + 1][i], tops[i]);
                float top = max3_abs(tops[0], tops[1], max3_abs(tops[2], tops[3], 0.f));
                if (__any(top > FINITE)) {                       // (an infinite V: its columns are infinite, the others keep their values)
                    top = 0.f;
#pragma unroll
                    for (int j = 0; j < 16; j++)
#pragma unroll
                        for (int i = 0; i < 4; i++) top = fmaxf(top, fabsf(O[hh][j][i]) <= FINITE ? fabsf(O[hh][j][i]) : 0.f);
                }
                const int up_e = min(267 - (int)(__float_as_uint(max_over_groups(top)) >> 23), 253);   // exponent field of the power of two, 13 or more
                const bool tag = fabsf(m) < TAG_BELOW;
                m_part = tag ? tagged_m(m, up_e) : m;
                back = tag ? __builtin_amdgcn_exp2f(m - m_part) : 1.f;                                 // 2^-1/4 .. 2^1/4
                up = tag ? __uint_as_float((unsigned)up_e << 23) * back : 1.0f / l;
            }
#pragma unroll
            for (int jj = 0; jj < 8; jj++) {
                f32x4 lo, hi;
                columns(O[hh], jj, up, lo, hi);
#pragma unroll
                for (int i = 0; i < 4; i++) lo[i] = seen ? lo[i] : 0.f, hi[i] = seen ? hi[i] : 0.f;
                if constexpr (HALF) {
                    half8 h;
#pragma unroll
                    for (int i = 0; i < 4; i++) h[i] = (_Float16)lo[i], h[4 + i] = (_Float16)hi[i];
                    *reinterpret_cast<half8*>(po + 32 * jj) = h;
                } else {
                    reinterpret_cast<f32x4*>(po + 32 * jj)[0] = lo;
                    reinterpret_cast<f32x4*>(po + 32 * jj)[1] = hi;
                }
            }
            if (g == 0) {
                pml[RB + lr] = seen ? l * back : 0.f;
                pml[lr] = seen ? m_part : NEG;
            }
        }
        return;
    }
    // Sixteen-row blocks compute the rows past the end too and leave out their stores alone: with the lanes of one or two rows these instructions
    // took 1.2 us instead of 0.4 (time stamps).
    if (NH == 2 && !row_ok) return;
#pragma unroll
    for (int hh = 0; hh < NH; hh++) {
        const float inv = 1.0f / Lsum[hh][0];
        bf16_t* dst = out + (size_t)(h0 + hh) * q_head_stride + (size_t)row * q_row_stride + 8 * g;
#pragma unroll
        for (int jj = 0; jj < 8; jj++) {
            f32x4 lo, hi;
            columns(O[hh], jj, inv, lo, hi);
            u32x4 pk = u32x4{pack2_bf(lo[0], lo[1]), pack2_bf(lo[2], lo[3]), pack2_bf(hi[0], hi[1]), pack2_bf(hi[2], hi[3])};
            if (NH == 1) asm volatile("" : "+v"(pk));            // (otherwise formed below the branch)
            if (NH == 2 || row_ok) *reinterpret_cast<u32x4*>(dst + 32 * jj) = pk;
        }
    }
}

// Combines the parts of the row blocks that were split: grid = (split blocks, KV heads, 4 heads of the group x 16-row halves of
// a block); thread (row, lane c of 16) of 16 x 256 outputs has the 16 bytes c of every 256 of
// a part's row.  out = sum_p f_p u_p O_p / sum_p f_p l_p, f_p = 2^(m_p - m), u_p = part_unit, parts in order; a
// thread's loads of O do not depend on the factors, so all parts are in flight together.
template <int RB, class PT>
__global__ __launch_bounds__(256) void attn_prefill_merge_kernel(const PT* __restrict__ part_o, const float* __restrict__ part_ml,
                                                                 bf16_t* __restrict__ out, int S, int q_pos0, int tmax, long slots_per_kv,
                                                                 long q_head_stride, int q_row_stride) {
    constexpr int PO = part_o_size(RB), PML = part_ml_floats(RB);
    const int c = (KT / RB) * tmax, p = (q_pos0 + RB - 1) / RB;
    const int rb = max(0, c - p) + blockIdx.x;                   // the first block with two parts is c - p
    const int np = (p + rb) / c + 1;
    const size_t slot0 = (size_t)blockIdx.y * slots_per_kv + (size_t)(parts_upto(p + rb, c) - parts_upto(p, c));
    const int hq = blockIdx.z / (RB / 16), cg = threadIdx.x & 15;
    {
        const int lr = 16 * (blockIdx.z % (RB / 16)) + (threadIdx.x >> 4);
        if (rb * RB + lr >= S) return;
        constexpr int VEC = 16 / sizeof(PT), NV = AD / 16 / VEC;  // values of a load, loads of a part
        typedef PT vec __attribute__((ext_vector_type(VEC)));
        const PT* po = part_o + (slot0 * 4 + hq) * (RB * AD) + lr * AD + cg * VEC;
        const float* pml = part_ml + (slot0 * 4 + hq) * (2 * RB) + lr;
        // AHEAD parts at a time, all their loads in flight together (an index past the last part loads the last again); the first ones are
        // requested before the maximum is known
        constexpr int AHEAD = 4;
        vec ov[AHEAD][NV];
        float pm[AHEAD], pl[AHEAD];
        auto load = [&](int p0) {
#pragma unroll
            for (int i = 0; i < AHEAD; i++) {
                const size_t pp = min(p0 + i, np - 1);
                pm[i] = pml[pp * PML], pl[i] = pml[pp * PML + RB];
#pragma unroll
                for (int j = 0; j < NV; j++) ov[i][j] = *reinterpret_cast<const vec*>(po + pp * PO + 16 * VEC * j);
            }
        };
        load(0);
        __builtin_amdgcn_sched_barrier(0);
        float m = NEG;
#pragma unroll
        for (int i = 0; i < AHEAD; i++) m = fmaxf(m, pm[i]);
        for (int p0 = AHEAD; p0 < np; p0 += AHEAD) {
            float mv[AHEAD];
#pragma unroll
            for (int i = 0; i < AHEAD; i++) mv[i] = pml[(size_t)min(p0 + i, np - 1) * PML];
#pragma unroll
            for (int i = 0; i < AHEAD; i++) m = fmaxf(m, mv[i]);
        }
        float l = 0.f;
        float acc[NV][VEC] = {};
        for (int p0 = 0;;) {
#pragma unroll
            for (int k = 0; k < AHEAD; k++) {
                if (p0 + k >= np) break;
                const float f = __builtin_amdgcn_exp2f(pm[k] - m), fu = f * part_unit<PT>(pm[k], pl[k]);
                l += f * pl[k];
#pragma unroll
                for (int j = 0; j < NV; j++)
#pragma unroll
                    for (int e = 0; e < VEC; e++) acc[j][e] += fu * (float)ov[k][j][e];
            }
            p0 += AHEAD;
            if (p0 >= np) break;
            load(p0);
        }
        const float inv = 1.0f / l;
        bf16_t* dst = out + (size_t)(blockIdx.y * (AH / AKV) + hq) * q_head_stride + (size_t)(rb * RB + lr) * q_row_stride + cg * VEC;
        typedef unsigned words __attribute__((ext_vector_type(VEC / 2)));
#pragma unroll
        for (int j = 0; j < NV; j++) {
            words pk;
#pragma unroll
            for (int e = 0; e < VEC / 2; e++) pk[e] = pack_bf(acc[j][2 * e] * inv, acc[j][2 * e + 1] * inv);
            *reinterpret_cast<words*>(dst + 16 * VEC * j) = pk;
        }
    }
}

}  // namespace

namespace {

inline bool two_heads_per_wave(int S) { return (S + 31) / 32 * AKV >= 288; }   // from 4577 rows on: 32-row blocks unsplit

// The key split of a launch: tmax = 0 (none) or the tiles per part, parts = grid width, split_blocks = blocks with several parts.
// Only launches that leave CUs without a workgroup are split (fewer than 2048 query rows: a short continuation of a long
// prefix, a short prompt), and only as far as the idle CUs go: all parts are resident at once, because a CU that has to run a second part
// pays the 6 us that a workgroup costs beyond its tiles (dispatch, Q and first-tile latency, the output stores) twice.
struct KeySplit {
    int nh = 1;            // heads per wavefront: row blocks of 16 nh rows
    int tmax = 0;
    long parts = 0;
    int split_blocks = 0;
    bool wide = false;     // parts in single precision
    long bytes() const { return parts * AKV * part_bytes(16 * nh, wide); }
};
// A form of split launch and its time, us: base + tile * (tiles per part) + part * (parts, both KV heads) + round * (groups of four parts that
// the merge takes one after the other).  It takes part sizes from min_tiles on that shorten the longest workgroup by min_gain tiles.
struct SplitForm {
    int nh, min_tiles, min_gain;
    bool wide;
    float base, tile, part, round;
};
// Takes the form if its best part size is faster than `us`, the best so far.  parts(t) falls with t: the smallest resident part size is found
// by bisection, and the few sizes from there on are priced (a launch of 20 us does not hide much of its host).
void consider(const SplitForm& f, int cus, int S, int L, int q_pos0, KeySplit& best, float& us) {
    const int RB = 16 * f.nh, nb = (S + RB - 1) / RB;
    if (S < 1 || nb * AKV >= cus || f.base + f.tile * f.min_tiles >= us) return;
    const int most = (std::min(L, q_pos0 + S) + KT - 1) / KT - f.min_gain;       // (the last block's tiles, less the gain)
    const long p = (q_pos0 + RB - 1) / RB, cpt = KT / RB;
    auto parts = [&](int t) { return parts_upto(p + nb, cpt * t) - parts_upto(p, cpt * t); };
    int t = f.min_tiles, hi = most + 1;
    if (t > most) return;
    if (parts(t) * AKV > cus)
        while (hi - t > 1) {                                     // parts(t) are too many, parts(hi) are not or hi is out of range
            const int mid = (t + hi) / 2;
            if (parts(mid) * AKV > cus) t = mid; else hi = mid;
        }
    else
        hi = t;
    for (t = hi; t <= std::min(most, hi + 8) && f.base + f.tile * t < us; t++) {
        const long n = parts(t), c = cpt * t;
        const float now = f.base + f.tile * t + f.part * AKV * n + f.round * (((p + nb + c - 1) / c + 3) / 4);
        if (now >= us) continue;
        us = now;
        best.nh = f.nh, best.tmax = t, best.parts = n, best.split_blocks = nb - (int)std::max(0L, c - p), best.wide = f.wide;
    }
}
// The form of a launch, by measurement (us at q_pos0 = 0, 16-row blocks (NH = 1) in their best form / 32-row blocks (NH = 2) with
// the split: S = 1280 25.3 / 27.3, 1408 27.7 / 27.7, 1536 32.3 / 30.0, 2048 47.0 / 37.2, 2560 59.9 / 51.4, 2944 68.5 / 63.3,
// 3072 71.0 / 69.8, 3200 76.3 / 75.5, 3328 79.3 / 82.5; unsplit 4096 108 / 114, 4608 138 / 131, 5120 167 / 149):
//   from about 4600 rows on     NH = 2, unsplit (enough 32-row blocks to balance themselves);
//   from about 1500 rows on     NH = 2 with the key split, where the launch leaves room for it and, for a whole prompt, up to
//                               3200 rows (a tile of a 32-row block costs less than two tiles of 16-row blocks, but its parts
//                               are twice the size): the smallest resident parts of six tiles or more, if they shorten the longest
//                               workgroup by four;
//   fewer rows                  the fastest of no split (NH = 1), NH = 1 with parts of six tiles or more in half precision, NH = 1 with parts
//                               of three tiles or more and NH = 2, both in single precision.
// Half precision is for launches that are split in earnest.  A few more tiles side by side, or more rows split for the sake of the
// larger block, are no reason to give up bits: without the split those rows are summed in single precision to the end.
// The times are fitted to 15 sizes of 1 - 1400 rows on 11 prefixes of 0 - 32000 keys, each form at up to nine part sizes; the choice is
// within 0.4 % of the best of these forms on average and 6 % at worst.  With short parts in half precision as well / as chosen: 17 rows on
// 700 keys 11.7 / 12.7 us, 333 on 300 / 1500 13.5 / 15.9 and 18.9 / 19.4, 600 13.4 / 15.3, 700 on 3000 32.7 / 36.6, 1185 on 1500 36.2 / 38.8.
KeySplit plan_split(int S, int L, int q_pos0) {
    KeySplit ks;
    if (two_heads_per_wave(S)) {                                 // (two heads: S >= 1472, or parts of several tiles, so L >= one tile)
        ks.nh = 2;
        return ks;
    }
    const int cus = cu_count();
    if (S >= 1472 && (q_pos0 > 0 || S <= 3200)) {
        float any = 1e30f;
        consider(SplitForm{2, 6, 4, false, 0.f, 1.f, 0.f, 0.f}, cus, S, L, q_pos0, ks, any);        // (priced by its tiles alone)
        if (ks.tmax) return ks;
    }
    float us = 4.2f + 1.2f * ((std::min(L, q_pos0 + S) + KT - 1) / KT);         // no split
    consider(SplitForm{1, 6, 6, false, 6.7f, 1.03f, 0.019f, 1.03f}, cus, S, L, q_pos0, ks, us);
    if (S < 1472) {
        consider(SplitForm{1, 3, 1, true, 7.7f, 0.97f, 0.030f, 1.05f}, cus, S, L, q_pos0, ks, us);
        consider(SplitForm{2, 3, 1, true, 10.4f, 1.51f, 0.037f, 0.61f}, cus, S, L, q_pos0, ks, us);
    }
    return ks;
}

}  // namespace

extern "C" {

// Bytes of workspace the key split of this launch uses (0: the launch is not split).  Without that much workspace
// qt_gqa_prefill_causal runs the same launch unsplit, with the same results up to rounding.
long qt_gqa_prefill_workspace_bytes_for(int S, int L, int q_pos0) {
    if (S < 0 || L < 1 || q_pos0 < 0) return -1;
    const KeySplit ks = plan_split(S, L, q_pos0);
    return ks.tmax ? ks.bytes() : 0;
}
// An upper bound of the above over every launch with at most L keys: a split launch has at most one part per CU, of 32 rows in single
// precision at most.
long qt_gqa_prefill_workspace_bytes(int L) { return L < 0 ? -1 : cu_count() * part_bytes(32, true); }

// q, out [8 heads][S rows][256] bf16 with head stride q_head_stride and row stride q_row_stride (elements; head-major rows have row
// stride 256, the token-major rows of a projection head stride 256 and row stride 2048, so neither has to be copied into the other),
// K, V [2][>=L][256] bf16 (head stride kv_head_stride):
// query i sits at absolute position q_pos0 + i and sees keys 0 .. q_pos0 + i (< L).  workspace: see above; may be null.
int qt_gqa_prefill_causal_strided(const void* q, const void* K, const void* V, void* out, void* workspace, long workspace_bytes, int S,
                          int L, int q_pos0, long q_head_stride, int q_row_stride, long kv_head_stride, hipStream_t stream) {
    if (!q || !K || !V || !out) return QT_ERR_NULL;
    if (S < 0 || L < 1 || q_pos0 < 0 || (long)q_pos0 + S > L || kv_head_stride < (long)L * AD || q_row_stride < AD)
        return QT_ERR_DIM;
    // the rows of different heads must not overlap: heads apart by whole row ranges, or side by side within a row
    if (q_head_stride < (long)S * q_row_stride && (q_head_stride < AD || q_row_stride < (AH - 1) * q_head_stride + AD)) return QT_ERR_DIM;
    if (S == 0) return QT_OK;
    for (const void* p : {q, K, V, (const void*)out, (const void*)workspace})
        if (reinterpret_cast<uintptr_t>(p) & 15u) return QT_ERR_ALIGN;
    if ((q_head_stride | q_row_stride | kv_head_stride) & 7) return QT_ERR_ALIGN;
    KeySplit ks = plan_split(S, L, q_pos0);
    if (ks.tmax && (!workspace || workspace_bytes < ks.bytes())) {          // no room for the parts: the unsplit form
        ks = KeySplit();
        ks.nh = two_heads_per_wave(S) ? 2 : 1;
    }
    const int RB = 16 * ks.nh;
    const dim3 grid((ks.tmax ? (unsigned)ks.parts : (unsigned)((S + RB - 1) / RB)) * AKV);
    auto launch = [&](auto nh, auto part_type) {
        constexpr int NH = decltype(nh)::value;
        using PT = decltype(part_type);
        PT* part_o = ks.tmax ? (PT*)workspace : nullptr;
        float* part_ml = ks.tmax ? reinterpret_cast<float*>(part_o + (size_t)ks.parts * AKV * part_o_size(RB)) : nullptr;
        hipLaunchKernelGGL((attn_prefill_kernel<NH, PT>), grid, dim3(512), 0, stream, (const bf16_t*)q, (const bf16_t*)K, (const bf16_t*)V,
                           (bf16_t*)out, S, L, q_pos0, q_head_stride, q_row_stride, kv_head_stride, ks.tmax, part_o, part_ml);
        if (ks.tmax)
            hipLaunchKernelGGL((attn_prefill_merge_kernel<16 * NH, PT>), dim3((unsigned)ks.split_blocks, AKV, (AH / AKV) * NH), dim3(256), 0, stream,
                               part_o, part_ml, (bf16_t*)out, S, q_pos0, ks.tmax, ks.parts, q_head_stride, q_row_stride);
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    if (ks.nh == 2 && ks.wide) launch(Two{}, float{});
    else if (ks.nh == 2) launch(Two{}, _Float16{});
    else if (ks.wide) launch(One{}, float{});
    else launch(One{}, _Float16{});
    QT_CHECK_LAUNCH();
    return QT_OK;
}
int qt_gqa_prefill_causal(const void* q, const void* K, const void* V, void* out, void* workspace, long workspace_bytes, int S,
                          int L, int q_pos0, long q_head_stride, long kv_head_stride, hipStream_t stream) {
    if (q_head_stride < (long)S * AD) return !q || !K || !V || !out ? QT_ERR_NULL : QT_ERR_DIM;
    return qt_gqa_prefill_causal_strided(q, K, V, out, workspace, workspace_bytes, S, L, q_pos0, q_head_stride, AD, kv_head_stride, stream);
}

}  // extern "C"
