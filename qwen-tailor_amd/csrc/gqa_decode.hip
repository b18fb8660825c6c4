// Ragged GQA decode / verify attention, head dim 256, 8 query heads on 2 KV heads, for gfx950.
// Replaces the Metal kernel attn_b_{Lmax}_m{M} (qwen35/batch.py:141-237): row r = b*M + j of the batch sits at position
// pos[b] + j of slot slots[b]; it attends the pool keys below pos[b] and the new keys of rows b*M .. b*M + j, which are
// read from the inputs (never from the pool) and appended to the pool at pos[b] + j.
//
// Split-K over one flat tile space: segment sg = (sequence b, kv head) owns max(1, ceil(pos[b] / 16)) tiles of 16 pool keys,
// the segments are laid end to end, and each of the launch's workgroups takes the same number of consecutive tiles (it may
// cross segment borders: it then emits one partial result per segment it touches).  Every workgroup therefore streams the
// same number of bytes whatever the mix of sequence lengths, K and V are read from HBM exactly once per step for all 4*M
// query rows that share the KV head, and the launch is one round of resident workgroups (one per CU).
//   loads  : a K or V tile (16 keys x 512 bytes) is fetched as whole rows, two rows per wavefront-wide load (nontemporal),
//            and parked row-major in LDS
//   scores : S^T[16 keys x 16 rows] = K_tile[16 x 256] . Q^T[256 x 16] on bf16 MFMA (16x16x32), K fragments from LDS
//   P . V  : O^T[256 x 16 rows] += V^T[256 x 16 keys] . P^T[16 keys x 16 rows] on bf16 MFMA (16x16x16): the transposed scores in
//            their accumulator layout ARE the B operand; the V tile is read back through the transposing LDS load
//            (ds_read_b64_tr_b16), which delivers the A operand (4 consecutive keys of one column).
//            P is split into two bf16 terms (p = hi + lo, error 2^-17), so the product keeps fp32-like accuracy.
// Each wavefront walks its tiles with a one-tile-deep register FIFO: a register is refilled with the next tile's row right
// after the LDS store that consumed it, so a tile's loads fly during the previous tile's arithmetic.  The loop issues
// loads only, in the order of their use, which keeps every vmcnt wait partial.
// Each wavefront keeps its own online-softmax state (m, l, O); the 4 wavefronts of a workgroup are merged through LDS and
// the workgroup writes one unnormalised partial (m, l, O) per row and segment; a second kernel merges the partials
// (batch.py:203-221).
// A kernel instance holds at most four query tokens per sequence (16 rows = one MFMA tile).  More tokens per sequence (M up
// to 16) run as passes of up to four: pass j0 = 0, 4, 8, 12 takes rows j0 .. j0+3 of every sequence at position pos[b] + j0 and
// finds the rows that the earlier passes appended among its pool keys (the passes are launches on one stream, in order).
#include "qt_common.h"
#include <type_traits>

using namespace qt;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int GQA = AH / AKV;          // 4 query heads per KV head
constexpr float SCALE = 0.0625f;       // 256^-0.5, batch.py:177
constexpr float NEG = -3.0e38f;
constexpr int VL_LD = AD + 16;         // row stride (elements) of the V tile in LDS: 544 bytes spread the 16 rows over the banks
constexpr int MO_LD = AD + 4;           // row stride (floats) of the O tiles in LDS: the 16 rows of a store start 4 banks apart
constexpr int KL_LD = AD + 8;          // row stride of the K tile: 528 bytes, the 16 rows of a fragment read start 4 banks apart

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }
// workgroup barrier for data that goes through LDS: loads and stores of global memory stay in flight across it (__syncthreads()
// would wait for all of them)
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// a copy the compiler cannot see through: what is derived from it is computed again where it is used instead of living in
// registers across the whole visit loop (about 30 lane-dependent addresses: they were spilled)
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// ---- the layer form: q / k RMSNorm and rotary embedding inside the attention kernel (qwen35/batch.py:505-512) ----------------
constexpr int QKV_W = AH * 2 * AD + 2 * AKV * AD;      // 5120: [(q_h | gate_h) x 8 | k x 2 | v x 2]
constexpr int ROPE_PAIRS = 32;                         // rotary pairs (i, i + 32), i < 32, of the first 64 features

// max over the four lanes n, n + 16, n + 32, n + 48 with the vector-ALU lane swaps (v_permlane32_swap exchanges the upper half of one
// register with the lower half of the other, v_permlane16_swap the odd 16-lane rows of one with the even rows of the other)
__device__ __forceinline__ float max_over_groups(float x) {
    const unsigned xi = __float_as_uint(x);
    const auto a = __builtin_amdgcn_permlane32_swap(xi, xi, false, false);
    const unsigned mi = __float_as_uint(fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
    const auto b = __builtin_amdgcn_permlane16_swap(mi, mi, false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// ... and the sum
__device__ __forceinline__ float sum_over_groups(float x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    const float s = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(s), __float_as_uint(s), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}
__device__ __forceinline__ float row16_max(float v) {            // over a 16-lane row
    v = fmaxf(v, dpp_mov<0xB1>(v));
    v = fmaxf(v, dpp_mov<0x4E>(v));
    v = fmaxf(v, dpp_mov<0x141>(v));
    return fmaxf(v, dpp_mov<0x140>(v));
}

// Online-softmax update of one tile of 16 keys from its transposed scores: lane (row n, group g) holds keys 4g .. 4g+3.
// Leaves the probabilities of those keys in p (fp32) and returns the row's rescale factor (the same in the row's four lanes).
__device__ __forceinline__ float softmax_tile(const f32x4& acc, int nvalid, bool causal, float& m_run, float& l_run, float (&p)[4], int lane) {
    const int n = lane & 15, g = lane >> 4;
    const int jq = n / GQA;                                      // query token of this row (rows >= 4*M are padding)
    float s[4], mx = NEG;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int key = 4 * g + i;
        const bool vis = key < nvalid && (!causal || key <= jq);
        s[i] = vis ? acc[i] * SCALE : NEG;
        mx = fmaxf(mx, s[i]);
    }
    mx = max_over_groups(mx);
    const float m_new = fmaxf(m_run, mx);
    const float corr = __expf(m_run - m_new);                    // m_run = NEG initially: exp(-huge) = 0
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        p[i] = s[i] > 0.5f * NEG ? __expf(s[i] - m_new) : 0.f;
        ps += p[i];
    }
    l_run = l_run * corr + ps;                                   // this lane's share; summed over g at the end
    m_run = m_new;
    return corr;
}

// O^T (256 x 16 rows, accumulator layout: block j, lane (row n, group g), columns 16 j + 4 g .. + 3) = c * O^T + V^T . P^T for the
// V tile in v_lds ([16 keys][VL_LD]).  p: this lane's probabilities (row n, keys 4g .. 4g+3), c: the row's rescale factor.  Taken in
// this order a row's factor and its output columns belong to the lane that holds its probabilities, so the factor goes through
// no LDS and a lane stores four adjacent columns.
__device__ __forceinline__ void pv_tile(f32x4 (&O)[16], const float (&p)[4], float c, const bf16_t* v_lds, int lane) {
    const int n = lane & 15, g = lane >> 4;
    s16x4 ph, pl;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const bf16_t h = f2bf(p[i]);
        ph[i] = (short)h;
        pl[i] = (short)f2bf(p[i] - bf2f(h));
    }
    if (__any(c != 1.0f)) {                                      // some row's maximum moved
#pragma unroll
        for (int j = 0; j < 16; j++) O[j] *= c;
    }
    // transposing load: within a group of 16 lanes, lane 4q + i receives element i of the 8-byte chunks addressed by lanes
    // q, q+4, q+8, q+12.  Lane j' = n of group g points at key 4g + n/4, columns 4 (n%4) .. + 3 of the block: lane n then
    // receives keys 4g .. 4g+3 of column n, the A operand.
    const bf16_t* vrow = v_lds + (4 * g + (n >> 2)) * VL_LD + 4 * (n & 3);
#pragma unroll
    for (int j = 0; j < 16; j++) {
        if (j % 8 == 0) __builtin_amdgcn_sched_barrier(0);       // (at most eight fragments in registers at a time)
        const s16x4 A = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(const_cast<bf16_t*>(vrow + 16 * j)));
        O[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(A, ph, O[j], 0, 0, 0);
        O[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(A, pl, O[j], 0, 0, 0);
    }
}

// inclusive prefix sum over the wavefront's lanes: four shifts within each 16-lane row, then the rows' totals as scalars
__device__ __forceinline__ int wave_prefix_sum(int v, int lane) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);           // row_shr:1, 2, 4, 8 (zeros shifted in)
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);
    const int r0 = __builtin_amdgcn_readlane(v, 15), r1 = __builtin_amdgcn_readlane(v, 31), r2 = __builtin_amdgcn_readlane(v, 47);
    return v + (lane < 16 ? 0 : lane < 32 ? r0 : lane < 48 ? r0 + r1 : r0 + r1 + r2);
}

constexpr int MAX_SEG = 2048;          // segments (2 per sequence) a launch can hold
// A workgroup pays for every segment it visits (the query rows, the merge of its four wavefronts, the partial result) about as much
// as for streaming five tiles.  Every segment therefore starts with that many empty positions in the flat tile space, so that a
// workgroup whose range crosses a segment border gets fewer tiles to stream.  Layer form, us, with 3 / 5 / 7 positions: 32 sequences of
// 1000 - 8000 keys 55.4 / 54.9 / 55.7, 64 of 200 - 2000 37.9 / 38.1 / 38.3, 16 of 512 - 32768 92.7 / 90.8 / 91.2, 5 x 3 rows of 90 - 900 17.0 /
// 16.7 / 16.9.
// A range that holds nothing but such positions of a segment does not visit it.  (When it did, for the new keys, a workgroup paid a visit, 3.3
// us, for no tile: 1 of 300 keys 14.0 us, 5 x 3 of 90 - 900 16.2, 16 of 100 - 1000 16.4, 64 of 50 - 200 17.5; without these visits and
// with a default split of 32 keys instead of 128 9.5 / 12.4 / 12.8 / 15.3.)
constexpr int VISIT_TILES = 5;


// tiles of a segment in the flat tile space; a row whose slot or position is out of range owns none (it is skipped by both kernels)
__device__ __forceinline__ int segment_tiles(int slot, int p0, int Lmax, int n_slots, int Mtot, int j0) {
    const bool ok = (unsigned)slot < (unsigned)n_slots && p0 >= 0 && p0 + Mtot <= Lmax;    // all of the sequence's rows fit, or none is taken
    return ok ? max(1, (p0 + j0 + 15) >> 4) + VISIT_TILES : 0;
}
// Prefix sums of the segments' tile counts -> seg_start[0 .. nseg] (LDS); returns the total.  Every thread of the workgroup (256)
// must call it; 256 segments per round.
__device__ __forceinline__ int build_segments(int* seg_start, const int* __restrict__ slots, const int* __restrict__ pos, int nseg,
                                              int Lmax, int n_slots, int Mtot, int j0) {
    __shared__ int wave_total[2][4];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    int carry = 0;
    if (tid == 0) seg_start[0] = 0;
    for (int base = 0, r = 0; base < nseg; base += 256, r ^= 1) {
        const int sg = base + tid;
        const int end = wave_prefix_sum(sg < nseg ? segment_tiles(slots[sg / AKV], pos[sg / AKV], Lmax, n_slots, Mtot, j0) : 0, lane);
        if (lane == 63) wave_total[r][w] = end;
        lds_barrier();
        int before = carry;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int t = wave_total[r][i];
            before += i < w ? t : 0;
            carry += t;
        }
        if (sg < nseg) seg_start[sg + 1] = end + before;
    }
    lds_barrier();
    return carry;
}
// tiles per workgroup for `total` tiles spread over nwg workgroups, at least min_tiles
__device__ __forceinline__ int tiles_per_wg(int total, int nwg, int min_tiles) { return max(min_tiles, (total + nwg - 1) / nwg); }

// partial results: slot id = workgroup + segment (unique, and consecutive for the workgroups that share a segment);
// part_o [slot][4*M rows][256] f32 (unnormalised), part_ml [slot][4*M][2] = (running max, running sum)
// LAYER: q is the layer's qkv rows [B*Mtot, 5120]; the query rows and the new keys are normed and roped here, the
// new values are read from the rows' v part, and k_new / v_new are not used.
template <int M, bool LAYER>
__global__ __launch_bounds__(256, 2) void attn_partial_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_new,
                                                           const bf16_t* __restrict__ v_new, bf16_t* Kp, bf16_t* Vp,
                                                           const int* __restrict__ slots, const int* __restrict__ pos,
                                                           float* __restrict__ part_o, float* __restrict__ part_ml,
                                                           int* __restrict__ seg_tab, int B, int Lmax, int min_tiles, int n_slots,
                                                           int Mtot, int j0, const bf16_t* __restrict__ q_norm,
                                                           const bf16_t* __restrict__ k_norm, const float2* __restrict__ rope_tab,
                                                           float eps) {
    // M = tokens of this pass (rows j0 .. j0 + M - 1 of each sequence's Mtot rows)
    constexpr int R = 4 * M;
    __shared__ int seg_start[MAX_SEG + 1];
    // one V tile and one K tile per wavefront, in one array: at the end the same memory holds the four wavefronts' scaled O
    // ([4][R rows][256] f32) for the merge
    __shared__ __align__(16) bf16_t tile_s[4 * 16 * (VL_LD + KL_LD)];
    __shared__ float m_s[4][16], l_s[4][16];
    static_assert(sizeof(bf16_t) * 4 * 16 * (VL_LD + KL_LD) >= sizeof(float) * 4 * 16 * MO_LD, "the four O tiles must fit into the K / V tiles");
    float* const mo = reinterpret_cast<float*>(tile_s);

    const int nseg = B * AKV;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    // Every wavefront holds a window of 64 segments in its lanes: lane i has the end, the slot and the position of segment win + i (ends
    // count in the flat tile space).  With up to 64 segments (32 sequences) the window is the whole table and comes from a prefix
    // sum over the lanes: nothing goes through LDS and no barrier is met.  With more, the ends are built in LDS and the window is
    // read where the workgroup's range begins.
    // (both forms of the kernel cut the tile space alike, so that the layer form sums its partial results in the order of the
    // plain one: same bits)
    int win = 0, lane_end = 0, lane_slot = 0, lane_pos = 0, total;
    auto load_rows = [&](int base) {
        if (base + lane < nseg) lane_slot = slots[(base + lane) / AKV], lane_pos = pos[(base + lane) / AKV];
    };
    if (nseg <= 64) {
        load_rows(0);
        lane_end = wave_prefix_sum(segment_tiles(lane < nseg ? lane_slot : -1, lane_pos, Lmax, n_slots, Mtot, j0), lane);
        total = __builtin_amdgcn_readlane(lane_end, 63);
        if (blockIdx.x == 0 && w == 0) {                         // the merge kernel reads the table instead of building it again
            if (lane == 0) seg_tab[0] = 0;
            if (lane < nseg) seg_tab[lane + 1] = lane_end;
        }
    } else {
        total = build_segments(seg_start, slots, pos, nseg, Lmax, n_slots, Mtot, j0);
        if (blockIdx.x == 0)
            for (int i = threadIdx.x; i <= nseg; i += 256) seg_tab[i] = seg_start[i];
    }
    const int per = tiles_per_wg(__builtin_amdgcn_readfirstlane(total), gridDim.x, min_tiles);
    const int wt0 = blockIdx.x * per, wt1 = min(wt0 + per, total);
    if (wt0 >= wt1) return;
    int sg0 = 0;                                                 // the segment that holds tile wt0
    if (nseg <= 64) {
        sg0 = __popcll(__ballot(lane < nseg && lane_end <= wt0));
    } else {
        for (int hi_ = nseg; sg0 < hi_;) {                       // (uniform binary search)
            const int mid = (sg0 + hi_) >> 1;
            if (__builtin_amdgcn_readfirstlane(seg_start[mid + 1]) <= wt0) sg0 = mid + 1; else hi_ = mid;
        }
    }
    auto move_window = [&](int base) {
        win = base;
        load_rows(base);
        lane_end = seg_start[min(base + lane, nseg - 1) + 1];
    };
    // A visit is the part of one segment's tiles that lies in this workgroup's range: its number (-1: there is none), slot, position of
    // the pass's first row, pool keys [lo, hi), and whether the range holds the segment's first tile.  All of it is scalar.  (A range that
    // holds only empty positions of a segment does not visit it.)
    auto find_visit = [&](int sg, int begin, int& v_sg, int& v_slot, int& v_p0, int& v_lo, int& v_hi, int& v_first) {
        // the first one at or after segment sg, which begins at `begin`
        int end = 0;
        for (; sg < nseg && begin + VISIT_TILES < wt1; sg++) {
            if (sg - win >= 64) move_window(sg);
            end = __builtin_amdgcn_readlane(lane_end, sg - win);
            if (end != begin) break;                             // (otherwise a skipped row)
        }
        const bool found = sg < nseg && begin + VISIT_TILES < wt1;
        const int at = found ? sg - win : 0;
        v_sg = __builtin_amdgcn_readfirstlane(found ? sg : -1);
        v_slot = __builtin_amdgcn_readlane(lane_slot, at);
        v_p0 = __builtin_amdgcn_readlane(lane_pos, at) + j0;
        v_first = __builtin_amdgcn_readfirstlane(wt0 <= begin + VISIT_TILES);
        v_lo = __builtin_amdgcn_readfirstlane(max(0, wt0 - begin - VISIT_TILES) * 16);
        v_hi = __builtin_amdgcn_readfirstlane(min((min(wt1, end) - begin - VISIT_TILES) * 16, v_p0));
    };
    auto end_of = [&](int sg) { return __builtin_amdgcn_readlane(lane_end, sg - win); };
    if (nseg > 64) move_window(sg0);
    int v_sg, v_slot, v_p0, v_lo, v_hi;
    int v_first;
    find_visit(sg0, nseg <= 64 ? (sg0 ? end_of(sg0 - 1) : 0) : __builtin_amdgcn_readfirstlane(seg_start[sg0]), v_sg, v_slot, v_p0, v_lo, v_hi, v_first);
    auto rows_of = [&](int sg, int slot) { return ((size_t)slot * AKV + sg % AKV) * Lmax * AD; };      // the (slot, head)'s rows in the pools
    auto tiles_in = [](int lo, int hi) { return hi > lo ? (hi - lo + 15) / 16 : 0; };

    bf16_t* const vl = tile_s + w * (16 * VL_LD);
    bf16_t* const kl = tile_s + 4 * (16 * VL_LD) + w * (16 * KL_LD);
    u32x4 a[8], vv[8];
    // Rows of a tile: key 2i (lower half wavefront) / 2i + 1 (upper half), 8 columns per lane, so one load covers two whole
    // 512-byte rows (a wavefront-wide load of 16 rows x 64 bytes streams about 15 % slower from HBM).  Keys past `hi` re-read the
    // tile's first key (they are masked / weighted by 0).  The tile's address is a scalar; a lane adds 32 bits.
    auto load_row = [](int ln, const bf16_t* tile0, int nkeys, int i) {
        const unsigned key = 2 * i + (ln >> 5);
        const unsigned off = ((int)key < nkeys ? key * (AD * 2) : 0u) + (ln & 31) * 16u;
        return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(tile0) + off));
    };
    auto load_first_tile = [&](int sg, int slot, int lo, int hi) {             // in the order of their use
        if (sg < 0 || w >= tiles_in(lo, hi)) return;
        const size_t at = rows_of(sg, slot) + (size_t)(lo + w * 16) * AD;
        const int nkeys = hi - (lo + w * 16), ln = opaque(lane);
#pragma unroll
        for (int i = 0; i < 8; i++) a[i] = load_row(ln, Kp + at, nkeys, i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; i++) vv[i] = load_row(ln, Vp + at, nkeys, i);
        __builtin_amdgcn_sched_barrier(0);
    };
    // layer form: the staged query rows lie in wavefront 0's V tile (the tiles are not in use yet), the staged new keys in an
    // array of their own (they are read after the tile loop).  With the query rows in an array of their own the workgroup's LDS
    // would pass half of a CU's: the compiler then plans for one workgroup per CU and all 512 registers, puts O into the
    // accumulation registers, and the rescale of O in the tile loop costs a register copy each way (+4 us per launch).
    __shared__ __align__(16) bf16_t k_s[LAYER ? 4 * KL_LD : 8];
    bf16_t* const q_s = tile_s;
    static_assert(16 * KL_LD <= 16 * VL_LD, "the staged query rows must fit into one V tile");

  if (v_sg < 0) return;                                          // (a range that lies in empty positions)
  // What a visit needs besides its tiles: the new values, and Q^T as the MFMA B operand: lane (row n, group g) holds q[row n][32 kb +
  // 8 g .. + 8]; row n = token (n / 4), head n % 4.  The first visit's first tile is requested in here.
  constexpr int NEW_REGS = (M + 1) / 2;
  u32x4 nv[NEW_REGS];
  bf16x8 bq[8];
  auto prepare = [&](auto first_visit) {
    const int v_b = v_sg / AKV, v_kvh = v_sg % AKV, v_ntiles = tiles_in(v_lo, v_hi);
    const size_t v_base = rows_of(v_sg, v_slot);
    // The wavefront with the fewest tiles also takes the M new keys of the sequence, where this workgroup holds the segment's first
    // tile; it asks for the new values now (keys 2 i and 2 i + 1 in the lower and upper half of the lanes; they are used after its tiles) and appends what it holds.
    const bool takes_new = v_first && w == (v_ntiles & 3);
#pragma unroll
    for (u32x4& x : nv) x = u32x4{0, 0, 0, 0};
    if (takes_new) {
        const bf16_t* vn = LAYER ? q + (size_t)(v_b * Mtot + j0) * QKV_W + AH * 2 * AD + AKV * AD + v_kvh * AD
                                 : v_new + ((size_t)(v_b * Mtot + j0) * AKV + v_kvh) * AD;
        const size_t stride = LAYER ? (size_t)QKV_W : (size_t)AKV * AD;
        const int ln = opaque(lane);
#pragma unroll
        for (int i = 0; i < NEW_REGS; i++)
            if (2 * i + (ln >> 5) < M) nv[i] = reinterpret_cast<const u32x4*>(vn + (size_t)(2 * i + (ln >> 5)) * stride)[ln & 31];
    }

    if constexpr (LAYER) {
        // The 4 M query rows are normed and roped once per workgroup: wavefront w takes token w (its four heads, a row per
        // 16-lane group, 16 consecutive elements per lane) and leaves the rows in LDS, where every wavefront picks up its
        // B operand.  The workgroup that holds the segment's first tile does the same for the M new keys (a key per 16-lane
        // group), which it also appends to the pool (batch.py:196-201).  Same arithmetic, value for value, as
        // attn_qkv_prep_kernel: sum of squares exact in double and rounded once, correctly rounded 1 / sqrt,
        // BF(w * BF(x * inv)), rotary products and sums rounded one by one; (cos, sin) from the table qt_rope_table_build wrote.
        // A wavefront's loads return in the order in which they were issued, so the first visit's rows are requested before
        // its first tile and the arithmetic runs while the tile is on its way from HBM; a later visit's tile was requested
        // while the visit before it was still at work.
        const int ln = opaque(lane), rr = ln >> 4, c = ln & 15;
        if (w >= M) {                                             // rows past 4 M: zeros
            *reinterpret_cast<u32x4*>(q_s + (4 * w + rr) * KL_LD + 16 * c) = u32x4{0, 0, 0, 0};
            *reinterpret_cast<u32x4*>(q_s + (4 * w + rr) * KL_LD + 16 * c + 8) = u32x4{0, 0, 0, 0};
        }
        // item it: the query rows of token it, or (it = M, on an idle wavefront if there is one) the new keys; one copy of the code
        const int items = M + (v_first ? 1 : 0);
        int it = w;
#pragma unroll 1
        do {
            const bool is_q = it < M, real = it < items;          // (a wavefront without an item goes along once: it has a tile to request)
            const int tok = is_q ? it : rr < M ? rr : 0;          // (of the keys' four groups the idle ones work on a copy of key 0)
            const u32x4* x = reinterpret_cast<const u32x4*>(q + (size_t)(v_b * Mtot + j0 + tok) * QKV_W +
                                                            (is_q ? (v_kvh * GQA + rr) * 2 * AD : AH * 2 * AD + v_kvh * AD) + 16 * c);
            const u32x4* wgt = reinterpret_cast<const u32x4*>((is_q ? q_norm : k_norm) + 16 * c);
            const f32x4* cs = reinterpret_cast<const f32x4*>(rope_tab + (size_t)(v_p0 + tok) * ROPE_PAIRS + 16 * (c & 1));
            u32x4 x0, x1, w0, w1;
            f32x4 cv[8];                                          // rotary pairs 16 (c & 1) .. + 15 (used by lanes c < 4 only)
            if (real) {
                x0 = x[0], x1 = x[1], w0 = wgt[0], w1 = wgt[1];
#pragma unroll
                for (int e = 0; e < 8; e++) cv[e] = cs[e];
            }
            __builtin_amdgcn_sched_barrier(0);
            if (decltype(first_visit)::value && it == w) load_first_tile(v_sg, v_slot, v_lo, v_hi);
            if (!real) break;
            float y[16], wt[16];
            unpack8(make_uint4(x0[0], x0[1], x0[2], x0[3]), reinterpret_cast<float(&)[8]>(y[0]));
            unpack8(make_uint4(x1[0], x1[1], x1[2], x1[3]), reinterpret_cast<float(&)[8]>(y[8]));
            unpack8(make_uint4(w0[0], w0[1], w0[2], w0[3]), reinterpret_cast<float(&)[8]>(wt[0]));
            unpack8(make_uint4(w1[0], w1[1], w1[2], w1[3]), reinterpret_cast<float(&)[8]>(wt[8]));
            double ss = 0.0;
#pragma unroll
            for (int e = 0; e < 16; e++) ss += (double)y[e] * y[e];
            const float inv = rsqrt_rn((float)row16_sum_d(ss) / (float)AD + eps);
#pragma unroll
            for (int e = 0; e < 16; e++) y[e] = BF(wt[e] * BF(y[e] * inv));
            // rotary pairs (i, i + 32), i < 32: lanes 0, 1 of a row hold the first halves, lanes 2, 3 their partners
            float other[16];
#pragma unroll
            for (int e = 0; e < 16; e++) other[e] = dpp_mov<0x4E>(y[e]);              // lane c ^ 2
            if (c < 4) {
#pragma clang fp contract(off)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const float cs_c = cv[e >> 1][2 * (e & 1)], cs_s = cv[e >> 1][2 * (e & 1) + 1];
                    const float own = y[e] * cs_c, oth = other[e] * cs_s;
                    y[e] = BF(c < 2 ? own - oth                   // y1 c - y2 s
                                    : oth + own);                 // y1 s + y2 c
                }
            }
            const u32x4 o0 = u32x4{pack2_bf(y[0], y[1]), pack2_bf(y[2], y[3]), pack2_bf(y[4], y[5]), pack2_bf(y[6], y[7])};
            const u32x4 o1 = u32x4{pack2_bf(y[8], y[9]), pack2_bf(y[10], y[11]), pack2_bf(y[12], y[13]), pack2_bf(y[14], y[15])};
            if (is_q) {                                           // (a pointer that may mean either array would be a flat access)
                *reinterpret_cast<u32x4*>(q_s + (4 * it + rr) * KL_LD + 16 * c) = o0;
                *reinterpret_cast<u32x4*>(q_s + (4 * it + rr) * KL_LD + 16 * c + 8) = o1;
            } else if (rr < M) {
                *reinterpret_cast<u32x4*>(k_s + rr * KL_LD + 16 * c) = o0;
                *reinterpret_cast<u32x4*>(k_s + rr * KL_LD + 16 * c + 8) = o1;
                *reinterpret_cast<u32x4*>(Kp + v_base + (size_t)(v_p0 + rr) * AD + 16 * c) = o0;
                *reinterpret_cast<u32x4*>(Kp + v_base + (size_t)(v_p0 + rr) * AD + 16 * c + 8) = o1;
            }
            it += 4;
        } while (it < items);
        lds_barrier();
        const int n = ln & 15, g = ln >> 4;
#pragma unroll
        for (int kb = 0; kb < 8; kb++) bq[kb] = as_bf16x8(*reinterpret_cast<const u32x4*>(q_s + n * KL_LD + 32 * kb + 8 * g));
        lds_barrier();                                            // every wavefront has its rows: wavefront 0 may park its first tile there
    } else {
        const int ln = opaque(lane), n = ln & 15, g = ln >> 4;
        const bool real = n < R;
        const bf16_t* qr = q + ((size_t)(v_b * Mtot + j0 + (real ? n / GQA : 0)) * AH + v_kvh * GQA + (n % GQA)) * AD;
#pragma unroll
        for (int kb = 0; kb < 8; kb++) {
            u32x4 x = reinterpret_cast<const u32x4*>(qr)[kb * 4 + g];
            if (!real) x = u32x4{0, 0, 0, 0};
            bq[kb] = as_bf16x8(x);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (decltype(first_visit)::value) load_first_tile(v_sg, v_slot, v_lo, v_hi);
    }
  };
  prepare(std::true_type{});
  while (true) {
    const int v_b = v_sg / AKV, v_kvh = v_sg % AKV, v_ntiles = tiles_in(v_lo, v_hi);
    const size_t v_base = rows_of(v_sg, v_slot);
    const bool takes_new = v_first && w == (v_ntiles & 3);
    float m_run = NEG, l_run = 0.f;
    f32x4 O[16];
#pragma unroll
    for (int j = 0; j < 16; j++) O[j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // the tile registers of the last step take the first tile of the next visit: its latency passes while this one is finished
    int n_sg, n_slot, n_p0, n_lo, n_hi;
    int n_first;
    find_visit(v_sg + 1, end_of(v_sg), n_sg, n_slot, n_p0, n_lo, n_hi, n_first);
    if (w < v_ntiles) {
        const int ln = opaque(lane), n = ln & 15, g = ln >> 4, hw = ln >> 5, cl = ln & 31;
        auto tile = [&](int t, auto refill) {
            const int nvalid = min(16, v_hi - (v_lo + t * 16)), nnext = v_hi - (v_lo + (t + 4) * 16);
            const size_t at = v_base + (size_t)(v_lo + (t + 4) * 16) * AD;
            // park both tiles row-major in LDS; every register is refilled with the next tile's row right after its store
#pragma unroll
            for (int i = 0; i < 8; i++) {
                *reinterpret_cast<u32x4*>(kl + (2 * i + hw) * KL_LD + 8 * cl) = a[i];
                if constexpr (decltype(refill)::value) a[i] = load_row(ln, Kp + at, nnext, i);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < 8; i++) {
                *reinterpret_cast<u32x4*>(vl + (2 * i + hw) * VL_LD + 8 * cl) = vv[i];
                if constexpr (decltype(refill)::value) vv[i] = load_row(ln, Vp + at, nnext, i);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (!decltype(refill)::value) load_first_tile(n_sg, n_slot, n_lo, n_hi);
            wave_lds_sync();
            f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};      // (two chains: half the dependent latency)
#pragma unroll
            for (int kb = 0; kb < 8; kb++) {                     // A operand: lane (key n, group g) holds k[key n][32 kb + 8 g .. + 8]
                const u32x4 ka = *reinterpret_cast<const u32x4*>(kl + n * KL_LD + 32 * kb + 8 * g);
                acc[kb & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(ka), bq[kb], acc[kb & 1], 0, 0, 0);
            }
            float p[4];
            const float c = softmax_tile(acc[0] + acc[1], nvalid, false, m_run, l_run, p, ln);
            pv_tile(O, p, c, vl, ln);
            wave_lds_sync();
        };
        // the last tile is taken outside the loop: inside, its refill would read some tile again (64 KiB per visited segment, 17 %
        // of the bytes of 64 sequences of 1100 keys)
        int t = w;
        for (; t + 4 < v_ntiles; t += 4) tile(t, std::true_type{});
        tile(t, std::false_type{});
    } else {
        load_first_tile(n_sg, n_slot, n_lo, n_hi);
    }
    const int ln = opaque(lane), n = ln & 15, g = ln >> 4;
    if (takes_new) {
        const int hw = ln >> 5, cl = ln & 31;
        // The M new keys of this sequence, straight from the inputs (batch.py:143-145), with the causal rule among them:
        // key i is visible to query token j only if i <= j.  Not pipelined: it runs once per sequence.  The rows are appended to the
        // pool here (batch.py:196-201): row j of the sequence goes to position p0 + j.
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
        if constexpr (LAYER) {                                    // the new keys as they were left in LDS (and appended)
#pragma unroll
            for (int kb = 0; kb < 8; kb++) {
                u32x4 x = *reinterpret_cast<const u32x4*>(k_s + (n & 3) * KL_LD + 32 * kb + 8 * g);
                if (n >= M) x = u32x4{0, 0, 0, 0};
                acc[kb & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(x), bq[kb], acc[kb & 1], 0, 0, 0);
            }
        } else {
            const u32x4* kr = reinterpret_cast<const u32x4*>(k_new + ((size_t)(v_b * Mtot + j0 + (n < M ? n : 0)) * AKV + v_kvh) * AD);
            u32x4 ka[8];
#pragma unroll
            for (int kb = 0; kb < 8; kb++) ka[kb] = kr[kb * 4 + g];
#pragma unroll
            for (int kb = 0; kb < 8; kb++) {
                if (n < M) reinterpret_cast<u32x4*>(Kp + v_base + (size_t)(v_p0 + n) * AD)[kb * 4 + g] = ka[kb];
                const u32x4 x = n < M ? ka[kb] : u32x4{0, 0, 0, 0};
                acc[kb & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(x), bq[kb], acc[kb & 1], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < NEW_REGS; i++)
            if (2 * i + hw < M) reinterpret_cast<u32x4*>(Vp + v_base + (size_t)(v_p0 + 2 * i + hw) * AD)[cl] = nv[i];
        float p[4];
        const float c = softmax_tile(acc[0] + acc[1], M, true, m_run, l_run, p, ln);
#pragma unroll
        for (int i = 0; i < 8; i++)                               // rows past the M new keys are zero: their weight is 0
            *reinterpret_cast<u32x4*>(vl + (2 * i + hw) * VL_LD + 8 * cl) = i < NEW_REGS ? nv[i < NEW_REGS ? i : 0] : u32x4{0, 0, 0, 0};
        wave_lds_sync();
        pv_tile(O, p, c, vl, ln);
        wave_lds_sync();
    }

    // ---- merge the 4 wavefronts (deterministic order); lane (n, g) holds columns 16 j + 4 g .. + 3 of row n
    l_run = sum_over_groups(l_run);
    if (g == 0) {
        m_s[w][n] = m_run;
        l_s[w][n] = l_run;
    }
    lds_barrier();                                               // also: every wavefront is done with its V tile
    const float f = __expf(m_run - fmaxf(fmaxf(m_s[0][n], m_s[1][n]), fmaxf(m_s[2][n], m_s[3][n])));
    // every wavefront leaves its scaled O in its own part of LDS; then each thread adds the four for R / 4 groups of four
    // columns, in a fixed order, and writes the partial result
    if (n < R) {
#pragma unroll
        for (int j = 0; j < 16; j++) *reinterpret_cast<f32x4*>(&mo[(w * R + n) * MO_LD + 16 * j + 4 * g]) = O[j] * f;
    }
    lds_barrier();
    const size_t pslot = (size_t)blockIdx.x + v_sg;
    float* po = part_o + pslot * R * AD;
    const int tid = 64 * w + ln;
#pragma unroll
    for (int i = tid; i < R * AD / 4; i += 256) {
        const float* src = mo + (i / (AD / 4)) * MO_LD + 4 * (i % (AD / 4));
        const auto part = [&](int ww) { return *reinterpret_cast<const f32x4*>(src + ww * (R * MO_LD)); };
        reinterpret_cast<f32x4*>(po)[i] = (part(0) + part(1)) + (part(2) + part(3));
    }
    if (tid < R) {
        const float mm = fmaxf(fmaxf(m_s[0][tid], m_s[1][tid]), fmaxf(m_s[2][tid], m_s[3][tid]));
        float ll = 0.f;
        for (int ww = 0; ww < 4; ww++) ll += l_s[ww][tid] * __expf(m_s[ww][tid] - mm);
        part_ml[(pslot * R + tid) * 2] = mm;
        part_ml[(pslot * R + tid) * 2 + 1] = ll;
    }
    lds_barrier();                                               // the LDS tiles are reused by the next visit
    if (n_sg < 0) break;
    v_sg = n_sg, v_slot = n_slot, v_p0 = n_p0, v_lo = n_lo, v_hi = n_hi, v_first = n_first;
    prepare(std::false_type{});
  }
}

// merge of the partial results: one workgroup of 256 threads per (segment, row).  The per-partial factors exp(m_s - m) are
// computed by one thread each; then wavefront w sums the partials s = w, w+4, ... (a lane owns 4 output columns, four
// partials' loads in flight) and the four wavefronts are added in order.
constexpr int MAX_SPLITS = 4096;
// GATE: out [R,2048] = BF(o * sigmoid_bf16(gate)) with the row's gate from its qkv row (qwen35/batch.py:513), value for value what
// attn_out_gate_kernel makes of the bf16 o that this kernel would store otherwise.
template <int M, bool GATE>
__global__ __launch_bounds__(256) void attn_merge_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                         const int* __restrict__ seg_tab, bf16_t* __restrict__ out, int B, int nwg,
                                                         int min_tiles, int Mtot, int j0, const bf16_t* __restrict__ qkv) {
    constexpr int R = 4 * M;
    __shared__ float fs_s[MAX_SPLITS];
    __shared__ float red_m[4], red_l[4];
    __shared__ __align__(16) float acc_s[4][AD];
    const int r = blockIdx.x % R, sg = blockIdx.x / R, kvh = sg % AKV, b = sg / AKV;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const size_t row = (size_t)(b * Mtot + j0 + r / GQA);
    const int head = kvh * GQA + (r % GQA);
    bf16_t gate_raw = 0;
    if constexpr (GATE) gate_raw = qkv[row * QKV_W + head * 2 * AD + AD + tid];   // requested first, needed last
    const int total = seg_tab[B * AKV], ss = seg_tab[sg], se = seg_tab[sg + 1];   // written by the partial kernel
    if (se == ss) return;                                        // a skipped row
    const int per = tiles_per_wg(total, nwg, min_tiles);
    const int wg0 = (ss + VISIT_TILES) / per, ns = (se - 1) / per - wg0 + 1;     // the workgroups that hold tiles of this segment
    const size_t base = (size_t)wg0 + sg;                        // their partials sit in consecutive slots
    const float* ml = part_ml + (base * R + r) * 2;              // slot stride 2 R floats
    const float* po = part_o + (base * R + r) * AD + lane * 4;   // slot stride R * AD floats
    // this wavefront's first four partials are requested beside the factors' inputs: one memory latency less with few partials (layer form,
    // 1 of 300 keys 10.4 -> 9.5 us, 16 of 100 - 1000 13.7 -> 12.8)
    f32x4 first[4];
#pragma unroll
    for (int i = 0; i < 4; i++) first[i] = *reinterpret_cast<const f32x4*>(po + (size_t)min(w + 4 * i, ns - 1) * R * AD);
    // (a thread's first pair stays in its registers: with up to 256 partials nothing is loaded a second time)
    float2 own = make_float2(NEG, 0.f);
    if (tid < ns) own = *reinterpret_cast<const float2*>(ml + (size_t)tid * 2 * R);
    float mx = own.x;
    for (int s = tid + 256; s < ns; s += 256) mx = fmaxf(mx, ml[(size_t)s * 2 * R]);
    mx = max_over_groups(row16_max(mx));
    if (lane == 0) red_m[w] = mx;
    __syncthreads();
    const float mm = fmaxf(fmaxf(red_m[0], red_m[1]), fmaxf(red_m[2], red_m[3]));
    float lp = 0.f;
    if (tid < ns) {
        const float f = __expf(own.x - mm);
        fs_s[tid] = f;
        lp = own.y * f;
    }
    for (int s = tid + 256; s < ns; s += 256) {
        const float f = __expf(ml[(size_t)s * 2 * R] - mm);
        fs_s[s] = f;
        lp += ml[(size_t)s * 2 * R + 1] * f;
    }
    lp = sum_over_groups(row16_sum(lp));
    if (lane == 0) red_l[w] = lp;
    __syncthreads();
    const float l = (red_l[0] + red_l[1]) + (red_l[2] + red_l[3]);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (w + 4 * i < ns) acc += first[i] * fs_s[w + 4 * i];
    int s = w + 16;
    for (; s + 12 < ns; s += 16) {
        f32x4 ov[4];
#pragma unroll
        for (int i = 0; i < 4; i++) ov[i] = *reinterpret_cast<const f32x4*>(po + (size_t)(s + 4 * i) * R * AD);
#pragma unroll
        for (int i = 0; i < 4; i++) acc += ov[i] * fs_s[s + 4 * i];
    }
    for (; s < ns; s += 4) acc += *reinterpret_cast<const f32x4*>(po + (size_t)s * R * AD) * fs_s[s];
    *reinterpret_cast<f32x4*>(&acc_s[w][lane * 4]) = acc;
    __syncthreads();
    const int d = tid;
    const float a = (acc_s[0][d] + acc_s[1][d]) + (acc_s[2][d] + acc_s[3][d]);
    const float ov = l == 0.f ? a : a / l;                                           // batch.py:216
    if constexpr (GATE) {
        out[(row * AH + head) * AD + d] = f2bf(BF(ov) * sigmoid_bf16(bf2f(gate_raw)));
    } else {
        out[(row * AH + head) * AD + d] = f2bf(ov);
    }
}

}  // namespace

extern "C" {

constexpr int MAX_WG = 1024;           // upper bound of the partial kernel's grid (one workgroup per CU)
constexpr int MAX_PASS_M = 4;          // query tokens per sequence in one pass (16 rows: one MFMA tile)
constexpr int MAX_M = 16;              // query tokens per sequence in one call (as many as the verify step of the recurrent layers takes)

static int partial_grid() {            // one workgroup per CU of the current device: measured faster than two (the stream is
                                       // bandwidth-bound with 64 KiB in flight per CU; a second workgroup only adds queueing)
    const int cus = qt::cu_count();
    return cus < MAX_WG ? cus : MAX_WG;
}

constexpr long SEG_TAB_BYTES = ((MAX_SEG + 1) * 4 + 15) / 16 * 16;   // the segment table, after the partial results

// bytes of workspace qt_gqa_attn_decode needs for (B sequences, M rows each, pool length Lmax); CH is accepted for callers
// written against the fixed-split form and does not change the size
long qt_gqa_attn_workspace_bytes(int B, int M, int Lmax, int CH) {
    if (B < 0 || M < 1 || Lmax < 1 || CH < 16) return -1;
    const int mp = M < MAX_PASS_M ? M : MAX_PASS_M;                // the passes of a call with more tokens reuse one pass's space
    return ((long)MAX_WG + (long)B * AKV) * (4 * mp) * (AD + 2) * 4 + SEG_TAB_BYTES;
}

// Both entry points: checks, grid size and the two launches.  The partial results of at most `slot_cap` slots
// (slot = workgroup + segment < grid + 2 B) start at part_o / part_ml; seg_tab holds 2 B + 1 ints.
struct LayerArgs {                      // the layer form's extra operands (null q_norm: the plain form)
    const bf16_t* q_norm;
    const bf16_t* k_norm;
    const float2* rope_tab;
    float eps;
};

static int attn_launch(const void* q, const void* k_new, const void* v_new, void* Kp, void* Vp, const int32_t* slots,
                       const int32_t* pos, void* out, float* part_o, float* part_ml, int* seg_tab, int max_grid, int B, int M,
                       int Lmax, int n_slots, int CH, hipStream_t stream, LayerArgs la = LayerArgs{nullptr, nullptr, nullptr, 0.f}) {
    const int min_tiles = CH / 16;                               // a workgroup takes at least CH keys
    const long max_tiles = (long)B * AKV * ((Lmax + 15) / 16);
    const long want = (max_tiles + min_tiles - 1) / min_tiles;
    const int nwg = (int)(want < max_grid ? want : max_grid);
    const dim3 g1((unsigned)nwg);
    const bool layer = la.q_norm != nullptr;
#define QT_ATTN_LAUNCH2(MM, LY)                                                                                           \
    hipLaunchKernelGGL((attn_partial_kernel<MM, LY>), g1, dim3(256), 0, stream, (const bf16_t*)q, (const bf16_t*)k_new,   \
                       (const bf16_t*)v_new, (bf16_t*)Kp, (bf16_t*)Vp, slots, pos, part_o, part_ml, seg_tab, B, Lmax, min_tiles,    \
                       n_slots, M, j0, la.q_norm, la.k_norm, la.rope_tab, la.eps);                                        \
    hipLaunchKernelGGL((attn_merge_kernel<MM, LY>), dim3((unsigned)(B * AKV * 4 * MM)), dim3(256), 0, stream, part_o, part_ml,      \
                       seg_tab, (bf16_t*)out, B, nwg, min_tiles, M, j0, (const bf16_t*)q);
#define QT_ATTN_LAUNCH(MM)                                                                                                \
    if (layer) { QT_ATTN_LAUNCH2(MM, true) } else { QT_ATTN_LAUNCH2(MM, false) }
    for (int j0 = 0; j0 < M; j0 += MAX_PASS_M) {                 // passes of up to four tokens per sequence
        switch (M - j0 < MAX_PASS_M ? M - j0 : MAX_PASS_M) {
            case 1: QT_ATTN_LAUNCH(1) break;
            case 2: QT_ATTN_LAUNCH(2) break;
            case 3: QT_ATTN_LAUNCH(3) break;
            default: QT_ATTN_LAUNCH(4) break;
        }
        QT_CHECK_LAUNCH();
    }
#undef QT_ATTN_LAUNCH
#undef QT_ATTN_LAUNCH2
    return QT_OK;
}

static int attn_check(const void* q, const void* k_new, const void* v_new, const void* Kp, const void* Vp, const int32_t* slots,
                      const int32_t* pos, const void* out, int B, int M, int Lmax, int n_slots, int CH) {
    if (!q || !k_new || !v_new || !Kp || !Vp || !slots || !pos || !out) return QT_ERR_NULL;
    if (B < 0 || Lmax < 1 || n_slots < 1 || CH < 16 || CH % 16) return QT_ERR_DIM;
    if (M < 1 || M > MAX_M || B * AKV > MAX_SEG) return QT_ERR_UNSUPPORTED;
    for (const void* p : {q, k_new, v_new, Kp, Vp})
        if (reinterpret_cast<uintptr_t>(p) & 15u) return QT_ERR_ALIGN;
    return QT_OK;
}

int qt_gqa_attn_decode(const void* q, const void* k_new, const void* v_new, void* Kp, void* Vp, const int32_t* slots,
                       const int32_t* pos, void* out, void* workspace, long workspace_bytes, int B, int M, int Lmax,
                       int n_slots, int CH, hipStream_t stream) {
    if (!workspace) return QT_ERR_NULL;
    if (const int rc = attn_check(q, k_new, v_new, Kp, Vp, slots, pos, out, B, M, Lmax, n_slots, CH)) return rc;
    if (B == 0) return QT_OK;
    if (reinterpret_cast<uintptr_t>(workspace) & 15u) return QT_ERR_ALIGN;
    if (workspace_bytes < qt_gqa_attn_workspace_bytes(B, M, Lmax, CH)) return -6;
    const size_t cap = (size_t)MAX_WG + (size_t)B * AKV;
    const int mp = M < MAX_PASS_M ? M : MAX_PASS_M;
    float* part_o = (float*)workspace;
    float* part_ml = part_o + cap * (4 * mp) * AD;
    int* seg_tab = reinterpret_cast<int*>(part_ml + cap * (4 * mp) * 2);
    return attn_launch(q, k_new, v_new, Kp, Vp, slots, pos, out, part_o, part_ml, seg_tab, partial_grid(), B, M, Lmax, n_slots, CH,
                       stream);
}

// The attention half of a full-attention layer at a decode / verify step in two launches per pass: q / k RMSNorm, rotary
// embedding, the split of the qkv rows, attn_b and the output gate (qwen35/batch.py:505-513).
long qt_rope_table_bytes(int n_pos) { return n_pos < 0 ? -1 : (long)n_pos * ROPE_PAIRS * (long)sizeof(float2); }

int qt_gqa_attn_layer_decode(const void* qkv, const void* q_norm, const void* k_norm, const void* rope_table, int table_positions,
                             void* Kp, void* Vp, const int32_t* slots, const int32_t* pos, void* out, void* workspace,
                             long workspace_bytes, int B, int M, int Lmax, int n_slots, int CH, float eps, hipStream_t stream) {
    if (!workspace || !q_norm || !k_norm || !rope_table) return QT_ERR_NULL;
    if (const int rc = attn_check(qkv, qkv, qkv, Kp, Vp, slots, pos, out, B, M, Lmax, n_slots, CH)) return rc;
    if (table_positions < Lmax) return QT_ERR_DIM;               // every position a row can sit at has its (cos, sin) pairs
    if (B == 0) return QT_OK;
    for (const void* p : {(const void*)workspace, q_norm, k_norm, rope_table, (const void*)out})
        if (reinterpret_cast<uintptr_t>(p) & 15u) return QT_ERR_ALIGN;
    if (workspace_bytes < qt_gqa_attn_workspace_bytes(B, M, Lmax, CH)) return -6;
    const size_t cap = (size_t)MAX_WG + (size_t)B * AKV;
    const int mp = M < MAX_PASS_M ? M : MAX_PASS_M;
    float* part_o = (float*)workspace;
    float* part_ml = part_o + cap * (4 * mp) * AD;
    int* seg_tab = reinterpret_cast<int*>(part_ml + cap * (4 * mp) * 2);
    return attn_launch(qkv, nullptr, nullptr, Kp, Vp, slots, pos, out, part_o, part_ml, seg_tab, partial_grid(), B, M, Lmax, n_slots,
                       CH, stream, LayerArgs{(const bf16_t*)q_norm, (const bf16_t*)k_norm, (const float2*)rope_table, eps});
}

// ---- the same operator for callers that cannot allocate: the partial results live in a static device array -------------------
constexpr int ST_MAX_B = 128;          // sequences per call of the allocation-free entry point
constexpr int ST_MAX_WG = 256;         // its partial kernel's grid is capped here (one workgroup per CU on MI355X)
constexpr size_t ST_CAP = (size_t)ST_MAX_WG + (size_t)ST_MAX_B * AKV;
constexpr size_t ST_BYTES = ST_CAP * 16 * (AD + 2) * 4 + SEG_TAB_BYTES;        // 8.1 MiB
static __device__ __align__(256) unsigned char scratch[ST_BYTES];

// Device address of `scratch` on the current device, looked up once per device (every GPU holds its own copy of the array
// at its own address).  In host code the array's name is only a handle for this lookup, never a pointer to pass on.
static int scratch_address(unsigned char** out) {
    constexpr int MAX_DEV = 64;
    static std::atomic<unsigned char*> cache[MAX_DEV];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEV) return QT_ERR_LAUNCH;
    unsigned char* p = cache[dev].load(std::memory_order_acquire);
    if (!p) {
        if (hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return QT_ERR_LAUNCH;
        cache[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return QT_OK;
}

int qt_gqa_attn_decode_static(const void* q, const void* k_new, const void* v_new, void* Kp, void* Vp, const int32_t* slots,
                              const int32_t* pos, void* out, int B, int M, int Lmax, int n_slots, int CH, hipStream_t stream) {
    if (const int rc = attn_check(q, k_new, v_new, Kp, Vp, slots, pos, out, B, M, Lmax, n_slots, CH)) return rc;
    if (B > ST_MAX_B) return QT_ERR_STATIC_MAX;
    if (B == 0) return QT_OK;
    unsigned char* base = nullptr;
    if (const int rc = scratch_address(&base)) return rc;
    // Nothing in the array has to start at zero: every partial slot and table entry a launch reads was written by that launch.
    const int mp = M < MAX_PASS_M ? M : MAX_PASS_M;
    float* part_o = reinterpret_cast<float*>(base);
    float* part_ml = part_o + ST_CAP * (4 * mp) * AD;
    int* seg_tab = reinterpret_cast<int*>(part_ml + ST_CAP * (4 * mp) * 2);
    const int grid = partial_grid() < ST_MAX_WG ? partial_grid() : ST_MAX_WG;
    return attn_launch(q, k_new, v_new, Kp, Vp, slots, pos, out, part_o, part_ml, seg_tab, grid, B, M, Lmax, n_slots, CH, stream);
}

}  // extern "C"
