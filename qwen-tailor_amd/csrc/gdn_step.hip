// Fused GatedDeltaNet decode / speculative-verify step for gfx950.
//
// One group of WPH wavefronts (4; 8 for a few whole heads) owns ROWS = 4 RS WPH value rows of one (sequence, head) and streams them
// HBM -> registers -> HBM exactly once: conv4 + SiLU, q/k L2 norm, gates, then for every value row r
//     s = S[r,:] * g;  kv = s.k;  delta = (v_r - kv) * beta;  s += k * delta;  y_r = s.q
// (qwen35/kernels.py:518-530).  Replaces the Metal kernels deltanet_b (qwen35/batch.py:36-135), deltanet_bm
// (qwen35/batch_spec.py:45-150) and deltanet_m{M} (qwen35/kernels.py:461-567).
//
// Memory layout (slot-major, as qwen35/batch.py:1-12): ssm pool [S+1][16][128][128] f32, one head = 64 KiB contiguous;
// a 16-lane group reads 256 contiguous bytes of a row per load, a wavefront 4 rows, the workgroup 16 rows = 8 KiB per
// load slot.  Both dot products of a row are taken from the state as loaded,
//     kv = g * (S_r . k),   y_r = g * (S_r . q) + delta * (k . q),
// so the two 16-lane DPP reductions of a row are independent and the row is touched once.
#include "qt_common.h"

using namespace qt;

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));   // native vector: nontemporal loads / stores take it

struct RawIn {          // the un-convolved inputs one prologue thread needs for one token: raw bf16 bits
    unsigned w0, w1, w2, x;
    uint2 c;
};

// input row t of channel ch for the chained tokens of one sequence: t < 0 reads the stored window (kernels.py:477-479)
__device__ __forceinline__ unsigned inp(const bf16_t* __restrict__ cs_in, const bf16_t* __restrict__ proj, int t, int ch) {
    return t < 0 ? cs_in[(t + 3) * CD + ch] : proj[(size_t)t * PW + ch];
}
// what does not depend on the sequence's slot ...
__device__ __forceinline__ void load_taps(RawIn& r, const bf16_t* __restrict__ cw, int ch) { r.c = *reinterpret_cast<const uint2*>(cw + (size_t)ch * 4); }
template <bool TAPS = true>
__device__ __forceinline__ void load_raw_proj(RawIn& r, const bf16_t* __restrict__ proj, const bf16_t* __restrict__ cw, int j, int ch) {
    r.x = proj[(size_t)j * PW + ch];
    if (TAPS) load_taps(r, cw, ch);
}
// ... and what does
__device__ __forceinline__ void load_raw_window(RawIn& r, const bf16_t* __restrict__ cs_in, const bf16_t* __restrict__ proj, int j, int ch) {
    r.w0 = inp(cs_in, proj, j - 3, ch);
    r.w1 = inp(cs_in, proj, j - 2, ch);
    r.w2 = inp(cs_in, proj, j - 1, ch);
}
// (a value that is converted in the block that loads it is waited for there: what is read again behind this is converted behind it)
__device__ __forceinline__ void pin(RawIn& r) { asm volatile("" : "+v"(r.w0), "+v"(r.w1), "+v"(r.w2), "+v"(r.x)); }
__device__ __forceinline__ void drop(const RawIn& r) { asm volatile("" ::"v"(r.x), "v"(r.c.x), "v"(r.c.y)); }
__device__ __forceinline__ float conv_raw(const RawIn& r) {
    return conv_silu(bf2f((bf16_t)r.w0), bf2f((bf16_t)r.w1), bf2f((bf16_t)r.w2), bf2f((bf16_t)r.x), r.c);
}
__device__ __forceinline__ void store_window(bf16_t* __restrict__ cs_out, const RawIn& r, int ch) {
    cs_out[ch] = (bf16_t)r.w1;          // kernels.py:531: the new window is the last three input rows
    cs_out[CD + ch] = (bf16_t)r.w2;
    cs_out[2 * CD + ch] = (bf16_t)r.x;
}
// where a sequence's window and state lie; snapshot j of the state goes to st_out + j*st_stride and of the conv window to cs_out +
// j*cs_stride (strides 0 = update in place).  ok = false: the row is skipped, and the places are none
struct Place {
    bool ok;
    int par;                            // which of two windows is read (looked up with the slot)
    const bf16_t* cs_in;
    bf16_t* cs_out;
    size_t cs_stride;
    const float* st_in;
    float* st_out;
    size_t st_stride;
};
// the value of lane I of the wavefront, which is the same for all of them
__device__ __forceinline__ float lane_value(float v, int i) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), i)); }

// M chained tokens of one (sequence, head, row split), by WPH wavefronts; place() tells where they lie.
// NORM (whole heads only): y receives the gated RMSNorm of the head's 128 outputs, BF(z sigmoid(z) gw (y inv)) with
// z = proj[6144 + h*128 + row] (qwen35/batch.py:321-331), instead of the outputs themselves: same bits as the stand-alone
// norm kernel applied to the stored outputs.
// Order of the loads: what depends on neither slot nor position first, while those two are looked up, then the window, then the state;
// nothing is waited for before the state has been requested.  (Slot, position and the inputs one after the other, and the inputs
// converted where they are loaded, the state's requests left about two memory latencies late.  Fused norm, us in a HIP graph at 1 / 8 / 16 /
// 20 / 64 rows 4.7 / 5.8 / 7.6 / 9.2 / 24.6, now 4.4 / 5.4 / 7.2 / 8.9 / 24.4; verify of 16 x 4 17.9, now 17.3.)
// TAPS_LATE: the taps behind the state, which the conv then waits for (the rule is at the launch of the verify step).
// WPH: four wavefronts share q, k, v and the gates; with more, q and k, v, and the gates have wavefronts of their own, and the state is in
// more hands: a little faster while most CUs have nothing to do.
template <int RS, int HPW = 1, bool NORM = false, int WPH = 4, bool TAPS_LATE = false, class PlaceFn>
__device__ __forceinline__ void gdn_tokens(const bf16_t* __restrict__ proj, const bf16_t* __restrict__ cw, const float* __restrict__ A_log,
                                           const float* __restrict__ dt_bias, bf16_t* __restrict__ y, int M, int h, int split,
                                           PlaceFn place, const float* __restrict__ gw = nullptr, float eps = 0.f) {
    constexpr int GRPS = 4 * WPH, ROWS = RS * GRPS;
    static_assert(!NORM || ROWS == DV, "the fused norm needs the whole head in one group of wavefronts");
    static_assert(WPH == 4 || (WPH >= 8 && ROWS == DV), "more wavefronts take whole heads");
    __shared__ double red_a[HPW][WPH];
    __shared__ __align__(16) float qk_a[HPW][2][DK];
    __shared__ float v_a[HPW][ROWS];
    __shared__ float gb_a[HPW][2];
    // HPW heads per workgroup: each group of WPH wavefronts runs one head, only the barriers are shared
    const int wg_w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), sub = HPW > 1 ? wg_w / WPH : 0, w = HPW > 1 ? wg_w % WPH : wg_w;
    double* red = red_a[sub];
    float (*qk_s)[DK] = qk_a[sub];
    float* v_s = v_a[sub];
    float* gb_s = gb_a[sub];

    const int lane = threadIdx.x & 63, tid = 64 * w + lane, grp = lane >> 4, c = lane & 15;
    const int row0 = split * ROWS;
    // wavefronts 0, 1: q channels, 2, 3: k channels; v channels: the first ROWS threads, or wavefronts 4 and 5; gates: wavefront GW
    constexpr int V0 = WPH > 4 ? 256 : 0, GW = WPH > 4 ? 6 : 3;
    const bool is_qk = WPH == 4 || w < 4, has_v = WPH == 4 ? tid < ROWS : (w == 4 || w == 5), is_g = w == GW;
    const int which = w >> 1;                                    // 0: a q channel, 1: a k channel
    const int ch_qk = which * KD + h * DK + (tid & 127);
    const int ch_v = 2 * KD + h * DV + row0 + tid - V0;
    const int ch_v_ld = has_v ? ch_v : ch_qk;                    // (four wavefronts: every load is unconditional)

    RawIn rq = {0, 0, 0, 0, {0, 0}}, rv = {0, 0, 0, 0, {0, 0}};
    if (is_qk) load_raw_proj<!TAPS_LATE>(rq, proj, cw, 0, ch_qk);
    if (WPH == 4 || has_v) load_raw_proj<!TAPS_LATE>(rv, proj, cw, 0, ch_v_ld);
    // gates: lane 1 the decay gate (reads a), lane 2 beta (reads b)
    const int g_at = CD + KD + HV * (lane == 1 ? 1 : 0) + h;
    unsigned gx = 0;
    if (WPH == 4 || is_g) gx = proj[g_at];
    const float gA = A_log[h], gdt = dt_bias[h];
    // fused norm: lane c < RS of a 16-lane group finishes the group's row i = c (row c*GRPS + w*4 + grp of the head)
    const int nrow = (c % RS) * GRPS + w * 4 + grp;
    unsigned nz = 0;
    float ngw = 0.f;
    if (NORM) {
        nz = proj[CD + h * DV + nrow];
        ngw = gw[nrow];
    }
    __builtin_amdgcn_sched_barrier(0);
    const Place at = place();
    // A skipped row costs its slot's lookup and these few loads (us: 64 of them 2.3, with the state's loads and the conv 7.5, without a load 1.8; 32 rows
    // and 32 skipped 16.6 / 17.9 / 17.1, 64 and 64 30.5 / 35.4 / 30.3).
    if (__builtin_expect(!at.ok, 0)) {
        // (they count as used on this way out as well: otherwise they would be moved below the branch, and wait for it)
        drop(rq);
        drop(rv);
        asm volatile("" ::"v"(gx), "v"(nz), "v"(ngw), "s"(gA), "s"(gdt), "s"(at.par));
        __builtin_amdgcn_endpgm();                               // (a return would join the way out of the whole step: two more branches for every row)
    }
    if (is_qk) load_raw_window(rq, at.cs_in, proj, 0, ch_qk);
    if (WPH == 4 || has_v) load_raw_window(rv, at.cs_in, proj, 0, ch_v_ld);
    __builtin_amdgcn_sched_barrier(0);           // keep the small loads ahead of the state loads in issue order

    f4 s[RS][2];
    {
        const f4* sin4 = reinterpret_cast<const f4*>(at.st_in + ((size_t)h * DV + row0) * DK);
#pragma unroll
        for (int i = 0; i < RS; i++) {
            const int row = i * GRPS + w * 4 + grp;
            s[i][0] = __builtin_nontemporal_load(sin4 + row * (DK / 4) + c);
            s[i][1] = __builtin_nontemporal_load(sin4 + row * (DK / 4) + 16 + c);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if (TAPS_LATE) load_taps(rq, cw, ch_qk), load_taps(rv, cw, ch_v_ld);
    pin(rq);
    pin(rv);
    asm volatile("" : "+v"(gx), "+v"(nz));

    const float sc = which == 0 ? BF(INV_SCALE * INV_SCALE) : BF(INV_SCALE);       // kernels.py:492
    for (int j = 0; j < M; j++) {
        if (j > 0) {
            if (is_qk) load_raw_proj(rq, proj, cw, j, ch_qk), load_raw_window(rq, at.cs_in, proj, j, ch_qk);
            if (WPH == 4 || has_v) load_raw_proj(rv, proj, cw, j, ch_v_ld), load_raw_window(rv, at.cs_in, proj, j, ch_v_ld);
            if (WPH == 4 || is_g) gx = proj[(size_t)j * PW + g_at];
        }
        bf16_t* cso = at.cs_out + (size_t)j * at.cs_stride;
        // conv + silu, exact sum of squares over the head's 128 q (waves 0,1) / k (waves 2,3) channels
        float u = 0.f;
        if (is_qk) {
            u = conv_raw(rq);
            const double tot = wave_sum_d((double)u * (double)u);
            if (lane == 0) red[w] = tot;
        }
        float vv = 0.f;
        if (has_v) {
            vv = conv_raw(rv);
        }
        float g = 0.f, beta = 0.f;
        if (is_g) {                                                              // kernels.py:511-515
            const float gv = bf2f((bf16_t)gx);
            g = lane_value(decay_gate(gA, BF(gv + gdt)), 1);
            beta = lane_value(sigmoid_bf16(gv), 2);
        }
        __syncthreads();
        if (is_qk) {
            if (split == 0) store_window(cso, rq, ch_qk);
            const float ss = (float)(red[which * 2] + red[which * 2 + 1]);
            const float r = rsqrt_rn(ss / (float)DK + qk_eps());
            qk_s[which][tid & 127] = BF(BF(u * r) * sc);                         // kernels.py:507-510
        }
        if (has_v) {
            v_s[tid - V0] = vv;
            store_window(cso, rv, ch_v);
        }
        if (is_g && lane == 0) {
            gb_s[0] = g;
            gb_s[1] = beta;
        }
        __syncthreads();

        // ---- the recurrence over this thread's 8 columns of RS rows
        float q8[8], k8[8];
        {
            const float4 a = reinterpret_cast<const float4*>(qk_s[0])[c], b = reinterpret_cast<const float4*>(qk_s[0])[16 + c];
            const float4 d = reinterpret_cast<const float4*>(qk_s[1])[c], e = reinterpret_cast<const float4*>(qk_s[1])[16 + c];
            q8[0] = a.x; q8[1] = a.y; q8[2] = a.z; q8[3] = a.w; q8[4] = b.x; q8[5] = b.y; q8[6] = b.z; q8[7] = b.w;
            k8[0] = d.x; k8[1] = d.y; k8[2] = d.z; k8[3] = d.w; k8[4] = e.x; k8[5] = e.y; k8[6] = e.z; k8[7] = e.w;
        }
        const float gg = gb_s[0], bb = gb_s[1];
        const float kq = dot8_row16(k8, q8);

        f4* so4 = reinterpret_cast<f4*>(at.st_out + (size_t)j * at.st_stride + ((size_t)h * DV + row0) * DK);
        bf16_t* yo = y + (size_t)j * KD + h * DV + row0;
        float yb[RS];
#pragma unroll
        for (int i = 0; i < RS; i++) {
            const int row = i * GRPS + w * 4 + grp;
            float sv[8] = {s[i][0].x, s[i][0].y, s[i][0].z, s[i][0].w, s[i][1].x, s[i][1].y, s[i][1].z, s[i][1].w};
            const float yv = gdn_row_step(sv, k8, q8, v_s[row], gg, bb, kq);
            s[i][0] = f4{sv[0], sv[1], sv[2], sv[3]};
            s[i][1] = f4{sv[4], sv[5], sv[6], sv[7]};
            __builtin_nontemporal_store(s[i][0], so4 + row * (DK / 4) + c);
            __builtin_nontemporal_store(s[i][1], so4 + row * (DK / 4) + 16 + c);
            if (!NORM) {
                if (c == 0) yo[row] = f2bf(yv);
            } else {
                yb[i] = BF(yv);
            }
        }
        if (NORM) {
            // sum of squares of the head's 128 stored outputs: this lane's RS rows, the wavefront's 4 groups, the WPH wavefronts
            double ss = 0.0;
#pragma unroll
            for (int i = 0; i < RS; i++) ss += (double)yb[i] * yb[i];
            ss = groups_sum_d(ss);
            __shared__ double red_y[HPW][WPH];
            if (lane == 0) red_y[sub][w] = ss;
            __syncthreads();
            double tot = 0.0;
#pragma unroll
            for (int i = 0; i < WPH; i += 4)
                tot += (red_y[sub][i] + red_y[sub][i + 1]) + (red_y[sub][i + 2] + red_y[sub][i + 3]);
            const float inv = rsqrt_rn((float)tot / 128.f + eps);
            float mine = yb[0];
#pragma unroll
            for (int i = 1; i < RS; i++) mine = ((c % RS) == i) ? yb[i] : mine;
            if (c < RS) yo[nrow] = gated_out(bf2f((bf16_t)nz), ngw * (mine * inv));
        }
    }
}

// The same for a verify step whose workgroups have a quarter of a head or less: TOKENS tokens share one prologue.  Token by token, the inputs of
// each token but the first were asked for behind the stores of the one before (a wavefront's loads and stores share a counter, so such a load is
// waited for together with microseconds of stores), and two barriers and the string conv - sum - root stood in every token.  Here the
// inputs of a group come ahead of the state, convs, norms and gates of all its tokens are formed at once, the next group's inputs are asked for
// ahead of this group's stores, and the windows are stored behind the state.  The same bits.
// us in a HIP graph, token by token / here: 1 x 2 4.6 / 4.45, 7 x 2 6.75 / 6.55, 1 x 4 7.7 / 6.1, 5 x 3 8.2 / 7.0, 5 x 5 11.6 / 9.9, 3 x 8 16.1 / 12.8, 2 x 16 24.8 / 19.0;
// groups of two 6.5 / 7.6 / 10.1 at 1 x 4 .. 5 x 5.  A single token has no other to share with and would only load and keep the rows of three more: 1 x 1
// 3.3 / 3.8, 4 x 1 4.0 / 4.5, 7 x 1 4.65 / 5.4: gdn_tokens takes it.  With half a head the launch alone gains, too (16 x 4 16.5 / 16.1), but a step of eight layers of 16 x 4 rows takes 382.2 us
// against 378.9, and with whole heads the registers cost more than it gives (32 x 2 18.9 / 19.5): both go token by token.
constexpr int TOKENS = 4;
struct GroupIn {                        // one channel's raw input rows t0 - 3 .. t0 + TOKENS - 1, and its taps
    unsigned in[TOKENS + 3];
    uint2 c;
};
__device__ __forceinline__ float conv_raw(const GroupIn& r, int t) {
    return conv_silu(bf2f((bf16_t)r.in[t]), bf2f((bf16_t)r.in[t + 1]), bf2f((bf16_t)r.in[t + 2]), bf2f((bf16_t)r.in[t + 3]), r.c);
}
__device__ __forceinline__ void store_window(bf16_t* __restrict__ cs_out, const GroupIn& r, int t, int ch) {
#pragma unroll
    for (int i = 0; i < 3; i++) cs_out[i * CD + ch] = (bf16_t)r.in[t + 1 + i];     // kernels.py:531
}
template <int RS, class PlaceFn>
__device__ __forceinline__ void gdn_token_groups(const bf16_t* __restrict__ proj, const bf16_t* __restrict__ cw, const float* __restrict__ A_log,
                                                 const float* __restrict__ dt_bias, bf16_t* __restrict__ y, int M, int h, int split, PlaceFn place) {
    constexpr int GRPS = 16, ROWS = RS * GRPS;
    __shared__ double red[TOKENS][4];
    __shared__ __align__(16) float qk_s[TOKENS][2][DK];
    __shared__ float v_s[TOKENS][ROWS];
    __shared__ float gb_s[TOKENS][2];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), tid = threadIdx.x, lane = tid & 63, grp = lane >> 4, c = lane & 15;
    const int row0 = split * ROWS;
    // wavefronts 0, 1: q channels, 2, 3: k channels; v channels: the first ROWS threads (every load is unconditional); gates: wavefront 3
    const bool has_v = tid < ROWS, is_g = w == 3;
    const int which = w >> 1;                                    // 0: a q channel, 1: a k channel
    const int ch_qk = which * KD + h * DK + (tid & 127), ch_v = has_v ? 2 * KD + h * DV + row0 + tid : ch_qk;
    // gates: lane 2 t the decay gate of token t (reads a), lane 2 t + 1 its beta (reads b)
    const int g_at = CD + KD + HV * ((lane & 1) ^ 1) + h, g_tok = min(lane >> 1, TOKENS - 1);
    GroupIn rq, rv;
    unsigned gx;
    auto ask = [&](int t0) {                                     // a group's own rows (past the last token: the last one)
#pragma unroll
        for (int t = 0; t < TOKENS; t++) {
            const size_t at = (size_t)min(t0 + t, M - 1) * PW;
            rq.in[3 + t] = proj[at + ch_qk];
            rv.in[3 + t] = proj[at + ch_v];
        }
        gx = proj[(size_t)min(t0 + g_tok, M - 1) * PW + g_at];
    };
    ask(0);
    rq.c = *reinterpret_cast<const uint2*>(cw + (size_t)ch_qk * 4);
    rv.c = *reinterpret_cast<const uint2*>(cw + (size_t)ch_v * 4);
    const float gA = A_log[h], gdt = dt_bias[h];
    __builtin_amdgcn_sched_barrier(0);
    const Place at = place();
    if (__builtin_expect(!at.ok, 0)) {                           // (a skipped row, see above)
#pragma unroll
        for (int t = 0; t < TOKENS; t++) asm volatile("" ::"v"(rq.in[3 + t]), "v"(rv.in[3 + t]));
        asm volatile("" ::"v"(rq.c.x), "v"(rq.c.y), "v"(rv.c.x), "v"(rv.c.y));
        asm volatile("" ::"v"(gx), "s"(gA), "s"(gdt), "s"(at.par));
        __builtin_amdgcn_endpgm();
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
        rq.in[i] = at.cs_in[i * CD + ch_qk];
        rv.in[i] = at.cs_in[i * CD + ch_v];
    }
    __builtin_amdgcn_sched_barrier(0);           // keep the small loads ahead of the state loads in issue order
    f4 s[RS][2];
    {
        const f4* sin4 = reinterpret_cast<const f4*>(at.st_in + ((size_t)h * DV + row0) * DK);
#pragma unroll
        for (int i = 0; i < RS; i++) {
            const int row = i * GRPS + w * 4 + grp;
            s[i][0] = __builtin_nontemporal_load(sin4 + row * (DK / 4) + c);
            s[i][1] = __builtin_nontemporal_load(sin4 + row * (DK / 4) + 16 + c);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    // (nothing is converted, and so waited for, before the state has been requested)
#pragma unroll
    for (int i = 0; i < TOKENS + 3; i++) asm volatile("" : "+v"(rq.in[i]), "+v"(rv.in[i]));
    asm volatile("" : "+v"(gx));

    const float sc = which == 0 ? BF(INV_SCALE * INV_SCALE) : BF(INV_SCALE);       // kernels.py:492
    // groups of one length: five tokens are three and two (as four and one the last token waits for four tokens' stores)
    const int groups = (M + TOKENS - 1) / TOKENS, step = (M + groups - 1) / groups;         // (3 or 4 where there are several)
    for (int t0 = 0; t0 < M; t0 += step) {
        const int n = min(step, M - t0);                                         // (the same for the whole workgroup)
        // conv + silu, exact sums of squares over the head's 128 q (waves 0, 1) / k (waves 2, 3) channels
        float u[TOKENS], vv[TOKENS], gate = 0.f;
#pragma unroll
        for (int t = 0; t < TOKENS; t++) {
            u[t] = vv[t] = 0.f;
            if (t >= n) continue;
            u[t] = conv_raw(rq, t);
            const double tot = wave_sum_d((double)u[t] * (double)u[t]);
            if (lane == 0) red[t][w] = tot;
            if (has_v) vv[t] = conv_raw(rv, t);
        }
        if (is_g) {                                                              // kernels.py:511-515
            const float gv = bf2f((bf16_t)gx);
            const float g = decay_gate(gA, BF(gv + gdt)), beta = sigmoid_bf16(gv);
            gate = (lane & 1) ? beta : g;
        }
        __syncthreads();
        if (is_g && lane < 2 * TOKENS) gb_s[g_tok][lane & 1] = gate;
#pragma unroll
        for (int t = 0; t < TOKENS; t++) {
            if (t >= n) continue;
            const float ss = (float)(red[t][which * 2] + red[t][which * 2 + 1]);
            const float r = rsqrt_rn(ss / (float)DK + qk_eps());
            qk_s[t][which][tid & 127] = BF(BF(u[t] * r) * sc);                   // kernels.py:507-510
            if (has_v) v_s[t][tid] = vv[t];
        }
        __syncthreads();
        const GroupIn oq = rq, ov = rv;
        if (t0 + step < M) {                                                     // the next group's inputs, ahead of this one's stores
            const bool full = step == TOKENS;
#pragma unroll
            for (int i = 0; i < 3; i++) {
                rq.in[i] = full ? rq.in[TOKENS + i] : rq.in[TOKENS - 1 + i];
                rv.in[i] = full ? rv.in[TOKENS + i] : rv.in[TOKENS - 1 + i];
            }
            ask(t0 + step);
        }
#pragma unroll
        for (int t = 0; t < TOKENS; t++) {
            if (t >= n) break;
            const int j = t0 + t;
            // ---- the recurrence over this thread's 8 columns of RS rows
            float q8[8], k8[8];
#pragma unroll
            for (int e = 0; e < 8; e += 4) {
                const f4 a = reinterpret_cast<const f4*>(qk_s[t][0])[4 * e + c], b = reinterpret_cast<const f4*>(qk_s[t][1])[4 * e + c];
#pragma unroll
                for (int i = 0; i < 4; i++) q8[e + i] = a[i], k8[e + i] = b[i];
            }
            const float gg = gb_s[t][0], bb = gb_s[t][1];
            const float kq = dot8_row16(k8, q8);
            f4* so4 = reinterpret_cast<f4*>(at.st_out + (size_t)j * at.st_stride + ((size_t)h * DV + row0) * DK);
            bf16_t* yo = y + (size_t)j * KD + h * DV + row0;
#pragma unroll
            for (int i = 0; i < RS; i++) {
                const int row = i * GRPS + w * 4 + grp;
                float sv[8] = {s[i][0].x, s[i][0].y, s[i][0].z, s[i][0].w, s[i][1].x, s[i][1].y, s[i][1].z, s[i][1].w};
                const float yv = gdn_row_step(sv, k8, q8, v_s[t][row], gg, bb, kq);
                s[i][0] = f4{sv[0], sv[1], sv[2], sv[3]};
                s[i][1] = f4{sv[4], sv[5], sv[6], sv[7]};
                __builtin_nontemporal_store(s[i][0], so4 + row * (DK / 4) + c);
                __builtin_nontemporal_store(s[i][1], so4 + row * (DK / 4) + 16 + c);
                if (c == 0) yo[row] = f2bf(yv);
            }
            bf16_t* cso = at.cs_out + (size_t)j * at.cs_stride;
            if (split == 0) store_window(cso, oq, t, ch_qk);
            if (has_v) store_window(cso, ov, t, ch_v);
        }
    }
}

template <int RS>
__device__ __forceinline__ void split_id(int& b, int& h, int& split) {
    constexpr int NSPLIT = 8 / RS;
    const unsigned id = xcd_remap(blockIdx.x, gridDim.x);
    b = id / (HV * NSPLIT);
    const unsigned rem = id % (HV * NSPLIT);
    h = rem / NSPLIT;
    split = rem % NSPLIT;
}

__device__ __forceinline__ Place decode_place(bf16_t* conv_pool, float* ssm_pool, int slot, int p, int n_slots) {
    const int par = p & 1;                                       // batch.py:49-52: read buffer pos&1, write the other
    const bool ok = (unsigned)slot < (unsigned)n_slots;
    float* st = ssm_pool + (size_t)slot * HV * DV * DK;
    return {ok, par, conv_pool + (size_t)(slot * 2 + par) * 3 * CD, conv_pool + (size_t)(slot * 2 + (par ^ 1)) * 3 * CD, 0, st, st, 0};
}

// batch.deltanet_b (qwen35/batch.py:128-135): one token per row, pools updated in place
template <int RS>
__global__ __launch_bounds__(256) void gdn_decode_kernel(const bf16_t* __restrict__ proj, bf16_t* conv_pool,
                                                         const bf16_t* __restrict__ cw, const float* __restrict__ A_log,
                                                         const float* __restrict__ dt_bias, float* ssm_pool,
                                                         const int* __restrict__ slots, const int* __restrict__ pos,
                                                         bf16_t* __restrict__ y, int n_slots) {
    int b, h, split;
    split_id<RS>(b, h, split);
    const int slot = slots[b], p = pos[b];
    gdn_tokens<RS>(proj + (size_t)b * PW, cw, A_log, dt_bias, y + (size_t)b * KD, 1, h, split,
                   [&] { return decode_place(conv_pool, ssm_pool, slot, p, n_slots); });
}

// the same step with HPW heads of one row per workgroup (WPH wavefronts per head, whole heads only): the workgroup streams
// HPW * 64 KiB of contiguous state
template <int HPW, bool NORM = false, int WPH = 4>
__global__ __launch_bounds__(64 * WPH * HPW) void gdn_decode_wide_kernel(const bf16_t* __restrict__ proj, bf16_t* conv_pool,
                                                                         const bf16_t* __restrict__ cw, const float* __restrict__ A_log,
                                                                         const float* __restrict__ dt_bias, float* ssm_pool,
                                                                         const int* __restrict__ slots, const int* __restrict__ pos,
                                                                         bf16_t* __restrict__ y, int n_slots,
                                                                         const float* __restrict__ gw = nullptr, float eps = 0.f) {
    const unsigned id = xcd_remap(blockIdx.x, gridDim.x);
    const int b = id / (HV / HPW), h = (id % (HV / HPW)) * HPW + (HPW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / (64 * WPH)) : 0);
    const int slot = slots[b], p = pos[b];
    gdn_tokens<32 / WPH, HPW, NORM, WPH>(proj + (size_t)b * PW, cw, A_log, dt_bias, y + (size_t)b * KD, 1, h, 0,
                                         [&] { return decode_place(conv_pool, ssm_pool, slot, p, n_slots); }, gw, eps);
}

// batch_spec.deltanet_bm (qwen35/batch_spec.py:142-150): M chained tokens per sequence, snapshot pools in place
template <int RS, bool TAPS_LATE = false, bool GROUPS = (RS < 4)>
__global__ __launch_bounds__(256) void gdn_verify_kernel(const bf16_t* __restrict__ proj, bf16_t* conv_pool,
                                                         const bf16_t* __restrict__ cw, const float* __restrict__ A_log,
                                                         const float* __restrict__ dt_bias, float* ssm_pool,
                                                         const int* __restrict__ sslots, const int* __restrict__ sels,
                                                         const int* __restrict__ pars, bf16_t* __restrict__ y, int M,
                                                         int n_entries) {
    int b, h, split;
    split_id<RS>(b, h, split);
    const int ss = sslots[b], sl = sels[b], pr = pars[b];
    auto place = [&] {
        const int par = pr & 1;
        const size_t hs = (size_t)HV * DV * DK;
        const bool ok = (unsigned)ss < (unsigned)n_entries && (unsigned)sl < (unsigned)M;
        return Place{ok, par, conv_pool + ((size_t)(ss * 2 + par) * M + sl) * 3 * CD,
                     conv_pool + (size_t)(ss * 2 + (par ^ 1)) * M * 3 * CD, (size_t)3 * CD, ssm_pool + ((size_t)ss * M + sl) * hs,
                     ssm_pool + (size_t)ss * M * hs, hs};
    };
    if constexpr (GROUPS)
        gdn_token_groups<RS>(proj + (size_t)b * M * PW, cw, A_log, dt_bias, y + (size_t)b * M * KD, M, h, split, place);
    else
        gdn_tokens<RS, 1, false, 4, TAPS_LATE>(proj + (size_t)b * M * PW, cw, A_log, dt_bias, y + (size_t)b * M * KD, M, h, split, place);
}
template <int RS>
constexpr auto gdn_verify_single_kernel = gdn_verify_kernel<RS, false, false>;   // token by token

// kernels.deltanet (qwen35/kernels.py:555-567): one sequence, starts from snapshot sel[0], writes M fresh snapshots
template <int RS, bool GROUPS = (RS < 4)>
__global__ __launch_bounds__(256) void gdn_solo_kernel(const bf16_t* __restrict__ proj, const bf16_t* __restrict__ cs_snap,
                                                       const bf16_t* __restrict__ cw, const float* __restrict__ A_log,
                                                       const float* __restrict__ dt_bias, const float* __restrict__ st_snap,
                                                       const int* __restrict__ sel, bf16_t* __restrict__ y,
                                                       bf16_t* __restrict__ cs_out, float* __restrict__ st_out, int M,
                                                       int n_snap) {
    int b, h, split;
    split_id<RS>(b, h, split);
    const int sl = sel[0];
    auto place = [&] {
        const size_t hs = (size_t)HV * DV * DK;
        const bool ok = (unsigned)sl < (unsigned)n_snap;
        return Place{ok, 0, cs_snap + (size_t)sl * 3 * CD, cs_out, (size_t)3 * CD, st_snap + sl * hs, st_out, hs};
    };
    if constexpr (GROUPS)
        gdn_token_groups<RS>(proj, cw, A_log, dt_bias, y, M, h, split, place);
    else
        gdn_tokens<RS>(proj, cw, A_log, dt_bias, y, M, h, split, place);
}
template <int RS>
constexpr auto gdn_solo_single_kernel = gdn_solo_kernel<RS, false>;

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// rows per workgroup: few sequences -> split a head over more workgroups so the chip still fills
inline int pick_rs(int nseq, int rows_split) {
    if (rows_split == 128 || rows_split == 64 || rows_split == 32 || rows_split == 16) return rows_split / 16;
    if (nseq >= 32) return 8;
    if (nseq >= 8) return 4;
    if (nseq >= 4) return 2;
    return 1;
}

// The decode step's shape: whole heads per workgroup (1, 2 or 4) while B x 16 heads give every CU a workgroup (measured, us at
// 1 / 2 / 4 heads: B = 16 6.7 / 7.7 / 11.4, 24 11.9 / 9.8 / 12.1, 32 12.4 / 12.3 / 13.5, 48 19.2 / 21.2 / 18.5, 64 25.6 / 24.8 /
// 23.7), below that a head split over 2, 4 or 8 workgroups (B = 8: 5.5 us at 2 or 4 parts, B = 4: 4.5 us at 4).
// Beyond one round of four-head workgroups (B > 64) small workgroups balance the rounds better: half a head each (B = 96
// 38.1 against 39.5 us, B = 128 50.7 against 52.1), a whole head where the fused norm needs one.
inline int decode_heads_per_wg(int B) {
    const long heads = (long)B * HV, cus = cu_count();
    return heads > 4 * cus ? 1 : heads > 2 * cus ? 4 : heads > cus ? 2 : 1;
}
inline int decode_rs(int B) {                                    // 16-row groups per workgroup when a head is split
    const long heads = (long)B * HV, cus = cu_count();
    if (heads > 4 * cus) return 4;
    int rs = 8;
    while (rs > 1 && heads * (8 / rs) * 2 <= cus) rs >>= 1;
    return rs;
}

}  // namespace

#define QT_DISPATCH_RS(rs, KERNEL, nseq, stream, ...)                                                  \
    switch (rs) {                                                                                       \
        case 8: hipLaunchKernelGGL(KERNEL<8>, dim3((nseq) * HV * 1), dim3(256), 0, stream, __VA_ARGS__); break; \
        case 4: hipLaunchKernelGGL(KERNEL<4>, dim3((nseq) * HV * 2), dim3(256), 0, stream, __VA_ARGS__); break; \
        case 2: hipLaunchKernelGGL(KERNEL<2>, dim3((nseq) * HV * 4), dim3(256), 0, stream, __VA_ARGS__); break; \
        default: hipLaunchKernelGGL(KERNEL<1>, dim3((nseq) * HV * 8), dim3(256), 0, stream, __VA_ARGS__); break; \
    }

extern "C" {

int qt_gdn_decode_step(const void* proj, void* conv_pool, const void* conv_w, const float* A_log, const float* dt_bias,
                       float* ssm_pool, const int32_t* slots, const int32_t* pos, void* y, int B, int n_slots,
                       int rows_per_wg, hipStream_t stream) {
    if (!proj || !conv_pool || !conv_w || !A_log || !dt_bias || !ssm_pool || !slots || !pos || !y) return QT_ERR_NULL;
    if (B < 0 || n_slots <= 0) return QT_ERR_DIM;
    if (B == 0) return QT_OK;
    if (!aligned16(ssm_pool) || (reinterpret_cast<uintptr_t>(conv_w) & 7u)) return QT_ERR_ALIGN;
    // Many rows: 2 or 4 whole heads of a row per workgroup (128 / 256 KiB of contiguous state per workgroup); measured at
    // B = 64: 23.3 us against 26.0 us with one head per workgroup.  Few rows: split heads so the chip still fills.  The shape
    // that wins at every batch size measured (4 .. 64 rows) is the largest one that still gives every CU a workgroup.
    const int hpw = rows_per_wg == 512 ? 4 : rows_per_wg == 256 ? 2 : rows_per_wg != 0 ? 1 : decode_heads_per_wg(B);
    if (hpw == 4) {
        hipLaunchKernelGGL(gdn_decode_wide_kernel<4>, dim3(B * (HV / 4)), dim3(1024), 0, stream, (const bf16_t*)proj,
                           (bf16_t*)conv_pool, (const bf16_t*)conv_w, A_log, dt_bias, ssm_pool, slots, pos, (bf16_t*)y, n_slots);
    } else if (hpw == 2) {
        hipLaunchKernelGGL(gdn_decode_wide_kernel<2>, dim3(B * (HV / 2)), dim3(512), 0, stream, (const bf16_t*)proj,
                           (bf16_t*)conv_pool, (const bf16_t*)conv_w, A_log, dt_bias, ssm_pool, slots, pos, (bf16_t*)y, n_slots);
    } else {
        const int rs = rows_per_wg ? pick_rs(B, rows_per_wg) : decode_rs(B);
        QT_DISPATCH_RS(rs, gdn_decode_kernel, B, stream, (const bf16_t*)proj, (bf16_t*)conv_pool, (const bf16_t*)conv_w, A_log,
                       dt_bias, ssm_pool, slots, pos, (bf16_t*)y, n_slots);
    }
    QT_CHECK_LAUNCH();
    return QT_OK;
}

// batch.deltanet_b followed by batch.gnorm_rows (qwen35/batch.py:128-135, 338-343) in one launch: `out` receives the gated
// RMSNorm of the step's outputs (same bits as the two launches), the outputs themselves are not stored.
int qt_gdn_decode_step_gnorm(const void* proj, void* conv_pool, const void* conv_w, const float* A_log, const float* dt_bias,
                             float* ssm_pool, const int32_t* slots, const int32_t* pos, const float* gw, float eps, void* out, int B,
                             int n_slots, hipStream_t stream) {
    if (!proj || !conv_pool || !conv_w || !A_log || !dt_bias || !ssm_pool || !slots || !pos || !gw || !out) return QT_ERR_NULL;
    if (B < 0 || n_slots <= 0) return QT_ERR_DIM;
    if (B == 0) return QT_OK;
    if (!aligned16(ssm_pool) || (reinterpret_cast<uintptr_t>(conv_w) & 7u)) return QT_ERR_ALIGN;
#define QT_GNORM_LAUNCH(HPW_, WPH_)                                                                                                  \
    hipLaunchKernelGGL((gdn_decode_wide_kernel<HPW_, true, WPH_>), dim3(B * (HV / HPW_)), dim3(64 * WPH_ * HPW_), 0, stream, (const bf16_t*)proj, \
                       (bf16_t*)conv_pool, (const bf16_t*)conv_w, A_log, dt_bias, ssm_pool, slots, pos, (bf16_t*)out, n_slots, gw, eps)
    const int hpw = decode_heads_per_wg(B);
    if (hpw == 4) QT_GNORM_LAUNCH(4, 4);
    else if (hpw == 2) QT_GNORM_LAUNCH(2, 4);
    else if (4L * B * HV <= cu_count()) QT_GNORM_LAUNCH(1, 8);   // (8 against 4 wavefronts a head, us: 1 row 4.4 / 4.7, 4 rows 4.9 / 5.0, 8 rows 5.9 / 5.4)
    else QT_GNORM_LAUNCH(1, 4);
    QT_CHECK_LAUNCH();
    return QT_OK;
}

int qt_gdn_verify_step(const void* proj, void* conv_pool, const void* conv_w, const float* A_log, const float* dt_bias,
                       float* ssm_pool, const int32_t* sslots, const int32_t* sels, const int32_t* pars, void* y, int B,
                       int M, int n_entries, int rows_per_wg, hipStream_t stream) {
    if (!proj || !conv_pool || !conv_w || !A_log || !dt_bias || !ssm_pool || !sslots || !sels || !pars || !y) return QT_ERR_NULL;
    if (B < 0 || n_entries <= 0) return QT_ERR_DIM;
    if (M < 1 || M > 16) return QT_ERR_UNSUPPORTED;
    if (B == 0) return QT_OK;
    if (!aligned16(ssm_pool) || (reinterpret_cast<uintptr_t>(conv_w) & 7u)) return QT_ERR_ALIGN;
    const int rs = pick_rs(B, rows_per_wg);
    // More than a head per CU, in workgroups of half a head or more: the taps behind the state, so that a workgroup waits for its whole state before
    // it computes and stores: fewer stores of one between the loads of another (us, taps late / ahead: 24 x 4 23.9 / 25.1, 18 x 4 19.6 / 20.8, 32 x
    // 2 17.9 / 18.7).  With less the conv beside the state's loads wins (8 x 4 11.4 / 10.4, 12 x 4 14.1 / 13.9, 16 x 8 33.0 / 31.2).
    const long cus = cu_count();
    if (rs >= 4 && (long)B * HV > cus) {
        const dim3 grid(B * HV * (8 / rs));
        if (rs == 8)
            hipLaunchKernelGGL((gdn_verify_kernel<8, true>), grid, dim3(256), 0, stream, (const bf16_t*)proj, (bf16_t*)conv_pool, (const bf16_t*)conv_w,
                               A_log, dt_bias, ssm_pool, sslots, sels, pars, (bf16_t*)y, M, n_entries);
        else
            hipLaunchKernelGGL((gdn_verify_kernel<4, true>), grid, dim3(256), 0, stream, (const bf16_t*)proj, (bf16_t*)conv_pool, (const bf16_t*)conv_w,
                               A_log, dt_bias, ssm_pool, sslots, sels, pars, (bf16_t*)y, M, n_entries);
        QT_CHECK_LAUNCH();
        return QT_OK;
    }
    // Quarters of a head in groups of tokens take 142 registers, so that three workgroups fit a CU, token by token 120 and four.  With that they go where it
    // makes a round of workgroups less (us, groups / token by token, rows_per_wg = 32: 13 x 4 17.4 / 15.1, 16 x 2 11.4 / 10.4, 16 x 4 21.9 / 17.2, 30 x 4
    // 35.1 / 32.8, 32 x 2 23.4 / 21.7; with as many rounds 12 x 4 12.6 / 12.8, 17 x 4 21.6 / 22.4, 24 x 4 24.6 / 26.4).
    auto rounds = [&](long per_cu) { return ((long)B * HV * 4 + per_cu * cus - 1) / (per_cu * cus); };
    if (M == 1 || (rs == 2 && rounds(3) > rounds(4))) {
        QT_DISPATCH_RS(rs, gdn_verify_single_kernel, B, stream, (const bf16_t*)proj, (bf16_t*)conv_pool, (const bf16_t*)conv_w, A_log,
                       dt_bias, ssm_pool, sslots, sels, pars, (bf16_t*)y, M, n_entries);
    } else {
        QT_DISPATCH_RS(rs, gdn_verify_kernel, B, stream, (const bf16_t*)proj, (bf16_t*)conv_pool, (const bf16_t*)conv_w, A_log,
                       dt_bias, ssm_pool, sslots, sels, pars, (bf16_t*)y, M, n_entries);
    }
    QT_CHECK_LAUNCH();
    return QT_OK;
}

int qt_gdn_deltanet(const void* proj, const void* conv_snap, const void* conv_w, const float* A_log, const float* dt_bias,
                    const float* ssm_snap, const int32_t* sel, void* y, void* cs_out, float* st_out, int M, int n_snap,
                    int rows_per_wg, hipStream_t stream) {
    if (!proj || !conv_snap || !conv_w || !A_log || !dt_bias || !ssm_snap || !sel || !y || !cs_out || !st_out) return QT_ERR_NULL;
    if (n_snap <= 0) return QT_ERR_DIM;
    if (M < 1 || M > 16) return QT_ERR_UNSUPPORTED;
    if (!aligned16(ssm_snap) || !aligned16(st_out) || (reinterpret_cast<uintptr_t>(conv_w) & 7u)) return QT_ERR_ALIGN;
    const int rs = pick_rs(1, rows_per_wg);
    if (M == 1) {
        QT_DISPATCH_RS(rs, gdn_solo_single_kernel, 1, stream, (const bf16_t*)proj, (const bf16_t*)conv_snap, (const bf16_t*)conv_w, A_log,
                       dt_bias, ssm_snap, sel, (bf16_t*)y, (bf16_t*)cs_out, st_out, M, n_snap);
    } else {
        QT_DISPATCH_RS(rs, gdn_solo_kernel, 1, stream, (const bf16_t*)proj, (const bf16_t*)conv_snap, (const bf16_t*)conv_w, A_log,
                       dt_bias, ssm_snap, sel, (bf16_t*)y, (bf16_t*)cs_out, st_out, M, n_snap);
    }
    QT_CHECK_LAUNCH();
    return QT_OK;
}

}  // extern "C"
