// The elementwise steps either side of the attention kernels of a full-attention layer, for gfx950: q / k RMSNorm, partial
// rotary embedding (the first 64 of 256 features, half-split pairing, theta = 1e7) and the output gate o * sigmoid(gate).
// Replaces the MLX graph ops of the reference's layer (qwen35/batch.py:505-513, qwen35/model.py:154-169):
//     qkv row = [ (q_h[256] | gate_h[256]) for h = 0..7 | k[2][256] | v[2][256] ]                         (5120 bf16)
//     q = rope(rms_norm(q_h, q_norm), pos),  k = rope(rms_norm(k, k_norm), pos),  v = v
//     out = o * sigmoid(gate)
// Arithmetic contract (fixed here so that a CPU restatement reproduces every bf16 value): sum of squares exact, rounded to
// float once; inv = correctly rounded 1/sqrt(ss/256 + eps); t = BF(x * inv); y = BF(w * t) (weight bf16); rotary angle
// theta = float(pos) * freq_i with freq_i = float(1e7^(-2 i / 64)); cos / sin = the double-precision libm values rounded to
// float; y1' = BF(y1 * c - y2 * s), y2' = BF(y1 * s + y2 * c), each product and the sum rounded to float separately;
// gate: BF(o * sigmoid_bf16(g)) with the bf16 sigmoid of the GatedDeltaNet path (qwen35/mslib.py:16-20).
#include "qt_common.h"

using namespace qt;

namespace {

constexpr int QKV_W = AH * 2 * AD + 2 * AKV * AD;      // 5120
constexpr int ROPE_DIM = 64;

__constant__ float rope_freq[ROPE_DIM / 2] = {
    1.0f, 0.604296386f, 0.365174115f, 0.220673412f, 0.133352146f, 0.0805842206f, 0.0486967526f, 0.0294272713f,
    0.0177827943f, 0.0107460786f, 0.00649381615f, 0.0039241896f, 0.00237137382f, 0.00143301254f, 0.000865964335f,
    0.000523299095f, 0.000316227757f, 0.0001910953f, 0.0001154782f, 6.97830619e-05f, 4.21696495e-05f,
    2.54829683e-05f, 1.5399266e-05f, 9.3057206e-06f, 5.62341347e-06f, 3.39820826e-06f, 2.05352512e-06f,
    1.24093776e-06f, 7.49894184e-07f, 4.5315835e-07f, 2.73841977e-07f, 1.65481708e-07f};

// One wavefront per row r = b * M + j (position pos[b] + j), four rows per workgroup.  The row's twelve 256-wide vectors (8 q heads, 2
// k heads, 2 v heads) are taken four at a time, one per 16-lane group: lane c of a group holds elements 8 c .. + 7 and 128 + 8 c ..
// + 7, so every load and store is 16 bytes per lane and all six loads of a row are in flight at once; a sum of squares needs
// four DPP steps, and no exchange leaves the wavefront.  The row's 32 (cos, sin) pairs come from the table of rope_table_kernel
// where it covers the position, else lanes 0..31 evaluate one each (double-precision libm, the expensive part: the same
// expression, so the same bits).
// Bound by the bytes it moves (12 KiB in and out per row).  With the table, 1024 / 2048 / 4096 / 8192 rows 7.6 / 11.1 / 17.8 / 29.3
// us with a workgroup per row, 8 bytes per lane and the sums over 64 lanes through LDS; now 5.4 / 8.6 / 13.9 / 25.0 us (4 TB/s).
// Nontemporal stores would take another 1 us off this kernel at 2048 rows, and cost the attention kernel that reads q next 18 us
// at 8192.
__global__ __launch_bounds__(256) void attn_qkv_prep_kernel(const bf16_t* __restrict__ qkv, const bf16_t* __restrict__ q_norm,
                                                            const bf16_t* __restrict__ k_norm, const int* __restrict__ pos,
                                                            bf16_t* __restrict__ q, bf16_t* __restrict__ k, bf16_t* __restrict__ v,
                                                            long R, int M, float eps, const float2* __restrict__ table,
                                                            int table_positions) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4), aligned(8)));      // the entry points ask for 8-byte alignment only
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    __shared__ __align__(16) float2 cs_s[4][ROPE_DIM / 2];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, rr = lane >> 4, c = lane & 15;
    const long r = (long)blockIdx.x * 4 + w;
    if (r >= R) return;
    // vector t of the group: q heads rr and 4 + rr, then (k0, k1, v0, v1)[rr]
    const bf16_t* row = qkv + r * QKV_W + 8 * c;
    u32x4 x[3][2], wn[2][2];
#pragma unroll
    for (int hf = 0; hf < 2; hf++) {
        x[0][hf] = *reinterpret_cast<const u32x4*>(row + rr * 2 * AD + 128 * hf);
        x[1][hf] = *reinterpret_cast<const u32x4*>(row + (4 + rr) * 2 * AD + 128 * hf);
        x[2][hf] = *reinterpret_cast<const u32x4*>(row + AH * 2 * AD + rr * AD + 128 * hf);
        wn[0][hf] = *reinterpret_cast<const u32x4*>(q_norm + 8 * c + 128 * hf);
        wn[1][hf] = *reinterpret_cast<const u32x4*>(k_norm + 8 * c + 128 * hf);
    }
    const int ip = pos[(unsigned)r / (unsigned)M] + (int)((unsigned)r % (unsigned)M);
    if (lane < ROPE_DIM / 2) {
        if (ip >= 0 && ip < table_positions) {                   // (table_positions = 0 without a table)
            cs_s[w][lane] = table[(size_t)ip * (ROPE_DIM / 2) + lane];
        } else {
            const float th = __fmul_rn((float)ip, rope_freq[lane]);
            cs_s[w][lane] = make_float2((float)cos((double)th), (float)sin((double)th));
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    f32x4 cs[4];                                                  // pairs 8 (c & 3) .. + 7: (cos, sin, cos, sin) each (lanes c < 8 use them)
#pragma unroll
    for (int i = 0; i < 4; i++) cs[i] = reinterpret_cast<const f32x4*>(&cs_s[w][8 * (c & 3)])[i];
    // v is a plain copy into the contiguous [R,2,256] layout
    if (rr >= 2) {
#pragma unroll
        for (int hf = 0; hf < 2; hf++) *reinterpret_cast<u32x4*>(v + (r * AKV + rr - 2) * AD + 8 * c + 128 * hf) = x[2][hf];
    }
#pragma unroll
    for (int t = 0; t < 3; t++) {
        const u32x4(&wt)[2] = wn[t == 2 ? 1 : 0];
        double ss = 0.0;
#pragma unroll
        for (int hf = 0; hf < 2; hf++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const double lo = (double)lo_bf(x[t][hf][j]), hi = (double)hi_bf(x[t][hf][j]);
                ss = fma(hi, hi, fma(lo, lo, ss));
            }
        const float inv = rsqrt_rn((float)row16_sum_d(ss) / (float)AD + eps);
        u32x4 y[2];
#pragma unroll
        for (int hf = 0; hf < 2; hf++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t n2 = pack2_bf(lo_bf(x[t][hf][j]) * inv, hi_bf(x[t][hf][j]) * inv);
                y[hf][j] = pack2_bf(lo_bf(wt[hf][j]) * lo_bf(n2), hi_bf(wt[hf][j]) * hi_bf(n2));
            }
        // rotary embedding of features 0..63: lanes 0..3 of a group hold x1 = features 0..31, lanes 4..7 their partners 32..63 (lane
        // c ^ 4 = the half row mirrored, then every quad reversed)
        u32x4 o;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int m = __builtin_amdgcn_update_dpp(0, (int)y[0][j], 0x141, 0xF, 0xF, true);
            o[j] = (unsigned)__builtin_amdgcn_update_dpp(0, m, 0x1B, 0xF, 0xF, true);
        }
        if (c < 8) {
            // The two products and their sum are rounded one by one.  Plain operators inside a contract(off) block: the
            // __fmul_rn / __fadd_rn helpers are ordinary operators compiled elsewhere, which the compiler contracts into one
            // fused multiply-add after inlining (a bf16 value in ~10^5 then rounds the other way).
#pragma clang fp contract(off)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float a0 = lo_bf(y[0][j]) * cs[j][0], b0 = lo_bf(o[j]) * cs[j][1];
                const float a1 = hi_bf(y[0][j]) * cs[j][2], b1 = hi_bf(o[j]) * cs[j][3];
                y[0][j] = c < 4 ? pack2_bf(a0 - b0, a1 - b1)     // y1 c - y2 s
                                : pack2_bf(b0 + a0, b1 + a1);    // y1 s + y2 c
            }
        }
        bf16_t* dst = t < 2 ? q + (r * AH + 4 * t + rr) * AD : k + (r * AKV + rr) * AD;
        if (t < 2 || rr < 2) {
#pragma unroll
            for (int hf = 0; hf < 2; hf++) *reinterpret_cast<u32x4*>(dst + 8 * c + 128 * hf) = y[hf];
        }
    }
}

// (cos, sin) of every rotary angle of positions 0 .. n_pos - 1, exactly the values the kernel above evaluates per row:
// table[p][i] = ((float)cos((double)th), (float)sin((double)th)), th = float(p) * rope_freq[i] rounded to float
__global__ __launch_bounds__(256) void rope_table_kernel(float2* __restrict__ table, int n_pos) {
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long)n_pos * (ROPE_DIM / 2)) return;
    const int p = (int)(t / (ROPE_DIM / 2)), i = (int)(t % (ROPE_DIM / 2));
    const float th = __fmul_rn((float)p, rope_freq[i]);
    table[t] = make_float2((float)cos((double)th), (float)sin((double)th));
}

// out[r][h*256 + d] = BF(o[r][h][d] * sigmoid_bf16(gate_h[d])), gate_h = qkv[r][h*512 + 256 ..]; 8 elements per thread.
// Moves 12 KiB per row.  With the sigmoid's boundary tests, IEEE division and fallbacks in every lane it was bound by the vector ALU
// (about 60 instructions an element, 19 us of issue at 8192 rows); with 18 an element, us in a graph over rotating rows: 64 rows 3.3 -> 2.3,
// 333 3.9 -> 2.9, 2048 8.7 -> 6.2, 8192 23.8 -> 17.6 (5.7 TB/s).
__global__ __launch_bounds__(256) void attn_out_gate_kernel(const bf16_t* __restrict__ o, const bf16_t* __restrict__ qkv,
                                                            bf16_t* __restrict__ out, long R) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;       // one 8-element group: AH * AD / 8 = 256 groups per row
    const long r = i >> 8;
    if (r >= R) return;
    const int c = (int)(i & 255), h = c >> 5, d = (c & 31) * 8;
    const uint4 ov = *reinterpret_cast<const uint4*>(o + (r * AH + h) * AD + d);
    const uint4 gv = *reinterpret_cast<const uint4*>(qkv + r * QKV_W + h * 2 * AD + AD + d);
    const uint32_t x[4] = {ov.x, ov.y, ov.z, ov.w}, g[4] = {gv.x, gv.y, gv.z, gv.w};
    uint32_t sg[4], p[4];
    u16x2 most = {0, 0};                                         // the largest magnitudes, as bits: a NaN is larger than any number
#pragma unroll
    for (int e = 0; e < 4; e++) {
        sg[e] = sigmoid_bf16_small2(g[e]);
        most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, g[e] & 0x7fff7fffu));
    }
    if (__builtin_expect(max(most.x, most.y) > (__float_as_uint(SIGMOID_FAST_MAX) >> 16), 0)) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (fabsf(lo_bf(g[e])) <= SIGMOID_FAST_MAX && fabsf(hi_bf(g[e])) <= SIGMOID_FAST_MAX) continue;
            sg[e] = pack2_bf(sigmoid_bf16_any(lo_bf(g[e])), sigmoid_bf16_any(hi_bf(g[e])));
        }
    }
#pragma unroll
    for (int e = 0; e < 4; e++) p[e] = pack2_bf(lo_bf(x[e]) * lo_bf(sg[e]), hi_bf(x[e]) * hi_bf(sg[e]));
    *reinterpret_cast<uint4*>(out + (r * AH + h) * AD + d) = make_uint4(p[0], p[1], p[2], p[3]);
}

}  // namespace

extern "C" {

// rope_table: null, or the (cos, sin) pairs of positions 0 .. table_positions - 1 as qt_rope_table_build writes them; rows at
// positions beyond the table evaluate their pairs themselves, with the same bits
int qt_attn_qkv_prep_table(const void* qkv, const void* q_norm, const void* k_norm, const int32_t* pos, const void* rope_table,
                           int table_positions, void* q, void* k, void* v, long R, int M, float eps, hipStream_t stream) {
    if (!qkv || !q_norm || !k_norm || !pos || !q || !k || !v) return QT_ERR_NULL;
    if (R < 0 || M < 1 || R % M || table_positions < 0) return QT_ERR_DIM;
    if (R == 0) return QT_OK;
    for (const void* p : {qkv, q_norm, k_norm, rope_table, (const void*)q, (const void*)k, (const void*)v})
        if (reinterpret_cast<uintptr_t>(p) & 7u) return QT_ERR_ALIGN;
    hipLaunchKernelGGL(attn_qkv_prep_kernel, dim3((unsigned)((R + 3) / 4)), dim3(256), 0, stream, (const bf16_t*)qkv, (const bf16_t*)q_norm,
                       (const bf16_t*)k_norm, pos, (bf16_t*)q, (bf16_t*)k, (bf16_t*)v, R, M, eps, (const float2*)rope_table,
                       rope_table ? table_positions : 0);
    QT_CHECK_LAUNCH();
    return QT_OK;
}
int qt_attn_qkv_prep(const void* qkv, const void* q_norm, const void* k_norm, const int32_t* pos, void* q, void* k, void* v, long R,
                     int M, float eps, hipStream_t stream) {
    return qt_attn_qkv_prep_table(qkv, q_norm, k_norm, pos, nullptr, 0, q, k, v, R, M, eps, stream);
}

int qt_rope_table_build(void* table, int n_pos, hipStream_t stream) {
    if (!table) return QT_ERR_NULL;
    if (n_pos < 0) return QT_ERR_DIM;
    if (reinterpret_cast<uintptr_t>(table) & 15u) return QT_ERR_ALIGN;
    if (n_pos == 0) return QT_OK;
    const long n = (long)n_pos * (ROPE_DIM / 2);
    hipLaunchKernelGGL(rope_table_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, (float2*)table, n_pos);
    QT_CHECK_LAUNCH();
    return QT_OK;
}

int qt_attn_out_gate(const void* o, const void* qkv, void* out, long R, hipStream_t stream) {
    if (!o || !qkv || !out) return QT_ERR_NULL;
    if (R < 0) return QT_ERR_DIM;
    if (R == 0) return QT_OK;
    for (const void* p : {o, qkv, (const void*)out})
        if (reinterpret_cast<uintptr_t>(p) & 15u) return QT_ERR_ALIGN;
    hipLaunchKernelGGL(attn_out_gate_kernel, dim3((unsigned)R), dim3(256), 0, stream, (const bf16_t*)o, (const bf16_t*)qkv,
                       (bf16_t*)out, R);
    QT_CHECK_LAUNCH();
    return QT_OK;
}

}  // extern "C"
