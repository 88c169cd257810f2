// qh_mmq81.hip -- the Q8_1 MMQ arithmetic mode (hip_gemm_q8_1_mmq): ggml-cuda's
// int8 MMQ rounding for Q4_K and Q6_K, bit-exact to the reference's CPU oracles
// gemm_q4k_q8_1_mmq[_stream_k] / gemm_q6k_q8_1_mmq[_stream_k]
// (src/dequant.rs:202-645):
//   * activations quantised per 32 values to Q8_1: max |x| and the sum over 8
//     lanes of 4 values, combined in XOR order 4, 2, 1; q = round(x * 127/max)
//     (half away from zero); scale 1 / (127/max), f16-rounded for Q4_K (with the
//     f16-rounded sum), kept in f32 for Q6_K (quantize_q8_1_mmq_d4);
//   * Q4_K: per 32-weight group, f16-rounded d*sc and -dmin*m, integer dot,
//     acc = fma(cs * scale, dot, acc); acc = fma(cm, sum, acc);
//   * Q6_K: per 128-value half, fragment = sum over 4 groups of fma(scale,
//     s1*dot1 + s2*dot2, .), acc = fma(d, fragment, acc);
//   * optional stream-K split (cuda_stream_k_cut): the accumulation restarts at
//     the cut superblock and the result is tail + prefix.
// The integer dots are exact, so they run on v_mfma_i32_16x16x32_i8 (K = 32 is
// one Q8_1 group); each lane then adds its four outputs in exactly that order.
// A workgroup (16 tokens x 128 columns, 8 wavefronts of 16 columns) quantises
// each 256-value block of its tokens once into LDS, one block ahead of its use.
// The calls share no scratch.  This is a compatibility mode for ggml-identical
// results, not the fast batched path (qh_gemm.hip).
#include "qh_internal.h"

#define QM_T 16   // tokens per workgroup
#define QM_W 8    // wavefronts per workgroup, 16 columns each
#define QM_C (16 * QM_W)

typedef int qm_i32x4 __attribute__((ext_vector_type(4)));
typedef float qm_f32x4 __attribute__((ext_vector_type(4)));
typedef float qm_f32x2 __attribute__((ext_vector_type(2)));

QH_DEV float qm_f16r(float v) { return (float)(_Float16)v; }  // round to nearest even, as f32_to_f16_round_to_even

// Stream-K cut of output (row, column): cuda_stream_k_cut (src/dequant.rs:338-374).
QH_DEV int qm_cut(int row, int column, int in_dim, int out_dim, int ref_rows, int mps) {
    if (ref_rows <= 0 || mps <= 0 || in_dim % 256) return -1;
    const long long bpt = in_dim / 256, tx = (ref_rows + 127) / 128, ty = (out_dim + 127) / 128, tc = tx * ty;
    const long long waves = (tc + mps - 1) / mps, eff = 100 * tc / (mps * waves);
    const long long grid = eff >= 90 ? tc : mps;
    if (grid == 0 || tc % grid == 0) return -1;
    const long long tile = (long long)(column / 128) * tx + row / 128, ts = tile * bpt, te = ts + bpt,
                    tot = tc * bpt;
    // the first boundary block * tot / grid inside (ts, te)
    long long b = (ts * grid) / tot + 1;
    for (; b < grid; b++) {
        const long long bd = b * tot / grid;
        if (bd >= te) break;
        if (bd > ts) return (int)(bd - ts);
    }
    return -1;
}

// Q8_1 of 8 of a 32-value group's values: the four threads of a quad hold
// values 4j .. 4j + 3 (v[0..3]) and 16 + 4j .. (v[4..7]), i.e. the reference's
// lanes j and j + 4, and the XOR order 4, 2, 1 is the add of the thread's own two
// lanes, then the quad's xor 2 and xor 1 (a sum's operand order does not matter).
template <bool Q6>
QH_DEV void qm_quantise(const float* v, uint32_t& q0, uint32_t& q1, float& scale, float& sum) {
    float pm[2], ps[2];
#pragma unroll
    for (int l = 0; l < 2; l++) {
        pm[l] = fmaxf(fmaxf(fmaxf(fmaxf(0.f, fabsf(v[4 * l])), fabsf(v[4 * l + 1])), fabsf(v[4 * l + 2])),
                      fabsf(v[4 * l + 3]));
        ps[l] = ((v[4 * l] + v[4 * l + 1]) + v[4 * l + 2]) + v[4 * l + 3];
    }
    float mx = fmaxf(pm[0], pm[1]), s = ps[0] + ps[1];
    mx = fmaxf(mx, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mx), 0x4E, 0xF, 0xF, false)));
    mx = fmaxf(mx, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mx), 0xB1, 0xF, 0xF, false)));
    s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x4E, 0xF, 0xF, false));
    s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0xB1, 0xF, 0xF, false));
    const float inv = mx == 0.f ? 0.f : __fdiv_rn(127.f, mx);
    uint32_t w[2];
#pragma unroll
    for (int l = 0; l < 2; l++) {
        int q[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float rq = inv != 0.f ? roundf(v[4 * l + i] * inv) : 0.f;
            rq = fminf(fmaxf(rq, -128.f), 127.f);
            q[i] = (int)rq;
        }
        w[l] = ((uint32_t)q[0] & 0xFFu) | (((uint32_t)q[1] & 0xFFu) << 8) | (((uint32_t)q[2] & 0xFFu) << 16) |
               ((uint32_t)q[3] << 24);
    }
    q0 = w[0];
    q1 = w[1];
    const float sc = inv == 0.f ? 0.f : __fdiv_rn(1.f, inv);
    scale = Q6 ? sc : qm_f16r(sc);
    sum = Q6 ? 0.f : qm_f16r(s);
}

// What bounds it: the f32 chain per output, four (Q4_K: cvt, mul, two fma) VALU
// operations per output and 32-value group, which no split of K may shorten (the
// order is the result); so tiles are small, 16 x 16 outputs per wavefront, to
// have enough wavefronts.  4096 x 4096 Q4_K at 128 tokens: one thread per output
// with byte loads and v_dot4 275 us, this kernel 30.9 us.
template <bool Q6>
__global__ __launch_bounds__(64 * QM_W) void qh_mmq_q81(const uint8_t* __restrict__ W, const float* __restrict__ x,
                                                        float* __restrict__ y, int in_dim, int out_dim, int rows,
                                                        int ref_rows, int mps) {
    constexpr int BB = Q6 ? 210 : 144, CH = Q6 ? 14 : 9, LAST = BB - 16, RS = 16 * CH;  // staged line: 16-byte slices
    constexpr int RP = Q6 ? RS + 16 : RS;  // line stride (240: 16 lines on distinct banks)
    constexpr int NL = (16 * CH + 63) / 64;
    // quantised tokens of two blocks in A-operand order: group g, k half kg (8
    // values), token m at 8 (64 g + 16 kg + m); their scales and sums [g][token]
    __shared__ __align__(16) unsigned char qa[2][8 * 512];
    __shared__ __align__(16) float qs[2][8 * QM_T], qm[2][8 * QM_T];
    __shared__ __align__(16) unsigned char wt[QM_W][16 * RP];
    __shared__ __align__(16) qm_f32x2 wsc[QM_W][Q6 ? 1 : 8 * 16];  // Q4_K: (d sc, -dmin m) of [group][column]
    const int T = threadIdx.x, lane = T & 63, w = T >> 6, n = lane & 15, kg = lane >> 4;
    const int row0 = blockIdx.y * QM_T, col0 = blockIdx.x * QM_C + 16 * w, nsb = in_dim / 256;
    // The whole tile lies in one 128 x 128 tile of the reference's launch, so
    // the cut is the workgroup's.
    const int cut = qm_cut(row0, blockIdx.x * QM_C, in_dim, out_dim, ref_rows, mps);

    // weight slices of this lane (columns past the matrix re-read its last one)
    const uint8_t* wp[NL];
#pragma unroll
    for (int h = 0; h < NL; h++) {
        const int q = 64 * h + lane < 16 * CH ? 64 * h + lane : 16 * CH - 1, r = q / CH, c = q - r * CH;
        const int col = col0 + r < out_dim ? col0 + r : out_dim - 1;
        wp[h] = W + (size_t)col * nsb * BB + (c == CH - 1 ? LAST : 16 * c);
    }
    typedef qh_u32x4 u32x4u __attribute__((aligned(1)));
    qh_u32x4 wr[NL];
    auto load_w = [&](int b) {
#pragma unroll
        for (int h = 0; h < NL; h++) wr[h] = *reinterpret_cast<const u32x4u*>(wp[h] + (size_t)b * BB);
    };
    // this thread's share of a block's tokens: token xt, group xg, quad lane xj
    const int xt = T >> 5, xg = (T >> 2) & 7, xj = T & 3;
    const bool xlive = row0 + xt < rows;
    const float4* xp = reinterpret_cast<const float4*>(x + (size_t)(xlive ? row0 + xt : rows - 1) * in_dim + 32 * xg + 4 * xj);
    float4 x0, x1;
    auto load_x = [&](int b) {
        x0 = xp[64 * b];
        x1 = xp[64 * b + 4];
    };
    auto put_x = [&](int b) {
        float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = xlive ? v[i] : 0.f;
        uint32_t q0, q1;
        float sc, sm;
        qm_quantise<Q6>(v, q0, q1, sc, sm);
        unsigned char* a = qa[b & 1] + 512 * xg + 128 * (xj >> 1) + 8 * xt + 4 * (xj & 1);
        *reinterpret_cast<uint32_t*>(a) = q0;
        *reinterpret_cast<uint32_t*>(a + 256) = q1;
        if (xj == 0) {
            qs[b & 1][QM_T * xg + xt] = sc;
            if constexpr (!Q6) qm[b & 1][QM_T * xg + xt] = sm;
        }
    };
    load_x(0);
    load_w(0);
    put_x(0);
    if (nsb > 1) load_x(1);
    __syncthreads();

    qm_f32x4 acc = {0.f, 0.f, 0.f, 0.f}, prefix = acc;
    const unsigned char* line = wt[w] + n * RP;
    for (int b = 0; b < nsb; b++) {
        // stage block b's weights (this wavefront's own lines), refill
#pragma unroll
        for (int h = 0; h < NL; h++) {
            const int q = 64 * h + lane, r = q / CH, c = q - r * CH;
            if (q < 16 * CH) *reinterpret_cast<qh_u32x4*>(wt[w] + r * RP + 16 * c) = wr[h];
        }
        if (b + 1 < nsb) load_w(b + 1);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if constexpr (!Q6) {
            // lane (column n, kg) rounds the scales of groups 2 kg and 2 kg + 1
            const qh_u32x4 h = *reinterpret_cast<const qh_u32x4*>(line);
            const float d = qh_f16(h.x), dmin = qh_f16(h.x >> 16);
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int g = 2 * kg + i, sh = 8 * (g & 3);  // get_scale_min_k4 (src/dequant.rs:1471-1480)
                const uint32_t s0 = (h.y >> sh) & 0xFFu, s1 = (h.z >> sh) & 0xFFu, s2 = (h.w >> sh) & 0xFFu;
                const uint32_t sc = g < 4 ? s0 & 63u : (s2 & 0x0Fu) | ((s0 >> 6) << 4);
                const uint32_t m = g < 4 ? s1 & 63u : (s2 >> 4) | ((s1 >> 6) << 4);
                wsc[w][16 * g + n] = qm_f32x2{qm_f16r(d * (float)sc), qm_f16r(-dmin * (float)m)};
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        if (b == cut) {
            prefix = acc;
            acc = qm_f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const unsigned char* A = qa[b & 1] + 128 * kg + 8 * n;
        const float* S = qs[b & 1] + 4 * kg;
        const qm_i32x4 zero = {0, 0, 0, 0};
        if constexpr (!Q6) {
            const float* M = qm[b & 1] + 4 * kg;
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const qh_u32x2 qq = *reinterpret_cast<const qh_u32x2*>(line + 16 + 32 * p + 8 * kg);
#pragma unroll
                for (int nib = 0; nib < 2; nib++) {
                    const int g = 2 * p + nib;
                    const qh_u32x2 bw = nib ? (qq >> 4) & 0x0F0F0F0Fu : qq & 0x0F0F0F0Fu;
                    const qm_i32x4 dot = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                        *reinterpret_cast<const long*>(A + 512 * g), __builtin_bit_cast(long, bw), zero, 0, 0, 0);
                    const qm_f32x2 c = wsc[w][16 * g + n];
                    const qm_f32x4 s4 = *reinterpret_cast<const qm_f32x4*>(S + QM_T * g);
                    const qm_f32x4 m4 = *reinterpret_cast<const qm_f32x4*>(M + QM_T * g);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float ds = c.x * s4[r];
                        acc[r] = fmaf(ds, (float)dot[r], acc[r]);
                        acc[r] = fmaf(c.y, m4[r], acc[r]);
                    }
                }
            }
        } else {
            const float d6 = qh_f16(*reinterpret_cast<const uint16_t*>(line + RS - 2));
            const qh_u32x4 sc = *reinterpret_cast<const qh_u32x4*>(line + 192);
            const uint32_t m1 = kg < 2 ? 0xFFFFFFFFu : 0u;  // values 0 .. 15 of the group, values 16 .. 31
#pragma unroll
            for (int f = 0; f < 2; f++) {
                const qh_u32x2 qh = *reinterpret_cast<const qh_u32x2*>(line + 128 + 32 * f + 8 * kg);
                qh_u32x2 ql[2];
                ql[0] = *reinterpret_cast<const qh_u32x2*>(line + 64 * f + 8 * kg);
                ql[1] = *reinterpret_cast<const qh_u32x2*>(line + 64 * f + 32 + 8 * kg);
                qm_f32x4 fs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int g = 4 * f + k;
                    // 6-bit quants less 32, byte by byte: (q | 128) - 32 never borrows
                    qh_u32x2 bw = ((ql[k & 1] >> (4 * (k >> 1))) & 0x0F0F0F0Fu) | (((qh >> (2 * k)) & 0x03030303u) << 4);
                    bw = ((bw | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
                    const long a = *reinterpret_cast<const long*>(A + 512 * g);
                    const qm_i32x4 d1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, __builtin_bit_cast(long, bw & m1), zero, 0, 0, 0);
                    const qm_i32x4 d2 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, __builtin_bit_cast(long, bw & ~m1), zero, 0, 0, 0);
                    const uint32_t sw = sc[g >> 1] >> (16 * (g & 1));
                    const int s1 = (int8_t)sw, s2 = (int8_t)(sw >> 8);
                    const qm_f32x4 s4 = *reinterpret_cast<const qm_f32x4*>(S + QM_T * g);
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        fs[r] = fmaf(s4[r], (float)(__mul24(s1, d1[r]) + __mul24(s2, d2[r])), fs[r]);
                }
#pragma unroll
                for (int r = 0; r < 4; r++) acc[r] = fmaf(d6, fs[r], acc[r]);
            }
        }
        // the next block's tokens; its buffer was last read before the previous barrier
        if (b + 1 < nsb) put_x(b + 1);
        if (b + 2 < nsb) load_x(b + 2);
        __syncthreads();
    }
    const int col = col0 + n;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int row = row0 + 4 * kg + r;
        if (row < rows && col < out_dim) y[(size_t)row * out_dim + col] = cut >= 0 ? acc[r] + prefix[r] : acc[r];
    }
}

hipError_t qh_launch_mmq_q81(uint32_t type, const uint8_t* W, const float* x, float* y, int in_dim, int out_dim,
                             int rows, int ref_rows, int mps, hipStream_t st) {
    if ((type != QT_Q4_K && type != QT_Q6_K) || in_dim % 256 || ((uintptr_t)x & 15u)) return hipErrorNotSupported;
    if (rows == 0 || out_dim == 0) return hipSuccess;
    const dim3 grid((unsigned)((out_dim + QM_C - 1) / QM_C), (unsigned)((rows + QM_T - 1) / QM_T));
    if (type == QT_Q4_K)
        hipLaunchKernelGGL(qh_mmq_q81<false>, grid, dim3(64 * QM_W), 0, st, W, x, y, in_dim, out_dim, rows, ref_rows, mps);
    else
        hipLaunchKernelGGL(qh_mmq_q81<true>, grid, dim3(64 * QM_W), 0, st, W, x, y, in_dim, out_dim, rows, ref_rows, mps);
    return hipGetLastError();
}
