// qh_mms.hip -- batched dequant-GEMM for 2 .. 16 tokens and few rows on
// v_mfma_f32_16x16x32_f16: Q4_K, Q5_K, Q6_K matrices that share one x.  The formats'
// B operands and the x images are qh_gemm.hip's.
//
// qh_mmq's tiles of 256 rows need K split over workgroups to fill the chip when a
// matrix has few rows: most of such a launch is filling pipelines, storing partials,
// an arrival counter and reading the partials back.  Here a workgroup takes 32
// rows and the whole of K: its 8 wavefronts take groups w, w + 8, ... and meet once,
// in LDS, to add their sums in order.
//   * A operand = tokens.  Lane (m = lane % 16, kg = lane / 16) reads its 8 elements
//     of a block of 32, hi then lo, as 32 bytes of the image straight into registers;
//     they serve both row tiles.
//   * weights: 16-byte slices global -> registers -> the wavefront's LDS lines ->
//     operands; a group's registers are refilled as they are used.
// Bound by latency and by the reads of x from L2 (16 KB per wavefront and group, which
// 2 row tiles share: with 1 tile twice as many workgroups read it, 4096 x 4096 Q4_K
// 9.5 us against 9.1, with 4 half the chip is idle, 12.8; images there already).
#include "qh_formats.h"
#include "qh_internal.h"

#define QS_RT 2  // row tiles of 16 per workgroup
#define QS_ROWS (16 * QS_RT)

struct QsArgs {
    const uint8_t* w[QS_MAXM];
    float* y[QS_MAXM];
    int rows[QS_MAXM], ldy[QS_MAXM];
    int type[QS_MAXM];
    uint32_t row_bytes[QS_MAXM];
    const unsigned char* img;
    uint32_t img_bytes;
    int n, in_dim, accum;
};

// As F::hdr, for lane quarter kg: a Q6_K scale is per 16 weights, so the scales of
// the block half this lane converts move to the bytes of the even K-blocks.
template <class F>
QH_DEV typename F::H qs_hdr(const unsigned char* r, int kg) {
    typename F::H h = F::hdr(r);
    if constexpr (std::is_same_v<F, GQ6K>) h.s = h.s >> (uint32_t)(8 * (kg >> 1));
    return h;
}

template <class F>
constexpr int qs_lds() {
    const int tiles = 8 * QS_ROWS * F::RS, red = 8 * QS_ROWS * 64;
    return tiles > red ? tiles : red;
}

template <class F>
__device__ __forceinline__ void qs_body(const QsArgs& a, int gi, int blk, unsigned char* lds) {
    constexpr int CH = F::CH, RS = F::RS, RT = QS_RT, ROWS = QS_ROWS, NL = (ROWS * CH + 63) / 64;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = lane & 15, kg = lane >> 4;
    const int rows = qg_uni(a.rows[gi]), ldy = qg_uni(a.ldy[gi]), row0 = blk * ROWS, ngroups = a.in_dim >> 8;
    const uint32_t row_bytes = (uint32_t)qg_uni((int)a.row_bytes[gi]);
    float* __restrict__ y = qg_uni(a.y[gi]);
    unsigned char* wl = lds + w * ROWS * RS;

    const int live = min(rows - row0, ROWS);
    const QhBuf wb = qh_buf(qg_uni(a.w[gi]) + (size_t)row0 * row_bytes, (uint32_t)(((uint64_t)live * row_bytes + 3) & ~(uint64_t)3));
    const QhBuf xb = qh_buf(a.img, a.img_bytes);
    struct In {
        qh_u32x4 w[NL], hi[8], lo[8], sums, rs;
    } in;
    auto load_w = [&](int g) {
        const uint32_t past = (uint32_t)(ngroups - 1 - g) & 0x80000000u;  // no traffic, zeros
#pragma unroll
        for (int h = 0; h < NL; h++) {
            const int q = 64 * h + lane, r = q / CH, c = q - CH * r;
            const uint32_t off = (uint32_t)r * row_bytes + (uint32_t)F::BYTES * (uint32_t)g + (c == CH - 1 ? F::LAST : 16u * c);
            in.w[h] = qh_ld128(wb, r < live ? off | past : 0x80000000u);
        }
    };
    // absent tokens read nothing
    const uint32_t xo = m < a.n ? 512u * kg + 32u * m : 0x80000000u;
    auto load_x = [&](int g, int half) {
        const uint32_t past = (uint32_t)(ngroups - 1 - g) & 0x80000000u;
        const uint32_t go = (uint32_t)XImg::BYTES * (uint32_t)g, xg = (xo | past) + go;
#pragma unroll
        for (int b = 4 * half; b < 4 * half + 4; b++) {
            in.hi[b] = qh_ld128(xb, xg + 2048u * b);
            in.lo[b] = qh_ld128(xb, xg + 2048u * b + 16u);
        }
        if (half == 0) {
            const uint32_t t = (go + XImg::RSF + 8u * kg) | past;  // tokens 4 kg .. + 3
            const qh_u32x2 r0 = qh_ld64(xb, t), r1 = qh_ld64(xb, t + 32u);
            in.rs = qh_u32x4{r0.x, r0.y, r1.x, r1.y};
        } else if constexpr (F::SUMS) {
            in.sums = qh_ld128(xb, (go + XImg::SUM + 16u * (m + 16 * (kg & 1))) | past);
        }
    };
    load_w(w);
    load_x(w, 0);
    load_x(w, 1);
    // this thread's result (token ot, row orow of the tile); a residual launch's y is on
    // its way from the start
    const int orow = threadIdx.x % ROWS, ot = threadIdx.x / ROWS;
    static_assert(ROWS * 16 == 512, "a result per thread");
    const bool mine = ot < a.n && orow < live;
    float* yp = y + (size_t)ot * ldy + row0 + orow;
    const float yv = a.accum && mine ? *yp : 0.f;
    __builtin_amdgcn_sched_barrier(0);

    const qh_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    qh_f32x4 tot[RT];
#pragma unroll
    for (int t = 0; t < RT; t++) tot[t] = zero;
    for (int g = w; g < ngroups; g += 8) {
#pragma unroll
        for (int h = 0; h < NL; h++) {
            const int q = 64 * h + lane, r = q / CH, c = q - CH * r;
            if (64 * h + 63 < ROWS * CH || q < ROWS * CH) *reinterpret_cast<qh_u32x4*>(wl + r * RS + 16 * c) = in.w[h];
        }
        load_w(g + 8);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        __builtin_amdgcn_sched_barrier(0);
        typename F::H hd[RT];
        qh_f32x4 ch[RT], cl[RT];
        const qh_u32x4 rs = in.rs;
        auto block = [&](auto BC) {
            constexpr int B = decltype(BC)::value;
#pragma unroll
            for (int t = 0; t < RT; t++) {
                const unsigned char* line = wl + (16 * t + m) * RS;
                if constexpr (B == 0) hd[t] = qs_hdr<F>(line, kg);
                const qh_f16x8 b = F::template cvt<2 * B>(F::template raw<2 * B>(line, kg), hd[t], nullptr);
                cl[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(qh_f16x8, in.lo[B]), b, B == 0 ? zero : cl[t], 0, 0, 0);
                ch[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(qh_f16x8, in.hi[B]), b, B == 0 ? zero : ch[t], 0, 0, 0);
            }
        };
        block(std::integral_constant<int, 0>{});
        block(std::integral_constant<int, 1>{});
        block(std::integral_constant<int, 2>{});
        block(std::integral_constant<int, 3>{});
        load_x(g + 8, 0);
        __builtin_amdgcn_sched_barrier(0);
        block(std::integral_constant<int, 4>{});
        block(std::integral_constant<int, 5>{});
        block(std::integral_constant<int, 6>{});
        block(std::integral_constant<int, 7>{});
        qh_f32x4 mm[RT];
        if constexpr (F::SUMS) {
#pragma unroll
            for (int t = 0; t < RT; t++) {
                const qh_u32x4 mn = __builtin_bit_cast(qh_u32x4, F::minh(hd[t], kg & 1));
                const uint32_t on = kg < 2 ? 0xFFFFFFFFu : 0u;  // K positions 16 .. 31 hold nothing
                mm[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(qh_f16x8, in.sums),
                                                               __builtin_bit_cast(qh_f16x8, mn & on), zero, 0, 0, 0);
            }
        }
        load_x(g + 8, 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < RT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float p = hd[t].d * (ch[t][i] + cl[t][i]);
                if constexpr (F::SUMS) p = fmaf(hd[t].dm * -32.0f, mm[t][i], p);
                tot[t][i] = fmaf(p, __uint_as_float(rs[i]), tot[t][i]);
            }
    }
    // ---- add the wavefronts' partial sums in order (the tiles' LDS is free)
    __syncthreads();
    float* red = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) red[((w * RT + t) * 4 + i) * 64 + lane] = tot[t][i];
    __syncthreads();
    if (mine) {
        const int at = ((orow >> 4) * 4 + (ot & 3)) * 64 + 16 * (ot >> 2) + (orow & 15);
        float s = red[at];
#pragma unroll
        for (int k = 1; k < 8; k++) s += red[k * RT * 256 + at];
        *yp = a.accum ? yv + s : s;
    }
}

// blockIdx.y = matrix; its type picks the body.
__global__ __launch_bounds__(512) void qh_mms(const QsArgs a) {
    __shared__ __align__(16) unsigned char lds[qs_lds<GQ6K>()];
    static_assert(qs_lds<GQ6K>() >= qs_lds<GQ5K>() && qs_lds<GQ6K>() >= qs_lds<GQ4K>(), "LDS");
    const int gi = (int)blockIdx.y, blk = (int)blockIdx.x;
    if (blk * QS_ROWS >= a.rows[gi]) return;  // uniform, before any barrier
    const int type = a.type[gi];
    if (type == QT_Q4_K) qs_body<GQ4K>(a, gi, blk, lds);
    else if (type == QT_Q5_K) qs_body<GQ5K>(a, gi, blk, lds);
    else qs_body<GQ6K>(a, gi, blk, lds);
}

// ---------------------------------------------------------------- launch

// One round of workgroups (in more, qh_mmq reads x less often: Q4_K 12288 x 4096 at 16
// tokens 17.7 us, here 21.3) and K up to 4096 (8192 x 8192 Q4_K 21.0 / 20.5, Q6_K 24.3
// / 24.6; 4096 x 14336 21 / 28).  Within that, us at 16 tokens with the image launch,
// qh_mmq / here: Q4_K 256 x 1024 8.8 / 8.0, 2048 x 2048 11.4 / 9.1, 4096 x 4096 13.3 /
// 11.5, 8192 x 4096 14.2 / 12.3; Q6_K 2048 x 2048 12.5 / 10.0, 4096 x 4096 16.6 / 14.3,
// 8192 x 4096 17.6 / 15.5; Q5_K 4096 x 4096 13.9 / 12.0.  Up to 8 tokens qh_mmq digitises
// x in its own launch in less time than the image launch costs: few weights (Q4_K 64 x
// 512 at 8 tokens 7.2 / 7.6) and a long K of few rows (1024 x 4096 at 4: 10.0 / 10.6) stay
// there, by fits of both times.  Images that are there already take 3 us off this
// kernel's time; the choice leaves that out, so that a call gives the same bits with and
// without them.
bool qs_pick(const QsMat* ms, int cnt, int in_dim, int n) {
    if (cnt < 1 || cnt > QS_MAXM || n > 16 || in_dim > 4096) return false;
    float mmq = 11.0f, group = 0.f, weights = 0.f;
    int blocks = 0;
    for (int i = 0; i < cnt; i++) {
        const uint32_t t = ms[i].type;
        if (t != QT_Q4_K && t != QT_Q5_K && t != QT_Q6_K) return false;
        blocks += (ms[i].rows + QS_ROWS - 1) / QS_ROWS;
        const float k = t == QT_Q4_K ? 0.163f : (t == QT_Q5_K ? 0.18f : 0.225f);  // per million weights
        const float gr = t == QT_Q4_K ? 0.47f : (t == QT_Q5_K ? 0.50f : 0.60f);   // per group of 256
        mmq += k * 1e-6f * (float)ms[i].rows * (float)in_dim;
        weights += (float)ms[i].rows * (float)in_dim;
        group = gr > group ? gr : group;
    }
    if (blocks > 256) return false;
    return n > 8 || (weights > 1048576.f && 5.2f + group * (float)(in_dim >> 8) < mmq);
}

hipError_t qs_run(const QsMat* ms, int cnt, const unsigned char* img, int n, int in_dim, int accum, hipStream_t st) {
    QsArgs a = {};
    int most = 0;
    for (int i = 0; i < cnt; i++) {
        a.w[i] = ms[i].w;
        a.y[i] = ms[i].y;
        a.rows[i] = ms[i].rows;
        a.ldy[i] = ms[i].ldy;
        a.type[i] = (int)ms[i].type;
        a.row_bytes[i] = (uint32_t)qh_type_size(ms[i].type, (size_t)in_dim);
        most = ms[i].rows > most ? ms[i].rows : most;
    }
    a.img = img;
    a.img_bytes = (uint32_t)((in_dim >> 8) * XImg::BYTES);
    a.n = n;
    a.in_dim = in_dim;
    a.accum = accum;
    hipLaunchKernelGGL(qh_mms, dim3((unsigned)((most + QS_ROWS - 1) / QS_ROWS), (unsigned)cnt), dim3(512), 0, st, a);
    return hipGetLastError();
}
