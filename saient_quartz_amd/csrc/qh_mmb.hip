// qh_mmb.hip -- batched dequant-GEMM of the 32-element block formats (Q4_0, Q4_1,
// Q5_0, Q5_1, Q8_0, IQ4_NL), 16 tokens per weight pass, without scratch: y[t][j] =
// sum_k W[j,k] x[t][k] on v_mfma_f32_16x16x32_f16.
//
// A workgroup takes 16 RT rows and 16 tokens; its W wavefronts split K (wavefront
// w takes groups w, w + W, ... of 8 blocks) and meet once, at the end, to add
// their partial sums in order.  Nothing lives in device scratch and there is one
// launch, so calls on different streams share nothing.
//   * A operand = tokens.  Lane (m = lane % 16, kg = lane / 16) loads its own 8
//     elements of every block of token m straight from x (32 consecutive floats
//     per token and block over the four kg) and splits them in registers: x' = x
//     2^s (s = 14 - exponent of the token's max|x| over half a group) = hi + lo,
//     two f16 rounded toward zero, 21-22 significant bits.  The operands serve
//     all RT row tiles.
//   * B operand = one block of 32 quants as integers, exact in f16; hi and lo
//     accumulate into the same f32 result, which the block's scale then
//     multiplies.  (Quants as f16 subnormals, q 2^-24, would need no subtraction
//     after the unpacking, but the matrix core aligns subnormal products more
//     coarsely: relative error 1e-6 instead of 2e-8 over a sum whose x span 2^10.)
//   * Minimums (Q4_1, Q5_1): one more product per half group, whose A operand
//     holds each lane's own partial sums of x' per block (k = (kg, block)) and
//     whose B operand holds the blocks' minimums: the matrix core does the
//     reduction too.
//   * Weights go global -> registers (16-byte slices, one group ahead) -> the
//     wavefront's LDS lines -> operands, as in qh_mmv16.hip.
// Bound by latency and the splitting of x, which every workgroup does for itself
// (about two thirds of the VALU work at RT = 1).
//
// Reference counterpart: dequant::gemm (src/dequant.rs:143-200), CPU only.
#include "qh_formats.h"
#include "qh_internal.h"

typedef _Float16 qb_f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 qb_f16x2 __attribute__((ext_vector_type(2)));
typedef float qb_f32x4 __attribute__((ext_vector_type(4)));
typedef qh_u32x2 qb_u32x2a4 __attribute__((aligned(4)));

#define QB_NT 16    // tokens per workgroup

// ---------------------------------------------------------------- operands

// 8 bytes at r + OFF, r a multiple of 4 and OFF a multiple of 2.
template <int OFF>
QH_DEV qh_u32x2 qb_rd8(const unsigned char* r) {
    if constexpr (OFF % 4 == 0) {
        return *reinterpret_cast<const qb_u32x2a4*>(r + OFF);
    } else {
        const uint32_t* p = reinterpret_cast<const uint32_t*>(r + OFF - 2);
        return qh_u32x2{__builtin_amdgcn_alignbyte(p[1], p[0], 2), __builtin_amdgcn_alignbyte(p[2], p[1], 2)};
    }
}
QH_DEV qb_f16x8 qb_op(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(qb_f16x8, qh_u32x4{a, b, c, d});
}
QH_DEV qb_f16x2 qb_h2(uint32_t u) { return __builtin_bit_cast(qb_f16x2, u); }
QH_DEV uint32_t qb_u(qb_f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
// bytes 0, 1 / 2, 3 of w as the f16 pair 1024 + byte, less `bias`
QH_DEV uint32_t qb_b01(uint32_t w, _Float16 bias) {
    return qb_u(qb_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04010400u)) - qb_f16x2{bias, bias});
}
QH_DEV uint32_t qb_b23(uint32_t w, _Float16 bias) {
    return qb_u(qb_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04030402u)) - qb_f16x2{bias, bias});
}
QH_DEV qb_f16x8 qb_bytes(qh_u32x2 w, float bias) {
    const _Float16 b = (_Float16)(1024.0f + bias);
    return qb_op(qb_b01(w.x, b), qb_b23(w.x, b), qb_b01(w.y, b), qb_b23(w.y, b));
}
// ---------------------------------------------------------------- formats
// BYTES per group of 8 blocks, CH 16-byte slices of it, RS the LDS line (a stride
// that puts 16 lines' 16-byte pieces on distinct banks).  bop<B>(line, kg):
// weights 8 kg .. + 7 of block B; scale<B>(line): what multiplies that product.
// The 32-element block formats (src/dequant.rs:1381-1463, :1527-1574; Q4_0 and
// Q4_1 by the public GGUF layout), eight blocks a group: KIND 0 Q4_0, 1 Q4_1, 2
// Q5_0, 3 Q5_1, 4 IQ4_NL, 5 Q8_0.  Elements 0 .. 15 of a block are the low
// nibbles (kg 0, 1), 16 .. 31 the high ones (kg 2, 3).
template <int KIND>
struct BBlk {
    static constexpr int BB = KIND == 5 ? 34 : (KIND == 0 || KIND == 4) ? 18 : (KIND == 1 ? 20 : (KIND == 2 ? 22 : 24));
    static constexpr int QS = (KIND == 0 || KIND >= 4) ? 2 : (KIND == 1 ? 4 : (KIND == 2 ? 6 : 8));  // quants
    static constexpr int BYTES = 8 * BB, CH = BYTES / 16;
    static constexpr int RS = KIND == 1 ? 176 : (KIND == 3 ? 208 : BYTES);
    static constexpr bool MINS = KIND == 1 || KIND == 3;
    template <int B>
    static QH_DEV qb_f16x8 bop(const unsigned char* r, int kg) {
        if constexpr (KIND == 5) {
            return qb_bytes(qb_rd8<BB * B + QS>(r + 8 * kg) ^ 0x80808080u, 128.0f);
        } else {
            qh_u32x2 q = (qb_rd8<BB * B + QS>(r + 8 * (kg & 1)) >> (4u * (uint32_t)(kg >> 1))) & 0x0F0F0F0Fu;
            if constexpr (KIND == 2 || KIND == 3) {
                const uint32_t hb = r[BB * B + QS - 4 + kg];  // the fifth bits of elements 8 kg .. + 7
                q = q | (qh_u32x2{qh_spread4(hb & 0xFu), qh_spread4(hb >> 4)} << 4);
            }
            if constexpr (KIND == 0) return qb_bytes(q, 8.0f);
            if constexpr (KIND == 2) return qb_bytes(q, 16.0f);
            if constexpr (KIND == 4) return qb_bytes(qh_u32x2{qh_iq4nl_lut(q.x), qh_iq4nl_lut(q.y)}, 128.0f);
            return qb_bytes(q, 0.0f);
        }
    }
    template <int B>
    static QH_DEV float scale(const unsigned char* r) {
        return qh_h2f(*reinterpret_cast<const uint16_t*>(r + BB * B));
    }
    // the minimums of half HF's blocks (nb: the group's blocks; past them lies another row)
    template <int HF>
    static QH_DEV qb_f16x8 minb(const unsigned char* r, int nb) {
        qb_f16x8 o = __builtin_bit_cast(qb_f16x8, qh_u32x4{0, 0, 0, 0});
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const uint16_t m = *reinterpret_cast<const uint16_t*>(r + BB * (4 * HF + b) + 2);
            o[b] = __builtin_bit_cast(_Float16, (uint16_t)(4 * HF + b < nb ? m : 0));
        }
        return o;
    }
};

// a less the low / high half of an f16 pair, exact (one v_fma_mix_f32)
typedef __fp16 qb_fp16x2 __attribute__((ext_vector_type(2)));
QH_DEV float qb_less_lo(float a, qb_fp16x2 h) {
    float r;
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(a));
    return r;
}
QH_DEV float qb_less_hi(float a, qb_fp16x2 h) {
    float r;
    asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(a));
    return r;
}

// The x operands of half a group (four blocks) of a lane: its 8 elements of
// each, and (MINS) its partial sums of them, as hi and lo f16.  Returns 2^-s of
// the lane's token.
struct QbX {
    qb_f16x8 hi[4], lo[4], shi, slo;
};
template <bool MINS>
QH_DEV float qb_split(const qh_u32x4 (*xr)[2], QbX& o) {
    float m = 0.f;
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            m = fmaxf(fmaxf(m, fabsf(__uint_as_float(xr[b][0][i]))), fabsf(__uint_as_float(xr[b][1][i])));
    m = fmaxf(m, __shfl_xor(m, 16));
    m = fmaxf(m, __shfl_xor(m, 32));
    int e = 0;
    (void)frexpf(m, &e);
    int s = m > 0.f ? 14 - e : 0;
    s = s > 126 ? 126 : (s < -126 ? -126 : s);
    const float scx = ldexpf(1.0f, s);
    uint32_t sh[2] = {0, 0}, sl[2] = {0, 0};
    float sm[4];
#pragma unroll
    for (int b = 0; b < 4; b++) {
        float a[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            a[i] = __uint_as_float(xr[b][0][i]) * scx;
            a[4 + i] = __uint_as_float(xr[b][1][i]) * scx;
        }
        uint32_t hp[4], lp[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const auto h = __builtin_amdgcn_cvt_pkrtz(a[2 * i], a[2 * i + 1]);
            const auto l = __builtin_amdgcn_cvt_pkrtz(qb_less_lo(a[2 * i], h), qb_less_hi(a[2 * i + 1], h));
            hp[i] = __builtin_bit_cast(uint32_t, h);
            lp[i] = __builtin_bit_cast(uint32_t, l);
        }
        o.hi[b] = qb_op(hp[0], hp[1], hp[2], hp[3]);
        o.lo[b] = qb_op(lp[0], lp[1], lp[2], lp[3]);
        if (MINS) sm[b] = (((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]))) * 0.03125f;
        __builtin_amdgcn_sched_barrier(0);  // x[b] is dead before the next one is split (registers)
    }
    if (__ballot(m == __builtin_inff())) {
        // x holds an infinity: its low part is Inf - Inf, so this token's lows go
        // and its products stay Inf (a NaN reaches every product by itself)
#pragma unroll
        for (int b = 0; b < 4; b++)
            if (m == __builtin_inff()) o.lo[b] = qb_op(0, 0, 0, 0);
    }
    if constexpr (MINS) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const auto h = __builtin_amdgcn_cvt_pkrtz(sm[2 * i], sm[2 * i + 1]);
            const auto l = __builtin_amdgcn_cvt_pkrtz(qb_less_lo(sm[2 * i], h), qb_less_hi(sm[2 * i + 1], h));
            sh[i] = __builtin_bit_cast(uint32_t, h);
            sl[i] = __builtin_bit_cast(uint32_t, l);
        }
        o.shi = qb_op(sh[0], sh[1], 0, 0);
        o.slo = qb_op(sl[0], sl[1], 0, 0);
    }
    return ldexpf(1.0f, -s);
}

// ---------------------------------------------------------------- kernel

template <class F, int RT, int W>
constexpr int qb_lds() {
    const int tiles = W * 16 * RT * F::RS, red = W * RT * 4 * 64 * 4;
    return (tiles > red ? tiles : red) + W * 16 * 4;
}

template <class F, int RT, int W>
__global__ __launch_bounds__(64 * W) void qh_mmb(const uint8_t* __restrict__ wts, const float* __restrict__ x,
                                              float* __restrict__ y, uint32_t row_bytes, int in_dim, int rows,
                                              int ntok) {
    constexpr int CH = F::CH, RS = F::RS, ROWS = 16 * RT;
    constexpr int NL = (ROWS * CH + 63) / 64;
    constexpr int TILE = ROWS * RS;
    __shared__ __align__(16) unsigned char lds[qb_lds<F, RT, W>()];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, n = lane & 15, kg = lane >> 4;
    const int row0 = (int)blockIdx.x * ROWS, t0 = (int)blockIdx.y * QB_NT, nt = min(ntok - t0, QB_NT);
    const int nblk = in_dim >> 5, ngroups = (nblk + 7) >> 3;
    unsigned char* wl = lds + w * TILE;
    float* rsl = reinterpret_cast<float*>(lds + qb_lds<F, RT, W>() - W * 16 * 4) + 16 * w;

    // x of this lane: token n, elements 8 kg .. of each block (past the
    // tokens or the row: out of range, zeros)
    const QhBuf xb = qh_buf(x + (size_t)t0 * in_dim, 4u * (uint32_t)nt * (uint32_t)in_dim);
    const uint32_t xo = n < nt ? 4u * ((uint32_t)n * (uint32_t)in_dim + 8u * (uint32_t)kg) : 0x80000000u;
    qh_u32x4 xr[4][2];
    auto load_x = [&](int h) {  // half-group h
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const uint32_t o = 4 * h + b < nblk ? xo + 512u * (uint32_t)h + 128u * b : 0x80000000u;
            xr[b][0] = qh_ld128(xb, o);
            xr[b][1] = qh_ld128(xb, o + 16u);
        }
    };
    // weight slices: row q / CH of the tile, slice q % CH.  In a last group of
    // fewer than 8 blocks the last slice ends with the row (no load runs past
    // the matrix) and is staged at its own bytes.
    const int live = min(rows - row0, ROWS);
    const QhBuf wb = qh_buf(wts + (size_t)row0 * row_bytes,
                            (uint32_t)(((uint64_t)live * row_bytes + 3) & ~(uint64_t)3));
    auto gbytes = [&](int g) { return F::BB * min(8, nblk - 8 * g); };
    qh_u32x4 wr[NL];
    auto load_w = [&](int g) {
        const int gb = gbytes(g);
#pragma unroll
        for (int h = 0; h < NL; h++) {
            const int q = 64 * h + lane, r = q / CH, c = q - CH * r;
            const uint32_t o = (uint32_t)r * row_bytes + (uint32_t)F::BYTES * (uint32_t)g + (uint32_t)min(16 * c, gb - 16);
            wr[h] = qh_ld128(wb, r < live && 16 * c < gb ? o : 0x80000000u);
        }
    };
    auto stage_w = [&](int g) {
        const int gb = gbytes(g);
#pragma unroll
        for (int h = 0; h < NL; h++) {
            const int q = 64 * h + lane, r = q / CH, c = q - CH * r;
            if (64 * h + 63 < ROWS * CH || q < ROWS * CH) {
                if (gb == F::BYTES) {
                    *reinterpret_cast<qh_u32x4*>(wl + r * RS + 16 * c) = wr[h];
                } else if (16 * c < gb) {  // 2-byte aligned
                    uint16_t* p = reinterpret_cast<uint16_t*>(wl + r * RS + min(16 * c, gb - 16));
#pragma unroll
                    for (int i = 0; i < 8; i++) p[i] = (uint16_t)(wr[h][i >> 1] >> (16 * (i & 1)));
                }
            }
        }
    };

    qb_f32x4 tot[RT];
#pragma unroll
    for (int t = 0; t < RT; t++) tot[t] = qb_f32x4{0.f, 0.f, 0.f, 0.f};
    load_x(2 * w);
    __builtin_amdgcn_sched_barrier(0);
    load_w(w);
    __builtin_amdgcn_sched_barrier(0);
    const qb_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    for (int g = w; g < ngroups; g += W) {
        auto half = [&](auto HC) {
            constexpr int HF = decltype(HC)::value;
            QbX X;
            const float r2 = qb_split<F::MINS>(xr, X);
            if (kg == 0) rsl[n] = r2;
            // the next half's x before the next group's weights: waiting for it leaves them in flight
            load_x(HF == 0 ? 2 * g + 1 : 2 * (g + W));
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (HF == 0) {
                stage_w(g);
                load_w(g + W);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const qb_f32x4 rs = *reinterpret_cast<const qb_f32x4*>(rsl + 4 * kg);
#pragma unroll
            for (int t = 0; t < RT; t++) {
                const unsigned char* line = wl + (16 * t + n) * RS;
                qb_f32x4 tg = zero, cp = zero;
                float sp = 0.f;
                // one block behind: the products of B while B - 1's are scaled
                auto sub = [&](auto BC) {
                    constexpr int B = decltype(BC)::value;
                    const qb_f16x8 b = F::template bop<4 * HF + B>(line, kg);
                    const float sc = F::template scale<4 * HF + B>(line);
                    qb_f32x4 c = __builtin_amdgcn_mfma_f32_16x16x32_f16(X.lo[B], b, zero, 0, 0, 0);
                    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(X.hi[B], b, c, 0, 0, 0);
                    if constexpr (B > 0) {
#pragma unroll
                        for (int i = 0; i < 4; i++) tg[i] = fmaf(sp, cp[i], tg[i]);
                    }
                    cp = c;
                    // a block past the row's end holds another row's scale: not its products (0 * Inf)
                    sp = 8 * g + 4 * HF + B < nblk ? sc : 0.f;
                    __builtin_amdgcn_sched_barrier(0);
                };
                sub(std::integral_constant<int, 0>{});
                sub(std::integral_constant<int, 1>{});
                sub(std::integral_constant<int, 2>{});
                sub(std::integral_constant<int, 3>{});
#pragma unroll
                for (int i = 0; i < 4; i++) tg[i] = fmaf(sp, cp[i], tg[i]);
                if constexpr (F::MINS) {
                    const qb_f16x8 mb = F::template minb<HF>(line, nblk - 8 * g);
                    qb_f32x4 c = __builtin_amdgcn_mfma_f32_16x16x32_f16(X.slo, mb, zero, 0, 0, 0);
                    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(X.shi, mb, c, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) tg[i] = fmaf(32.0f, c[i], tg[i]);
                }
#pragma unroll
                for (int i = 0; i < 4; i++) tot[t][i] = fmaf(tg[i], rs[i], tot[t][i]);
            }
        };
        half(std::integral_constant<int, 0>{});
        half(std::integral_constant<int, 1>{});
    }
    // ---- add the wavefronts' partial sums in order (the tiles' LDS is free)
    __syncthreads();
    float* red = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) red[((w * RT + t) * 4 + i) * 64 + lane] = tot[t][i];
    __syncthreads();
    for (int o = threadIdx.x; o < ROWS * QB_NT; o += 64 * W) {
        const int r = o % ROWS, t = o / ROWS;  // row of the tile, token
        if (t < nt && row0 + r < rows) {
            const int at = ((r >> 4) * 4 + (t & 3)) * 64 + 16 * (t >> 2) + (r & 15);
            float a = red[at];
#pragma unroll
            for (int k = 1; k < W; k++) a += red[k * RT * 256 + at];
            y[(size_t)(t0 + t) * rows + row0 + r] = a;
        }
    }
}

// Rows per workgroup and wavefronts: 16 rows x 8 wavefronts while that is at most
// two workgroups per CU (4096 x 4096 Q8_0 at 16 tokens: 12.7 us, 14.8 with 32 x
// 4; 16 GEMV launches took 90), else 32 rows x 4 wavefronts, which split x half
// as often (14336 x 4096: 26.8 us against 41.6; at 512 tokens 0.52 ms).
template <int KIND>
static void launch_mmb(const uint8_t* W, const float* x, float* y, uint32_t row_bytes, int in_dim, int rows, int n,
                       hipStream_t st) {
    using F = BBlk<KIND>;
    const int tb = (n + QB_NT - 1) / QB_NT;
    if ((int64_t)((rows + 15) / 16) * tb <= 512)
        hipLaunchKernelGGL((qh_mmb<F, 1, 8>), dim3((unsigned)((rows + 15) / 16), (unsigned)tb), dim3(512), 0, st, W, x, y,
                           row_bytes, in_dim, rows, n);
    else
        hipLaunchKernelGGL((qh_mmb<F, 2, 4>), dim3((unsigned)((rows + 31) / 32), (unsigned)tb), dim3(256), 0, st, W, x, y,
                           row_bytes, in_dim, rows, n);
}

// n >= 2 tokens of a 32-element block type; hipErrorNotSupported for other types.
hipError_t qh_launch_mmb(uint32_t type, const uint8_t* W, const float* x, float* y, int in_dim, int out_dim, int n,
                         hipStream_t st) {
    if (n < 2 || in_dim % 32 || in_dim > (1 << 20)) return hipErrorNotSupported;
    const uint32_t rb = (uint32_t)qh_type_size(type, (size_t)in_dim);
    for (int t0 = 0; t0 < n; t0 += 16 * 32768) {  // the grid's second dimension
        const int nt = n - t0 < 16 * 32768 ? n - t0 : 16 * 32768;
        const float* xs = x + (size_t)t0 * in_dim;
        float* ys = y + (size_t)t0 * out_dim;
        switch (type) {
            case QT_Q4_0: launch_mmb<0>(W, xs, ys, rb, in_dim, out_dim, nt, st); break;
            case QT_Q4_1: launch_mmb<1>(W, xs, ys, rb, in_dim, out_dim, nt, st); break;
            case QT_Q5_0: launch_mmb<2>(W, xs, ys, rb, in_dim, out_dim, nt, st); break;
            case QT_Q5_1: launch_mmb<3>(W, xs, ys, rb, in_dim, out_dim, nt, st); break;
            case QT_IQ4_NL: launch_mmb<4>(W, xs, ys, rb, in_dim, out_dim, nt, st); break;
            case QT_Q8_0: launch_mmb<5>(W, xs, ys, rb, in_dim, out_dim, nt, st); break;
            default: return hipErrorNotSupported;
        }
    }
    return hipGetLastError();
}
