// qh_mmw.hip -- batched dequant-GEMM for more than 32 tokens (a prompt) on
// v_mfma_f32_32x32x16_f16: Q4_K, Q5_K, Q6_K, IQ3_S, IQ2_XXS.  The formats' B
// operands (integer weight times integer scale, exact in f16) and the split of x
// into two f16 are qh_gemm.hip's; here a workgroup's tile is wide in tokens, so
// that a weight is converted once for 64 tokens instead of 32 and read from
// memory once for all of them.
//
// A workgroup of 8 wavefronts computes 32 MT TW tokens x 32 CT CW rows of W (CW =
// 8 / TW), each wavefront MT x CT tiles of 32 x 32; hi and lo products accumulate
// into the same registers.
//   * x: images of 32 tokens x 256 elements written once by qw_image in A-operand
//     order stream from L2 straight into LDS (buffer loads to LDS), KS blocks of 16
//     elements per step, three buffers: one being read, two on their way.  One
//     barrier per step orders them.
//   * weights: 16-byte slices global -> registers one group (256) ahead -> LDS.
//   * after a group, tot += (d P - dmin M) 2^-s in f32, P the group's products and
//     M the minimums' (one more MFMA on the x sums).
// Bound by the vector instructions that convert weights (about 8 per 4 weights and
// tile) beside two matrix instructions per product: Q4_K 14336 x 4096 at 512 tokens
// 129 us (0.47 PFLOP/s, twice that in matrix instructions; qh_mmq's 16 passes of 32
// tokens 197), at 256 78 (103), at 160 72 (93); Q6_K 138 (232), 84 (120), 83 (109).
//   * K is split over workgroups when the tiles alone do not fill the chip; the
//     last wavefront to arrive at a tile adds the splits in order (qh_mmq's way).
#include "qh_formats.h"
#include "qh_internal.h"

// x image of one (32-token tile, group): block j (16 elements) at 2048 j: hi, then
// lo at + 1024, in A-operand order (token t, half c: 16 (t + 32 c)); the x sums'
// operand (hi: half 0, lo: half 1) at SUM; 2^-s per token at RSF.
struct WImg {
    static constexpr int SUM = 32768, RSF = 33792, BYTES = 33920;
};
#define QW_NB 3  // x buffers in LDS

// One (group, token tile) per workgroup: thread t, c = token t / 32, chunk t % 32.
__global__ __launch_bounds__(1024) void qw_image(const float* __restrict__ x, const float* __restrict__ x2,
                                                 unsigned char* __restrict__ img, int n, int in_dim) {
    const int g = blockIdx.x, tt = blockIdx.y, ngroups = in_dim >> 8;
    const int lane = threadIdx.x & 63, xt = threadIdx.x >> 5, xc = threadIdx.x & 31;
    const int t = 32 * tt + xt;
    if (t >= n) return;  // whole half-wavefronts
    const size_t t0 = (size_t)(32 * tt) * in_dim;
    const uint32_t nb = 4u * (uint32_t)(n - 32 * tt < 32 ? n - 32 * tt : 32) * (uint32_t)in_dim;
    const uint32_t off = 4u * ((uint32_t)xt * (uint32_t)in_dim + 256u * (uint32_t)g + 8u * (uint32_t)xc);
    const QhBuf xb = qh_buf(x + t0, nb);
    qh_u32x4 xr[2] = {qh_ld128(xb, off), qh_ld128(xb, off + 16u)}, ur[2] = {};
    if (x2) {
        const QhBuf ub = qh_buf(x2 + t0, nb);
        ur[0] = qh_ld128(ub, off);
        ur[1] = qh_ld128(ub, off + 16u);
    }
    float v[8];
    qg_chunk(xr, ur, x2 != nullptr, v);
    const QgSplit s = qg_split<true>(v, lane);
    unsigned char* im = img + ((size_t)tt * ngroups + g) * WImg::BYTES;
    unsigned char* p = im + 2048 * (xc >> 1) + 16 * (xt + 32 * (xc & 1));
    *reinterpret_cast<qh_u32x4*>(p) = qh_u32x4{s.hi[0], s.hi[1], s.hi[2], s.hi[3]};
    *reinterpret_cast<qh_u32x4*>(p + 1024) = qh_u32x4{s.lo[0], s.lo[1], s.lo[2], s.lo[3]};
    if ((xc & 3) == 0) {
        uint16_t* q = reinterpret_cast<uint16_t*>(im + WImg::SUM + 16 * xt) + (xc >> 2);
        q[0] = (uint16_t)s.sum;
        q[256] = (uint16_t)(s.sum >> 16);
    }
    if (xc == 0) reinterpret_cast<float*>(im + WImg::RSF)[xt] = s.bad ? __builtin_nanf("") : ldexpf(1.0f, -s.s);
}

// All but this wavefront's newest N vector loads and every LDS access so far are
// done (then, qw_meet: in every wavefront); no memory access moves across.  One
// asm, so that the count of newer loads is exactly what stands after it in the
// source.
template <int N>
QH_DEV void qw_wait() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory"); }
template <int N>
QH_DEV void qw_meet() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory"); }
// A value the compiler cannot derive others from ahead of time (offsets made from
// it are computed where they are used instead of being held in registers).
QH_DEV int qw_fresh(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

template <class F, int MT, int CT, int TW>
struct QwShape {
    static constexpr int TT = MT * TW, CW = 8 / TW;  // token tiles of a workgroup, wavefronts side by side
    static constexpr int COLS = 32 * CT * CW;
    static constexpr int KS = 4, NST = 4;      // blocks per step, steps per group
    static constexpr int XI = TT * KS * 2 / 8;  // 1 KB x loads per wavefront and step
    static constexpr int XB = TT * KS * 2048;
    static constexpr int NLW = (COLS * F::CH + 511) / 512;
    static constexpr int WB = COLS * F::RS;
    static constexpr int GRIDB = F::GRID ? IQT_BYTES : 0;
    static constexpr int RSB = 2 * TT * 128;  // 2^-s of two groups
    static constexpr int LDS = QW_NB * XB + WB + RSB + GRIDB;
};

struct QwArgs {
    const uint8_t* w;
    const unsigned char* img;
    float* y;
    float* part;
    unsigned int* cnt;
    uint32_t wbytes, img_bytes, row_bytes;
    int in_dim, rows, n, ldy, accum, splits, tblocks;
};

template <class F, int MT, int CT, int TW>
__global__ __launch_bounds__(512) void qh_mmw(const QwArgs a) {
    using S = QwShape<F, MT, CT, TW>;
    constexpr int TT = S::TT, CW = S::CW, KS = S::KS, NST = S::NST, XI = S::XI, CH = F::CH, RS = F::RS, NLW = S::NLW;
    __shared__ __align__(1024) unsigned char lds[S::LDS];
    unsigned char* wl = lds + QW_NB * S::XB;
    float* rsl = reinterpret_cast<float*>(wl + S::WB);
    unsigned char* gridl = wl + S::WB + S::RSB;
    if constexpr (F::GRID != 0) qg_iq_tables<F::GRID>(gridl, threadIdx.x, 512);
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int R = lane & 31, hh = lane >> 5, tw = w / CW, cw = w - tw * CW;
    // Workgroup ids go round the 8 XCDs: the token blocks of one (row block, split)
    // follow each other on one XCD, whose L2 then serves its weights to all of them.
    const int id = blockIdx.x, j8 = id >> 3;
    const int pair = (id & 7) + 8 * (j8 / a.tblocks), tb = j8 % a.tblocks;
    const int blocks = (a.rows + S::COLS - 1) / S::COLS;
    if (pair >= blocks * a.splits) return;  // uniform, before any barrier
    const int cb = pair / a.splits, sp = pair - cb * a.splits;
    const int ngroups = a.in_dim >> 8;
    const int g0 = ngroups * sp / a.splits, g1 = ngroups * (sp + 1) / a.splits;

    const QhBuf wb = qh_buf(a.w, a.wbytes);
    const QhBuf ib = qh_buf(a.img, a.img_bytes);
    qh_u32x4 wr[NLW];
    float rsr;
    // group g's weights and 2^-s (threads < 32 TT), to registers
    auto load_g = [&](int g) {
        const uint32_t past = (uint32_t)(g1 - 1 - g) & 0x80000000u;
        const int t = qw_fresh(tid);
#pragma unroll
        for (int h = 0; h < NLW; h++) {  // slice q % CH of the tile's row q / CH
            const int q = 512 * h + t, r = q / CH, c = q - CH * r, row = cb * S::COLS + r;
            const uint32_t o = (uint32_t)row * a.row_bytes + (c == CH - 1 ? F::LAST : 16u * c) + (uint32_t)F::BYTES * (uint32_t)g;
            wr[h] = qh_ld128(wb, o | past | (q < S::COLS * CH && row < a.rows ? 0u : 0x80000000u));
        }
        const uint32_t o = (uint32_t)((tb * TT + (t >> 5)) * ngroups + g) * (uint32_t)WImg::BYTES + WImg::RSF + 4u * R;
        rsr = __uint_as_float(qh_ld32(ib, o | past | (t < 32 * TT ? 0u : 0x80000000u)));
    };
    auto stage_g = [&](int g) {
        const int t = qw_fresh(tid);
#pragma unroll
        for (int h = 0; h < NLW; h++) {
            const int q = 512 * h + t, r = q / CH, c = q - CH * r;
            if (512 * h + 511 < S::COLS * CH || q < S::COLS * CH)
                *reinterpret_cast<qh_u32x4*>(wl + r * RS + 16 * c) = wr[h];
        }
        if (t < 32 * TT) rsl[(g & 1) * 32 * TT + t] = rsr;
    };
    // x of step k (blocks k KS ..) of group g into a buffer: load i of the step's
    // 2 TT KS goes to its 1 KB i; a wavefront takes XI of them
    auto load_x = [&](int g, int k, int buf) {
        const uint32_t past = (uint32_t)(g1 - 1 - g) & 0x80000000u;
#pragma unroll
        for (int ii = 0; ii < XI; ii++) {
            const int i = w * XI + ii, tt = i / (2 * KS), rem = i - tt * 2 * KS;
            const uint32_t so = ((uint32_t)((tb * TT + tt) * ngroups + g) * (uint32_t)WImg::BYTES) +
                                1024u * (uint32_t)(2 * KS * k + rem);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ib.rs, (__attribute__((address_space(3))) void*)(lds + buf * S::XB + 1024 * i),
                                                     16, (int)(16u * lane + (so | past)), 0, 0, 0);
        }
    };

    qh_f32x16 c[MT][CT], tot[MT][CT];
    const qh_f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int q = 0; q < CT; q++) tot[m][q] = zero;
    // Stages over the blocks J = 0, 1, ... of 16 elements of the whole K range: the
    // products of J, the conversion of J + 1, the weight bytes of J + 2 from LDS; each
    // half (lo, hi) of x of J + 1 follows the products that used J's.  A group's 16
    // blocks are unrolled: with a loop over the steps the compiler's own waits at the
    // joins also wait for the x loads in flight (14336 x 4096 Q4_K at 128 tokens 58
    // against 48 us).
    qh_f16x8 hi[MT], lo[MT], b[2][CT];
    typename F::Raw raw[2][CT];
    // headers of the group being converted, of the next one and, read again where the
    // group ends (not held through it), of the group to finish
    typename F::H hd[CT], hn[CT], he[CT];
    const unsigned char* line[CT];
#pragma unroll
    for (int q = 0; q < CT; q++) line[q] = wl + ((cw * CT + q) * 32 + R) * RS;
    int buf = 0;  // x buffer of the step being read
    auto read_x = [&](auto JC, int part, qh_f16x8* v) {
        constexpr int J = decltype(JC)::value;
        const unsigned char* xa = lds + buf * S::XB + tw * MT * KS * 2048 + 2048 * (J % KS) + 1024 * part + 16 * lane;
#pragma unroll
        for (int m = 0; m < MT; m++) v[m] = __builtin_bit_cast(qh_f16x8, qh_lds128(xa + m * KS * 2048));
    };
    auto read_w = [&](auto JC) {
        constexpr int J = decltype(JC)::value % 16;
#pragma unroll
        for (int q = 0; q < CT; q++) raw[J & 1][q] = F::template raw<J>(line[q], hh);
    };
    auto convert = [&](auto JC, const typename F::H* h) {
        constexpr int J = decltype(JC)::value % 16;
#pragma unroll
        for (int q = 0; q < CT; q++) b[J & 1][q] = F::template cvt<J>(raw[J & 1][q], h[q], gridl);
    };

    load_g(g0);
    load_x(g0, 0, 0);
    load_x(g0, 1, 1);
    stage_g(g0);
    // meets: the x loads of the step at hand (issued two steps ago) have landed;
    // newer are the next step's and what step 0 issued since (the sums' loads are
    // not counted: waiting for them too is harmless)
    constexpr int NG = NLW + 1, SK = 3;
    qw_meet<XI>();
    load_x(g0, 2, 2);
    load_g(g0 + 1);
#pragma unroll
    for (int q = 0; q < CT; q++) hd[q] = F::hdr(line[q]);
    read_x(std::integral_constant<int, 0>{}, 1, lo);
    read_x(std::integral_constant<int, 0>{}, 0, hi);
    read_w(std::integral_constant<int, 0>{});
    read_w(std::integral_constant<int, 1>{});
    convert(std::integral_constant<int, 0>{}, hd);
    for (int g = g0; g < g1; g++) {
        qh_u32x4 sums[MT];
        auto block = [&](auto JC) {
            constexpr int J = decltype(JC)::value, k = J / KS;
            constexpr std::integral_constant<int, J + 1> J1{};
            constexpr std::integral_constant<int, J + 2> J2{};
            // where a group's bytes have all been read (its last two blocks are in
            // registers), the next group's take their place
            if constexpr (J == 14) {
#pragma unroll
                for (int q = 0; q < CT; q++) he[q] = F::hdr(line[q]);
                if (g + 1 < g1) {
                    qw_meet<63>();
                    stage_g(g + 1);
                }
            }
            // where a step ends, first the next step's x (this step's buffer has been
            // read by every wavefront), and the loads two steps on
            if constexpr (J % KS == KS - 1) {
                constexpr int kn = (k + 1) % NST, k2 = kn + 2, gn = J == 15 ? 1 : 0;
                qw_meet<XI + ((kn == 1 || kn == 2) ? NG : 0)>();
                buf = buf + 1 >= QW_NB ? 0 : buf + 1;
                load_x(g + gn + (k2 >= NST ? 1 : 0), k2 % NST, buf + 2 >= QW_NB ? buf + 2 - QW_NB : buf + 2);
                if constexpr (kn == 0) {
                    load_g(g + 2);
#pragma unroll
                    for (int q = 0; q < CT; q++) hn[q] = F::hdr(line[q]);
                    read_w(std::integral_constant<int, 16>{});
                }
                if constexpr (kn == SK && F::SUMS) {
#pragma unroll
                    for (int m = 0; m < MT; m++)
                        sums[m] = qh_ld128(ib, (uint32_t)((tb * TT + tw * MT + m) * ngroups + g) * (uint32_t)WImg::BYTES +
                                                   WImg::SUM + 16u * lane);
                }
            }
            if constexpr (J != 14) read_w(J2);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < CT; q++)
#pragma unroll
                for (int m = 0; m < MT; m++)
                    c[m][q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo[m], b[J & 1][q], J == 0 ? zero : c[m][q], 0, 0, 0);
            read_x(J1, 1, lo);
            convert(J1, J == 15 ? hn : hd);
#pragma unroll
            for (int q = 0; q < CT; q++)
#pragma unroll
                for (int m = 0; m < MT; m++)
                    c[m][q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi[m], b[J & 1][q], c[m][q], 0, 0, 0);
            read_x(J1, 0, hi);
            __builtin_amdgcn_sched_barrier(0);
        };
        block(std::integral_constant<int, 0>{});
        block(std::integral_constant<int, 1>{});
        block(std::integral_constant<int, 2>{});
        block(std::integral_constant<int, 3>{});
        block(std::integral_constant<int, 4>{});
        block(std::integral_constant<int, 5>{});
        block(std::integral_constant<int, 6>{});
        block(std::integral_constant<int, 7>{});
        block(std::integral_constant<int, 8>{});
        block(std::integral_constant<int, 9>{});
        block(std::integral_constant<int, 10>{});
        block(std::integral_constant<int, 11>{});
        block(std::integral_constant<int, 12>{});
        block(std::integral_constant<int, 13>{});
        block(std::integral_constant<int, 14>{});
        block(std::integral_constant<int, 15>{});
        // the group's end: tot += (d P - 32 dmin M) 2^-s: register i is token 8 (i / 4) +
        // 4 hh + i % 4 of the tile
        const float* rs = rsl + (g & 1) * 32 * TT + tw * MT * 32 + 4 * hh;
#pragma unroll
        for (int m = 0; m < MT; m++) {
            float r[16];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const qh_u32x4 v = qh_lds128(reinterpret_cast<const unsigned char*>(rs + 32 * m + 8 * i));
#pragma unroll
                for (int e = 0; e < 4; e++) r[4 * i + e] = __uint_as_float(v[e]);
            }
#pragma unroll
            for (int q = 0; q < CT; q++) {
                if constexpr (F::SUMS) {
                    const qh_f32x16 mm = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(qh_f16x8, sums[m]),
                                                                                 F::minw(he[q]), zero, 0, 0, 0);
                    const float dm = he[q].dm * -32.0f;
#pragma unroll
                    for (int i = 0; i < 16; i++)
                        tot[m][q][i] = fmaf(fmaf(dm, mm[i], he[q].d * c[m][q][i]), r[i], tot[m][q][i]);
                } else {
#pragma unroll
                    for (int i = 0; i < 16; i++) tot[m][q][i] = fmaf(he[q].d * c[m][q][i], r[i], tot[m][q][i]);
                }
                __builtin_amdgcn_sched_barrier(0);  // one tile's minimum products at a time (registers)
            }
        }
#pragma unroll
        for (int q = 0; q < CT; q++) hd[q] = hn[q];
    }
    qw_wait<0>();  // the loads past the end (zeros) still write LDS

    // results
    const int t0 = (tb * TT + tw * MT) * 32 + 4 * hh, col0 = cb * S::COLS + cw * CT * 32 + R;
    auto put = [&](int m, int q, const qh_f32x16& v) {
        const int col = col0 + 32 * q;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = t0 + 32 * m + 8 * (i >> 2) + (i & 3);
            if (t < a.n && col < a.rows) {
                float* yp = a.y + (size_t)t * a.ldy + col;
                *yp = a.accum ? *yp + v[i] : v[i];
            }
        }
    };
    if (a.splits == 1) {
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int q = 0; q < CT; q++) put(m, q, tot[m][q]);
        return;
    }
    // Split K: as qh_mmq_body, per wavefront (agent-scope stores, arrival counter,
    // the last one adds the splits in order).
    constexpr int PW = MT * CT * 1024;
    const size_t slot = (size_t)((cb * a.tblocks + tb) * 8 + w);
    float* mine = a.part + (slot * a.splits + sp) * PW + lane;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int q = 0; q < CT; q++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                __hip_atomic_store(mine + ((m * CT + q) * 16 + i) * 64, tot[m][q][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    qw_wait<0>();
    unsigned old = 0;
    if (lane == 0) old = __hip_atomic_fetch_add(&a.cnt[slot], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    old = (unsigned)__builtin_amdgcn_readfirstlane((int)old);
    if (old != (unsigned)(a.splits - 1)) return;
    const QhBuf pb = qh_buf(a.part, 4u * QG_PART_FLOATS);
    const uint32_t base = 4u * (uint32_t)(slot * a.splits * PW) + 4u * lane;
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int q = 0; q < CT; q++) tot[m][q] = zero;
    constexpr int KP = 64 / (MT * CT * 16);  // splits in flight together: a round trip to memory per KP
    for (int k0 = 0; k0 < a.splits; k0 += KP) {
        uint32_t u[KP][MT * CT][16];
#pragma unroll
        for (int k = 0; k < KP; k++)
#pragma unroll
            for (int j = 0; j < MT * CT; j++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    u[k][j][i] = __builtin_amdgcn_raw_buffer_load_b32(
                        pb.rs, (int)((base + 4u * (uint32_t)((k0 + k) * PW + (j * 16 + i) * 64)) | (k0 + k < a.splits ? 0u : 0x80000000u)), 0, 16);
#pragma unroll
        for (int k = 0; k < KP; k++)
#pragma unroll
            for (int j = 0; j < MT * CT; j++)
#pragma unroll
                for (int i = 0; i < 16; i++) tot[j / CT][j % CT][i] += __uint_as_float(u[k][j][i]);
    }
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int q = 0; q < CT; q++) put(m, q, tot[m][q]);
    if (lane == 0) __hip_atomic_store(&a.cnt[slot], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // next call
}

// ---------------------------------------------------------------- launch

template <class F, int MT, int CT, int TW>
static void launch_mmw(const QwArgs& a, hipStream_t st) {
    const int blocks = (a.rows + QwShape<F, MT, CT, TW>::COLS - 1) / QwShape<F, MT, CT, TW>::COLS;
    hipLaunchKernelGGL((qh_mmw<F, MT, CT, TW>), dim3((unsigned)((blocks * a.splits + 7) / 8 * 8 * a.tblocks)), dim3(512), 0, st,
                       a);
}

// Estimated times (us) of one matrix of mw million weights on n tokens: qh_mmq in
// 32-token passes, and this kernel with tiles of 64 and 128 tokens.  Fits of
// measurements on MI355X (us, qh_mmq / 64 / 128): Q4_K 14336 x 4096 at 128 tokens
// 53 / 48 / 66, 256: 103 / 84 / 78, 512: 197 / 155 / 129; 4096 x 4096 at 128: 27 /
// 28 / 37, 512: 68 / 53 / 60; Q6_K 4096 x 14336 at 77: 62 / 55 / 72, 512: 225 / 162
// / 152; IQ3_S 14336 x 4096 at 100: 79 / 60 / 88, 512: 278 / 187 / 163;
// Q5_K 1000 x 2048 at 300: 17 / 22 / 33.  A split costs its partials and a round of
// the merge (4096 x 14336 at 64 tokens and 16 splits: Q4_K 43 against 34 with 4 at
// 14336 x 4096; IQ3_S at 65 and 8: 74 against 58 with 2).
enum { QW_NONE = 0, QW_64 = 1, QW_128 = 2 };
static int qw_splits(int64_t blocks, int ngroups) {
    return blocks * 8 <= (int64_t)QG_PART_TILES * QG_WAVES ? qg_pick_splits((int)blocks, ngroups, ngroups, QG_TARGET_WGS) : 1;
}
static int qw_pick(uint32_t type, int rows, int ngroups, int n) {
    const bool iq = type == QT_IQ3_S || type == QT_IQ2_XXS;
    // per million weights and pass of 32, 64 and 128 tokens; per split
    const float k32 = type == QT_Q6_K ? 0.25f : (type == QT_IQ3_S ? 0.28f : (type == QT_IQ2_XXS ? 0.24f : 0.20f));
    const float k64 = type == QT_Q6_K ? 0.325f : (type == QT_IQ3_S ? 0.355f : (type == QT_IQ2_XXS ? 0.32f : 0.285f));
    const float k128 = type == QT_Q6_K ? 0.57f : (type == QT_IQ3_S ? 0.60f : (type == QT_IQ2_XXS ? 0.55f : 0.51f));
    const float ks = iq ? 2.5f : 0.7f;
    const float mw = (float)rows * (float)ngroups * 256e-6f;
    const int c32 = (n + 31) / 32, c64 = (n + 63) / 64, c128 = (n + 127) / 128;
    const int64_t cb = (rows + 255) / 256;
    const float t32 = 13.f + k32 * mw * (float)c32;
    const float t64 = 15.f + ks * (float)qw_splits(cb * c64, ngroups) + k64 * mw * (float)c64;
    const float t128 = 22.f + ks * (float)qw_splits(cb * c128, ngroups) + k128 * mw * (float)c128;
    if (t32 <= t64 && t32 <= t128) return QW_NONE;
    return t64 <= t128 ? QW_64 : QW_128;
}

// Y[t][0 .. rows) (+)= W X[t] (X = silu(X) X2 with X2) for n > 32 tokens, one
// weight pass per launch; hipErrorNotSupported where qh_mmq is the faster one.
// `have`: whose images the previous matrix of the same grouped call left in the
// image array; updated.
hipError_t qw_run(uint32_t type, const uint8_t* W, const float* X, const float* X2, float* Y, int n, int rows, int in_dim,
                  int accum, const QgScratch& sc, QwImgs* have, hipStream_t st) {
    const int ngroups = in_dim / 256;
    const uint32_t row_bytes = (uint32_t)qh_type_size(type, (size_t)in_dim);
    const int shape = n > 32 ? qw_pick(type, rows, ngroups, n) : QW_NONE;
    if (shape == QW_NONE || (int64_t)rows * row_bytes >= ((int64_t)1 << 31) - 4096) return hipErrorNotSupported;
    const int tile = shape == QW_128 ? 128 : 64;
    // tokens whose images fit the array, in whole tiles
    const int64_t cap = (int64_t)QG_IMG_BYTES / ((int64_t)ngroups * WImg::BYTES) * 32 / tile * tile;
    if (cap < tile) return hipErrorNotSupported;
    for (int t0 = 0; t0 < n; t0 += (int)cap) {
        const int nt = n - t0 < cap ? n - t0 : (int)cap, tiles = (nt + 31) / 32;
        const float* x = X + (size_t)t0 * in_dim;
        const float* x2 = X2 ? X2 + (size_t)t0 * in_dim : nullptr;
        if (have->x != x || have->x2 != x2 || have->n != nt) {
            hipLaunchKernelGGL(qw_image, dim3((unsigned)ngroups, (unsigned)tiles), dim3(1024), 0, st, x, x2, sc.img, nt, in_dim);
            *have = QwImgs{x, x2, nt};
        }
        QwArgs a = {};
        a.w = W;
        a.img = sc.img;
        a.y = Y + (size_t)t0 * rows;
        a.part = sc.part;
        a.cnt = sc.cnt;
        a.wbytes = (uint32_t)(((uint64_t)rows * row_bytes + 3) & ~(uint64_t)3);
        a.img_bytes = (uint32_t)((int64_t)tiles * ngroups * WImg::BYTES);
        a.row_bytes = row_bytes;
        a.in_dim = in_dim;
        a.rows = rows;
        a.n = nt;
        a.ldy = rows;
        a.accum = accum;
        a.tblocks = (nt + tile - 1) / tile;
        const int64_t blocks = (int64_t)((rows + 255) / 256) * a.tblocks;  // both shapes: 256 rows
        a.splits = qw_splits(blocks, ngroups);
        const int64_t pw = 8 * (shape == QW_128 ? 4 : 2) * 1024;  // floats of a workgroup's partial
        while (a.splits > 1 && blocks * a.splits * pw > QG_PART_FLOATS) a.splits--;
#define QW_GO(F)                                     \
    if (shape == QW_128) launch_mmw<F, 2, 2, 2>(a, st); \
    else launch_mmw<F, 2, 1, 1>(a, st)
        switch (type) {
            case QT_Q4_K: QW_GO(GQ4K); break;
            case QT_Q5_K: QW_GO(GQ5K); break;
            case QT_IQ3_S: QW_GO(GIQ3S); break;
            case QT_IQ2_XXS: QW_GO(GIQ2XXS); break;
            default: QW_GO(GQ6K); break;
        }
#undef QW_GO
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
