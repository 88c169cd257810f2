// qh_dequant.hip -- bit-exact GGUF block decode on the GPU (hip_dequant).
//
// Each function restates the matching dequant_* of src/dequant.rs with the same
// f32 operations in the same order (contraction disabled), so every decoded value
// is bit-identical to Quartz's CPU decode.  The IQ codebooks live here as
// device globals initialised from iq_grids.h.
#define QH_GRIDS_NO_STATIC
#include "iq_grids.h"
#include "qh_formats.h"
#include "qh_internal.h"

__device__ uint64_t qh_g_iq2xxs[256] = {QH_IQ2XXS_GRID_VALUES};
__device__ uint64_t qh_g_iq2xs[512] = {QH_IQ2XS_GRID_VALUES};
__device__ uint64_t qh_g_iq2s[1024] = {QH_IQ2S_GRID_VALUES};
__device__ uint32_t qh_g_iq3s[512] = {QH_IQ3S_GRID_VALUES};

#pragma clang fp contract(off)

QH_DEV uint32_t qh_rd16(const uint8_t* p) { return (uint32_t)p[0] | ((uint32_t)p[1] << 8); }
QH_DEV uint32_t qh_rd32(const uint8_t* p) { return qh_rd16(p) | (qh_rd16(p + 2) << 16); }

QH_DEV void qh_gsm_k4(int j, const uint8_t* s, uint32_t& sc, uint32_t& m) {  // src/dequant.rs:1471-1480
    if (j < 4) {
        sc = s[j] & 63u;
        m = s[j + 4] & 63u;
    } else {
        sc = (s[j + 4] & 0x0Fu) | ((uint32_t)(s[j - 4] >> 6) << 4);
        m = (uint32_t)(s[j + 4] >> 4) | ((uint32_t)(s[j] >> 6) << 4);
    }
}

__device__ void qh_decode_block(uint32_t t, const uint8_t* b, float* o) {
    switch (t) {
        case QT_F32: o[0] = qh_bits(qh_rd32(b)); return;
        case QT_F16: o[0] = qh_f16(qh_rd16(b)); return;
        case QT_BF16: o[0] = qh_bits(qh_rd16(b) << 16); return;
        case QT_Q8_0: {  // :1450-1463
            const float d = qh_f16(qh_rd16(b));
            for (int i = 0; i < 32; i++) o[i] = d * (float)(int8_t)b[2 + i];
            return;
        }
        case QT_Q5_0: {  // :1381-1409
            const float d = qh_f16(qh_rd16(b));
            const uint32_t qh = qh_rd32(b + 2);
            for (int j = 0; j < 16; j++) {
                const uint32_t xh0 = ((qh >> j) << 4) & 0x10u, xh1 = (qh >> (j + 12)) & 0x10u;
                o[j] = (float)((int32_t)((b[6 + j] & 0x0Fu) | xh0) - 16) * d;
                o[j + 16] = (float)((int32_t)((uint32_t)(b[6 + j] >> 4) | xh1) - 16) * d;
            }
            return;
        }
        case QT_Q5_1: {  // :1419-1443
            const float d = qh_f16(qh_rd16(b)), m = qh_f16(qh_rd16(b + 2));
            const uint32_t qh = qh_rd32(b + 4);
            for (int j = 0; j < 16; j++) {
                const uint32_t xh0 = ((qh >> j) << 4) & 0x10u, xh1 = (qh >> (j + 12)) & 0x10u;
                o[j] = (float)((b[8 + j] & 0x0Fu) | xh0) * d + m;
                o[j + 16] = (float)((uint32_t)(b[8 + j] >> 4) | xh1) * d + m;
            }
            return;
        }
        case QT_Q4_0: {  // GGUF layout
            const float d = qh_f16(qh_rd16(b));
            for (int j = 0; j < 16; j++) {
                o[j] = (float)((int32_t)(b[2 + j] & 0x0Fu) - 8) * d;
                o[j + 16] = (float)((int32_t)(b[2 + j] >> 4) - 8) * d;
            }
            return;
        }
        case QT_Q4_1: {  // GGUF layout
            const float d = qh_f16(qh_rd16(b)), m = qh_f16(qh_rd16(b + 2));
            for (int j = 0; j < 16; j++) {
                o[j] = (float)(b[4 + j] & 0x0Fu) * d + m;
                o[j + 16] = (float)(b[4 + j] >> 4) * d + m;
            }
            return;
        }
        case QT_IQ4_NL: {  // :1557-1574
            const float T[16] = {-127.f, -104.f, -83.f, -65.f, -49.f, -35.f, -22.f, -10.f,
                                 1.f,    13.f,   25.f,  38.f,  53.f,  69.f,  89.f,  113.f};
            const float d = qh_f16(qh_rd16(b));
            for (int k = 0; k < 16; k++) {
                o[k] = d * T[b[2 + k] & 0x0F];
                o[k + 16] = d * T[b[2 + k] >> 4];
            }
            return;
        }
        case QT_Q4_K: {  // :1482-1519
            const float d = qh_f16(qh_rd16(b)), dmin = qh_f16(qh_rd16(b + 2));
            const uint8_t* sc = b + 4;
            const uint8_t* qs = b + 16;
            for (int it = 0; it < 4; it++) {
                uint32_t s1, mb1, s2, mb2;
                qh_gsm_k4(2 * it, sc, s1, mb1);
                qh_gsm_k4(2 * it + 1, sc, s2, mb2);
                const float d1 = d * (float)s1, m1 = dmin * (float)mb1;
                const float d2 = d * (float)s2, m2 = dmin * (float)mb2;
                for (int l = 0; l < 32; l++) o[64 * it + l] = d1 * (float)(qs[32 * it + l] & 0x0F) - m1;
                for (int l = 0; l < 32; l++) o[64 * it + 32 + l] = d2 * (float)(qs[32 * it + l] >> 4) - m2;
            }
            return;
        }
        case QT_Q5_K: {  // :1146-1181
            const float d = qh_f16(qh_rd16(b)), dmin = qh_f16(qh_rd16(b + 2));
            const uint8_t* sc = b + 4;
            const uint8_t* qh = b + 16;
            const uint8_t* qs = b + 48;
            uint32_t u1 = 1, u2 = 2;
            for (int jb = 0; jb < 4; jb++) {
                const uint8_t* ql = qs + 32 * jb;
                uint32_t s1, mm1, s2, mm2;
                qh_gsm_k4(2 * jb, sc, s1, mm1);
                const float d1 = d * (float)s1, m1 = dmin * (float)mm1;
                qh_gsm_k4(2 * jb + 1, sc, s2, mm2);
                const float d2 = d * (float)s2, m2 = dmin * (float)mm2;
                for (int l = 0; l < 32; l++)
                    o[64 * jb + l] = d1 * ((float)(ql[l] & 0xF) + ((qh[l] & u1) ? 16.0f : 0.0f)) - m1;
                for (int l = 0; l < 32; l++)
                    o[64 * jb + 32 + l] = d2 * ((float)(ql[l] >> 4) + ((qh[l] & u2) ? 16.0f : 0.0f)) - m2;
                u1 <<= 2;
                u2 <<= 2;
            }
            return;
        }
        case QT_Q6_K: {  // :1583-1631
            const float d = qh_f16(qh_rd16(b + 208));
            for (int h = 0; h < 2; h++) {
                const uint8_t* ql = b + 64 * h;
                const uint8_t* qh = b + 128 + 32 * h;
                const int8_t* sc = (const int8_t*)(b + 192 + 8 * h);
                float* y = o + 128 * h;
                for (int l = 0; l < 32; l++) {
                    const int is = l / 16;
                    const int q1 = (int)((ql[l] & 0x0F) | (((qh[l] >> 0) & 3) << 4)) - 32;
                    const int q2 = (int)((ql[l + 32] & 0x0F) | (((qh[l] >> 2) & 3) << 4)) - 32;
                    const int q3 = (int)((ql[l] >> 4) | (((qh[l] >> 4) & 3) << 4)) - 32;
                    const int q4 = (int)((ql[l + 32] >> 4) | (((qh[l] >> 6) & 3) << 4)) - 32;
                    y[l] = d * (float)sc[is] * (float)q1;
                    y[l + 32] = d * (float)sc[is + 2] * (float)q2;
                    y[l + 64] = d * (float)sc[is + 4] * (float)q3;
                    y[l + 96] = d * (float)sc[is + 6] * (float)q4;
                }
            }
            return;
        }
        case QT_Q2_K: {  // :1113-1144
            const uint8_t* scales = b;
            const uint8_t* qs = b + 16;
            const float d = qh_f16(qh_rd16(b + 80)), dmin = qh_f16(qh_rd16(b + 82));
            int is = 0, k = 0;
            for (int n = 0; n < 2; n++) {
                const uint8_t* q = qs + 32 * n;
                for (int j = 0; j < 4; j++) {
                    const int shift = 2 * j;
                    uint32_t sc = scales[is++];
                    float dl = d * (float)(sc & 0xF), ml = dmin * (float)(sc >> 4);
                    for (int l = 0; l < 16; l++) o[k++] = dl * (float)((q[l] >> shift) & 3) - ml;
                    sc = scales[is++];
                    dl = d * (float)(sc & 0xF);
                    ml = dmin * (float)(sc >> 4);
                    for (int l = 0; l < 16; l++) o[k++] = dl * (float)((q[l + 16] >> shift) & 3) - ml;
                }
            }
            return;
        }
        case QT_IQ2_XXS: {  // :1011-1041
            const float d = qh_f16(qh_rd16(b));
            const uint8_t* qs = b + 2;
            int k = 0;
            for (int ib32 = 0; ib32 < 8; ib32++) {
                const uint32_t a1 = qh_rd32(qs + 8 * ib32 + 4);
                const float db = d * (0.5f + (float)(a1 >> 28)) * 0.25f;
                for (int l = 0; l < 4; l++) {
                    const uint64_t g = qh_g_iq2xxs[qs[8 * ib32 + l]];
                    const uint32_t signs = qh_ksigns((a1 >> (7 * l)) & 127u);
                    for (int j = 0; j < 8; j++) {
                        const float s = (signs & (1u << j)) ? -1.0f : 1.0f;
                        o[k++] = db * (float)(int8_t)(g >> (8 * j)) * s;
                    }
                }
            }
            return;
        }
        case QT_IQ2_XS: {  // :1043-1075
            const float d = qh_f16(qh_rd16(b));
            const uint8_t* qs = b + 2;
            const uint8_t* scales = b + 66;
            int k = 0;
            for (int ib32 = 0; ib32 < 8; ib32++) {
                const float db0 = d * (0.5f + (float)(scales[ib32] & 0xF)) * 0.25f;
                const float db1 = d * (0.5f + (float)(scales[ib32] >> 4)) * 0.25f;
                for (int l = 0; l < 4; l++) {
                    const uint32_t q = qh_rd16(qs + 2 * (4 * ib32 + l));
                    const uint64_t g = qh_g_iq2xs[q & 511u];
                    const uint32_t signs = qh_ksigns(q >> 9);
                    const float db = l < 2 ? db0 : db1;
                    for (int j = 0; j < 8; j++) {
                        const float s = (signs & (1u << j)) ? -1.0f : 1.0f;
                        o[k++] = db * (float)(int8_t)(g >> (8 * j)) * s;
                    }
                }
            }
            return;
        }
        case QT_IQ2_S: {  // :1077-1110
            const float d = qh_f16(qh_rd16(b));
            const uint8_t* qs = b + 2;
            const uint8_t* qh = b + 66;
            const uint8_t* scales = b + 74;
            int k = 0;
            for (int ib32 = 0; ib32 < 8; ib32++) {
                const float db0 = d * (0.5f + (float)(scales[ib32] & 0xF)) * 0.25f;
                const float db1 = d * (0.5f + (float)(scales[ib32] >> 4)) * 0.25f;
                for (int l = 0; l < 4; l++) {
                    const float db = l < 2 ? db0 : db1;
                    const uint32_t idx = qs[4 * ib32 + l] | (((uint32_t)qh[ib32] << (8 - 2 * l)) & 0x300u);
                    const uint64_t g = qh_g_iq2s[idx];
                    const uint32_t signs = qs[32 + 4 * ib32 + l];
                    for (int j = 0; j < 8; j++) {
                        const float s = (signs & (1u << j)) ? -1.0f : 1.0f;
                        o[k++] = db * (float)(int8_t)(g >> (8 * j)) * s;
                    }
                }
            }
            return;
        }
        case QT_IQ3_S: {  // :1184-1237
            const float d = qh_f16(qh_rd16(b));
            const uint8_t* qs = b + 2;
            const uint8_t* qh = b + 66;
            const uint8_t* sg = b + 74;
            const uint8_t* scales = b + 106;
            int k = 0;
            for (int it = 0; it < 4; it++) {
                const float db1 = d * (1.0f + 2.0f * (float)(scales[it] & 0xF));
                const float db2 = d * (1.0f + 2.0f * (float)(scales[it] >> 4));
                for (int half = 0; half < 2; half++) {
                    const float db = half ? db2 : db1;
                    const uint32_t qhb = qh[2 * it + half];
                    const int qbase = 16 * it + 8 * half, sbase = 8 * it + 4 * half;
                    for (int l = 0; l < 4; l++) {
                        const uint32_t i0 = qs[qbase + 2 * l] | ((qhb << (8 - 2 * l)) & 256u);
                        const uint32_t i1 = qs[qbase + 2 * l + 1] | ((qhb << (7 - 2 * l)) & 256u);
                        const uint32_t g1 = qh_g_iq3s[i0], g2 = qh_g_iq3s[i1];
                        const uint32_t s = sg[sbase + l];
                        for (int j = 0; j < 4; j++)
                            o[k++] = db * (float)(int8_t)(g1 >> (8 * j)) * ((s & (1u << j)) ? -1.0f : 1.0f);
                        for (int j = 0; j < 4; j++)
                            o[k++] = db * (float)(int8_t)(g2 >> (8 * j)) * ((s & (1u << (j + 4))) ? -1.0f : 1.0f);
                    }
                }
            }
            return;
        }
        default: return;
    }
}

// Elements 16u .. 16u + 15 of a Q4_K or Q6_K block (u < 16), with the same f32
// operations as qh_decode_block, so 16 threads decode a block bit-identically
// to one thread decoding all of it.  False for other types.
__device__ bool qh_decode_part16(uint32_t t, const uint8_t* b, int u, float* o) {
    if (t == QT_Q4_K) {  // sub-block j = u / 2, positions 16 (u % 2) ..
        const int j = u >> 1, l0 = 16 * (u & 1);
        const float d = qh_f16(qh_rd16(b)), dmin = qh_f16(qh_rd16(b + 2));
        uint32_t s, mb;
        qh_gsm_k4(j, b + 4, s, mb);
        const float d1 = d * (float)s, m1 = dmin * (float)mb;
        const uint8_t* qs = b + 16 + 32 * (j >> 1) + l0;
        for (int l = 0; l < 16; l++) o[l] = d1 * (float)((j & 1) ? (qs[l] >> 4) : (qs[l] & 0x0F)) - m1;
        return true;
    }
    if (t == QT_Q6_K) {  // half h = u / 8, quarter r = (u / 2) % 4, positions 16 (u % 2) ..
        const int h = u >> 3, r = (u >> 1) & 3, l0 = 16 * (u & 1), is = l0 / 16;
        const float d = qh_f16(qh_rd16(b + 208));
        const uint8_t* ql = b + 64 * h + (r & 1) * 32;
        const uint8_t* qh = b + 128 + 32 * h;
        const int8_t* sc = (const int8_t*)(b + 192 + 8 * h);
        for (int l = l0; l < l0 + 16; l++) {
            const int q = (int)(((r < 2) ? (ql[l] & 0x0F) : (ql[l] >> 4)) | (((qh[l] >> (2 * r)) & 3) << 4)) - 32;
            o[l - l0] = d * (float)sc[is + 2 * r] * (float)q;
        }
        return true;
    }
    return false;
}

// Little-endian words at any byte address (GGUF fields are 1- or 2-byte
// aligned; gfx950 loads them as they stand).
typedef uint32_t qd_u32 __attribute__((aligned(1)));
typedef uint16_t qd_u16 __attribute__((aligned(1)));
typedef qh_u32x4 qd_u32x4 __attribute__((aligned(1)));
typedef qh_u32x2 qd_u32x2 __attribute__((aligned(1)));
typedef float qd_f32x4 __attribute__((ext_vector_type(4), aligned(4)));
QH_DEV uint32_t qd_rd32(const uint8_t* p) { return *reinterpret_cast<const qd_u32*>(p); }
QH_DEV uint32_t qd_rd16(const uint8_t* p) { return *reinterpret_cast<const qd_u16*>(p); }
QH_DEV uint32_t qd_byte(uint32_t w, int k) { return (w >> (8 * k)) & 0xFFu; }

// Elements 4u .. 4u + 3 of block b: the words they need (qd_raw, loads only) and
// the decode with qh_decode_block's f32 operations on them (qd_decode4), apart
// so that a thread's loads for several units are in flight together.
struct QdRaw {
    uint32_t h0, h1, h2, h3;  // scale fields
    uint32_t q, e;            // quants, and the format's second plane
};

template <uint32_t T>
QH_DEV QdRaw qd_raw(const uint8_t* b, int u) {
    QdRaw r = {};
    if constexpr (T == QT_F32) {
        const qh_u32x4 v = *reinterpret_cast<const qd_u32x4*>(b + 16 * u);
        r.h0 = v.x; r.h1 = v.y; r.h2 = v.z; r.h3 = v.w;
    } else if constexpr (T == QT_F16 || T == QT_BF16) {
        const qh_u32x2 v = *reinterpret_cast<const qd_u32x2*>(b + 8 * u);
        r.h0 = v.x; r.h1 = v.y;
    } else if constexpr (T == QT_Q8_0) {
        r.h0 = qd_rd16(b);
        r.q = qd_rd32(b + 2 + 4 * u);
    } else if constexpr (T == QT_Q4_0 || T == QT_IQ4_NL) {
        r.h0 = qd_rd16(b);
        r.q = qd_rd32(b + 2 + 4 * (u & 3));
    } else if constexpr (T == QT_Q4_1) {
        r.h0 = qd_rd32(b);
        r.q = qd_rd32(b + 4 + 4 * (u & 3));
    } else if constexpr (T == QT_Q5_0) {
        r.h0 = qd_rd16(b);
        r.e = qd_rd32(b + 2);
        r.q = qd_rd32(b + 6 + 4 * (u & 3));
    } else if constexpr (T == QT_Q5_1) {
        r.h0 = qd_rd32(b);
        r.e = qd_rd32(b + 4);
        r.q = qd_rd32(b + 8 + 4 * (u & 3));
    } else if constexpr (T == QT_Q4_K || T == QT_Q5_K) {
        const qh_u32x4 v = *reinterpret_cast<const qd_u32x4*>(b);
        r.h0 = v.x; r.h1 = v.y; r.h2 = v.z; r.h3 = v.w;
        if constexpr (T == QT_Q5_K) r.e = qd_rd32(b + 16 + 4 * (u & 7));
        r.q = qd_rd32(b + (T == QT_Q5_K ? 48 : 16) + 32 * (u >> 4) + 4 * (u & 7));
    } else if constexpr (T == QT_Q6_K) {
        const int h = u >> 5, k = (u >> 3) & 3, l = 4 * (u & 7);
        r.h0 = qd_rd16(b + 208);
        r.h1 = b[192 + 8 * h + 2 * k + (l >> 4)];
        r.q = qd_rd32(b + 64 * h + 32 * (k & 1) + l);
        r.e = qd_rd32(b + 128 + 32 * h + l);
    } else if constexpr (T == QT_Q2_K) {
        r.h0 = qd_rd32(b + 80);
        r.h1 = b[u >> 2];
        r.q = qd_rd32(b + 16 + 32 * (u >> 5) + 4 * (u & 7));
    } else if constexpr (T == QT_IQ2_XXS) {  // group l = (u / 2) % 4 of sub-block u / 8, its half u % 2
        r.h0 = qd_rd16(b);
        r.q = b[2 + 8 * (u >> 3) + ((u >> 1) & 3)];
        r.e = qd_rd32(b + 6 + 8 * (u >> 3));
    } else if constexpr (T == QT_IQ2_XS) {
        r.h0 = qd_rd16(b);
        r.h1 = b[66 + (u >> 3)];
        r.q = qd_rd16(b + 2 + 2 * (u >> 1));
    } else if constexpr (T == QT_IQ2_S) {
        r.h0 = qd_rd16(b);
        r.h1 = b[74 + (u >> 3)];
        r.q = b[2 + (u >> 1)] | ((uint32_t)b[66 + (u >> 3)] << 8);
        r.e = b[34 + (u >> 1)];
    } else if constexpr (T == QT_IQ3_S) {
        r.h0 = qd_rd16(b);
        r.h1 = b[106 + (u >> 4)];
        r.q = b[2 + u] | ((uint32_t)b[66 + (u >> 3)] << 8);
        r.e = b[74 + (u >> 1)];
    }
    return r;
}

template <uint32_t T>
QH_DEV qh_u32x4 qd_decode4(const QdRaw& r, int u) {
    float o[4];
    if constexpr (T == QT_F32) return qh_u32x4{r.h0, r.h1, r.h2, r.h3};
    if constexpr (T == QT_F16) {
        o[0] = qh_f16(r.h0); o[1] = qh_f16(r.h0 >> 16); o[2] = qh_f16(r.h1); o[3] = qh_f16(r.h1 >> 16);
    } else if constexpr (T == QT_BF16) {
        return qh_u32x4{r.h0 << 16, r.h0 & 0xFFFF0000u, r.h1 << 16, r.h1 & 0xFFFF0000u};
    } else if constexpr (T == QT_Q8_0) {
        const float d = qh_f16(r.h0);
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = d * (float)(int8_t)qd_byte(r.q, i);
    } else if constexpr (T == QT_Q4_0 || T == QT_Q4_1 || T == QT_Q5_0 || T == QT_Q5_1 || T == QT_IQ4_NL) {
        const int hi = (u >> 2) & 1;  // elements 16 .. 31: the high nibbles
        const uint32_t w = hi ? (r.q >> 4) & 0x0F0F0F0Fu : r.q & 0x0F0F0F0Fu;
        const float d = qh_f16(r.h0);
        if constexpr (T == QT_IQ4_NL) {
            // the 16 codebook bytes as two v_perm tables of 8, picked by bit 3
            const uint32_t s = w & 0x07070707u;
            const uint32_t lo = __builtin_amdgcn_perm(0xF6EADDCFu, 0xBFAD9881u, s);
            const uint32_t up = __builtin_amdgcn_perm(0x71594535u, 0x26190D01u, s);
            const uint32_t m = ((w >> 3) & 0x01010101u) * 0xFFu;
            const uint32_t v = (lo & ~m) | (up & m);
#pragma unroll
            for (int i = 0; i < 4; i++) o[i] = d * (float)(int8_t)qd_byte(v, i);
        } else {
            uint32_t v = w;
            if constexpr (T == QT_Q5_0 || T == QT_Q5_1)  // the fifth bits: 4 consecutive bits of qh
                v |= qh_spread4((r.e >> (16 * hi + 4 * (u & 3))) & 0xFu) << 4;
            const float m = (T == QT_Q4_1 || T == QT_Q5_1) ? qh_f16(r.h0 >> 16) : 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int q = (int)qd_byte(v, i);
                if constexpr (T == QT_Q4_0) o[i] = (float)(q - 8) * d;
                else if constexpr (T == QT_Q5_0) o[i] = (float)(q - 16) * d;
                else o[i] = (float)q * d + m;
            }
        }
    } else if constexpr (T == QT_Q4_K || T == QT_Q5_K) {
        const int j = u >> 3;  // sub-block
        const float d = qh_f16(r.h0), dmin = qh_f16(r.h0 >> 16);
        // bytes j % 4 of the three scale words (qh_gsm_k4)
        const uint32_t s0 = qd_byte(r.h1, j & 3), s1 = qd_byte(r.h2, j & 3), s2 = qd_byte(r.h3, j & 3);
        const uint32_t sc = j < 4 ? s0 & 63u : (s2 & 0x0Fu) | ((s0 >> 6) << 4);
        const uint32_t mb = j < 4 ? s1 & 63u : (s2 >> 4) | ((s1 >> 6) << 4);
        const float d1 = d * (float)sc, m1 = dmin * (float)mb;
        const uint32_t w = (j & 1) ? (r.q >> 4) & 0x0F0F0F0Fu : r.q & 0x0F0F0F0Fu;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float q = (float)qd_byte(w, i);
            if constexpr (T == QT_Q5_K) q = q + (((r.e >> (8 * i + j)) & 1u) ? 16.0f : 0.0f);
            o[i] = d1 * q - m1;
        }
    } else if constexpr (T == QT_Q6_K) {
        const int k = (u >> 3) & 3;
        const float d = qh_f16(r.h0), ds = d * (float)(int8_t)r.h1;
        const uint32_t lo = k < 2 ? r.q & 0x0F0F0F0Fu : (r.q >> 4) & 0x0F0F0F0Fu;
        const uint32_t v = lo | (((r.e >> (2 * k)) & 0x03030303u) << 4);
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = ds * (float)((int)qd_byte(v, i) - 32);
    } else if constexpr (T == QT_Q2_K) {
        const float d = qh_f16(r.h0), dmin = qh_f16(r.h0 >> 16);
        const float dl = d * (float)(r.h1 & 0xF), ml = dmin * (float)(r.h1 >> 4);
        const uint32_t w = (r.q >> (2 * ((u >> 3) & 3))) & 0x03030303u;
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = dl * (float)qd_byte(w, i) - ml;
    } else {
        const float d = qh_f16(r.h0);
        float db;
        uint32_t g, s;  // 4 codebook bytes and their sign bits
        if constexpr (T == QT_IQ2_XXS) {
            db = d * (0.5f + (float)(r.e >> 28)) * 0.25f;
            g = reinterpret_cast<const uint32_t*>(qh_g_iq2xxs)[2 * r.q + (u & 1)];
            s = qh_ksigns((r.e >> (7 * ((u >> 1) & 3))) & 127u);
        } else if constexpr (T == QT_IQ2_XS) {
            db = d * (0.5f + (float)((u & 4) ? r.h1 >> 4 : r.h1 & 0xF)) * 0.25f;
            g = reinterpret_cast<const uint32_t*>(qh_g_iq2xs)[2 * (r.q & 511u) + (u & 1)];
            s = qh_ksigns(r.q >> 9);
        } else if constexpr (T == QT_IQ2_S) {
            db = d * (0.5f + (float)((u & 4) ? r.h1 >> 4 : r.h1 & 0xF)) * 0.25f;
            const uint32_t i = (r.q & 0xFFu) | (((r.q >> 8) << (8 - 2 * ((u >> 1) & 3))) & 0x300u);
            g = reinterpret_cast<const uint32_t*>(qh_g_iq2s)[2 * i + (u & 1)];
            s = r.e;
        } else {  // IQ3_S: entry u % 8 of sub-block u / 8
            db = d * (1.0f + 2.0f * (float)(((u >> 3) & 1) ? r.h1 >> 4 : r.h1 & 0xF));
            g = qh_g_iq3s[(r.q & 0xFFu) | (((r.q >> 8) << (8 - (u & 7))) & 256u)];
            s = r.e;
        }
        s >>= 4 * (u & 1);
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = db * (float)(int8_t)qd_byte(g, i) * ((s & (1u << i)) ? -1.0f : 1.0f);
    }
    return qh_u32x4{__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]), __float_as_uint(o[3])};
}

#pragma clang fp contract(on)

// Four consecutive elements per thread and step, QD_UNITS steps 256 units apart:
// a wavefront's stores are 1 KB of consecutive output and its loads fall in a few
// cache lines, so the kernel is bound by the output's write bandwidth: Q6_K
// 14336 x 4096, 48 MB in and 235 MB out, 51.6 us (5.5 TB/s).  One thread per
// block, through a private array, with byte loads and stores a block apart,
// took 1193 us.
#define QD_UNITS 4
template <uint32_t T>
__global__ __launch_bounds__(256) void qh_dequant4(const uint8_t* __restrict__ W, float* __restrict__ out,
                                                   size_t n_units, uint32_t blk_bytes, uint32_t lg) {
    // lg = log2(units per block); formats of one element per block have blocks
    // of four here
    size_t u0 = (size_t)blockIdx.x * (256 * QD_UNITS) + threadIdx.x;
    QdRaw r[QD_UNITS];
    int ui[QD_UNITS];
#pragma unroll
    for (int k = 0; k < QD_UNITS; k++) {
        const size_t u = u0 + 256 * k < n_units ? u0 + 256 * k : n_units - 1;
        ui[k] = (int)(u & ((1u << lg) - 1u));
        r[k] = qd_raw<T>(W + (u >> lg) * blk_bytes, ui[k]);
    }
#pragma unroll
    for (int k = 0; k < QD_UNITS; k++) {
        const size_t u = u0 + 256 * k;
        if (u < n_units) {
            const qh_u32x4 v = qd_decode4<T>(r[k], ui[k]);
            reinterpret_cast<qd_f32x4*>(out)[u] = qd_f32x4{__uint_as_float(v.x), __uint_as_float(v.y),
                                                           __uint_as_float(v.z), __uint_as_float(v.w)};
        }
    }
}

// The last n % 4 elements of the one-element formats.
__global__ void qh_dequant_tail(uint32_t type, const uint8_t* __restrict__ W, float* __restrict__ out, int n,
                                uint32_t blk_bytes) {
    if ((int)threadIdx.x < n) qh_decode_block(type, W + (size_t)threadIdx.x * blk_bytes, out + threadIdx.x);
}

template <uint32_t T>
static void launch_dequant(const uint8_t* W, float* out, size_t n_elems, hipStream_t st) {
    const int qk = qh_block_elems(T);
    const uint32_t bb = qh_block_bytes(T);
    const uint32_t lg = qk == 256 ? 6 : (qk == 32 ? 3 : 0);
    const size_t n_units = n_elems / 4;
    const size_t per = 256 * QD_UNITS, most = (size_t)1 << 30;  // workgroups per launch below 2^31
    for (size_t u = 0; u < n_units; u += most * per) {
        const size_t n = n_units - u < most * per ? n_units - u : most * per;
        hipLaunchKernelGGL(qh_dequant4<T>, dim3((unsigned)((n + per - 1) / per)), dim3(256), 0, st,
                           W + (u >> lg) * (qk == 1 ? 4 * bb : bb), out + 4 * u, n, qk == 1 ? 4 * bb : bb, lg);
    }
    if (n_elems % 4)
        hipLaunchKernelGGL(qh_dequant_tail, dim3(1), dim3(64), 0, st, T, W + (n_elems & ~(size_t)3) * bb,
                           out + (n_elems & ~(size_t)3), (int)(n_elems % 4), bb);
}

hipError_t qh_launch_dequant(uint32_t type, const uint8_t* W, float* out, size_t n_elems, hipStream_t st) {
    if (n_elems < (size_t)qh_block_elems(type)) return hipSuccess;
    switch (type) {
        case QT_F32: launch_dequant<QT_F32>(W, out, n_elems, st); break;
        case QT_F16: launch_dequant<QT_F16>(W, out, n_elems, st); break;
        case QT_BF16: launch_dequant<QT_BF16>(W, out, n_elems, st); break;
        case QT_Q4_0: launch_dequant<QT_Q4_0>(W, out, n_elems, st); break;
        case QT_Q4_1: launch_dequant<QT_Q4_1>(W, out, n_elems, st); break;
        case QT_Q5_0: launch_dequant<QT_Q5_0>(W, out, n_elems, st); break;
        case QT_Q5_1: launch_dequant<QT_Q5_1>(W, out, n_elems, st); break;
        case QT_Q8_0: launch_dequant<QT_Q8_0>(W, out, n_elems, st); break;
        case QT_IQ4_NL: launch_dequant<QT_IQ4_NL>(W, out, n_elems, st); break;
        case QT_Q2_K: launch_dequant<QT_Q2_K>(W, out, n_elems, st); break;
        case QT_Q4_K: launch_dequant<QT_Q4_K>(W, out, n_elems, st); break;
        case QT_Q5_K: launch_dequant<QT_Q5_K>(W, out, n_elems, st); break;
        case QT_Q6_K: launch_dequant<QT_Q6_K>(W, out, n_elems, st); break;
        case QT_IQ2_XXS: launch_dequant<QT_IQ2_XXS>(W, out, n_elems, st); break;
        case QT_IQ2_XS: launch_dequant<QT_IQ2_XS>(W, out, n_elems, st); break;
        case QT_IQ2_S: launch_dequant<QT_IQ2_S>(W, out, n_elems, st); break;
        case QT_IQ3_S: launch_dequant<QT_IQ3_S>(W, out, n_elems, st); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
