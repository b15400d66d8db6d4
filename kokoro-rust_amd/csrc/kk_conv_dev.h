// kk_conv_dev.h -- what the MFMA convolution kernels share (kk_conv.hip, kk_conv_narrow.hip): the
// producers' staging of input slabs with the layer's prologue, the residual operands, the residual
// rules and the stores of the epilogues.  Device code; include it in .hip files only.
#pragma once
#include "kk_common.h"
#include "kk_kernels.h"
#include "kk_walk.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace kk {

namespace {

constexpr int kCK = 64;       // input channels per LDS slab
constexpr int kRS = kCK + 8;  // LDS row stride (bf16 elements, 144 bytes)
constexpr int kNJ = 8;        // 16-column MFMA tiles per wave (wave N = 128)
constexpr int kMaxHalo = 64;    // largest (k - 1) * dil the staging covers
constexpr int kSmallHalo = 16;  // layers with (k - 1) * dil up to this run fewer producer passes
constexpr int kNP = 256;      // producer threads per block

typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
    const bf16x2_t v = __builtin_convertvector((f32x2_t){a, b}, bf16x2_t);  // v_cvt_pk_bf16_f32 (RNE)
    return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ uint32_t pack_f16x2(float a, float b) {
    const f16x2_t v = __builtin_convertvector((f32x2_t){a, b}, f16x2_t);  // v_cvt_pk_f16_f32 (RNE)
    return __builtin_bit_cast(uint32_t, v);
}

// Read-only tables (tiles, item spans) through the constant address space: uniform indices become
// scalar loads, which leave the vector-memory counter -- and the producers' prefetch -- alone.
template <typename T>
__device__ __forceinline__ T ld_const(const T* p, int64_t i) {
    return ((const __attribute__((address_space(4))) T*)p)[i];
}

// Per-device flags (device ordinals below 64), safe to set from several host threads.
struct DeviceFlags {
    std::atomic<uint64_t> bits{0};
    bool test(int dev) const { return dev >= 0 && dev < 64 && ((bits.load() >> dev) & 1u); }
    void set(int dev) {
        if (dev >= 0 && dev < 64) bits.fetch_or(1ull << dev);
    }
};

// One (tile, M-block) unit of work.  Rows fit in 32 bits (checked on the host).
struct Unit {
    int tile, n0, in0, i_lo, i_hi, m0, item, nv;
};

// An empty asm that reads its operands: whatever produces them (e.g. their loads) completes here,
// once and outside any branch.  Without it, a first use inside a branch that may be skipped makes
// the wait-count pass (whose state merges conservatively at join points) wait for every later load.
__device__ __forceinline__ void ready(const float4& v) { asm volatile("" ::"v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w)); }
__device__ __forceinline__ void ready(uint32_t v) { asm volatile("" ::"v"(v)); }
// Copy a (uniform) value into a VGPR, so it is not rematerialized from memory inside a loop.
__device__ __forceinline__ int vgpr(int x) {
    int v;
    asm volatile("v_mov_b32 %0, %1" : "=v"(v) : "s"(x));
    return v;
}
__device__ __forceinline__ float vgpr_f(float x) { return __int_as_float(vgpr(__float_as_int(x))); }

// Producer side: one slab = rows [in0, in0 + tw) x channels [c0, c0 + 64) of the input.  Producer
// thread pt owns channel quad q = (pt % 16) * 4 of rows pt / 16 + j * RP (j < RB).  A Slot holds one
// slab's raw input and the per-channel prologue constants in registers; load() issues every global
// load of the slab (addresses outside the unit's item are clamped to a row of the item, so the
// number of loads is fixed and the producers' wait counts are static), convert() applies the
// prologue and writes bf16 rows into an LDS buffer.  Rows outside the item, and channels >= cin,
// are staged as 0 (the conv's zero padding of the activated signal).
template <int PRO, bool IN_H, int BN, int MAXH>
struct Slot {
    static constexpr int RP = kNP / 16;                   // rows per pass
    static constexpr int RB = (BN + MAXH + RP - 1) / RP;  // passes (MAXH: the largest halo served)
    static constexpr bool WIDE = PRO != PRO_BF16 && !IN_H;    // f32 source: 4 dwords per quad
    static constexpr int NW = WIDE ? 4 : 2;
    static constexpr bool ADAIN = PRO == PRO_ADAIN_LEAKY || PRO == PRO_ADAIN_SNAKE;
    static constexpr bool SNAKE = PRO == PRO_ADAIN_SNAKE;
    uint32_t raw[RB][NW];
    float4 k01, k23;  // AdaIN coefficients (sc, sh) of channels c..c+1 and c+2..c+3
    float4 ar, ai;    // Snake alpha / (2 pi) and 1 / alpha

    // Slab (u, c0): row in0 + r (r = rr + j RP < tw) is read clamped into the item's rows and
    // channel c0 + q as channel 0 past cin (the conversion zeroes both).  Addresses are 32-bit byte
    // offsets from the item's first row (a uniform base), one clamp and one 24-bit multiply-add per
    // row.
    __device__ __forceinline__ void load(const ConvParams& p, const Unit& u, int c0, int tw, int q, int rr) {
        const int c = c0 + q;
        const int cl = c < p.cin ? c : 0;
        constexpr int ES = WIDE ? 4 : 2;  // bytes per element
        const char* base = (const char*)p.x + (int64_t)u.i_lo * p.x_ld * ES;
        const uint32_t ld = (uint32_t)p.x_ld;
        const int r0 = u.in0 - u.i_lo, rmax = u.i_hi - 1 - u.i_lo;  // row offsets from the item start
#pragma unroll
        for (int j = 0; j < RB; j++) {
            // rows past the slab's window re-read its first row (a cache hit, no HBM traffic); the
            // first BN / RP passes lie inside every window (tw >= BN), with no test
            const int r = ((j + 1) * RP <= BN || rr + j * RP < tw) ? rr + j * RP : 0;
            const uint32_t row = (uint32_t)max(min(r0 + r, rmax), 0);
            const uint32_t off = (__umul24(row, ld) + (uint32_t)cl) * ES;
            if constexpr (WIDE) {
                const uint4 x = *(const uint4*)(base + off);
                raw[j][0] = x.x, raw[j][1] = x.y, raw[j][2] = x.z, raw[j][3] = x.w;
            } else {
                const uint2 h = *(const uint2*)(base + off);
                raw[j][0] = h.x, raw[j][1] = h.y;
            }
        }
        if constexpr (ADAIN) {
            const float4* kp = (const float4*)(p.coef + (int64_t)u.item * p.cin + cl);
            k01 = kp[0], k23 = kp[1];
        }
        if constexpr (SNAKE) {
            ar = *(const float4*)(p.alpha_rev + cl);
            ai = *(const float4*)(p.alpha_inv + cl);
        }
    }

    // Converts the slab into LDS rows [r][kRS]: the layer's prologue once per element, rows outside
    // the item (gap masking) and channels past cin as zero, branch-free per row.
    __device__ __forceinline__ void convert(const ConvParams& p, uint16_t* xs, const Unit& u, int c0, int tw, int q,
                                            int rr) const {
        const int c = c0 + q;
#pragma unroll
        for (int j = 0; j < RB; j++)
#pragma unroll
            for (int e = 0; e < NW; e++) ready(raw[j][e]);
        if constexpr (ADAIN) ready(k01), ready(k23);
        if constexpr (SNAKE) ready(ar), ready(ai);
        const float sc[4] = {k01.x, k01.z, k23.x, k23.z}, sh[4] = {k01.y, k01.w, k23.y, k23.w};
        // Snake in its cosine form, with the AdaIN affine folded into both operands (four channel
        // constants per slab, three VALU operations and one cosine per element):
        //   v + sin^2(a v) / a = (v + h) - h cos(2 a v),  h = 1 / (2 a),
        //   2 a v / (2 pi) = x (sc a / pi) + sh a / pi   (__builtin_amdgcn_cosf(t) = cos(2 pi t)).
        float tsc[4], tsh[4], vsh[4], nh[4];
        if constexpr (SNAKE) {
            const float arv[4] = {ar.x, ar.y, ar.z, ar.w}, aiv[4] = {ai.x, ai.y, ai.z, ai.w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float a_pi = 2.0f * arv[e], h = 0.5f * aiv[e];  // a / pi, 1 / (2 a)
                tsc[e] = sc[e] * a_pi, tsh[e] = sh[e] * a_pi, vsh[e] = sh[e] + h, nh[e] = -h;
            }
        }
        // Per-slab limits, held in VGPRs for the whole loop (the kernel is short of SGPRs, and a
        // limit rematerialized from the kernel arguments costs a scalar load and a wait per row):
        // live rows r in [r_lo, r_hi), live channels e < n_ch of this quad.
        const int r_lo = vgpr(u.i_lo - u.in0), r_hi = vgpr(min(tw, u.i_hi - u.in0)), n_ch = p.cin - c;
        const uint32_t r_n = (uint32_t)(r_hi - r_lo);
        const float slope = vgpr_f(p.slope);
        uint16_t* xrow = xs + rr * kRS + q;
#pragma unroll
        for (int j = 0; j < RB; j++) {
            const int r = rr + j * RP;
            const bool live = (uint32_t)(r - r_lo) < r_n;
            uint2 out;
            if constexpr (PRO == PRO_BF16) {
                out = make_uint2(raw[j][0], raw[j][1]);  // bf16 input: channels >= cin hold 0
            } else {
                float v[4];
                if constexpr (WIDE) {
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = __uint_as_float(raw[j][e]);
                } else {
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        v[2 * e] = (float)__builtin_bit_cast(_Float16, (uint16_t)(raw[j][e] & 0xffffu));
                        v[2 * e + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(raw[j][e] >> 16));
                    }
                }
                float w[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    float x = v[e];
                    if constexpr (PRO == PRO_LEAKY) {
                        x = x < 0.f ? x * slope : x;
                    } else if constexpr (PRO == PRO_ADAIN_LEAKY) {
                        x = __builtin_fmaf(x, sc[e], sh[e]);
                        x = x < 0.f ? x * slope : x;
                    } else if constexpr (PRO == PRO_ADAIN_SNAKE) {
                        const float c = __builtin_amdgcn_cosf(__builtin_fmaf(x, tsc[e], tsh[e]));
                        x = __builtin_fmaf(c, nh[e], __builtin_fmaf(x, sc[e], vsh[e]));
                    }
                    // the Snake layers' cin is a multiple of the slab width (checked on the host)
                    if constexpr (!SNAKE) x = e < n_ch ? x : 0.f;
                    w[e] = x;
                }
                out = make_uint2(pack_bf16x2(w[0], w[1]), pack_bf16x2(w[2], w[3]));
            }
            if constexpr (PRO == PRO_BF16) {
                if (!live) out = make_uint2(0, 0);
            } else {
                if (!live || n_ch <= 0) out = make_uint2(0, 0);
            }
            // (a branch per row would keep the compiler from scheduling across rows)
            if ((j + 1) * RP <= BN || r < tw) *(uint2*)(xrow + j * RP * kRS) = out;
        }
    }
};

// ConvT epilogue geometry (kernels/kokoro.cu:452-467 for the reflection pad).  GEMM row m = phase
// ph x cout + co of input column t is output column o = stride t + ph - pad; the wave's 64 rows lie in
// one phase (cout is a multiple of 64).  EPI_CONVT writes y[o] = conv + b + r0[o] for o in the
// item's output span; EPI_CONVT_REFLECT applies ReflectionPad1d((1,0)) per item on the padded
// domain (padded[s] = ups[s + 1], padded[s + 1 + j] = ups[s + j]): it writes row o + 1 for
// o < len - 1, and the item's first row again from o = 1.
struct ConvTGeo {
    int64_t os, ol;  // the item's output span (rows written from ups: [os, os + ol))
    int ph, co;      // this lane's phase and first output channel
};

// Residual operands a stride-1 epilogue reads per 4 output rows.
template <int EPI>
constexpr int kNumRes = EPI == EPI_MEAN3_LEAKY_BF16 ? 3
                        : (EPI == EPI_ACCUM || EPI == EPI_RESID || EPI == EPI_RESID_UP2 || EPI == EPI_ADD_FROM) ? 1
                                                                                                                 : 0;

// Row pointers of one unit: every tensor the epilogue touches, advanced to the unit's first row
// (uniform), so a lane's element offset within the unit fits 32 bits.
struct EpiBase {
    void* y;
    const float *r0, *r1, *r2;
    __amdgpu_buffer_rsrc_t ry;   // y from the unit's first row, as a buffer resource (see store4)
    __amdgpu_buffer_rsrc_t rr0, rr1, rr2;  // EPI_ADD_FROM, EPI_MEAN3_LEAKY_BF16: r0..r2 likewise
};

// fp16 residual operands travel as their raw bits (4 halves in .x and .y) from the load to
// finish4, which widens them: converting at the load would wait for it there.
__device__ __forceinline__ float4 raw_h4(uint2 v) { return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), 0.f, 0.f); }
__device__ __forceinline__ float4 widen_h4(float4 raw) {
    const f16x2_t a = __builtin_bit_cast(f16x2_t, __float_as_uint(raw.x));
    const f16x2_t b = __builtin_bit_cast(f16x2_t, __float_as_uint(raw.y));
    return make_float4((float)a.x, (float)a.y, (float)b.x, (float)b.y);
}

// h + v for the four fp16 values of a raw residual (halves 0, 1 in .x, 2, 3 in .y): one
// v_fma_mix_f32 each, h widened in the instruction, h * one + v with one rounding -- the value that
// widening h and adding it in f32 gives.  `one` is 1.0 held in a VGPR (a literal 1.0 would turn
// the fma back into a widen and an add).
__device__ __forceinline__ float4 add_h4(float4 raw, float4 v, float one) {
    const f16x2_t a = __builtin_bit_cast(f16x2_t, __float_as_uint(raw.x));
    const f16x2_t b = __builtin_bit_cast(f16x2_t, __float_as_uint(raw.y));
    return make_float4(__builtin_fmaf((float)a.x, one, v.x), __builtin_fmaf((float)a.y, one, v.y),
                       __builtin_fmaf((float)b.x, one, v.z), __builtin_fmaf((float)b.y, one, v.w));
}
// The same with both operands raw fp16 residuals.
__device__ __forceinline__ float4 add_hh4(float4 raw_a, float4 raw_b, float one) {
    const f16x2_t b0 = __builtin_bit_cast(f16x2_t, __float_as_uint(raw_b.x));
    const f16x2_t b1 = __builtin_bit_cast(f16x2_t, __float_as_uint(raw_b.y));
    return add_h4(raw_a, make_float4((float)b0.x, (float)b0.y, (float)b1.x, (float)b1.y), one);
}

// x / 3 rounded to nearest, equal to the division x / 3.0f for every finite x (checked over all of
// them, tests/test_div3.py): q = x RN(1/3), the exact remainder as n = 3 q - x (one FMA), then
// Markstein's correction q - n RN(1/3) (one FMA).  The remainder is taken negated so that a zero
// x keeps its sign: x = -0 gives q = -0, n = +0 and -0 + -0 = -0 (with r = x - 3 q, r = +0 and
// the correction would give +0).  Three FMA-unit operations instead of the ~10 of a correctly
// rounded division.
__device__ __forceinline__ float div3(float x) {
    constexpr float kThird = 1.0f / 3.0f;
    const float q = __fmul_rn(x, kThird);
    const float n = __builtin_fmaf(3.0f, q, -x);
    return __builtin_fmaf(-n, kThird, q);
}

// Raw buffer resources (stride 0) of the epilogue's rows: byte offsets are 32-bit, and an offset
// past the range drops a store (see store4)
constexpr int kBufRecords = 0x7fffffff;         // the resource's range in bytes
constexpr uint32_t kDropOffset = 0x80000000u;   // past it: the store is dropped
constexpr int kCpolNT = 2;                      // cache policy: nontemporal
constexpr int kBufFormat = 0x00020000;          // descriptor word 3: 32-bit data format, no swizzle

// Residual operands of output row t, channels m..m+3 (`yo`, `ro`: element offsets from the unit's
// first row in y and r0..r2).
template <int EPI, bool OUT_H>
__device__ __forceinline__ void load_res(const ConvParams& p, const EpiBase& eb, uint32_t yo, uint32_t ro, int64_t t,
                                         int m, float4* r) {
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    if constexpr (EPI == EPI_ACCUM && OUT_H) {
        // the fp16 rows this epilogue overwrites, streamed like its stores (a buffer load: 32-bit
        // offsets, no 64-bit address arithmetic)
        const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(eb.ry, (int)(yo * 2u), 0, kCpolNT);
        r[0] = raw_h4(make_uint2(v.x, v.y));
    } else if constexpr (EPI == EPI_MEAN3_LEAKY_BF16) {
        const u32x2_t v0 = __builtin_amdgcn_raw_buffer_load_b64(eb.rr0, (int)(ro * 2u), 0, 0);
        const u32x2_t v1 = __builtin_amdgcn_raw_buffer_load_b64(eb.rr1, (int)(ro * 2u), 0, 0);
        const u32x2_t v2 = __builtin_amdgcn_raw_buffer_load_b64(eb.rr2, (int)(ro * 2u), 0, 0);
        r[0] = raw_h4(make_uint2(v0.x, v0.y));
        r[1] = raw_h4(make_uint2(v1.x, v1.y));
        r[2] = raw_h4(make_uint2(v2.x, v2.y));
    } else if constexpr (EPI == EPI_ACCUM || EPI == EPI_RESID) {
        // the rows this epilogue overwrites: streamed (nontemporal), like its stores
        const f32x4 v = __builtin_nontemporal_load((const f32x4*)((const float*)eb.y + yo));
        r[0] = make_float4(v.x, v.y, v.z, v.w);
    } else if constexpr (EPI == EPI_RESID_UP2) {
        r[0] = *(const float4*)(p.r0 + (t >> 1) * p.r0_ld + m);
    } else if constexpr (EPI == EPI_ADD_FROM && OUT_H) {
        const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(eb.rr0, (int)(ro * 2u), 0, 0);
        r[0] = raw_h4(make_uint2(v.x, v.y));
    } else if constexpr (EPI == EPI_ADD_FROM) {
        r[0] = *(const float4*)(eb.r0 + ro);
    }
}

// The residual rule applied to v (conv + bias) of 4 channels of one output row: the values to
// store (the statistics describe these: what the next layer reads).  With fp16 output, `pk` gets
// the fp16 bits.
template <int EPI, bool OUT_H>
__device__ __forceinline__ float4 finish4(const ConvParams& p, float4 v, const float4* r, uint2& pk, float one) {
    if constexpr (EPI == EPI_GELU_BF16) {
        // gelu_new x (1 + tanh u) / 2, u = sqrt(2 / pi) (x + 0.044715 x^3), once per element, as
        // x sigmoid(2 u) = x / (1 + 2^(-2 u log2 e)): one exp2 and one reciprocal (~1 ulp each, far
        // below the bf16 rounding that follows), no cancellation for negative x, and the limits
        // come out exact (2^(+inf) = inf -> -0, 2^(-inf) = 0 -> x).  Stored as the bf16 operand
        // the next linear's MFMA reads (round to nearest even, as its f32 prologue would do).
        constexpr float k2ul = 2.0f * 0.797884560802865355f * 1.44269504088896341f;
        float g[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float x = g[e];
            const float t = __builtin_amdgcn_exp2f(-k2ul * __builtin_fmaf(0.044715f * x, x * x, x));
            g[e] = x * __builtin_amdgcn_rcpf(1.0f + t);
        }
        pk = make_uint2(pack_bf16x2(g[0], g[1]), pack_bf16x2(g[2], g[3]));
        return v;
    } else if constexpr (EPI == EPI_MEAN3_LEAKY_BF16) {
        // ((rb0 + rb1) + (rb2_resid + conv)) / 3 (src/gpu_batch.rs:395-401) from the three fp16
        // residual streams, then the next layer's prologue (leaky ReLU, round to nearest even bf16):
        // the same operand bits that layer's PRO_LEAKY staging would produce
        const float4 ab = add_hh4(r[0], r[1], one), cv = add_h4(r[2], v, one);
        const float o[4] = {div3(ab.x + cv.x), div3(ab.y + cv.y), div3(ab.z + cv.z), div3(ab.w + cv.w)};
        // leaky ReLU as max(o, slope o): equal to o < 0 ? slope o : o for 0 < slope <= 1 (the
        // launch refuses other slopes), zeros' signs included
        const float slope = p.slope;
        float w[4];
#pragma unroll
        for (int e = 0; e < 4; e++) w[e] = __builtin_fmaxf(o[e], o[e] * slope);
        pk = make_uint2(pack_bf16x2(w[0], w[1]), pack_bf16x2(w[2], w[3]));
        return make_float4(o[0], o[1], o[2], o[3]);
    } else if constexpr (OUT_H && EPI == EPI_STORE) {
        // fp16 storage; the statistics describe the stored fp16 values (what the next layer reads;
        // ~2^-12 relative from the f32 values the reference's f32 h would give, far below the next
        // layer's bf16 operand rounding)
        pk = make_uint2(pack_f16x2(v.x, v.y), pack_f16x2(v.z, v.w));
        return v;
    }
    float4 o = v;
    if constexpr (EPI == EPI_ACCUM || EPI == EPI_ADD_FROM) {
        // an fp16 residual stream: the sum in f32, stored rounded to fp16 (statistics as above)
        if constexpr (OUT_H) {
            o = add_h4(r[0], v, one);
            pk = make_uint2(pack_f16x2(o.x, o.y), pack_f16x2(o.z, o.w));
        } else {
            const float4 y = r[0];
            o = make_float4(y.x + v.x, y.y + v.y, y.z + v.z, y.w + v.w);
        }
    } else if constexpr (EPI == EPI_RESID || EPI == EPI_RESID_UP2) {
        const float4 y = r[0];
        const float s = p.scale;
        o = make_float4((v.x + y.x) * s, (v.y + y.y) * s, (v.z + y.z) * s, (v.w + y.w) * s);
    }
    return o;
}

// Stores one row's result at element offset `yo` from the unit's first row of y, if `ok`.
// Buffer stores: a store of a lane that must not write gets a byte offset past the resource's
// range and is dropped by the hardware's range check, so no branch surrounds the store.  (Branches
// around stores make the compiler's vector-memory wait counts assume the store was skipped and
// wait for it on the other path: a residual load issued after a store would be waited for together
// with that store.)  Nontemporal: the layer's output is read again only by the next launch, so it
// streams through L2 instead of evicting the weights the A fragments reload every tap (1.4% of the
// Snake convs' time on the benchmark configuration).
template <bool OUT_H>
__device__ __forceinline__ void store4(const EpiBase& eb, uint32_t yo, bool ok, float4 o, uint2 pk) {
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    const uint32_t off = ok ? yo * (OUT_H ? 2u : 4u) : kDropOffset;
    if constexpr (OUT_H) {
        __builtin_amdgcn_raw_buffer_store_b64((u32x2_t){pk.x, pk.y}, eb.ry, (int)off, 0, kCpolNT);
    } else {
        __builtin_amdgcn_raw_buffer_store_b128(
            (u32x4_t){__float_as_uint(o.x), __float_as_uint(o.y), __float_as_uint(o.z), __float_as_uint(o.w)}, eb.ry,
            (int)off, 0, kCpolNT);
    }
}

// store4 with the byte offset given (kDropOffset: no store)
template <bool OUT_H>
__device__ __forceinline__ void store4b(const EpiBase& eb, uint32_t off, float4 o, uint2 pk) {
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    if constexpr (OUT_H) {
        __builtin_amdgcn_raw_buffer_store_b64((u32x2_t){pk.x, pk.y}, eb.ry, (int)off, 0, kCpolNT);
    } else {
        __builtin_amdgcn_raw_buffer_store_b128(
            (u32x4_t){__float_as_uint(o.x), __float_as_uint(o.y), __float_as_uint(o.z), __float_as_uint(o.w)}, eb.ry,
            (int)off, 0, kCpolNT);
    }
}

}  // namespace

}  // namespace kk
