// kk_conv_narrow.hip -- the MFMA convolutions of launches that leave most of the chip idle.
//
// kk_conv.hip's kernel gives a wave a 64 x 128 output tile and a block 256 x 128 or 128 x 256: the
// right trade where a launch has several such units per CU, but a short item's layer is a handful of
// units (a 40-frame item's decoder convolutions: 4 to 8 of 256 CUs), each a serial chain of
// hundreds of MFMA steps and one wave's epilogue over 64 x 128 values.  Here a block computes 32 or
// 64 output rows of 64 or 128 columns of one 128-column span of a tile (a "wave column" of
// kk_conv.hip): 2 or 4 consumer waves of 32 x 32 or 32 x 64 outputs, 4 producer waves staging the
// input slabs (the same staging code), and all of them in the epilogue; one block per unit.
// * What bounds it: the fixed part of a launch (3.5 us to start, 1 us for the unit's dependent table
//   loads, 1.5 to 2.7 us until the first slab is staged, 1 to 1.5 us of epilogue) and, per 64-channel
//   tap, a wave's 4 NJ dependent-pair MFMAs (264 cycles at NJ = 2; 410 measured).  Parameters
//   reloaded from the kernel arguments inside the loop, LDS reads issued ahead of the MFMAs instead
//   of between them, and loops whose early exits made the compiler's wait counts conservative cost
//   680 cycles per tap before.
// * Weight fragments are loaded kNwRing taps ahead into a ring of register sets (flat over slabs
//   and taps); a tap's LDS fragments one tap ahead; the producers hold 2 to 4 slabs in flight.
// * The arithmetic is kk_conv.hip's, value for value: every accumulator starts at the bias and runs
//   the same sequence of v_mfma_f32_32x32x16_bf16 (slab, tap, 16-channel step), the residual rules
//   are the shared finish4, and the statistics partials are summed in that epilogue's order (per
//   channel and column group cg: columns cg, cg + 4, ... in sequence, then the four groups), so a
//   layer's outputs and partials do not depend on which kernel ran it.
// launch_conv's rule (kNarrowUnits) says which launches come here.
#include "kk_conv_dev.h"

namespace kk {

namespace {

constexpr int kNwRing = 4;  // taps of weight fragments in flight

// A uniform value copied into SGPRs that the compiler cannot rematerialize from memory.
__device__ __forceinline__ int pin(int x) {
    int v;
    asm volatile("s_mov_b32 %0, %1" : "=s"(v) : "s"(x));
    return v;
}
__device__ __forceinline__ int64_t pin(int64_t x) {
    int64_t v;
    asm volatile("s_mov_b64 %0, %1" : "=s"(v) : "s"(x));
    return v;
}
template <class T>
__device__ __forceinline__ const T* pin(const T* x) {
    // (through the global address space: an address from an asm is otherwise a flat one)
    return (const T*)(const __attribute__((address_space(1))) T*)pin((int64_t)x);
}

// f(0), ..., f(N - 1) with compile-time arguments.
template <class F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void each(F&& f) {
    each_of(f, std::make_integer_sequence<int, N>{});
}

// Slabs of input in flight (register slots of the producers): as many as the register file takes
// without spilling next to the consumers' ring.
template <int PRO, bool IN_H, int BN, int MAXH>
constexpr int kNwSlots = PRO == PRO_BF16 ? 4 : BN == 64 && PRO == PRO_F32 ? (MAXH <= kSmallHalo ? 4 : 3)
                         : MAXH <= kSmallHalo && (IN_H || BN == 64) ? 3 : 2;

// BN: the block's columns, 128, or 64 for launches without statistics (a partial is one 128-column
// span's).
// WM: 32 WM output rows per block, 2 WM consumer waves.
template <int PRO, int EPI, bool STATS, bool IN_H, bool OUT_H, int MAXH, int BN, int WM>
__global__ __launch_bounds__(128 * WM + kNP) void conv_narrow_kernel(ConvGroup grp) {
    static_assert(kNwRing % 2 == 0, "the B double buffer alternates with the ring");
    static_assert(BN == 128 || (BN == 64 && !STATS), "a statistics partial is one 128-column span's");
    constexpr int BM = 32 * WM, NC = 128 * WM, NT = NC + kNP;
    constexpr int NJ = BN / 64;        // 32-column MFMA tiles per consumer wave
    constexpr int LD = BM + 4;         // LDS row stride of the output tile (f32), one column's rows
    constexpr int CQ = BM / 4;         // epilogue threads per column, 32 columns at a time
    constexpr int NI = BN / 32;        // epilogue columns per thread
    static_assert(32 * CQ <= NT, "epilogue threads");
    constexpr bool CONVT = EPI == EPI_CONVT || EPI == EPI_CONVT_REFLECT;
    constexpr int NR = CONVT ? 1 : kNumRes<EPI>;
    constexpr int NRA = NR > 0 ? NR : 1;
    constexpr bool HSTATS = STATS && OUT_H && !CONVT;  // as kk_conv.hip's epilogue
    extern __shared__ __align__(16) uint16_t xs[];
    // the group's layer of this block, its unit: M-block fastest, then the tile's wave column
    int gi = 0;
    while (gi + 1 < grp.n && (int)blockIdx.x >= grp.first[gi + 1]) gi++;
    // The loops' parameters pinned in SGPRs: reloaded from the kernel arguments (which the compiler
    // prefers) they cost a scalar load and its wait, ~200 cycles, per tap and per slab.
    ConvParams p = grp.p[gi];
    p.x = pin(p.x), p.x_ld = pin(p.x_ld), p.cin = pin(p.cin), p.k = pin(p.k), p.dil = pin(p.dil);
    p.w = pin(p.w), p.m_pad = pin(p.m_pad), p.cin_pad = pin(p.cin_pad);
    if constexpr (PRO == PRO_ADAIN_LEAKY || PRO == PRO_ADAIN_SNAKE) p.coef = pin(p.coef);
    if constexpr (PRO == PRO_ADAIN_SNAKE) p.alpha_rev = pin(p.alpha_rev), p.alpha_inv = pin(p.alpha_inv);
    const int mb = p.m_pad / BM, wnt = p.tile_wn * (128 / BN);
    const int v = blockIdx.x - grp.first[gi];
    const int wcol = (v / mb) % wnt;
    Unit u;
    u.tile = v / (mb * wnt);
    u.m0 = (v % mb) * BM;
    u.item = ld_const(p.tiles.item, u.tile);
    u.n0 = (int)ld_const(p.tiles.t0, u.tile) + wcol * BN;
    u.nv = max(min(ld_const(p.tiles.n, u.tile) - wcol * BN, BN), 0);
    u.i_lo = (int)ld_const(p.in_start, u.item);
    u.i_hi = u.i_lo + (int)ld_const(p.in_len, u.item);
    u.in0 = u.n0 - p.pad;
    if (u.nv == 0) {  // the tile ends before this wave column: empty records
        if constexpr (STATS && !CONVT) {
            const int ch = u.m0 + threadIdx.x;
            if (threadIdx.x < BM && ch < p.cout)
                p.part[((int64_t)u.tile * wnt + wcol) * p.cout + ch] = StatPart{0.f, 0.f, 0.f, 0.f};
        }
        return;
    }
    const int tw = BN + (p.k - 1) * p.dil;
    const int slab_elems = tw * kRS;
    const int nsl = p.cin_pad / kCK;
    float* T = (float*)xs;  // the output tile [column][LD], over the slabs once they are consumed

    if (threadIdx.x >= NC) {
        // ------------------------------------------------------------ producer waves
        // Slab g is staged before the barrier that ends the consumers' slab g - 1; NS register slots:
        // while slab g + 1 is converted the loads of the NS - 1 slabs after it are in flight (a load
        // takes 1 to 1.4 us here, the MFMAs of a slab 0.05 to 0.3; past the last slab, that one again).
        const int pt = threadIdx.x - NC;
        const int q = (pt & 15) * 4, rr = pt >> 4;
        using S = Slot<PRO, IN_H, BN, MAXH>;
        constexpr int NS = kNwSlots<PRO, IN_H, BN, MAXH>;
        S slot[NS];
        const int last = nsl - 1;
#pragma unroll
        for (int i = 0; i < NS; i++) slot[i].load(p, u, min(i, last) * kCK, tw, q, rr);
        auto stage = [&](int i, int g) {
            slot[i].convert(p, xs + (g & 1) * slab_elems, u, g * kCK, tw, q, rr);
            slot[i].load(p, u, min(g + NS, last) * kCK, tw, q, rr);
            __syncthreads();
        };
        // whole rounds of the slots, then the rest (a break inside a round would make the wait counts
        // assume it)
        int g = 0;
        for (; g + NS <= nsl; g += NS) {
#pragma unroll
            for (int i = 0; i < NS; i++) stage(i, g + i);
        }
#pragma unroll
        for (int i = 0; i < NS - 1; i++)
            if (g + i < nsl) stage(i, g + i);
        __syncthreads();  // the consumers' last slab
    } else {
        // ------------------------------------------------------------ consumer waves
        // wave (wm, wn) of WM x 2: rows m0 + 32 wm .. + 31, columns 32 NJ wn .. of the unit (NJ MFMA
        // tiles); lane layouts as in kk_conv.hip
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        const int wm = wave % WM, wn = wave / WM;
        const int l32 = lane & 31, lh = lane >> 5;
        const int taps = nsl * p.k;
        // The ring's load iterator: the uniform byte offset of tap lk's fragments (past the last tap,
        // the last one again: the number of loads in flight is static) and the lane's four offsets
        // from it, through a buffer resource (no address arithmetic per load).
        const uint32_t c16 = (uint32_t)p.m_pad * 32u;  // bytes of one 16-channel group of A
        const uint32_t step_k = (uint32_t)(p.cin_pad / 16) * c16;
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)p.w, 0, (int)(step_k * (uint32_t)p.k), kBufFormat);
        uint32_t a_off[4];
#pragma unroll
        for (int kc = 0; kc < 4; kc++)
            a_off[kc] = ((uint32_t)(u.m0 + wm * 32 + l32) * 2u + (uint32_t)lh) * 16u + (uint32_t)kc * c16;
        uint32_t a_pos = 0;
        const uint32_t a_last = (uint32_t)(p.k - 1) * step_k + (uint32_t)(nsl - 1) * 4u * c16;
        int lk = 0, left = taps;
        auto load_a = [&](bf16x8& dst, int kc) {
            typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
            const u32x4_t t = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)a_off[kc], (int)a_pos, 0);
            dst = __builtin_bit_cast(bf16x8, t);
        };
        auto next_a = [&]() {
            lk++, left--, a_pos += step_k;
            const bool wrap = lk == p.k;  // the next slab's first tap
            a_pos = wrap ? a_pos + 4u * c16 - (uint32_t)p.k * step_k : a_pos;
            lk = wrap ? 0 : lk;
            a_pos = left > 0 ? a_pos : a_last;
        };
        // B fragments of a whole tap: 16-channel step kc, columns 32 NJ wn + 32 j + l32 of the unit
        const int boff = (wn * 32 * NJ + l32) * kRS + lh * 8;
        auto read_b = [&](bf16x8 (&dst)[4][NJ], const uint16_t* buf) {
            const uint16_t* bp = buf + boff;
#pragma unroll
            for (int kc = 0; kc < 4; kc++)
#pragma unroll
                for (int j = 0; j < NJ; j++) dst[kc][j] = *(const bf16x8*)(bp + j * 32 * kRS + kc * 16);
        };
        bf16x8 A[kNwRing][4], B[2][4][NJ];
#pragma unroll
        for (int r = 0; r < kNwRing; r++) {
#pragma unroll
            for (int kc = 0; kc < 4; kc++) load_a(A[r][kc], kc);
            next_a();
            __builtin_amdgcn_sched_barrier(0);  // in the order of their use: the loop's waits count them
        }
        // element 4 g + e of an accumulator is row 8 g + 4 lh + e of the wave's 32, starting at the
        // bias (ConvT: added in the scatter)
        f32x16 acc[NJ];
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float bv = CONVT ? 0.f : row_bias(p.bias, u.m0 + wm * 32 + 8 * g + 4 * lh + e, p.m);
#pragma unroll
                for (int j = 0; j < NJ; j++) acc[j][4 * g + e] = bv;
            }
        __syncthreads();  // slab 0 staged
        read_b(B[0], xs);
        __builtin_amdgcn_sched_barrier(0);
        int kk = 0;
        uint32_t bi = 0, tap_off = 0;  // the slab's buffer, the tap's row offset in it (elements)
        auto tap = [&](auto rc) {
            constexpr int r = decltype(rc)::value;
            // The next tap's B fragments are read under this tap's MFMAs (an LDS read takes ~130 cycles,
            // a step's MFMAs 32 NJ), four steps at a time and on every path, so that the wait counts
            // are static.  At the slab's last tap every read of the slab has completed: the barrier
            // hands its buffer back, and the next slab is there to be read (past the last slab a stale
            // read, in bounds and unused).
            const bool fin = kk + 1 == p.k;
            bf16x8(&bc)[4][NJ] = B[r & 1];
            bf16x8(&bn)[4][NJ] = B[1 - (r & 1)];
            if (fin) __syncthreads();
            bi = fin ? (uint32_t)slab_elems - bi : bi;
            tap_off = fin ? 0u : tap_off + (uint32_t)(p.dil * kRS);
            kk = fin ? 0 : kk + 1;
            __builtin_amdgcn_sched_barrier(0);
            read_b(bn, xs + bi + tap_off);
#pragma unroll
            for (int kc = 0; kc < 4; kc++) {
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[r][kc], bc[kc][j], acc[j], 0, 0, 0);
                load_a(A[r][kc], kc);
            }
            next_a();
            // (MFMA, LDS read) pairs, each step's weight load after its MFMAs: issued before the MFMAs
            // the reads left the matrix core idle for ~130 cycles per tap
#pragma unroll
            for (int kc = 0; kc < 4; kc++) {
#pragma unroll
                for (int j = 0; j < NJ; j++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
                }
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // weight load
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // whole rounds of the ring, then the rest
        for (int n = taps / kNwRing; n > 0; n--) each<kNwRing>(tap);
        each<kNwRing - 1>([&](auto rc) {
            if (decltype(rc)::value < taps % kNwRing) tap(rc);
        });
        // the slabs are consumed (the last barrier): the output tile goes over them
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *(float4*)(T + ((wn * NJ + j) * 32 + l32) * LD + wm * 32 + 8 * g + 4 * lh) =
                    make_float4(acc[j][4 * g], acc[j][4 * g + 1], acc[j][4 * g + 2], acc[j][4 * g + 3]);
    }
    __syncthreads();

    // ---------------------------------------------------------------- epilogue, all the waves
    // thread: rows m .. m + 3 of columns cb + 32 i (CQ lanes cover one column's rows); threads past
    // 32 CQ (BM = 32) have no columns
    const int cq = threadIdx.x % CQ, cb = threadIdx.x / CQ;
    const bool et = 32 * CQ == NT || threadIdx.x < 32 * CQ;
    const int m = u.m0 + 4 * cq;
    const bool mok = m < p.m;
    const float one = vgpr_f(1.0f);
    int lo = 0, hi = u.nv;  // the columns that store
    if (!et) {
    } else if constexpr (CONVT) {
        const int64_t os = ld_const(p.out_start, u.item);
        const int64_t ol = ld_const(p.out_len, u.item) - (EPI == EPI_CONVT_REFLECT ? 1 : 0);
        const int mm = mok ? m : u.m0;
        const int ph = mm / p.cout, co = mm - ph * p.cout;  // the block's 64 rows lie in one phase
        const ConvTCols cc = convt_cols(u.n0, u.nv, p.stride_t, p.pad_t, ph, os, ol, EPI == EPI_CONVT_REFLECT, mok);
        lo = cc.lo, hi = cc.hi;
        EpiBase eb;
        eb.y = OUT_H ? (void*)((uint16_t*)p.y + cc.ubase * p.y_ld) : (void*)(p.y + cc.ubase * p.y_ld);
        eb.ry = __builtin_amdgcn_make_buffer_rsrc(eb.y, 0, kBufRecords, kBufFormat);
        const float4 cbv = *(const float4*)(p.bias + co);
        // residual: r0 at the output row; an invalid column reads the unit's first row
        auto res_at = [&](int64_t row) {
            if constexpr (OUT_H)
                return widen_h4(raw_h4(*(const uint2*)((const uint16_t*)p.r0 + row * p.r0_ld + co)));
            else
                return *(const float4*)(p.r0 + row * p.r0_ld + co);
        };
        float4 r[NI];
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int col = cb + 32 * i;
            const bool ok = col >= lo && col < hi;
            r[i] = res_at(ok ? cc.ubase + cc.rel0 + (int64_t)p.stride_t * col : cc.ubase);
        }
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int col = cb + 32 * i;
            const bool ok = col >= lo && col < hi;
            float4* tp = (float4*)(T + col * LD + 4 * cq);
            const float4 a = *tp;
            const float4 w = make_float4(a.x + cbv.x, a.y + cbv.y, a.z + cbv.z, a.w + cbv.w);
            const float4 o = make_float4(r[i].x + w.x, r[i].y + w.y, r[i].z + w.z, r[i].w + w.w);
            const uint2 pk = OUT_H ? make_uint2(pack_f16x2(o.x, o.y), pack_f16x2(o.z, o.w)) : make_uint2(0u, 0u);
            const uint32_t yo = (uint32_t)(cc.rel0 + p.stride_t * col) * (uint32_t)p.y_ld + (uint32_t)co;
            store4<OUT_H>(eb, yo, ok, o, pk);
            if (EPI == EPI_CONVT_REFLECT && col == cc.refl) {
                // this column (output row os + 1) also fills the item's first row, = ubase here
                const float4 f0 = res_at(os);
                const float4 f = make_float4(w.x + f0.x, w.y + f0.y, w.z + f0.z, w.w + f0.w);
                const uint2 fk = OUT_H ? make_uint2(pack_f16x2(f.x, f.y), pack_f16x2(f.z, f.w)) : make_uint2(0u, 0u);
                store4<OUT_H>(eb, (uint32_t)co, true, f, fk);
            }
            if constexpr (STATS) *tp = o;
        }
    } else {
        EpiBase eb;
        const int64_t n0 = u.n0;
        eb.y = OUT_H ? (void*)((uint16_t*)p.y + n0 * p.y_ld) : (void*)(p.y + n0 * p.y_ld);
        eb.ry = __builtin_amdgcn_make_buffer_rsrc(eb.y, 0, kBufRecords, kBufFormat);
        eb.r0 = eb.r1 = eb.r2 = nullptr;
        if constexpr (EPI == EPI_ADD_FROM) {
            eb.r0 = OUT_H ? (const float*)((const uint16_t*)p.r0 + n0 * p.r0_ld) : p.r0 + n0 * p.r0_ld;
            eb.rr0 = __builtin_amdgcn_make_buffer_rsrc((void*)eb.r0, 0, kBufRecords, kBufFormat);
        }
        if constexpr (EPI == EPI_MEAN3_LEAKY_BF16) {
            eb.rr0 = __builtin_amdgcn_make_buffer_rsrc((void*)((const uint16_t*)p.r0 + n0 * p.r0_ld), 0, kBufRecords,
                                                       kBufFormat);
            eb.rr1 = __builtin_amdgcn_make_buffer_rsrc((void*)((const uint16_t*)p.r1 + n0 * p.r0_ld), 0, kBufRecords,
                                                       kBufFormat);
            eb.rr2 = __builtin_amdgcn_make_buffer_rsrc((void*)((const uint16_t*)p.r2 + n0 * p.r0_ld), 0, kBufRecords,
                                                       kBufFormat);
        }
        const uint32_t yld = (uint32_t)p.y_ld, rld = (uint32_t)p.r0_ld;
        float4 res[NI][NRA];
        if constexpr (NR > 0) {
#pragma unroll
            for (int i = 0; i < NI; i++) {
                // an invalid column or row reads column 0, row m0 of the unit
                const int col = cb + 32 * i;
                const bool ok = col < u.nv && mok;
                const uint32_t mo = ok ? m : u.m0, co = ok ? col : 0;
                load_res<EPI, OUT_H>(p, eb, co * yld + mo, co * rld + mo, n0 + co, (int)mo, res[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int col = cb + 32 * i;
            float* tp = T + col * LD;
            const float4 a = *(const float4*)(tp + 4 * cq);
            uint2 pk = make_uint2(0u, 0u);
            const float4 o = finish4<EPI, OUT_H>(p, a, res[i], pk, one);
            store4<OUT_H>(eb, (uint32_t)col * yld + (uint32_t)m, col < u.nv && mok, o, pk);
            // the stored values back into the tile for the statistics (a column's 16 lanes are in one
            // wave: its f32 values are read before its row is overwritten)
            if constexpr (HSTATS)
                *(uint2*)(tp + 2 * cq) = pk;
            else if constexpr (STATS)
                *(float4*)(tp + 4 * cq) = o;
        }
    }
    if constexpr (STATS) {
        __syncthreads();
        if (threadIdx.x >= 4 * BM) return;
        // one channel and column group per thread: columns cg + 4 k in sequence
        const int lane = threadIdx.x & 63, cl = (threadIdx.x >> 6) * 16 + (lane & 15), cg = lane >> 4;
        float s1 = 0.f, s2 = 0.f, sft;
        if constexpr (HSTATS) {
            const _Float16* th = (const _Float16*)T;
            const _Float16 s = th[cl];
            const f16x2_t sp = {s, s}, one2 = {(_Float16)1.0f, (_Float16)1.0f};
            sft = (float)s;
            _Float16 hv[32];  // all the reads first: one LDS latency, then the chain
#pragma unroll
            for (int k = 0; k < 32; k++) hv[k] = th[(4 * k + cg) * (2 * LD) + cl];
#pragma unroll
            for (int k = 0; k < 32; k += 2) {
                const int c0 = 4 * k + cg, c1 = c0 + 4;
                f16x2_t d = {hv[k], hv[k + 1]};
                d = d - sp;
                const uint32_t keep = (c0 < u.nv ? 0x0000ffffu : 0u) | (c1 < u.nv ? 0xffff0000u : 0u);
                d = __builtin_bit_cast(f16x2_t, __builtin_bit_cast(uint32_t, d) & keep);
                s1 = __builtin_amdgcn_fdot2(d, one2, s1, false);
                s2 = __builtin_amdgcn_fdot2(d, d, s2, false);
            }
        } else {
            sft = T[cl];
            if constexpr (CONVT) {  // the writing columns are the channel's phase's, not this thread's rows'
                const int64_t os = ld_const(p.out_start, u.item);
                const int64_t ol = ld_const(p.out_len, u.item) - (EPI == EPI_CONVT_REFLECT ? 1 : 0);
                const ConvTCols cc = convt_cols(u.n0, u.nv, p.stride_t, p.pad_t, (u.m0 + cl) / p.cout, os, ol,
                                                EPI == EPI_CONVT_REFLECT, u.m0 + cl < p.m);
                lo = cc.lo, hi = cc.hi;
            }
            float tv[32];  // all the reads first
#pragma unroll
            for (int k = 0; k < 32; k++) tv[k] = T[(4 * k + cg) * LD + cl];
#pragma unroll
            for (int k = 0; k < 32; k++) {
                const int c = 4 * k + cg;
                const float d = c >= lo && c < hi ? tv[k] - sft : 0.f;
                s1 += d;
                s2 = __builtin_fmaf(d, d, s2);
            }
        }
        s1 += __shfl_xor(s1, 16, 64);
        s2 += __shfl_xor(s2, 16, 64);
        s1 += __shfl_xor(s1, 32, 64);
        s2 += __shfl_xor(s2, 32, 64);
        const int mc = u.m0 + cl;
        if (cg == 0 && mc < p.m) {
            if constexpr (CONVT) {
                const int ph = mc / p.cout;
                const float nc = (float)max(hi - lo, 0);
                p.part[((int64_t)u.tile * p.stride_t + ph) * p.cout + (mc - ph * p.cout)] =
                    nc > 0.f ? StatPart{s1, s2, sft, nc} : StatPart{0.f, 0.f, 0.f, 0.f};
            } else if (mc < p.cout) {
                p.part[((int64_t)u.tile * wnt + wcol) * p.cout + mc] = StatPart{s1, s2, sft, (float)u.nv};
            }
        }
    }
}

template <int PRO, int EPI, bool STATS, bool IN_H, bool OUT_H>
hipError_t launch_narrow_t(const ConvGroup& g, int64_t blocks, int max_halo, int bn, int bm, hipStream_t s) {
    const size_t smem = std::max(2 * (size_t)(bn + max_halo) * kRS * sizeof(uint16_t), (size_t)bn * (bm + 4) * sizeof(float));
    static_assert(2 * (128 + kMaxHalo) * kRS * sizeof(uint16_t) <= 64 * 1024, "no dynamic LDS attribute needed");
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(4 * bm + kNP), smem, s, g);
        return hipGetLastError();
    };
    auto go_halo = [&](auto bn_c, auto wm_c) {
        constexpr int BN = decltype(bn_c)::value, WM = decltype(wm_c)::value;
        if constexpr (PRO == PRO_ADAIN_SNAKE)  // the other layers' halos are small (narrow_has)
            if (max_halo > kSmallHalo) return go(conv_narrow_kernel<PRO, EPI, STATS, IN_H, OUT_H, kMaxHalo, BN, WM>);
        return go(conv_narrow_kernel<PRO, EPI, STATS, IN_H, OUT_H, kSmallHalo, BN, WM>);
    };
    constexpr std::integral_constant<int, 1> c1{};
    constexpr std::integral_constant<int, 2> c2{};
    constexpr std::integral_constant<int, 64> n64{};
    constexpr std::integral_constant<int, 128> n128{};
    if constexpr (!STATS)
        if (bn == 64) return bm == 32 ? go_halo(n64, c1) : go_halo(n64, c2);
    return bm == 32 ? go_halo(n128, c1) : go_halo(n128, c2);
}

}  // namespace

hipError_t launch_conv_narrow(ConvGroup& g, int pro, int epi, bool stats, bool in_h, bool out_h, hipStream_t s) {
    // The smallest blocks that leave the launch at most one block per CU: 64 columns without
    // statistics, then 32 rows while they fill at most half of the CUs (a block's K loop is bound by
    // its own waves: 32 rows take 0.18 us per tap of 64 channels where 64 rows take 0.21; past 128
    // blocks the second copy of the staging costs as much).
    int64_t units = 0;
    for (int i = 0; i < g.n; i++) units += conv_units64(g.p[i]);
    const int bn = stats || 2 * units > 256 ? 128 : 64;
    const int bm = units * (128 / bn) * 2 <= 128 ? 32 : 64;
    int64_t blocks = 0;
    int max_halo = 0;
    for (int i = 0; i < g.n; i++) {
        const ConvParams& p = g.p[i];
        const bool convt = epi == EPI_CONVT || epi == EPI_CONVT_REFLECT;
        if (p.m_pad % 64 != 0 || p.tile_wn < 1 || (convt && (p.tile_wn != 1 || p.cout % 64 != 0)))
            return hipErrorInvalidValue;
        g.first[i] = (int)blocks;
        blocks += p.tiles.count * p.tile_wn * (128 / bn) * (p.m_pad / bm);
        max_halo = std::max(max_halo, (p.k - 1) * p.dil);
    }
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7fffffff || max_halo > (pro == PRO_ADAIN_SNAKE ? kMaxHalo : kSmallHalo)) return hipErrorInvalidValue;
#define KK_NARROW(P, E, ST, IH, OH)                                              \
    if (pro == P && epi == E && stats == ST && in_h == IH && out_h == OH) \
        return launch_narrow_t<P, E, ST, IH, OH>(g, blocks, max_halo, bn, bm, s);
    KK_NARROW(PRO_ADAIN_SNAKE, EPI_STORE, true, false, true)
    KK_NARROW(PRO_ADAIN_SNAKE, EPI_ACCUM, true, true, false)
    KK_NARROW(PRO_ADAIN_SNAKE, EPI_ACCUM, false, true, false)
    KK_NARROW(PRO_ADAIN_SNAKE, EPI_STORE, true, true, true)
    KK_NARROW(PRO_ADAIN_SNAKE, EPI_ADD_FROM, true, true, true)
    KK_NARROW(PRO_ADAIN_SNAKE, EPI_ACCUM, true, true, true)
    KK_NARROW(PRO_ADAIN_SNAKE, EPI_ACCUM, false, true, true)
    KK_NARROW(PRO_ADAIN_SNAKE, EPI_MEAN3_LEAKY_BF16, false, true, true)
    KK_NARROW(PRO_ADAIN_LEAKY, EPI_STORE, true, false, false)
    KK_NARROW(PRO_ADAIN_LEAKY, EPI_RESID, false, false, false)
    KK_NARROW(PRO_ADAIN_LEAKY, EPI_RESID_UP2, false, false, false)
    KK_NARROW(PRO_F32, EPI_STORE, false, false, false)
    KK_NARROW(PRO_BF16, EPI_STORE, true, false, false)
    KK_NARROW(PRO_F32, EPI_RESID, false, false, false)
    KK_NARROW(PRO_BF16, EPI_RESID, false, false, false)
    KK_NARROW(PRO_F32, EPI_GELU_BF16, false, false, true)
    KK_NARROW(PRO_LEAKY, EPI_CONVT, true, false, true)
    KK_NARROW(PRO_BF16, EPI_CONVT_REFLECT, true, false, true)
#undef KK_NARROW
    return hipErrorInvalidValue;
}

}  // namespace kk
