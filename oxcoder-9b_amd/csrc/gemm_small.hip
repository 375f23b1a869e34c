// Prefill GEMM for a few dozen tokens (gfx950): the exact integers and the fp32 epilogue of gemm_q8k.hip
// with no weight bytes through LDS.
//
// What bounds it.  With at most 64 tokens a weight meets one or two 32-token MFMA tiles, so a call is bound by the
// vector instructions that unpack the weights and scale the sums (~370 per wave, super-block and two tiles, against
// 34 MFMAs), then by reading the weights; which bytes of the activations a wave loads does not matter (a copy that
// always loads the same 2 KB runs as long).  The tile kernels of gemm_q8k.hip (128 tokens x 64 rows, the planes of each
// super-block staged in LDS behind a barrier) multiply four tiles there, most of them padding.  At 9 / 40 tokens:
// 24576x4096 Q4_K 40.0 / 43.5 -> 15.0 / 31.5 us, 4096x12288 Q6_K 22.9 / 27.4 -> 15.6 / 25.5 us, 4096x4096 Q4_K 10.7 /
// 11.8 -> 5.5 / 9.5 us.  From 65 tokens on (two token blocks, each unpacking the weights) the tile kernels are faster:
// at 65 tokens, quantizer included, 47.6 against 52.0 us for two 12288x4096 Q4_K and 34.6 against 46.8 for 4096x12288 Q6_K.
//
// Work split.  A workgroup owns 32 * RW weight rows and up to 64 tokens; RW row waves times SM_KW waves that split the
// super-blocks of its K range.  Each wave loads the raw blocks of its 32 rows, unpacks them in registers straight into
// MFMA operands (lane l holds row l % 32, K half l / 32 of each step) and multiplies them with every token tile, so
// there is no barrier until the end; the row waves read the same activations at the same time, which the L1
// serves.  The K waves' sums meet in LDS and are added in order.  Grids too small for the GPU also split K over
// workgroups, by the rule and into the partial planes of gemm_q8k.hip.  The order of a sum depends on (R, C, M)
// alone, never on RW, so a matrix gives the same bits alone and in a group, with and without the fragment
// copy.
//
// Weights are the MFMA's A operand and tokens its B operand: a lane then holds one token and 16 rows of
// the result, so the activation scale is one register and the rows' d / dmin are read from LDS once
// per super-block for all token tiles.
#include "kq_device.h"
#include "kq_internal.h"

namespace kq {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));

constexpr int SM_ROWS = 32;
constexpr int SM_LD = 36;       // floats per token row of the LDS sums: 16-byte rows, spread over the banks
constexpr int SM_KW = 2;        // waves that split a workgroup's super-blocks
constexpr int SM_CUS = 256;     // CUs of an MI355X (fixed, so a launch's shape does not depend on the device)
constexpr int SM_RW = 4;        // row waves of a workgroup, at most

struct SmOut {
    float* y[3];                // the output, or the matrix's partial planes (one per split, M rows of R floats)
    int64_t ldy[3], plane[3];   // row stride; distance between the planes of two splits
};
#define KQ_SM_PIN()                          \
    do {                                     \
        asm volatile("" ::: "memory");       \
        __builtin_amdgcn_sched_barrier(0);   \
    } while (0)

template <class T> __device__ __forceinline__ T sm_pick(int m, T a, T b, T c) { return m == 0 ? a : m == 1 ? b : c; }
template <class A, class B> __device__ __forceinline__ uint32_t sm_mul(A a, B b) {
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b));
}

// One lane's raw part of a block: row l % 32, the bytes its K half (l / 32) needs.
template <int TYPE> struct SmW;
template <> struct SmW<TYPE_Q4_K> { u32x4 hdr, q[4]; };
template <> struct SmW<TYPE_Q6_K> { u32x4 ql[4], qh[2], sc; uint32_t qle[4], qhe[2], sce, sh; };

// Raw buffer loads: a descriptor over the workgroup's rows (or tokens) in scalar registers, a 32-bit lane offset
// that stays the same for every super-block and a scalar offset, so the loop holds no 64-bit lane addresses
// (strength-reduced ones cost 40 registers and made the two-tile form spill).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sm_rsrc(const uint8_t* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ u32x4 sm_ld16(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)v, (int)s, 0));
}
__device__ __forceinline__ uint32_t sm_ld4(__amdgpu_buffer_rsrc_t r, uint32_t v, uint32_t s) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, (int)v, (int)s, 0);
}

// o: this lane's block in the super-block column; sg: the column.
__device__ __forceinline__ void sm_load(SmW<TYPE_Q4_K>& w, __amdgpu_buffer_rsrc_t r, uint32_t o, uint32_t sg, int half) {
    w.hdr = sm_ld16(r, o, sg);
    const uint32_t oq = o + 16u * half;
#pragma unroll
    for (int p = 0; p < 4; p++) w.q[p] = sm_ld16(r, oq, sg + 16 + 32 * p);
}
// Dword-aligned fields, funnel-shifted by the block's start & 3; the last dword (bytes 208..211 from the
// aligned base) passes the block end by 2 bytes only for blocks starting at 0 (mod 4), never row 7 of a tile.
__device__ __forceinline__ void sm_load(SmW<TYPE_Q6_K>& w, __amdgpu_buffer_rsrc_t r, uint32_t o, uint32_t sg, int half) {
    w.sh = o & 3u;                      // a super-block column starts at a multiple of 16
    const uint32_t ob = o - w.sh, oh = ob + 16u * half;
#pragma unroll
    for (int i = 0; i < 4; i++) {       // ql bytes 64 (i / 2) + 32 (i % 2) + 16 half
        w.ql[i] = sm_ld16(r, oh, sg + 32 * i);
        w.qle[i] = sm_ld4(r, oh, sg + 32 * i + 16);
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        w.qh[i] = sm_ld16(r, oh, sg + 128 + 32 * i);
        w.qhe[i] = sm_ld4(r, oh, sg + 144 + 32 * i);
    }
    w.sc = sm_ld16(r, ob, sg + 192);
    w.sce = sm_ld4(r, ob, sg + 208);
}

__device__ __forceinline__ u32x4 sm_funnel(const u32x4& v, uint32_t e, uint32_t sh) {
    return u32x4{__builtin_amdgcn_alignbyte(v.y, v.x, sh), __builtin_amdgcn_alignbyte(v.z, v.y, sh),
                 __builtin_amdgcn_alignbyte(v.w, v.z, sh), __builtin_amdgcn_alignbyte(e, v.w, sh)};
}

// Operands of one super-block, K step by K step: planes(ks, wh, wl) for ks = 0..7 (32 elements each).
template <int TYPE> struct SmUnpack;
template <> struct SmUnpack<TYPE_Q4_K> {
    static constexpr int SHIFT = 3;     // I1 = 8 (x . H) + (x . L)
    uint32_t a[2], b[2], m[2];          // scale >> 3, scale & 7, min of sub-blocks 0..3 and 4..7, a byte each
    u32x4 q[4];
    float d, dm;
    __device__ __forceinline__ SmUnpack(const SmW<TYPE_Q4_K>& w, int) {
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = w.q[i];
        const uint32_t s0 = w.hdr.y, s1 = w.hdr.z, s2 = w.hdr.w;
        const uint32_t sc[2] = {s0 & 0x3f3f3f3fu, (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u)};
#pragma unroll
        for (int i = 0; i < 2; i++) {
            a[i] = (sc[i] >> 3) & 0x07070707u;
            b[i] = sc[i] & 0x07070707u;
        }
        m[0] = s1 & 0x3f3f3f3fu;
        m[1] = ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u);
        d = f16_lo(w.hdr.x);
        dm = f16_hi(w.hdr.x);
    }
    __device__ __forceinline__ void planes(int ks, v4i& h, v4i& l) const {
        const uint32_t sel = 0x0c000c00u + 0x00010001u * (ks & 3);   // byte ks & 3 in both 16-bit halves
        const uint32_t as = __builtin_amdgcn_perm(0u, a[ks >> 2], sel), bs = __builtin_amdgcn_perm(0u, b[ks >> 2], sel);
        const u32x4 v = q[ks >> 1];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t n = (ks & 1 ? w[i] >> 4 : w[i]) & 0x0f0f0f0fu;
            h[i] = (int)sm_mul(n, as);
            l[i] = (int)sm_mul(n, bs);
        }
    }
    // Min-term operand: half h holds sub-blocks 4h .. 4h+3, f16 [-64 m] then [-m] (0x64mm is 1024 + m exactly)
    __device__ __forceinline__ v8h mins(int half) const {
        const h16x2 off = {(_Float16)1024.0f, (_Float16)1024.0f};
        const h16x2 f64 = {(_Float16)-64.0f, (_Float16)-64.0f}, f1 = {(_Float16)-1.0f, (_Float16)-1.0f};
        const uint32_t mm = half ? m[1] : m[0];
        const h16x2 a = __builtin_bit_cast(h16x2, __builtin_amdgcn_perm(0x64646464u, mm, 0x04010400u)) - off;
        const h16x2 b = __builtin_bit_cast(h16x2, __builtin_amdgcn_perm(0x64646464u, mm, 0x04030402u)) - off;
        return __builtin_bit_cast(v8h, u32x4{__builtin_bit_cast(uint32_t, (h16x2)(a * f64)), __builtin_bit_cast(uint32_t, (h16x2)(b * f64)),
                                             __builtin_bit_cast(uint32_t, (h16x2)(a * f1)), __builtin_bit_cast(uint32_t, (h16x2)(b * f1))});
    }
};
template <> struct SmUnpack<TYPE_Q6_K> {
    static constexpr int SHIFT = 8;     // I = 256 (x . H) + (x . L)
    u32x4 ql[4], qh[2], sc;
    int half;
    float d;
    __device__ __forceinline__ SmUnpack(const SmW<TYPE_Q6_K>& w, int hf) : half(hf) {
#pragma unroll
        for (int i = 0; i < 4; i++) ql[i] = sm_funnel(w.ql[i], w.qle[i], w.sh);
#pragma unroll
        for (int i = 0; i < 2; i++) qh[i] = sm_funnel(w.qh[i], w.qhe[i], w.sh);
        sc = sm_funnel(w.sc, w.sce, w.sh);
        d = f16_lo(w.sce >> (8 * w.sh));
    }
    // step ks = 4h + k: elements 128h + 32k + 16 half + i, scale 8h + 2k + half
    __device__ __forceinline__ void planes(int ks, v4i& h, v4i& l) const {
        const int hh = ks >> 2, k = ks & 3;
        const uint32_t scw = hh ? (k < 2 ? sc.z : sc.w) : (k < 2 ? sc.x : sc.y);
        const int s = (int)(int8_t)(uint8_t)(scw >> (16 * (k & 1) + 8 * half));
        const s16x2 s2 = __builtin_bit_cast(s16x2, (uint32_t)(s & 0xffff) * 0x10001u);
        const s16x2 c2 = __builtin_bit_cast(s16x2, (uint32_t)((128 - 32 * s) & 0xffff) * 0x10001u);
        const u32x4 lv = ql[2 * hh + (k & 1)], hv = qh[hh];
        const uint32_t lw[4] = {lv.x, lv.y, lv.z, lv.w}, hw[4] = {hv.x, hv.y, hv.z, hv.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t lq = (k >> 1 ? lw[i] >> 4 : lw[i]) & 0x0f0f0f0fu;
            const uint32_t hq = (k == 0 ? hw[i] << 4 : k == 1 ? hw[i] << 2 : k == 2 ? hw[i] : hw[i] >> 2) & 0x30303030u;
            const uint32_t q6 = lq | hq;
            const uint32_t e = __builtin_amdgcn_perm(0u, q6, 0x0c020c00u);   // bytes 0, 2 -> 16-bit lanes
            const uint32_t o = __builtin_amdgcn_perm(0u, q6, 0x0c030c01u);   // bytes 1, 3
            const uint32_t ve = __builtin_bit_cast(uint32_t, (s16x2)(__builtin_bit_cast(s16x2, e) * s2 + c2));
            const uint32_t vo = __builtin_bit_cast(uint32_t, (s16x2)(__builtin_bit_cast(s16x2, o) * s2 + c2));
            h[i] = (int)__builtin_amdgcn_perm(vo, ve, 0x07030501u);
            l[i] = (int)(__builtin_amdgcn_perm(vo, ve, 0x06020400u) ^ 0x80808080u);
        }
    }
};

// Min-term operand of one token, from bsums 8h .. 8h+7: B_s = bsum[2s] + bsum[2s+1] of sub-blocks s = 4h .. 4h+3
// as f16 [B_s >> 6] then [B_s & 63] (exact: |B_s| <= 4096).
__device__ __forceinline__ v8h sm_bsums(const u32x4& v) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    int B[4];
#pragma unroll
    for (int i = 0; i < 4; i++) B[i] = (int)(int16_t)(w[i] & 0xffffu) + (int)(int16_t)(w[i] >> 16);
    auto pk = [](int a, int b) { return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz((float)a, (float)b)); };
    return __builtin_bit_cast(v8h, u32x4{pk(B[0] >> 6, B[1] >> 6), pk(B[2] >> 6, B[3] >> 6),
                                         pk(B[0] & 63, B[1] & 63), pk(B[2] & 63, B[3] & 63)});
}

// Leading scalars, preloaded into registers: what the prologue needs of up to three matrices of one type (t12: first
// workgroups of matrices 1 and 2, f1 | f2 << 16; gps: their super-blocks per split, a byte each; GM: G | M << 8); the
// outputs follow.  Workgroup (x: rows, y: token tile, z: split).
template <int TYPE, int MT, bool FRAG>
__global__ void __launch_bounds__(64 * SM_RW * SM_KW)
k_gemm_small(const uint8_t* __restrict__ w0, const uint8_t* __restrict__ w1, const uint8_t* __restrict__ w2,
             const uint8_t* __restrict__ XQ, const uint8_t* __restrict__ XF, int R0, int R1, int R2, uint32_t t12,
             uint32_t GM, uint32_t gps3, SmOut out) {
    constexpr int BS = TYPE == TYPE_Q4_K ? Q4K_BYTES : Q6K_BYTES;
    __shared__ __attribute__((aligned(16))) float part[SM_RW * SM_KW][32 * MT][SM_LD];
    const int lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kw = wave % SM_KW, rw = wave / SM_KW;
    const int rows = blockDim.x / (64 * SM_KW) * 32;
    const int wg = blockIdx.x, m0 = blockIdx.y * (32 * MT);
    const int G = (int)(GM & 0xffu), M = (int)(GM >> 8);
    const int f1 = (int)(t12 & 0xffffu), f2 = (int)(t12 >> 16);
    const int mi = wg >= f1 ? (wg >= f2 ? 2 : 1) : 0;
    const int R = sm_pick(mi, R0, R1, R2);
    const int r0 = (wg - sm_pick(mi, 0, f1, f2)) * rows;      // the workgroup's first row, and this wave's
    const int n0 = r0 + 32 * rw < R ? r0 + 32 * rw : R - 8;
    const uint8_t* const W = sm_pick(mi, w0, w1, w2);

    // the split's super-blocks, then this wave's
    const int gps = (int)(gps3 >> (8 * mi)) & 0xff;
    const int s0 = blockIdx.z * gps, s1 = s0 + gps < G ? s0 + gps : G;
    if (s0 >= G) return;                                      // a matrix of fewer splits than the launch's most
    const int gpw = (s1 - s0 + SM_KW - 1) / SM_KW;
    const int gbeg = s0 + kw * gpw, gend = gbeg + gpw < s1 ? gbeg + gpw : s1;
    const int row = n0 + l32 < R ? n0 + l32 : R - 1;          // rows past R are loaded clamped, not stored
    // a workgroup's rows and tokens are far below 2 GB (at most 32 rows and 64 tokens of 61440 columns)
    const __amdgpu_buffer_rsrc_t wr = sm_rsrc(W + (int64_t)(n0 >> 3) * G * 8 * BS,
                                              (uint32_t)(R - n0 < SM_ROWS ? R - n0 : SM_ROWS) * G * BS);
    const uint32_t wlane = (uint32_t)(((row >> 3) - (n0 >> 3)) * G * 8 + (row & 7)) * BS;
    const uint32_t xrow = (uint32_t)G * Q8K_BYTES;
    const int mrows = M - m0 < 32 * MT ? M - m0 : 32 * MT;
    const __amdgpu_buffer_rsrc_t xr = sm_rsrc(XQ + (int64_t)m0 * xrow, (uint32_t)mrows * xrow);
    const __amdgpu_buffer_rsrc_t fr = sm_rsrc(FRAG ? XF + (int64_t)(m0 / 32) * G * 8192 : XQ, FRAG ? (uint32_t)MT * G * 8192 : 0u);
    uint32_t xlane[MT];             // this lane's token of each tile (tokens past M clamped)
#pragma unroll
    for (int t = 0; t < MT; t++) xlane[t] = (uint32_t)(32 * t + l32 < mrows ? 32 * t + l32 : mrows - 1) * xrow;
    uint32_t flane[MT];             // past the descriptor for tokens past M: zeros, and no bytes loaded
#pragma unroll
    for (int t = 0; t < MT; t++) flane[t] = 32 * t + l32 < mrows ? (uint32_t)lane * 16u : 0x7fff0000u;
    // MFMA operand of token tile t, step ks of super-block g
    auto load_a = [&](int t, int g, int ks) {
        if constexpr (FRAG)
            return __builtin_bit_cast(v4i, sm_ld16(fr, flane[t], (uint32_t)(t * G + g) * 8192u + 1024u * ks));
        else
            return __builtin_bit_cast(v4i, sm_ld16(xr, xlane[t] + 4u + 32u * ks + 16u * half, (uint32_t)g * Q8K_BYTES));
    };

    float y[MT][16];
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int a = 0; a < 16; a++) y[t][a] = 0.0f;

    if (gbeg < gend) {
        SmW<TYPE> raw;
        v4i xv[MT][8];
        u32x4 bs[MT];
        float dx[MT];
        auto load_x = [&](int t, int g) {
            const uint32_t sx = (uint32_t)g * Q8K_BYTES;
            dx[t] = __builtin_bit_cast(float, sm_ld4(xr, xlane[t], sx));
            if constexpr (TYPE == TYPE_Q4_K) bs[t] = sm_ld16(xr, xlane[t] + 16u * half, sx + 260u);
        };
        sm_load(raw, wr, wlane, (uint32_t)gbeg * (8 * BS), half);
#pragma unroll
        for (int t = 0; t < MT; t++) {
#pragma unroll
            for (int ks = 0; ks < 8; ks++)
                xv[t][ks] = load_a(t, gbeg, ks);
            load_x(t, gbeg);
        }
        float* const sd = &part[wave][0][0];    // this wave's d and dmin of the 32 rows, until its sums go there
        for (int g = gbeg; g < gend; g++) {
            const int gn = g + 1 < gend ? g + 1 : gend - 1;
            SmUnpack<TYPE> up(raw, half);
            v8h am[MT];
            float dxg[MT];
#pragma unroll
            for (int t = 0; t < MT; t++) {
                dxg[t] = dx[t];
                if constexpr (TYPE == TYPE_Q4_K) am[t] = sm_bsums(bs[t]);
            }
            sd[l32] = up.d;
            if constexpr (TYPE == TYPE_Q4_K) sd[32 + l32] = up.dm;
            // The next super-block's loads are issued here and after each operand's last use.  The empty
            // instructions keep them and the MFMAs where they are written: left alone, the compiler sinks the
            // loads to the end of the step and the L plane's MFMAs behind the H plane's (holding every plane).
            KQ_SM_PIN();
            sm_load(raw, wr, wlane, (uint32_t)gn * (8 * BS), half);
#pragma unroll
            for (int t = 0; t < MT; t++) load_x(t, gn);
            KQ_SM_PIN();
            // Step ks's MFMAs are dealt among the unpack of step ks + 1: a wave's MFMAs issued back to back
            // block its VALU work until the last one starts
            v16i ah[MT], al[MT];
            v4i h, l;
            up.planes(0, h, l);
#pragma unroll
            for (int ks = 0; ks < 8; ks++) {
                v4i hn = h, ln = l;
                if (ks < 7) up.planes(ks + 1, hn, ln);
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    ah[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(h, xv[t][ks], ks ? ah[t] : v16i{}, 0, 0, 0);
                    al[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(l, xv[t][ks], ks ? al[t] : v16i{}, 0, 0, 0);
                    xv[t][ks] = load_a(t, gn, ks);
                }
                constexpr int VALU = (TYPE == TYPE_Q4_K ? 18 : 46) / (2 * MT);
#pragma unroll
                for (int i = 0; i < 2 * MT; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // one MFMA
                    __builtin_amdgcn_sched_group_barrier(0x002, VALU, 0);   // its share of the VALU work
                }
#pragma unroll
                for (int t = 0; t < MT; t++) asm volatile("" : "+v"(ah[t]), "+v"(al[t]));
                asm volatile("" : "+v"(hn), "+v"(ln));
                KQ_SM_PIN();
                h = hn;
                l = ln;
            }
            v8h wmin;
            if constexpr (TYPE == TYPE_Q4_K) wmin = up.mins(half);
            v16f cm[MT];
            if constexpr (TYPE == TYPE_Q4_K)
#pragma unroll
                for (int t = 0; t < MT; t++) cm[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wmin, am[t], v16f{}, 0, 0, 0);   // -I2
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f32x4 dv = *reinterpret_cast<const f32x4*>(sd + 8 * q + 4 * half);
                f32x4 dmv = dv;
                if constexpr (TYPE == TYPE_Q4_K) dmv = *reinterpret_cast<const f32x4*>(sd + 32 + 8 * q + 4 * half);
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const int a = 4 * q + j;
                        const float f = __fmul_rn(dv[j], (float)((ah[t][a] << SmUnpack<TYPE>::SHIFT) + al[t][a]));
                        const float v = TYPE == TYPE_Q4_K ? __builtin_fmaf(dmv[j], cm[t][a], f) : f;
                        y[t][a] = __builtin_fmaf(dxg[t], v, y[t][a]);
                    }
                if constexpr (MT == 2) KQ_SM_PIN();     // one quarter's scales in registers at a time
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }

    // rows 8q + 4 half + i of token l32, then the waves' sums added in wave order
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int q = 0; q < 4; q++)
            *reinterpret_cast<f32x4*>(&part[wave][32 * t + l32][8 * q + 4 * half]) =
                f32x4{y[t][4 * q], y[t][4 * q + 1], y[t][4 * q + 2], y[t][4 * q + 3]};
    __syncthreads();
    float* const Y = sm_pick(mi, out.y[0], out.y[1], out.y[2]) + blockIdx.z * sm_pick(mi, out.plane[0], out.plane[1], out.plane[2]);
    const int64_t ldy = sm_pick(mi, out.ldy[0], out.ldy[1], out.ldy[2]);
    const int quads = rows / 4;     // consecutive threads store consecutive rows of a token
    for (int i = threadIdx.x; i < 32 * MT * quads; i += blockDim.x) {
        const int tok = i / quads, r = (i - tok * quads) * 4;
        const int pw = (r >> 5) * SM_KW;
        f32x4 s = *reinterpret_cast<const f32x4*>(&part[pw][tok][r & 31]);
#pragma unroll
        for (int w = 1; w < SM_KW; w++) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(&part[pw + w][tok][r & 31]);
            s = f32x4{__fadd_rn(s.x, v.x), __fadd_rn(s.y, v.y), __fadd_rn(s.z, v.z), __fadd_rn(s.w, v.w)};
        }
        if (m0 + tok < M && r0 + r < R) *reinterpret_cast<f32x4_a4*>(Y + (int64_t)(m0 + tok) * ldy + r0 + r) = s;
    }
}

// Workgroup numbers of a launch travel as 16-bit fields.
constexpr int64_t SM_WGS_MAX = 0xffff;

static int64_t sm_wgs(int R, int rw) { return (R + 32 * rw - 1) / (32 * rw); }

bool gemm_small_fits(int R, int M) { return M <= GEMM_SMALL_MAX && sm_wgs(R, 1) < SM_WGS_MAX; }

void launch_gemm_small_group(int n, const uint8_t* const* w, const int* R, int C, int type, const uint8_t* xq,
                             const uint8_t* xf, int M, float* const* y, const int64_t* ldy, float* const* part,
                             const int* gps, hipStream_t s) {
    int64_t total = 0;
    for (int i = 0; i < n; i++) total += sm_wgs(R[i], 1);
    if (n > 1 && total >= SM_WGS_MAX) {
        for (int i = 0; i < n; i++)
            launch_gemm_small_group(1, w + i, R + i, C, type, xq, xf, M, y + i, ldy + i, part + i, gps + i, s);
        return;
    }
    const int G = C / QK;
    // Row waves per workgroup: the number with the fewest bytes per super-block in the busiest CU, where each of the
    // CU's workgroups loads its rows' blocks and the tokens once (24576x4096 Q4_K: 3, one workgroup on each of 256 CUs,
    // 31.5 us at 40 tokens; 1 row wave and 4 K waves 31.2, 4096x12288 Q6_K 25.5 against 28.9 us).
    int rw = 1;
    int64_t best = INT64_MAX;
    for (int c = 1; c <= SM_RW; c++) {
        int64_t wgs = 0;
        for (int i = 0; i < n; i++) wgs += sm_wgs(R[i], c) * ((G + gps[i] - 1) / gps[i]);
        const int64_t cost = (wgs + SM_CUS - 1) / SM_CUS * (32 * c * block_bytes(type) + M * QK);
        if (cost < best) {
            best = cost;
            rw = c;
        }
    }
    SmOut out{};
    const uint8_t* wp[3] = {w[0], w[0], w[0]};
    int Rp[3] = {R[0], R[0], R[0]}, first[3] = {0, 0xffff, 0xffff}, wgs = 0, splits = 1;
    uint32_t gps3 = 0;
    for (int i = 0; i < n; i++) {
        wp[i] = w[i];
        Rp[i] = R[i];
        out.y[i] = part[i] ? part[i] : y[i];
        out.ldy[i] = part[i] ? R[i] : ldy[i];
        out.plane[i] = (int64_t)M * R[i];
        first[i] = wgs;
        wgs += (int)sm_wgs(R[i], rw);
        gps3 |= (uint32_t)gps[i] << (8 * i);
        const int S = (G + gps[i] - 1) / gps[i];
        splits = S > splits ? S : splits;
    }
    const uint32_t t12 = (uint32_t)first[1] | (uint32_t)first[2] << 16, GM = (uint32_t)G | (uint32_t)M << 8;
    const int mt = xf && M > 32 ? 2 : 1;
    const dim3 grid(wgs, (M + 32 * mt - 1) / (32 * mt), splits), block(64 * SM_KW * rw);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, s, wp[0], wp[1], wp[2], xq, xf, Rp[0], Rp[1], Rp[2], t12, GM, gps3, out);
    };
    if (type == TYPE_Q4_K) {
        if (!xf) go(k_gemm_small<TYPE_Q4_K, 1, false>);
        else if (mt == 2) go(k_gemm_small<TYPE_Q4_K, 2, true>);
        else go(k_gemm_small<TYPE_Q4_K, 1, true>);
    } else {
        if (!xf) go(k_gemm_small<TYPE_Q6_K, 1, false>);
        else if (mt == 2) go(k_gemm_small<TYPE_Q6_K, 2, true>);
        else go(k_gemm_small<TYPE_Q6_K, 1, true>);
    }
}

}  // namespace kq
