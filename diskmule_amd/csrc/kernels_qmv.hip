// kernels_qmv.hip -- fp16-MFMA quantized matvec for gfx950 (decode, the
// batches of up to 16 tokens the int8 kernels do not take).
//
// y[b][r] = sum_c W[r][c] * x[b][c] for Q4_K / Q6_K rows (src/cpu.rs:345-399
// semantics, fp32 accumulation).
//
// Operands of v_mfma_f32_16x16x32_f16, all exact:
//  * B (weights): 16 rows x 32 columns per step.  A Q4_K weight enters as the
//    fp16 integer sc*q (0..945), built from the packed bits with the
//    "1024 + q" exponent trick and one packed fp16 FMA (exact: the result is
//    representable and the FMA rounds once).  Q6_K's sc*(q-32) needs up to 13
//    bits: the scale is split into 8*sh + sl and sh*(q-32) and sl*(q-32),
//    both exact, go to an MFMA each.  The super-block scale d (and dmin)
//    multiply the fp32 block result afterwards.
//  * A (activations): 16 rows = 8 tokens x {hi, lo}.  Each 256-value block of
//    a token is scaled by a power of two so |x| < 2^15, then x = hi + lo with
//    hi, lo fp16 (22 significant bits).  Products are exact; MFMA accumulates
//    in fp32, and the block's result is multiplied back by 2^e.
//  * Q4_K's "- dmin * m * x" term is a ninth MFMA step per block whose B
//    column carries 64*m and whose A row carries the sub-block sums of x
//    (scaled by 2^-6, hi/lo), accumulated separately and scaled by dmin.
//
// Lanes: n = lane & 15 is the weight row within a 16-row tile (B column)
// and the A row; kg = lane >> 4 picks which quarter of each 32-column step
// the lane supplies.  C[m][n] sits in lane n + 16*(m/4), element m%4, so
// lane (n, g4) accumulates tokens 2*g4 and 2*g4+1 of row n.
//
// Data movement: see qmv_kernel.
#include "dm_device.h"
#include "dm_plan.h"
#include "dm_qmv.h"

namespace dm {

namespace {

constexpr uint32_t kBias16 = 0x64006400u;    // fp16 pair (1024, 1024)
constexpr uint32_t kBiasBytes = 0x64646464u;  // source of the 0x64 high bytes

__device__ __forceinline__ half2_t as_h2(uint32_t u) { return __builtin_bit_cast(half2_t, u); }
__device__ __forceinline__ uint32_t as_u(half2_t h) { return __builtin_bit_cast(uint32_t, h); }

__device__ __forceinline__ half2_t h2_fma(half2_t a, half2_t b, half2_t c) {
    return __builtin_elementwise_fma(a, b, c);
}

// (v, v) as fp16 from a small integer (exact: |v| < 2048).
__device__ __forceinline__ half2_t h2_int(int v) {
    const _Float16 h = (_Float16)(short)v;
    half2_t r;
    r[0] = h;
    r[1] = h;
    return r;
}

__device__ __forceinline__ half2_t h2_splat(float v) {
    half2_t h;
    h[0] = (_Float16)v;
    h[1] = (_Float16)v;
    return h;
}

__device__ __forceinline__ float f16_lo(uint32_t bits) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)(bits & 0xffffu));
}

__device__ __forceinline__ floatx4 mfma(half8 a, half8 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ half8 frag(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    u32x4 v = {a, b, c, d};
    return __builtin_bit_cast(half8, v);
}

// Power-of-two exponent e with max|x| * 2^-e in [2^14, 2^15) (0 for an
// all-zero or non-finite block, whose result is then non-finite anyway).
__device__ __forceinline__ int block_exponent(float mx) {
    int e = 0;
    if (mx > 0.0f && __builtin_isfinite(mx)) {
        int ex;
        (void)frexpf(mx, &ex);  // mx = f * 2^ex, f in [0.5, 1)
        e = ex - 15;
        if (e < -126) e = -126;
        if (e > 127) e = 127;
    }
    return e;
}

// How a wave holds one block of 8 tokens' activations as loaded: value j of
// load (u, r) (token group u of 4, round r) of lane 16 i + 4 kg + c is column
// round_column(kg, r) + 4 c + j of token 4 u + i, so a load reads runs of 64
// bytes.  (One 16-byte piece per lane in fragment order reads 64 lines with
// one load: 16 waves of them took 3 us of a 6.4 us kernel.)  The quad (r, c)
// of lane group kg belongs to step quad_step(r, c), half quad_half(r, c) of
// the lane's 8 values.
template <uint32_t TYPE>
__device__ __forceinline__ constexpr uint32_t round_bytes() { return TYPE == kQ4_K ? 64 : 128; }  // between rounds
template <uint32_t TYPE>
__device__ __forceinline__ uint32_t round_column(uint32_t kg) {  // of round 0
    return TYPE == kQ4_K ? 64 * kg : 128 * (kg >> 1) + 16 * (kg & 1u);
}
template <uint32_t TYPE> constexpr uint32_t quad_step(uint32_t r, uint32_t c) {
    return TYPE == kQ4_K ? 4 * (r & 1u) + c : 2 * r + (c >> 1);
}
template <uint32_t TYPE> constexpr uint32_t quad_half(uint32_t r, uint32_t c) {
    return TYPE == kQ4_K ? r >> 1 : c & 1u;
}

typedef float floatx2 __attribute__((ext_vector_type(2)));

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}
// DPP controls.  (After the exchanges by 1 and 2 the mirrors of 8 and 16
// lanes act as exchanges by 4 and 8.)
constexpr int kXor1 = 0xb1, kXor2 = 0x4e, kHalfMirror = 0x141, kMirror = 0x140;

__device__ __forceinline__ float row_max(float v) {  // over rows of 16 lanes
    v = fmaxf(v, dpp<kXor1>(v));
    v = fmaxf(v, dpp<kXor2>(v));
    v = fmaxf(v, dpp<kHalfMirror>(v));
    return fmaxf(v, dpp<kMirror>(v));
}
__device__ __forceinline__ float quad_sum(float v) {  // over groups of 4 lanes
    v += dpp<kXor1>(v);
    return v + dpp<kXor2>(v);
}
__device__ __forceinline__ float row_sum(float v) {
    v = quad_sum(v);
    v += dpp<kHalfMirror>(v);
    return v + dpp<kMirror>(v);
}

// (v0, v1) as fp16 hi + lo: 22 significant bits.
__device__ __forceinline__ void split_pair(float v0, float v1, uint32_t &hi, uint32_t &lo) {
    const half2_t h = __builtin_convertvector(floatx2{v0, v1}, half2_t);
    const half2_t l = __builtin_convertvector(floatx2{v0 - (float)h[0], v1 - (float)h[1]}, half2_t);
    hi = as_u(h);
    lo = as_u(l);
}

}  // namespace

// ---------------------------------------------------------------------------
// Raw bytes of one block of one row as a lane holds them, and the block's
// contribution to the lane's accumulators.
// ---------------------------------------------------------------------------
template <uint32_t TYPE> struct Raw;
template <> struct Raw<kQ4_K> {
    u32x4 hdr, q0, q1;  // d|dmin|scales, then qs bytes [32kg, 32kg+32)
};
template <> struct Raw<kQ6_K> {
    u32x4 a1, a2, a3;                  // aligned dwords under ql/ql+32/qh
    u32x2 a4;                          // and under the lane's half of the scales
    uint32_t e1, e2, e3, e4, e4b, e5;  // the dword after each (for the byte shift); e4, e4b hold d
    uint32_t s;                    // block start mod 4
};

// (a & mask) | b: one instruction when mask and b are in registers, as the
// callers arrange (as literals they would make it two).
__device__ __forceinline__ uint32_t and_or(uint32_t a, uint32_t mask, uint32_t b) { return (a & mask) | b; }

// The block's contribution to acc[g][j] (tokens 8 g + 2 kg + j), up[g][j] the
// 2^e of the tokens' scaled activations.
template <int NT>
__device__ __forceinline__ void block_dot(const Raw<kQ4_K> &raw, const half8 (&a)[8][NT],
                                          const uint32_t (&amin)[NT], uint32_t kg, const float (&up)[NT][2],
                                          float (&acc)[NT][2]) {
    const u32x4 hdr = raw.hdr;
    const float dscale = f16_lo(hdr[0]);
    const float mscale = f16_lo(hdr[0] >> 16);
    // (scale, min) bytes of sub-blocks 2kg and 2kg+1 (src/cpu.rs:607-616): for
    // sub-block j < 4 the low 6 bits of scales[j], scales[j+4]; for j >= 4
    // nibbles of scales[j+4] with the top bits of scales[j-4], scales[j].
    const uint32_t sh16 = 16 * (kg & 1u);
    const uint32_t m_low = kg < 2 ? 0x3f3fu : 0u, m_nib = kg < 2 ? 0u : 0x0f0fu, m_top = kg < 2 ? 0u : 0x3030u;
    const uint32_t b1 = hdr[1] >> sh16, b2 = hdr[2] >> sh16, b3 = hdr[3] >> sh16;
    const uint32_t sc = and_or(b1 >> 2, m_top, and_or(b3, m_nib, b1 & m_low));
    const uint32_t mn = and_or(b2 >> 2, m_top, and_or(b3 >> 4, m_nib, b2 & m_low));
    // bytes as fp16: 1024 + byte under the exponent of 1024, less 1024
    const half2_t minus = h2_splat(-1024.0f);
    const half2_t sl = as_h2(__builtin_amdgcn_perm(kBiasBytes, sc, 0x04000400u)) + minus;
    const half2_t shi = as_h2(__builtin_amdgcn_perm(kBiasBytes, sc, 0x04010401u)) + minus;
    const half2_t bl = sl * minus;
    const half2_t sh = shi * h2_splat(0.0625f);
    const half2_t bh = shi * h2_splat(-64.0f);
    uint32_t bias = kBias16, mask_lo = 0x000f000fu, mask_hi = 0x00f000f0u;
    asm("" : "+v"(bias));
    asm("" : "+s"(mask_lo), "+s"(mask_hi));
    floatx4 cm[NT];
#pragma unroll
    for (int g = 0; g < NT; g++) cm[g] = floatx4{0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const uint32_t d = t < 4 ? raw.q0[t] : raw.q1[t - 4];
        const uint32_t d8 = d >> 8;
        const uint32_t p0 = as_u(h2_fma(as_h2(and_or(d, mask_lo, bias)), sl, bl));
        const uint32_t p1 = as_u(h2_fma(as_h2(and_or(d8, mask_lo, bias)), sl, bl));
        const uint32_t p2 = as_u(h2_fma(as_h2(and_or(d, mask_hi, bias)), sh, bh));
        const uint32_t p3 = as_u(h2_fma(as_h2(and_or(d8, mask_hi, bias)), sh, bh));
        const half8 b = frag(p0, p1, p2, p3);
#pragma unroll
        for (int g = 0; g < NT; g++) cm[g] = mfma(a[t][g], b, cm[g]);
    }
    // min step: B = (64 m_lo, 64 m_hi, 0...), A = sub-block sums * 2^-6.
    const half2_t m64 = (as_h2(__builtin_amdgcn_perm(kBiasBytes, mn, 0x04010400u)) + minus) * h2_splat(64.0f);
    const half8 bmin = frag(as_u(m64), 0u, 0u, 0u);
#pragma unroll
    for (int g = 0; g < NT; g++) {
        const floatx4 cmin = mfma(frag(amin[g], 0u, 0u, 0u), bmin, floatx4{0, 0, 0, 0});
#pragma unroll
        for (int j = 0; j < 2; j++) {
            float v = dscale * (cm[g][2 * j] + cm[g][2 * j + 1]);
            v = __builtin_fmaf(-mscale, cmin[2 * j] + cmin[2 * j + 1], v);
            acc[g][j] = __builtin_fmaf(up[g][j], v, acc[g][j]);
        }
    }
}

template <int NT>
__device__ __forceinline__ void block_dot(const Raw<kQ6_K> &raw, const half8 (&a)[8][NT],
                                          const uint32_t (&amin)[NT], uint32_t kg, const float (&up)[NT][2],
                                          float (&acc)[NT][2]) {
    const uint32_t s = raw.s;
    uint32_t L1[4], L2[4], H[4], T[5];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        L1[i] = funnel(raw.a1[i], i < 3 ? raw.a1[i + 1] : raw.e1, s);
        L2[i] = funnel(raw.a2[i], i < 3 ? raw.a2[i + 1] : raw.e2, s);
        H[i] = funnel(raw.a3[i], i < 3 ? raw.a3[i + 1] : raw.e3, s);
    }
    const float dscale = f16_lo(funnel(raw.e4, raw.e4b, s));
    // int8 scales sc[8h + 2k + c], k = 0..3: bytes c and c+2 of scale words
    // 2h (k = 0, 1) and 2h+1 (k = 2, 3).  sc = 8 sh + sl, sl in 0..7.
    const uint32_t c = kg & 1u;
    const uint32_t w01 = funnel(raw.a4[0], raw.a4[1], s) >> (8 * c), w23 = funnel(raw.a4[1], raw.e5, s) >> (8 * c);
    floatx4 ch[NT], cl[NT];
#pragma unroll
    for (int g = 0; g < NT; g++) ch[g] = cl[g] = floatx4{0, 0, 0, 0};
    const half2_t off = h2_splat(-1056.0f);
    uint32_t nib = 0x0f0f0f0fu, top = 0x30303030u, bytes = kBiasBytes;
    asm("" : "+s"(nib), "+s"(top));
    asm("" : "+v"(bytes));
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int sck = (int)(int8_t)((k < 2 ? w01 : w23) >> (16 * (k & 1)));
        const half2_t f_hi = h2_int(sck >> 3), f_lo = h2_int(sck & 7);
        const half2_t o_hi = f_hi * off, o_lo = f_lo * off;
#pragma unroll
        for (int t = 2 * k; t < 2 * k + 2; t++) {
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int half_dw = 0; half_dw < 2; half_dw++) {
                const int dw = 2 * (t & 1) + half_dw;
                const uint32_t src = (k & 1) ? L2[dw] : L1[dw];
                // bits 2k..2k+1 of each qh byte moved to bits 4..5
                const uint32_t hsh = k == 0 ? H[dw] << 4 : (k == 1 ? H[dw] << 2 : (k == 2 ? H[dw] : H[dw] >> 2));
                const uint32_t q4 = and_or((k & 2) ? (src >> 4) : src, nib, hsh & top);  // four 6-bit q
                // fp16 pairs (1024 + q) of bytes (0, 2) and (1, 3)
                const half2_t p0 = as_h2(__builtin_amdgcn_perm(q4, bytes, 0x00060004u));
                const half2_t p1 = as_h2(__builtin_amdgcn_perm(q4, bytes, 0x00070005u));
                hi[2 * half_dw] = as_u(h2_fma(p0, f_hi, o_hi));
                hi[2 * half_dw + 1] = as_u(h2_fma(p1, f_hi, o_hi));
                lo[2 * half_dw] = as_u(h2_fma(p0, f_lo, o_lo));
                lo[2 * half_dw + 1] = as_u(h2_fma(p1, f_lo, o_lo));
            }
            const half8 b_hi = frag(hi[0], hi[1], hi[2], hi[3]), b_lo = frag(lo[0], lo[1], lo[2], lo[3]);
#pragma unroll
            for (int g = 0; g < NT; g++) {
                ch[g] = mfma(a[t][g], b_hi, ch[g]);
                cl[g] = mfma(a[t][g], b_lo, cl[g]);
            }
        }
    }
#pragma unroll
    for (int g = 0; g < NT; g++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float v = __builtin_fmaf(8.0f, ch[g][2 * j] + ch[g][2 * j + 1], cl[g][2 * j] + cl[g][2 * j + 1]);
            acc[g][j] = __builtin_fmaf(up[g][j], dscale * v, acc[g][j]);
        }
}

// ---------------------------------------------------------------------------
// Weight staging.  A wave fetches one block of each row of a 16-row tile as
// whole 16-byte chunks (row r of the tile: `chunks` chunks from the dword at
// or below the block; Q4_K blocks start 16-aligned), consecutive lanes on
// consecutive chunks of a row; each lane then takes its operand pieces from
// there.
// ---------------------------------------------------------------------------
typedef uint32_t v4u __attribute__((ext_vector_type(4)));  // 16-byte aligned (LDS)

// One block of each row of a tile, straight from memory to the wave's LDS
// ring: `loads` buffer loads of 64 (the last: the remaining) lanes whose
// 16-byte results go to consecutive places from m0 on.  Written as
// instructions: as builtins the compiler would make every LDS read wait for
// all of them.  The caller counts them (s_waitcnt vmcnt).  All 64 lanes of
// the wave are active.
#define DM_SLOT4(m, o0, o1, o2, rs)                                                                          \
    "s_mov_b32 m0, " m "\n\ts_nop 0\n\tbuffer_load_dwordx4 " o0 ", " rs ", 0 offen lds\n\t"                    \
    "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 " o1 ", " rs ", 0 offen lds\n\t"              \
    "s_add_u32 m0, m0, 0x400\n\ts_mov_b64 exec, 0xffff\n\tbuffer_load_dwordx4 " o2 ", " rs ", 0 offen lds\n\t" \
    "s_mov_b64 exec, -1\n\t"
#define DM_SLOT6(m, o0, o1, o2, o3, rs)                                                                      \
    "s_mov_b32 m0, " m "\n\ts_nop 0\n\tbuffer_load_dwordx4 " o0 ", " rs ", 0 offen lds\n\t"                    \
    "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 " o1 ", " rs ", 0 offen lds\n\t"              \
    "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 " o2 ", " rs ", 0 offen lds\n\t"              \
    "s_add_u32 m0, m0, 0x400\n\ts_mov_b32 exec_hi, 0\n\tbuffer_load_dwordx4 " o3 ", " rs ", 0 offen lds\n\t" \
    "s_mov_b64 exec, -1\n\t"

__device__ __forceinline__ void load_slot(uint32_t lds, const uint32_t (&o)[3], v4u rs) {
    asm volatile(DM_SLOT4("%0", "%1", "%2", "%3", "%4")::"s"(lds), "v"(o[0]), "v"(o[1]), "v"(o[2]), "s"(rs)
                 : "memory", "scc");
}
__device__ __forceinline__ void load_slot(uint32_t lds, const uint32_t (&o)[4], v4u rs) {
    asm volatile(DM_SLOT6("%0", "%1", "%2", "%3", "%4", "%5")::"s"(lds), "v"(o[0]), "v"(o[1]), "v"(o[2]),
                 "v"(o[3]), "s"(rs)
                 : "memory", "scc");
}

template <uint32_t TYPE> struct StageQ {
    static constexpr uint32_t bytes = TYPE == kQ4_K ? 144 : 210;  // of one block
    static constexpr uint32_t chunks = TYPE == kQ4_K ? 9 : (210 + 2 + 15) / 16;
    static constexpr uint32_t items = 16 * chunks;        // chunks of one tile
    static constexpr uint32_t loads = (items + 63) / 64;  // 16-byte loads per lane
};

// Lane (n, kg)'s raw bytes of the block at byte `off` of row n's run.
__device__ __forceinline__ void take_raw(const v4u *stage, uint32_t ch, uint32_t n, uint32_t kg, uint32_t off,
                                         Raw<kQ4_K> &raw) {
    const v4u *sr = stage + n * ch + off / 16;
    raw.hdr = __builtin_bit_cast(u32x4, sr[0]);
    raw.q0 = __builtin_bit_cast(u32x4, sr[1 + 2 * kg]);
    raw.q1 = __builtin_bit_cast(u32x4, sr[2 + 2 * kg]);
}

__device__ __forceinline__ void take_raw(const v4u *stage, uint32_t ch, uint32_t n, uint32_t kg, uint32_t off,
                                         Raw<kQ6_K> &raw) {
    // dwords of row n from the one holding the block's first byte
    const uint32_t *sw = (const uint32_t *)(stage + n * ch) + (off >> 2);
    const uint32_t h = kg >> 1, c = kg & 1u;
    const uint32_t o1 = 16 * h + 4 * c, o2 = o1 + 8, o3 = 32 + 8 * h + 4 * c;
    raw.s = off & 3u;
    raw.a1 = u32x4{sw[o1], sw[o1 + 1], sw[o1 + 2], sw[o1 + 3]};
    raw.a2 = u32x4{sw[o2], sw[o2 + 1], sw[o2 + 2], sw[o2 + 3]};
    raw.a3 = u32x4{sw[o3], sw[o3 + 1], sw[o3 + 2], sw[o3 + 3]};
    raw.a4 = u32x2{sw[48 + 2 * h], sw[49 + 2 * h]};
    raw.e5 = sw[50 + 2 * h];
    raw.e1 = sw[o1 + 4];
    raw.e2 = sw[o2 + 4];
    raw.e3 = sw[o3 + 4];
    raw.e4 = sw[52];
    raw.e4b = sw[53];
}

namespace {

// Workgroup barrier ordering LDS only: the waves' weight loads in flight are
// not waited for, as __syncthreads() would.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr uint64_t kMeetEmpty = ~0ull;  // no published pair (two NaNs publish() never writes)

struct QmvArgs {
    const uint8_t *w, *w2;  // w2: the up matrix (MODE 2)
    const float *x;
    float *y;
    uint64_t *meet;  // K-split meeting places, kMeetEmpty between launches
    uint32_t rows, columns, row_bytes, batch;
    uint32_t wave_k;      // waves of a workgroup that split K (1 to 16)
    uint32_t k_parts;     // workgroups that split K (1, 2, 4 or 8)
    uint32_t row_groups;  // workgroups that split the row tiles
    uint32_t phases;      // fragment sets a wave goes through per pass (PHASED)
    int normalize;
    float epsilon;
};

// The routed experts of a MoE layer call (GROUPED): pair i of `pairs` is
// selection i % k of token i / k, expert ids[i]; expert e's matrix is at
// w_of[e] (the up rows at w2_offset bytes from it).  Nothing is done unless
// go[0 .. go_count) are all 1.  Input row of a pair: its token's (k = 0: its
// own); output row: the pair's.
struct QmvExperts {
    const uint64_t *w_of;
    uint64_t w2_offset;
    const uint32_t *ids, *go;
    uint32_t go_count, pairs, k, x_rows;
};
constexpr uint32_t kGroupExperts = 256, kGroupPairs = 128;

// Two tokens' sums of one row as one word; a NaN becomes the canonical one,
// so no published pair equals kMeetEmpty.
__device__ __forceinline__ uint64_t pack_pair(float a, float b) {
    const uint32_t ua = a == a ? __float_as_uint(a) : 0x7fc00000u, ub = b == b ? __float_as_uint(b) : 0x7fc00000u;
    return (uint64_t)ub << 32 | ua;
}

// Tiles of a wave group between two cross-wave sums of all 8 NT tokens, whose
// LDS (red) leaves room for the ring; fewer tokens take less, and then more
// tiles share a sum.
template <int MODE, bool PHASED> constexpr uint32_t pass_tiles() { return (MODE == 2 ? 2 : 4) / (PHASED ? 2 : 1); }
template <int NT, int MODE, uint32_t W, bool PHASED> constexpr uint32_t red_floats() {
    return W * pass_tiles<MODE, PHASED>() * (MODE == 2 ? 2 : 1) * NT * 2 * 64;
}
// Slots of a wave's ring (one being read, the others in flight): what the
// 160 KiB of LDS (GROUPED: of two workgroups) hold, at most 5 or 4 (first_loads).
template <uint32_t TYPE, int NT, int MODE, uint32_t W, bool PHASED, bool GROUPED = false>
constexpr uint32_t ring_depth() {
    constexpr uint32_t fit = ((GROUPED ? 155 * 512 : 156 * 1024) - red_floats<NT, MODE, W, PHASED>() * 4 - (PHASED ? W * 2048 : 0)) /
                             (W * StageQ<TYPE>::items * 16);
    constexpr uint32_t most = TYPE == kQ4_K ? 5 : 4;
    return fit < most ? fit : most;
}

// The prologue's loads, in one block with their wait: the wave's first
// activations (8 loads from the bytes xo0 and xo1 of x on; for XB = 2 also
// those of the next block), then the first SLOTS slots of its ring, then the
// wait for the activations alone.  Offsets and descriptors are per slot.
#define DM_X(a, v, off) "buffer_load_dwordx4 %[" a "], %[" v "], %[xr], 0 offen offset:" off "\n\t"
#define DM_XQ4                                                                                            \
    DM_X("a0", "v0", "0") DM_X("a1", "v0", "64") DM_X("a2", "v0", "128") DM_X("a3", "v0", "192")          \
    DM_X("a4", "v1", "0") DM_X("a5", "v1", "64") DM_X("a6", "v1", "128") DM_X("a7", "v1", "192")
#define DM_XQ6                                                                                            \
    DM_X("a0", "v0", "0") DM_X("a1", "v0", "128") DM_X("a2", "v0", "256") DM_X("a3", "v0", "384")         \
    DM_X("a4", "v1", "0") DM_X("a5", "v1", "128") DM_X("a6", "v1", "256") DM_X("a7", "v1", "384")
#define DM_XQ4B                                                                                           \
    DM_X("b0", "v0", "1024") DM_X("b1", "v0", "1088") DM_X("b2", "v0", "1152") DM_X("b3", "v0", "1216")   \
    DM_X("b4", "v1", "1024") DM_X("b5", "v1", "1088") DM_X("b6", "v1", "1152") DM_X("b7", "v1", "1216")
#define DM_XQ6B                                                                                           \
    DM_X("b0", "v0", "1024") DM_X("b1", "v0", "1152") DM_X("b2", "v0", "1280") DM_X("b3", "v0", "1408")   \
    DM_X("b4", "v1", "1024") DM_X("b5", "v1", "1152") DM_X("b6", "v1", "1280") DM_X("b7", "v1", "1408")
#define DM_OUT(c, q)                                                                              \
    [c##0] "=&v"(x[q][0]), [c##1] "=&v"(x[q][1]), [c##2] "=&v"(x[q][2]), [c##3] "=&v"(x[q][3]),   \
        [c##4] "=&v"(x[q][4]), [c##5] "=&v"(x[q][5]), [c##6] "=&v"(x[q][6]), [c##7] "=&v"(x[q][7])
#define DM_Q4(d) DM_SLOT4("%[l]", "%[o" #d "0]", "%[o" #d "1]", "%[o" #d "2]", "%[r" #d "]")
#define DM_Q6(d) DM_SLOT6("%[l]", "%[o" #d "0]", "%[o" #d "1]", "%[o" #d "2]", "%[o" #d "3]", "%[r" #d "]")
#define DM_NEXT(bytes) "s_add_u32 %[l], %[l], " #bytes "\n\t"
#define DM_IN3(d) [o##d##0] "v"(o[d][0]), [o##d##1] "v"(o[d][1]), [o##d##2] "v"(o[d][2]), [r##d] "s"(rs[d])
#define DM_IN4(d) DM_IN3(d), [o##d##3] "v"(o[d][3])
#define DM_ARGS [xr] "s"(xr), [v0] "v"(xo0), [v1] "v"(xo1)
template <uint32_t TYPE, int XB, uint32_t SLOTS, uint32_t NL>
__device__ __forceinline__ void first_loads(floatx4 (&x)[XB][8], v4u xr, uint32_t xo0, uint32_t xo1, uint32_t lds,
                                            const uint32_t (&o)[SLOTS][NL], const v4u (&rs)[SLOTS]) {
    if constexpr (TYPE == kQ4_K && XB == 1 && SLOTS == 2) {
        asm volatile(DM_XQ4 DM_Q4(0) DM_NEXT(2304) DM_Q4(1) "s_waitcnt vmcnt(6)"
                     : DM_OUT(a, 0), [l] "+&s"(lds)
                     : DM_ARGS, DM_IN3(0), DM_IN3(1)
                     : "memory", "scc");
    } else if constexpr (TYPE == kQ4_K && XB == 1 && SLOTS == 4) {
        asm volatile(DM_XQ4 DM_Q4(0) DM_NEXT(2304) DM_Q4(1) DM_NEXT(2304) DM_Q4(2) DM_NEXT(2304) DM_Q4(3) "s_waitcnt vmcnt(12)"
                     : DM_OUT(a, 0), [l] "+&s"(lds)
                     : DM_ARGS, DM_IN3(0), DM_IN3(1), DM_IN3(2), DM_IN3(3)
                     : "memory", "scc");
    } else if constexpr (TYPE == kQ4_K && XB == 1 && SLOTS == 3) {
        asm volatile(DM_XQ4 DM_Q4(0) DM_NEXT(2304) DM_Q4(1) DM_NEXT(2304) DM_Q4(2) "s_waitcnt vmcnt(9)"
                     : DM_OUT(a, 0), [l] "+&s"(lds)
                     : DM_ARGS, DM_IN3(0), DM_IN3(1), DM_IN3(2)
                     : "memory", "scc");
    } else if constexpr (TYPE == kQ4_K && XB == 2 && SLOTS == 2) {
        asm volatile(DM_XQ4 DM_XQ4B DM_Q4(0) DM_NEXT(2304) DM_Q4(1) "s_waitcnt vmcnt(6)"
                     : DM_OUT(a, 0), DM_OUT(b, 1), [l] "+&s"(lds)
                     : DM_ARGS, DM_IN3(0), DM_IN3(1)
                     : "memory", "scc");
    } else if constexpr (TYPE == kQ6_K && XB == 1 && SLOTS == 1) {
        asm volatile(DM_XQ6 DM_Q6(0) "s_waitcnt vmcnt(4)"
                     : DM_OUT(a, 0), [l] "+&s"(lds)
                     : DM_ARGS, DM_IN4(0)
                     : "memory", "scc");
    } else if constexpr (TYPE == kQ6_K && XB == 1 && SLOTS == 2) {
        asm volatile(DM_XQ6 DM_Q6(0) DM_NEXT(3584) DM_Q6(1) "s_waitcnt vmcnt(8)"
                     : DM_OUT(a, 0), [l] "+&s"(lds)
                     : DM_ARGS, DM_IN4(0), DM_IN4(1)
                     : "memory", "scc");
    } else if constexpr (TYPE == kQ6_K && XB == 1 && SLOTS == 3) {
        asm volatile(DM_XQ6 DM_Q6(0) DM_NEXT(3584) DM_Q6(1) DM_NEXT(3584) DM_Q6(2) "s_waitcnt vmcnt(12)"
                     : DM_OUT(a, 0), [l] "+&s"(lds)
                     : DM_ARGS, DM_IN4(0), DM_IN4(1), DM_IN4(2)
                     : "memory", "scc");
    } else if constexpr (TYPE == kQ6_K && XB == 2 && SLOTS == 1) {
        asm volatile(DM_XQ6 DM_XQ6B DM_Q6(0) "s_waitcnt vmcnt(4)"
                     : DM_OUT(a, 0), DM_OUT(b, 1), [l] "+&s"(lds)
                     : DM_ARGS, DM_IN4(0)
                     : "memory", "scc");
    } else {
        static_assert(TYPE == 0, "no such prologue");
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Main kernel.  A wave owns a run of up to KB blocks of K: it builds the
// activation fragments of those columns in registers once, then streams its
// run of one 16-row tile after another, so the fragments are never read
// again.  The weights go from memory straight to the wave's LDS ring
// (buffer loads with the LDS destination), DEPTH - 1 blocks ahead of the one
// being computed.  The workgroup's wave_k waves cover a K part together
// (their loads are the whole rows of a tile) and its waves / wave_k wave groups
// take alternate tiles; every pass_tiles tiles the waves' results meet in
// LDS and are written.
// Grid: k_parts x row_groups workgroups, one per CU.  With k_parts > 1 the
// parts' sums meet pairwise in memory: a workgroup exchanges its pair of
// sums with the meeting place; the first to come finds it empty and is done,
// the second adds what it finds and goes on to the next level (a + b is the
// same in either order, so the result does not depend on who is first).
// MODE 0: y = W x.  MODE 2: gate/up pair on RMSNorm(x), act = silu(gate) * up
// (k_parts = 1).
//
// What bounds it: bytes in flight.  110 KiB of ring hold two or three tiles'
// blocks per wave, and each wave asks for the next only when it has finished
// one, so a tall matrix streams at 4.7 TB/s; the fragments' prologue (x, split,
// first weights) is about 3 us of every launch.  Measured on MI355X against
// the form with a launch that prepared the fragments in memory and waves that
// read them again for every tile: Q4_K 12288 x 4096, 8 tokens 16.8 -> 10.2
// us, 16 tokens 25.2 -> 15.0; Q6_K 4096 x 12288, 8 tokens 20.6 -> 13.9;
// 4096 x 4096 Q4_K 10.7 -> 7.0; Q6_K 151936 x 4096 200 -> 112 us.  16 waves
// of one block beat 8 of two (12.6 us at 12288 x 4096): four waves per SIMD
// hide each other's LDS and MFMA latency.
// ---------------------------------------------------------------------------
template <uint32_t TYPE, int NT, int MODE, int KB, uint32_t W, bool PHASED, bool GROUPED>
__device__ __forceinline__ void qmv_body(const QmvArgs &p, uint32_t part, uint32_t rg, uint32_t x_rows,
                                         const uint32_t *x_row, const uint32_t *y_row) {
    constexpr uint32_t BB = StageQ<TYPE>::bytes;
    constexpr uint32_t RR = MODE == 2 ? 2 : 1;  // matrices streamed
    constexpr uint32_t DEPTH = ring_depth<TYPE, NT, MODE, W, PHASED, GROUPED>();
    static_assert(DEPTH >= 2, "a slot in flight while one is read");
    using ST = StageQ<TYPE>;
    constexpr uint32_t CH = ST::chunks, NL = ST::loads;
    constexpr uint32_t SLOT = ST::items;      // chunks of a ring slot
    constexpr uint32_t PI = pass_tiles<MODE, PHASED>() * RR;  // items of a wave per pass (of 8 NT tokens)
    __shared__ v4u red_all[red_floats<NT, MODE, W, PHASED>() / 4];
    __shared__ v4u split_all[PHASED ? W * 128 : 1];
    __shared__ uint32_t s_min[W * 64];  // 8 tokens x {hi, lo} x 4 lane groups
    __shared__ float red_ss[MODE == 2 ? W * 16 : 1];
    __shared__ float s_up[W * KB * 16];  // 2^e of each wave's blocks and tokens
    extern __shared__ v4u ring_all[];
    float *red = (float *)red_all;

    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t n = lane & 15u, kg = lane >> 4;
    const uint32_t wk = p.wave_k, wt = (blockDim.x >> 6) / wk, kw = wave % wk, wg = wave / wk;
    const uint32_t blocks = p.columns / 256, tiles = (p.rows + 15) / 16;
    const uint32_t t_begin = (uint32_t)((uint64_t)rg * tiles / p.row_groups);
    const uint32_t t_end = (uint32_t)((uint64_t)(rg + 1) * tiles / p.row_groups);
    const uint32_t phases = PHASED ? p.phases : 1u, units = wk * p.k_parts * phases;
    v4u *ring = ring_all + wave * DEPTH * SLOT;
    const uint32_t ring_lds =
        __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) v4u *)ring);

    // Buffer descriptors over whole dwords: the last dword of the matrix may
    // extend up to 3 bytes past its end (inside the allocation's
    // granularity); loads beyond it read 0.
    const uint32_t records = (p.row_bytes * p.rows + 3u) & ~3u;
    auto descriptor = [&](const uint8_t *base) {
        return v4u{(uint32_t)(uintptr_t)base, (uint32_t)((uintptr_t)base >> 32) & 0xffffu, records, 0x00020000u};
    };
    const v4u rsrc = descriptor(p.w), rsrc2 = descriptor(MODE == 2 ? p.w2 : p.w);

    // Position in the wave's sequence: pass (pass_tiles tiles of each
    // wave group), phase, item (tile of the pass, matrix).
    struct Pos {
        uint32_t tile0, phase, i;  // first tile of the pass
    };
    // Token pairs kept per item of red (a power of two), and how many more
    // items a pass has for it.
    const uint32_t pairs = (p.batch + 1) / 2, pp = pairs <= 1 ? 1u : pairs <= 2 ? 2u : pairs <= 4 ? 4u : 8u;
    const uint32_t more = NT * 4 / pp, pass_items = PI * more;
    const uint32_t pass_step = pass_tiles<MODE, PHASED>() * more * wt;
    auto items = [&](uint32_t tile0) {  // items per wave and phase of the pass at tile0
        const uint32_t left = t_end - tile0, t = left < pass_step ? left : pass_step;
        return (t + wt - 1) / wt * RR;
    };
    auto advance = [&](Pos &q) {
        if (++q.i < items(q.tile0)) return;
        q.i = 0;
        if (PHASED) {
            if (++q.phase < phases) return;
            q.phase = 0;
        }
        q.tile0 += pass_step;
    };
    auto k_begin = [&](uint32_t phase) { return run_begin((part * phases + phase) * wk + kw, units, blocks); };
    auto k_end = [&](uint32_t phase) { return run_begin((part * phases + phase) * wk + kw + 1, units, blocks); };

    // Chunk j * 64 + lane of a block of a tile: offset from the wave's first
    // block of the tile's first row (16 c is a multiple of the 4 bytes the
    // sum is aligned to).
    uint32_t lane_off[NL];
#pragma unroll
    for (uint32_t j = 0; j < NL; j++) {
        const uint32_t item = j * 64 + lane, r = item / CH, c = item % CH;
        lane_off[j] = r * p.row_bytes + 16 * c;
    }
    // The loads of block b of the wave's run of q's item; a block past the run
    // or a tile past the end reads past the matrix (zeros), so that the loads
    // in flight can be counted.
    auto slot_loads = [&](const Pos &q, uint32_t b, uint32_t (&off)[NL], v4u &rs) {
        const uint32_t tile = q.tile0 + (q.i / RR) * wt + wg;
        const uint32_t blk = k_begin(q.phase) + b;
        const uint32_t base = q.tile0 < t_end && tile < t_end && blk < k_end(q.phase)
                                  ? tile * 16 * p.row_bytes + blk * BB
                                  : 0xffffffffu;
#pragma unroll
        for (uint32_t j = 0; j < NL; j++) off[j] = __builtin_elementwise_add_sat(lane_off[j], base) & ~3u;
        rs = MODE == 2 && (q.i % RR) ? rsrc2 : rsrc;
    };
    // nxt, nxt_b: the next block to request.
    Pos nxt{t_begin, 0, 0};
    uint32_t nxt_b = 0, issue_slot = 0;
    auto next_block = [&]() {
        if (++nxt_b == KB) {
            nxt_b = 0;
            advance(nxt);
        }
    };
    auto issue_next = [&]() {
        uint32_t off[NL];
        v4u rs;
        slot_loads(nxt, nxt_b, off, rs);
        // (the slot's last reads have returned)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        load_slot(ring_lds + issue_slot * (SLOT * 16), off, rs);
        issue_slot = issue_slot + 1 == DEPTH ? 0 : issue_slot + 1;
        next_block();
    };

    half8 a[KB][8][NT];
    uint32_t amin[KB][NT];  // the min step's fragment (its other columns are zero)
    float ss[NT * 2];       // MODE 2: the lane's part of its tokens' sums of squares
    // The fragments of block b, tokens 8 g .. 8 g + 7: the values are scaled
    // and split as they were loaded (x4[4 u + r], see round_column) and go
    // through LDS to the lanes that hold the token's A rows, a round (2 KiB)
    // at a time: the quad (kg, c) of token i is at slot (4 kg + c) ^ i of 16
    // (so neither side meets bank conflicts), hi pairs then lo pairs.  The
    // area is the ring slot the prologue leaves free, or (PHASED) LDS of its
    // own; a wave reads only what it wrote.
    const uint32_t li = lane >> 4, lk = (lane >> 2) & 3u, lc = lane & 3u;
    uint32_t *sp = PHASED ? (uint32_t *)split_all + wave * 512 : (uint32_t *)(ring + (DEPTH - 1) * SLOT);
    uint32_t *smn = s_min + wave * 64;
    auto split = [&](int g, int b, uint32_t phase, const floatx4 (&x4)[8]) {
        const bool used = k_begin(phase) + b < k_end(phase);
        float down[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            float mx = 0.0f, q = 0.0f;
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float v = x4[4 * u + r][j];
                    mx = fmaxf(mx, fabsf(v));
                    if (MODE == 2) q = __builtin_fmaf(v, v, q);
                }
            if (MODE == 2 && used) ss[2 * g + u] += q;
            const int e = block_exponent(row_max(mx));
            down[u] = ldexpf(1.0f, -e);
            // every lane of the row holds the same scale
            s_up[(wave * KB + b) * 16 + 8 * g + 4 * u + li] = ldexpf(1.0f, e);
        }
        uint32_t hi[8][2], lo[8][2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            float sum[2] = {0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const floatx4 v = x4[4 * u + r] * down[u];
                // fragment order of a quad: columns 0, 2, 1, 3 (the byte pairs of a weight dword)
                split_pair(v[0], v[2], hi[4 * u + r][0], lo[4 * u + r][0]);
                split_pair(v[1], v[3], hi[4 * u + r][1], lo[4 * u + r][1]);
                if (TYPE == kQ4_K) sum[r >> 1] += (v[0] + v[1]) + (v[2] + v[3]);
            }
            if constexpr (TYPE == kQ4_K) {
                // sub-blocks 2 kg, 2 kg + 1; 2^-6 keeps |sum| inside fp16
                uint32_t h, l;
                split_pair(quad_sum(sum[0]) * 0.015625f, quad_sum(sum[1]) * 0.015625f, h, l);
                smn[(4 * u + li) * 8 + lk] = h;
                smn[(4 * u + li) * 8 + 4 + lk] = l;
            }
        }
        const uint32_t token = n >> 1, half = n & 1u;
        uint32_t f[8][4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const uint32_t i = 4 * u + li;
                *(v4u *)&sp[i * 64 + ((4 * lk + lc) ^ i) * 4] =
                    v4u{hi[4 * u + r][0], hi[4 * u + r][1], lo[4 * u + r][0], lo[4 * u + r][1]};
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (uint32_t c = 0; c < 4; c++) {
                const u32x2 v = *(const u32x2 *)&sp[token * 64 + ((4 * kg + c) ^ token) * 4 + half * 2];
                f[quad_step<TYPE>(r, c)][2 * quad_half<TYPE>(r, c)] = v[0];
                f[quad_step<TYPE>(r, c)][2 * quad_half<TYPE>(r, c) + 1] = v[1];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int t = 0; t < 8; t++) a[b][t][g] = frag(f[t][0], f[t][1], f[t][2], f[t][3]);
        if constexpr (TYPE == kQ4_K) amin[b][g] = smn[token * 8 + half * 4 + kg];
    };
    // Byte of x that load (u, 0) of a block takes (tokens past the batch read
    // past the end: zeros).
    auto x_byte = [&](int g, uint32_t blk, int u) {
        const uint32_t i = 8 * g + 4 * u + li;
        const uint32_t at = ((GROUPED ? x_row[i] : i) * p.columns + blk * 256 + round_column<TYPE>(lk) + 4 * lc) * 4;
        return GROUPED && i >= p.batch ? 0xfffff000u : at;
    };
    const uint32_t x_bytes = x_rows * p.columns * 4;
    const v4u xr = v4u{(uint32_t)(uintptr_t)p.x, (uint32_t)((uintptr_t)p.x >> 32) & 0xffffu, x_bytes, 0x00020000u};
    const __amdgpu_buffer_rsrc_t xrs = make_rsrc(p.x, x_bytes);
    auto load_x = [&](int g, int b, uint32_t phase, floatx4 (&x4)[8]) {
#pragma unroll
        for (int i = 0; i < 8; i++)
            x4[i] = __builtin_bit_cast(
                floatx4, rsrc_load16(xrs, x_byte(g, k_begin(phase) + b, i / 4) + (i % 4) * round_bytes<TYPE>()));
    };
    auto store_ss = [&](uint32_t phase) {
        if constexpr (MODE == 2) {
#pragma unroll
            for (int i = 0; i < NT * 2; i++) {
                const float v = row_sum(ss[i]);
                if ((lane & 15u) == 0) {
                    float &slot = red_ss[wave * 16 + 4 * i + li];
                    slot = phase == 0 ? v : slot + v;
                }
            }
        }
    };

#pragma unroll
    for (int i = 0; i < NT * 2; i++) ss[i] = 0.0f;
    Pos cur{t_begin, 0, 0};
    {
        // The first activations are requested before the weights, and waited
        // for without them: a wave's loads complete in the order they were
        // issued.
        constexpr int XB = W == 16 ? KB : 1;  // blocks of x requested here
        floatx4 x4[XB][8];
        uint32_t off[DEPTH - 1][NL];
        v4u rs[DEPTH - 1];
#pragma unroll
        for (uint32_t d = 0; d + 1 < DEPTH; d++) {
            slot_loads(nxt, nxt_b, off[d], rs[d]);
            next_block();
        }
        issue_slot = DEPTH - 1;
        first_loads<TYPE, XB>(x4, xr, x_byte(0, k_begin(0), 0), x_byte(0, k_begin(0), 1), ring_lds, off, rs);
#pragma unroll
        for (int b = 0; b < XB; b++) split(0, b, 0, x4[b]);
#pragma unroll
        for (int g = 0; g < NT; g++)
#pragma unroll
            for (int b = g == 0 ? XB : 0; b < KB; b++) {
                load_x(g, b, 0, x4[0]);
                split(g, b, 0, x4[0]);
            }
    }
    store_ss(0);

    bool first_pass = true;
    uint32_t slot = 0;
    while (cur.tile0 < t_end) {
        const uint32_t tile0 = cur.tile0;
#pragma clang loop unroll(disable)
        do {
            if (PHASED && cur.i == 0 && !(first_pass && cur.phase == 0)) {
                // the next phase's fragments (K longer than the registers of
                // the workgroups that split it hold)
#pragma unroll
                for (int i = 0; i < NT * 2; i++) ss[i] = 0.0f;
#pragma unroll
                for (int g = 0; g < NT; g++)
#pragma unroll
                    for (int b = 0; b < KB; b++) {
                        floatx4 x4[8];
                        load_x(g, b, cur.phase, x4);
                        split(g, b, cur.phase, x4);
                    }
                if (first_pass) store_ss(cur.phase);
            }
            float acc[NT][2];
#pragma unroll
            for (int g = 0; g < NT; g++) acc[g][0] = acc[g][1] = 0.0f;
            const uint32_t k0 = k_begin(cur.phase), nb = k_end(cur.phase) - k0;
            const uint32_t tile = cur.tile0 + (cur.i / RR) * wt + wg;
            const uint32_t row_at = (tile * 16 + n) * p.row_bytes + k0 * BB;
#pragma unroll
            for (int b = 0; b < KB; b++) {
                issue_next();
                // The loads of this slot are the oldest in flight: all but
                // the DEPTH - 1 blocks requested after them have landed.
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NL * (DEPTH - 1)) : "memory");
                if ((uint32_t)b < nb) {
                    // read only by the wave that wrote them
                    float up[NT][2];
#pragma unroll
                    for (int g = 0; g < NT; g++)
#pragma unroll
                        for (int j = 0; j < 2; j++) up[g][j] = s_up[(wave * KB + b) * 16 + 8 * g + 2 * kg + j];
                    Raw<TYPE> raw;
                    // a Q6_K block starts 0 or 2 bytes into its first dword
                    take_raw(ring + slot * SLOT, CH, n, kg, (row_at + b * BB) & 3u, raw);
                    block_dot<NT>(raw, a[b], amin[b], kg, up, acc);
                }
                slot = slot + 1 == DEPTH ? 0 : slot + 1;
            }
            // row n, token pair 4 g + kg: two runs of 16 rows
            float *sl = &red[(wave * pass_items + cur.i) * pp * 32 + n];
#pragma unroll
            for (int g = 0; g < NT; g++) {
                if (4 * g + kg >= pp) continue;
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    float &s = sl[(4 * g + kg) * 32 + j * 16];
                    s = !PHASED || cur.phase == 0 ? acc[g][j] : s + acc[g][j];
                }
            }
            advance(cur);
        } while (cur.tile0 == tile0);
        first_pass = false;

        // The cross-wave sums and the output of the pass: thread = row rn of
        // a tile, tokens tk and tk + 1.
        lds_barrier();
        const uint32_t left = t_end - tile0, nt = left < pass_step ? left : pass_step;
        for (uint32_t idx = threadIdx.x; idx < nt * 16 * pairs; idx += blockDim.x) {
            const uint32_t rn = idx & 15u, pair = (idx >> 4) / nt, tl = (idx >> 4) - pair * nt;
            const uint32_t group = tl % wt, sl = tl / wt, tk = 2 * pair, row = (tile0 + tl) * 16 + rn;
            float v[RR][2];
#pragma unroll
            for (uint32_t m = 0; m < RR; m++) {
                v[m][0] = v[m][1] = 0.0f;
#pragma clang loop unroll_count(4)
                for (uint32_t k = 0; k < wk; k++) {
                    const float *r = &red[(((group * wk + k) * pass_items + sl * RR + m) * pp + pair) * 32 + rn];
                    v[m][0] += r[0];
                    v[m][1] += r[16];
                }
            }
            if constexpr (MODE == 2) {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    // RMSNorm factor inv = (ss/n + eps).sqrt().recip() (src/cpu.rs:98-142)
                    float q = 0.0f;
#pragma clang loop unroll_count(4)
                    for (uint32_t k = 0; k < wk; k++) q += red_ss[k * 16 + tk + j];
                    const float sc = p.normalize ? 1.0f / __builtin_sqrtf(q / (float)p.columns + p.epsilon) : 1.0f;
                    const float gate = v[0][j] * sc, u = v[1][j] * sc;
                    if constexpr (GROUPED) {
                        // routed-expert activation (src/glm52/expert.rs:260-267)
                        v[0][j] = (gate / (1.0f + expf(-gate))) * u;
                    } else {
                        // silu(gate) * up, stable sigmoid (src/qwen35/cpu.rs:982-993)
                        const float ex = expf(-fabsf(gate));
                        const float sig = (gate >= 0.0f ? 1.0f : ex) / (1.0f + ex);
                        v[0][j] = gate * sig * u;
                    }
                }
            } else {
                bool mine = true;
                uint64_t *place = p.meet + ((size_t)(tile0 + tl) * (p.k_parts - 1) * pairs + pair) * 16 + rn;
                for (uint32_t span = 1, nodes = p.k_parts / 2; span < p.k_parts; span *= 2, nodes /= 2) {
                    uint64_t *at = place + (size_t)(part / (2 * span)) * pairs * 16;
                    const uint64_t other = __hip_atomic_exchange(at, pack_pair(v[0][0], v[0][1]), __ATOMIC_RELAXED,
                                                                 __HIP_MEMORY_SCOPE_AGENT);
                    if (other == kMeetEmpty) {
                        mine = false;
                        break;
                    }
                    __hip_atomic_store(at, kMeetEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    v[0][0] += __uint_as_float((uint32_t)other);
                    v[0][1] += __uint_as_float((uint32_t)(other >> 32));
                    place += (size_t)nodes * pairs * 16;
                }
                if (!mine) continue;
            }
            if (row < p.rows) {
                p.y[(size_t)(GROUPED ? y_row[tk] : tk) * p.rows + row] = v[0][0];
                if (tk + 1 < p.batch) p.y[(size_t)(GROUPED ? y_row[tk + 1] : tk + 1) * p.rows + row] = v[0][1];
            }
        }
        lds_barrier();  // red is written again in the next pass
    }
    // the ring's last loads have landed before the workgroup's LDS is freed
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <uint32_t TYPE, int NT, int MODE, int KB, uint32_t W, bool PHASED>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(W / 4, W / 4)))
qmv_kernel(const QmvArgs p) {
    qmv_body<TYPE, NT, MODE, KB, W, PHASED, false>(p, blockIdx.x % p.k_parts, blockIdx.x / p.k_parts, p.batch, nullptr,
                                                   nullptr);
}

// The routed experts of up to kGroupPairs pairs in one launch (MODE 2 with
// the GLM activation, then MODE 0): each expert's matrix is streamed once
// for all its tokens, up to 8 at a time.  Every workgroup finds from the ids
// which experts are selected and takes its share of one of them: with n
// (expert, 8 tokens) entries, gridDim.x / n workgroups each.  The grid is two
// 8-wave workgroups per CU, so one's prologue runs beside the other's
// stream, and at least one per pair (experts_grid).
template <uint32_t TYPE, int MODE, int KB, uint32_t W>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(KB > 2 ? 2 : 4, KB > 2 ? 2 : 4)))
qmv_experts_kernel(const QmvArgs args, const QmvExperts ex) {
    __shared__ uint32_t s_count[kGroupExperts], s_pair[8], s_x[8], s_entry[4];
    const uint32_t tid = threadIdx.x;
    // The first wave reads every word it needs at once.
    uint32_t id0 = 0, id1 = 0, go = 1;
    if (tid < 64) {
        if (tid < ex.pairs) id0 = ex.ids[tid];
        if (tid + 64 < ex.pairs) id1 = ex.ids[tid + 64];
        if (tid < ex.go_count) go = ex.go[tid];
    }
    for (uint32_t e = tid; e < kGroupExperts; e += blockDim.x) s_count[e] = 0;
    if (tid < 8) s_pair[tid] = s_x[tid] = 0;
    if (tid == 0) s_entry[0] = 0;
    lds_barrier();
    if (tid < 64 && __builtin_amdgcn_ballot_w64(go == 0) == 0) {
        if (tid < ex.pairs) atomicAdd(&s_count[id0], 1u);
        if (tid + 64 < ex.pairs) atomicAdd(&s_count[id1], 1u);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        // entries of experts 4 tid .. + 3, their running sum over the lanes
        uint32_t n[4], sum = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            n[j] = (s_count[4 * tid + j] + 7) / 8;
            sum += n[j];
        }
        uint32_t upto = sum;
#pragma unroll
        for (int d = 1; d < 64; d *= 2) {
            const uint32_t v = __shfl_up(upto, d, 64);
            if ((int)tid >= d) upto += v;
        }
        const uint32_t total = __shfl(upto, 63, 64);
        const uint32_t share = experts_share(gridDim.x, total);
        const uint32_t entry = blockIdx.x / share;
        if (entry < total) {
            uint32_t base = upto - sum, mine = ~0u, from = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (entry >= base && entry < base + n[j]) {
                    mine = 4 * tid + j;
                    from = 8 * (entry - base);
                }
                base += n[j];
            }
            const int owner = __builtin_ctzll(__builtin_amdgcn_ballot_w64(mine != ~0u));
            const uint32_t expert = __shfl(mine, owner, 64), first = __shfl(from, owner, 64);
            // the entry's pairs, in order
            const bool h0 = tid < ex.pairs && id0 == expert, h1 = tid + 64 < ex.pairs && id1 == expert;
            const uint64_t b0 = __builtin_amdgcn_ballot_w64(h0), b1 = __builtin_amdgcn_ballot_w64(h1);
            const uint64_t below = (1ull << tid) - 1;
            const uint32_t r0 = __builtin_popcountll(b0 & below);
            const uint32_t r1 = __builtin_popcountll(b0) + __builtin_popcountll(b1 & below);
            if (h0 && r0 >= first && r0 < first + 8) {
                s_pair[r0 - first] = tid;
                s_x[r0 - first] = ex.k ? tid / ex.k : tid;
            }
            if (h1 && r1 >= first && r1 < first + 8) {
                s_pair[r1 - first] = tid + 64;
                s_x[r1 - first] = ex.k ? (tid + 64) / ex.k : tid + 64;
            }
            if (tid == 0) {
                const uint32_t left = __builtin_popcountll(b0) + __builtin_popcountll(b1) - first;
                s_entry[0] = left < 8 ? left : 8;
                s_entry[1] = expert;
                s_entry[2] = share;
            }
        }
    }
    lds_barrier();
    const uint32_t count = __builtin_amdgcn_readfirstlane(s_entry[0]);
    if (count == 0) return;
    const uint32_t expert = __builtin_amdgcn_readfirstlane(s_entry[1]);
    const uint32_t share = __builtin_amdgcn_readfirstlane(s_entry[2]);
    QmvArgs p = args;
    const uint64_t at = ex.w_of[expert];  // the same for every lane: kept in scalar registers
    const uint32_t at_lo = __builtin_amdgcn_readfirstlane((uint32_t)at);
    const uint32_t at_hi = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32));
    p.w = (const uint8_t *)((uint64_t)at_hi << 32 | at_lo);
    p.w2 = p.w + ex.w2_offset;
    p.batch = count;
    p.row_groups = share;
    qmv_body<TYPE, 1, MODE, KB, W, false, true>(p, 0, blockIdx.x % share, ex.x_rows, s_x, s_pair);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

bool qmv_supported(uint32_t type, size_t rows, size_t columns, const void *w, size_t batch) {
    if (type == kQ8_0) {
        // Q8_0 has the int8 kernel only: batch 1-4 (records permitting),
        // whole 8-block super-blocks (272 bytes, 16-byte aligned rows),
        // 32-bit offsets with slack.
        if (columns == 0 || columns % 256 || batch < 1 || batch > 4 || rows == 0) return false;
        const uint64_t row_bytes = (uint64_t)(columns / 256) * 272;
        if (row_bytes * (rows + 2) + 1024 >= 0xffffffffull || ((uintptr_t)w & 15u)) return false;
        return qmv8_supported(type, rows, columns, batch);
    }
    if (type != kQ4_K && type != kQ6_K) return false;
    if (columns == 0 || columns % 256 || batch < 1 || batch > 16) return false;
    const uint64_t row_bytes = (uint64_t)(columns / 256) * (type == kQ4_K ? 144 : 210);
    // Offsets are 32-bit: the matrix plus two rows of slack must fit.
    if (rows == 0 || row_bytes * (rows + 2) + 1024 >= 0xffffffffull) return false;
    if ((uint64_t)batch * columns * 4 >= 0xffffffffull) return false;
    // (both forms: a gate/up pair asks through here too)
    if (columns / 256 > 0xffff && !(qmv_runs_fit((uint32_t)(columns / 256), (uint32_t)batch, 0) &&
                                    qmv_runs_fit((uint32_t)(columns / 256), (uint32_t)batch, 2)))
        return false;
    const uintptr_t a = (uintptr_t)w;
    if (type == kQ4_K ? (a & 15u) : (a & 3u)) return false;
    return true;
}

namespace {

template <uint32_t TYPE, int NT, int MODE, int KB, uint32_t W, bool PHASED = false>
hipError_t run(dmhip_ctx *ctx, const QmvPlan &p, QmvArgs &a) {
    // no more wave groups than a workgroup has tiles
    const uint32_t tiles = (a.rows + 15) / 16, per = (tiles + p.row_groups - 1) / p.row_groups;
    const uint32_t groups = W / p.wave_k, waves = (groups < per ? groups : per) * p.wave_k;
    const uint32_t lds = waves * ring_depth<TYPE, NT, MODE, W, PHASED>() * StageQ<TYPE>::items * 16;
    auto kernel = qmv_kernel<TYPE, NT, MODE, KB, W, PHASED>;
    static LdsLimit limit;
    hipError_t e = limit.ensure((const void *)kernel, lds);
    if (e != hipSuccess) return e;
    return launch_kernel(ctx, kernel, dim3(p.k_parts * p.row_groups), dim3(64 * waves), lds, a);
}

template <uint32_t TYPE, int MODE>
hipError_t dispatch(dmhip_ctx *ctx, uint32_t rows, uint32_t columns, const void *w, const void *w2, uint32_t batch,
                    const float *x, int normalize, float epsilon, float *y) {
    const uint32_t blocks = columns / 256;
    const uint32_t cus = ctx->compute_units > 0 ? (uint32_t)ctx->compute_units : 256u;
    const QmvPlan p = qmv_plan(rows, blocks, batch, MODE, cus, kQmvMeetWords);
    QmvArgs a{(const uint8_t *)w, (const uint8_t *)w2, x, y, ctx->qmv_meet, rows, columns,
              blocks * StageQ<TYPE>::bytes, batch, p.wave_k, p.k_parts, p.row_groups, p.phases, normalize, epsilon};
    if (p.phases > 1)
        return batch <= 8 ? run<TYPE, 1, MODE, 2, 8, true>(ctx, p, a) : run<TYPE, 2, MODE, 2, 8, true>(ctx, p, a);
    if (batch > 8) return p.kb == 1 ? run<TYPE, 2, MODE, 1, 8>(ctx, p, a) : run<TYPE, 2, MODE, 2, 8>(ctx, p, a);
    // (16 waves; a gate/up pair, which holds a block per wave there, has 8 of 3 blocks besides)
    if constexpr (MODE == 2) {
        if (p.waves == 8) return run<TYPE, 1, MODE, 3, 8>(ctx, p, a);
    } else {
        if (p.kb == 2) return run<TYPE, 1, MODE, 2, 16>(ctx, p, a);
    }
    return run<TYPE, 1, MODE, 1, 16>(ctx, p, a);
}

}  // namespace

// Experts' rows: fragments of up to 3 blocks per wave, 8 waves.
constexpr uint32_t kGroupBlocks = 24;

bool qmv_experts_supported(uint32_t type, size_t rows, size_t columns, size_t experts, size_t pairs, size_t x_rows) {
    if ((type != kQ4_K && type != kQ6_K) || columns % 256 || columns == 0 || rows == 0) return false;
    if (columns / 256 > kGroupBlocks || experts > kGroupExperts || pairs > kGroupPairs) return false;
    const uint64_t row_bytes = (uint64_t)(columns / 256) * (type == kQ4_K ? 144 : 210);
    return row_bytes * (rows + 2) + 1024 < 0xffffffffull && (uint64_t)x_rows * columns * 4 < 0xffff0000ull;
}

namespace {

template <uint32_t TYPE, int MODE, int KB, uint32_t W>
hipError_t run_experts(dmhip_ctx *ctx, const QmvArgs &a, const QmvExperts &ex, uint32_t waves, uint32_t grid) {
    const uint32_t lds = waves * ring_depth<TYPE, 1, MODE, W, false, true>() * StageQ<TYPE>::items * 16;
    auto kernel = qmv_experts_kernel<TYPE, MODE, KB, W>;
    static LdsLimit limit;
    hipError_t e = limit.ensure((const void *)kernel, lds);
    if (e != hipSuccess) return e;
    return launch_kernel(ctx, kernel, dim3(grid), dim3(64 * waves), lds, a, ex);
}

template <uint32_t TYPE, int MODE>
hipError_t dispatch_experts(dmhip_ctx *ctx, uint32_t rows, uint32_t columns, const float *x, float *y,
                            const QmvExperts &ex) {
    const uint32_t blocks = columns / 256, kb = (blocks + 7) / 8, wave_k = (blocks + kb - 1) / kb;
    const uint32_t waves = 8 / wave_k * wave_k;
    const uint32_t cus = ctx->compute_units > 0 ? (uint32_t)ctx->compute_units : 256u;
    const QmvArgs a{nullptr, nullptr, x, y, nullptr, rows, columns, blocks * StageQ<TYPE>::bytes, 0, wave_k, 1, 1, 1, 0, 0.0f};
    const uint32_t grid = experts_grid(cus, ex.pairs);
    // (rows of 3 or 6 blocks keep 6 waves busy, whose ring has room for
    // another slot each)
    if (waves == 6 && kb == 1) return run_experts<TYPE, MODE, 1, 6>(ctx, a, ex, waves, grid);
    if (kb == 1) return run_experts<TYPE, MODE, 1, 8>(ctx, a, ex, waves, grid);
    if (kb == 2) return run_experts<TYPE, MODE, 2, 8>(ctx, a, ex, waves, grid);
    return run_experts<TYPE, MODE, 3, 8>(ctx, a, ex, waves, grid);
}

}  // namespace

hipError_t launch_qmv_experts(dmhip_ctx *ctx, uint32_t type, uint32_t rows, uint32_t columns, bool gate_up,
                              uint64_t up_offset, const uint64_t *w_of, const uint32_t *ids, const uint32_t *go,
                              uint32_t tokens, uint32_t k, const float *x, float *y) {
    const uint32_t pairs = tokens * k;
    const QmvExperts ex{w_of, up_offset, ids, go, tokens, pairs, gate_up ? k : 0, gate_up ? tokens : pairs};
    if (gate_up)
        return type == kQ4_K ? dispatch_experts<kQ4_K, 2>(ctx, rows, columns, x, y, ex)
                             : dispatch_experts<kQ6_K, 2>(ctx, rows, columns, x, y, ex);
    return type == kQ4_K ? dispatch_experts<kQ4_K, 0>(ctx, rows, columns, x, y, ex)
                         : dispatch_experts<kQ6_K, 0>(ctx, rows, columns, x, y, ex);
}

// The activations of a batch as fp16 fragments in memory.  No launch stores
// them there (they are built in registers, and the K-split partials go to
// ctx->qmv_meet): it is the allocation-free entry point's limit on a shape,
// kept so that it accepts and rejects the same ones.
size_t qmv_noalloc_bytes(uint32_t type, size_t columns, size_t batch) {
    const size_t spb = type == kQ4_K ? 9 : 8;
    const size_t xp_bytes = (columns / 256) * spb * 4 * 2 * batch * 8 * sizeof(_Float16);
    return ((xp_bytes + 255) & ~(size_t)255) + 64 * sizeof(float);
}

hipError_t launch_qmv(dmhip_ctx *ctx, uint32_t type, uint32_t rows, uint32_t columns, const void *w,
                      uint32_t batch, const float *x, float *y, ArgmaxState *argmax,
                      uint32_t *index_out) {
    if (qmv8_supported(type, rows, columns, batch)) {
        if (!argmax) return launch_qmv8(ctx, type, rows, columns, w, batch, x, y, nullptr, nullptr);
        // the int8 kernel's last workgroup publishes the argmax itself; at
        // most one candidate per 16-row tile otherwise
        const size_t candidates = (size_t)(rows + 15) / 16 + 4;
        if (ctx->partials.ensure(candidates * sizeof(ArgmaxPartial)) != DMHIP_OK) return hipErrorOutOfMemory;
        uint32_t count = 0;
        return launch_qmv8(ctx, type, rows, columns, w, batch, x, y, (ArgmaxPartial *)ctx->partials.ptr, &count,
                           ArgmaxFinish{argmax, index_out, ctx->argmax_ticket,
                                        (unsigned long long *)(ctx->argmax_ticket + 2)});
    }
    const hipError_t e = type == kQ4_K
                             ? dispatch<kQ4_K, 0>(ctx, rows, columns, w, nullptr, batch, x, 0, 0.0f, y)
                             : dispatch<kQ6_K, 0>(ctx, rows, columns, w, nullptr, batch, x, 0, 0.0f, y);
    if (e != hipSuccess || !argmax) return e;
    return launch_argmax(ctx->stream, y, rows, argmax, index_out);
}

hipError_t launch_qmv_gate_up(dmhip_ctx *ctx, uint32_t type, uint32_t rows, uint32_t columns,
                              const void *gate, const void *up, uint32_t batch, const float *x,
                              float *act, int normalize, float epsilon) {
    return type == kQ4_K
               ? dispatch<kQ4_K, 2>(ctx, rows, columns, gate, up, batch, x, normalize, epsilon, act)
               : dispatch<kQ6_K, 2>(ctx, rows, columns, gate, up, batch, x, normalize, epsilon, act);
}

// A kernel of this file: resolving it loads the file's code object.
const void *module_anchor_qmv() { return (const void *)qmv_kernel<kQ4_K, 1, 0, 1, 16, false>; }

}  // namespace dm
