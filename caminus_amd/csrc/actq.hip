// Fused activation fake-quant for gfx950, forward and backward: per row of K values (K % 128 == 0, K <= 8192) a 128-point
// Hadamard rotation per chunk in bf16 steps, one int4-style scale per row, codes packed two per byte. Replaces actq_fwd_{f32,bf16},
// actq_fwd_codes_{f32,bf16}, actq_bwd_{f32,bf16}, silu_mul_actq_{fwd,bwd} and block_entry_{fwd,bwd} (kernels/actq.hip:40-53,
// 96-218, 247-333).
//
// Rows of at most 4096 values with 16-byte aligned operands, forward and backward, plain and SiLU-fused: one wave per row, above 2048
// values two, in batches that fill the chip (actq_fwd_wave_k, actq_bwd_wave_k), the fused forms with the gates' tables in LDS. The
// RMSNorm-fused block entry of rows of at most 1024 values: a wave per row as well, four or sixteen rows sharing the projections
// (block_entry_fwd_quad, block_entry_fwd_rows16, block_entry_bwd_quad). Everything else (longer rows, unaligned operands, small batches
// of rows above 2048 values):
// One 256-thread workgroup per row. A half-wave (32 lanes) transforms one 128-chunk: lane l holds elements 4l .. 4l + 3,
// butterfly stages 1-2 in registers, 4 .. 64 across lanes; half-wave h takes chunks h, h + 8, ... (the reference's wave h of
// 32), NR = ceil(K / 1024) rounds of them stay in registers across the row-wide reductions. Kernels are instantiated per
// NR, so a row of 2048 values runs two rounds and not the eight the limit allows.
//
// Sums of the backward pass (dL/ds, the tie count, the RMSNorm dot) follow one fixed tree: a lane adds its terms in chunk
// order with fmaf, the 32 lanes of a half-wave combine by xor 16, 8, 4, 2, 1, the eight half-wave sums are added in order.
#include "common.cuh"
#include <mutex>
#include <type_traits>

#define HSCALE 0.08837890625f      // bf16(1 / sqrt(128))

#define CAMX_EACH4(OP) OP(x) OP(y) OP(z) OP(w)

// fp32 -> bf16 -> fp32. _any: a NaN stays a NaN but its sign and payload are the hardware's (for values that only feed further
// arithmetic, where nothing but NaN-ness survives); _canon: a NaN becomes 0x7fc00000, as the stored bf16 tensors have it
CAMX_DEV f32x4 rbf4_any(f32x4 v) {
    const uint32_t a = hw_pk_bf16(v.x, v.y), b = hw_pk_bf16(v.z, v.w);
    f32x4 r;
    r.x = __builtin_bit_cast(float, a << 16); r.y = __builtin_bit_cast(float, a & 0xffff0000u);
    r.z = __builtin_bit_cast(float, b << 16); r.w = __builtin_bit_cast(float, b & 0xffff0000u);
    return r;
}
CAMX_DEV f32x4 rbf4_canon(f32x4 v) { return unpack_bf16x4(pack_f2bf_x4(v)); }
CAMX_DEV f32x4 scaled4(f32x4 v) { v.x *= HSCALE; v.y *= HSCALE; v.z *= HSCALE; v.w *= HSCALE; return v; }

// A source gives four values at element k of a row (operator()), or, for the wave-per-row kernel, eight: fetch() issues the
// loads (NW 128-bit words), value8() turns them into floats later, so that the next row's loads fly during this row's arithmetic.
CAMX_DEV void unpack_bf16x8(u32x4 w, f32x4 & a, f32x4 & b) { a = unpack_bf16x4((u32x2){w.x, w.y}); b = unpack_bf16x4((u32x2){w.z, w.w}); }
struct PlainF32 {
    static constexpr bool bf16_valued = false, lds_tables = false; static constexpr int NW = 2;
    static CAMX_DEV u32x4 absent(int) { return (u32x4){0u, 0u, 0u, 0u}; }           // what stands for the words of a chunk behind the row
    CAMX_DEV void set_small(const uint16_t *) {}
    const float * x; int K;
    CAMX_DEV f32x4 operator()(int row, int k) const { return *(const f32x4 *)(x + (size_t)row * K + k); }
    CAMX_DEV f32x4 operator()(int row, int k, u32x2 &) const { return (*this)(row, k); }
    CAMX_DEV void fetch(int row, int k, u32x4 (&w)[NW]) const { const u32x4 * p = (const u32x4 *)(x + (size_t)row * K + k); w[0] = p[0]; w[1] = p[1]; }
    CAMX_DEV u32x4 packed8(const u32x4 (&w)[NW], u32x4 &) const {                   // autocast's bf16 input
        const f32x4 a = __builtin_bit_cast(f32x4, w[0]), b = __builtin_bit_cast(f32x4, w[1]);
        return (u32x4){hw_pk_bf16(a.x, a.y), hw_pk_bf16(a.z, a.w), hw_pk_bf16(b.x, b.y), hw_pk_bf16(b.z, b.w)};
    }
};
struct PlainBF16 {
    static constexpr bool bf16_valued = true, lds_tables = false; static constexpr int NW = 1;
    static CAMX_DEV u32x4 absent(int) { return (u32x4){0u, 0u, 0u, 0u}; }           // what stands for the words of a chunk behind the row
    CAMX_DEV void set_small(const uint16_t *) {}
    const uint16_t * x; int K;
    CAMX_DEV f32x4 operator()(int row, int k) const { return unpack_bf16x4(*(const u32x2 *)(x + (size_t)row * K + k)); }
    CAMX_DEV f32x4 operator()(int row, int k, u32x2 &) const { return (*this)(row, k); }
    CAMX_DEV void fetch(int row, int k, u32x4 (&w)[NW]) const { w[0] = *(const u32x4 *)(x + (size_t)row * K + k); }
    CAMX_DEV u32x4 packed8(const u32x4 (&w)[NW], u32x4 &) const { return w[0]; }
};
// the bf16 words {t[g0], t[g1]} and {t[g2], t[g3]} of four packed bf16 gates from the full table in device memory
CAMX_DEV u32x2 silu_lookup4(u32x2 gw, const uint16_t * lut) {
    return (u32x2){(uint32_t)lut[gw.x & 0xffffu] | ((uint32_t)lut[gw.x >> 16] << 16), (uint32_t)lut[gw.y & 0xffffu] | ((uint32_t)lut[gw.y >> 16] << 16)};
}
// Byte offsets of two packed gates' entries in the 16-bit small table, for the wave-per-row kernels: the sign falls out of a shift that
// also scales the magnitude to bytes. most: the largest magnitude offset so far; SWS_LAST in it says that a gate is a zero, whose entry
// that is, or outside the table: small_outside8 then tells which (a compare per eight gates instead of four per two). 16384 x 2048 with
// half the gates zeros: forward 43.8 us, backward 96.2; 45.5 and 100.3 with zeros on the full tables' path. Chunks behind the row stand
// as gates of 1 for the same reason: 16384 x 512 32.3 and 68.5 us, as zeros 38.9 and 75.4.
constexpr uint16_t SWS_LAST = 2 * SWS_SPAN;
CAMX_DEV uint32_t small_offset2(uint32_t w, u16x2 & most) {
    const u16x2 a = __builtin_bit_cast(u16x2, w) << (u16x2){1, 1};
    const u16x2 i = __builtin_elementwise_min(a - (u16x2){(uint16_t)(2 * SWS_A0), (uint16_t)(2 * SWS_A0)}, (u16x2){SWS_LAST, SWS_LAST});      // below the table: wraps, clamps
    most = __builtin_elementwise_max(most, i);
    return ((w >> 2) & 0x20002000u) | __builtin_bit_cast(uint32_t, i);
}
// whether one of eight packed gates is not in the small table (zeros are: less one they wrap to the largest number)
CAMX_DEV bool small_outside8(u32x4 w) {
    u16x2 low = {0xffff, 0xffff}, high = {0, 0};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t wi = w[i];
        const u16x2 a = __builtin_bit_cast(u16x2, wi & 0x7fff7fffu);
        low = __builtin_elementwise_min(low, a - (u16x2){1, 1}); high = __builtin_elementwise_max(high, a);
    }
    return (low.x < SWS_A0 - 1) | (low.y < SWS_A0 - 1) | (high.x >= SWS_A0 + SWS_SPAN) | (high.y >= SWS_A0 + SWS_SPAN);
}
CAMX_DEV uint32_t small_pair(const uint16_t * small, uint32_t o) {
    return (uint32_t)*(const uint16_t *)((const uint8_t *)small + (o & 0xffffu)) | ((uint32_t)*(const uint16_t *)((const uint8_t *)small + (o >> 16)) << 16);
}
struct SiluMulSrc {
    static constexpr bool bf16_valued = true;      // the activation is rounded to bf16 as it is formed
    static constexpr bool lds_tables = true;       // the wave-per-row kernels hold the small tables in LDS
    CAMX_DEV void set_small(const uint16_t * p) { small = p; }
    const uint16_t * gu; int ld, F;
    const uint16_t * lut;                          // bf16(silu g) for every bf16 g (the table silu_mul_bf16 uses: the same activation bits)
    const uint16_t * small;                        // its small form in LDS, or null
    CAMX_DEV f32x4 operator()(int row, int k, u32x2 & keep) const {          // keep: the four bf16(silu g), for the backward's sink
        const uint16_t * r = gu + (size_t)row * ld;
        const u32x2 gw = *(const u32x2 *)(r + k);
        const f32x4 u = unpack_bf16x4(*(const u32x2 *)(r + F + k));
        keep = silu_lookup4(gw, lut);
        const f32x4 sl = unpack_bf16x4(keep);
        return rbf4_any((f32x4){sl.x * u.x, sl.y * u.y, sl.z * u.z, sl.w * u.w});      // (feeds the rotation: of a NaN only its NaN-ness survives)
    }
    CAMX_DEV f32x4 operator()(int row, int k) const { u32x2 keep; return (*this)(row, k, keep); }
    static CAMX_DEV u32x4 absent(int w) { return w ? (u32x4){0u, 0u, 0u, 0u} : (u32x4){0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u}; }      // gates of 1, multipliers of 0: +0 without a zero gate's check
    static constexpr int NW = 2;                   // the wave-per-row form: eight gates, eight multipliers
    CAMX_DEV void fetch(int row, int k, u32x4 (&w)[NW]) const { const uint16_t * r = gu + (size_t)row * ld + k; w[0] = *(const u32x4 *)r; w[1] = *(const u32x4 *)(r + F); }
    CAMX_DEV u32x4 packed8(const u32x4 (&w)[NW], u32x4 & keep) const {              // (feeds the rotation: of a NaN only its NaN-ness survives)
        u16x2 most = {0, 0};
        const uint32_t o0 = small_offset2(w[0].x, most), o1 = small_offset2(w[0].y, most), o2 = small_offset2(w[0].z, most), o3 = small_offset2(w[0].w, most);
        if (__builtin_expect(most.x == SWS_LAST || most.y == SWS_LAST, 0) && __builtin_expect(small_outside8(w[0]), 0)) {
            const u32x2 k0 = silu_lookup4((u32x2){w[0].x, w[0].y}, lut), k1 = silu_lookup4((u32x2){w[0].z, w[0].w}, lut);
            keep = (u32x4){k0.x, k0.y, k1.x, k1.y};
        } else keep = (u32x4){small_pair(small, o0), small_pair(small, o1), small_pair(small, o2), small_pair(small, o3)};
        f32x4 sa, sb, ua, ub;
        unpack_bf16x8(keep, sa, sb); unpack_bf16x8(w[1], ua, ub);
        return (u32x4){hw_pk_bf16(sa.x * ua.x, sa.y * ua.y), hw_pk_bf16(sa.z * ua.z, sa.w * ua.w), hw_pk_bf16(sb.x * ub.x, sb.y * ub.y), hw_pk_bf16(sb.z * ub.z, sb.w * ub.w)};
    }
};
struct RmsSrc {
    static constexpr bool bf16_valued = false;
    const float * x; const float * w; float rstd; int d;
    CAMX_DEV f32x4 operator()(int row, int k) const {
        const f32x4 xv = *(const f32x4 *)(x + (size_t)row * d + k), wv = *(const f32x4 *)(w + k);
        f32x4 a; a.x = xv.x * rstd * wv.x; a.y = xv.y * rstd * wv.y; a.z = xv.z * rstd * wv.z; a.w = xv.w * rstd * wv.w;
        return a;
    }
    CAMX_DEV f32x4 operator()(int row, int k, u32x2 &) const { return (*this)(row, k); }
};
// u = bf16(H128 . bf16(source)) for the NR rounds of this half-wave, which takes chunks hw, hw + 8, ..; returns the lane's max |u| over its active chunks
template <int NR, typename Src>
CAMX_DEV float actq_rotate(Src src, int row, int l, int hw, int nch, f32x4 (&u)[NR], u32x2 * keep = nullptr) {
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const int ch = hw + 8 * c;
        f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        u32x2 kp = {0u, 0u};
        if (ch < nch) v = src(row, ch * 128 + 4 * l, kp);
        if (keep) keep[c] = kp;
        u[c] = v;
    }
    float amax = 0.0f;
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const f32x4 in = Src::bf16_valued ? u[c] : rbf4_any(u[c]);                // autocast's bf16 input
        const f32x4 v = rbf4_any(scaled4(hadamard128_l4(in, l, false)));
        u[c] = v;
        if (hw + 8 * c < nch) amax = fmaxf(amax, absmax4(v));
    }
    return amax;
}

// The row's scale and what the lanes need to divide by it. For |p| < 2^k, p = u * rcp(s) (rcp: 1 ulp; one more rounding) is within
// 2.5 * 2^(k - 23) of the exact quotient and the IEEE quotient within 2^(k - 24), and half-integers are floats: when p is farther than
// their sum from every half-integer, rintf of the two agree. Rows whose quotients stay below 16 (every int4 row with clip near 1) ask
// for 1e-5 (the sum: 5.8e-6), others below 256 for 3e-4 (9.2e-5), below 4096 for 2e-3 (1.5e-3; more than eight bits, or a clip far below
// 1: 4096 x 4096 fp32 values at qmax 127 and clip 0.4 take 20.9 us, 23.9 with every lane of such a row dividing, 22.1 with the lanes
// that hold a quotient above 256). A lane that holds a closer value divides, and so does every lane of a row whose largest quotient is not
// below 4096 or not a number (an infinite amax). A NaN among the four values needs no look of its own: its p is a NaN as its quotient
// is, and the maximum passes over it. (A scale above 2^126 has a subnormal reciprocal, which may be taken as zero: |u| is at most
// HSCALE times the largest float or infinite, so the quotients of such a row are below 0.36 and round to the same zeros.)
struct RowScale {
    float s, rcp, lo, hi, most;                          // most: how far p may lie from its integer
    CAMX_DEV RowScale(float s_, float amax, int qmax) : s(s_), rcp(__builtin_amdgcn_rcpf(s_)), lo((float)(-qmax - 1)), hi((float)qmax) {
        const float p = amax * rcp;
        most = p < 16.0f ? 0.49999f : p < 256.0f ? 0.4997f : p < 4096.0f ? 0.498f : -1.0f;
    }
    // clamp(rintf(u / s), lo, hi) of four values; the median of a NaN and two numbers is the smaller number, lo, as fminf(fmaxf(NaN, lo), hi) is
    CAMX_DEV f32x4 quant4(f32x4 u) const {
        const f32x4 p = {u.x * rcp, u.y * rcp, u.z * rcp, u.w * rcp};
        f32x4 r = {rintf(p.x), rintf(p.y), rintf(p.z), rintf(p.w)};
        const float off = fmaxf(fmaxf(fabsf(p.x - r.x), fabsf(p.y - r.y)), fmaxf(fabsf(p.z - r.z), fabsf(p.w - r.w)));
        if (off > most || most < 0.0f) { r.x = rintf(u.x / s); r.y = rintf(u.y / s); r.z = rintf(u.z / s); r.w = rintf(u.w / s); }
        return (f32x4){__builtin_amdgcn_fmed3f(r.x, lo, hi), __builtin_amdgcn_fmed3f(r.y, lo, hi), __builtin_amdgcn_fmed3f(r.z, lo, hi), __builtin_amdgcn_fmed3f(r.w, lo, hi)};
    }
    // the low four bits of four quantized values, packed. For values in [-8, 7]: q + 8 is the code with its top bit turned over, and
    // the digits q + 8 of a base-16 number are summed exactly in fp32 (four multiply-adds and one conversion instead of eleven instructions)
    CAMX_DEV uint32_t nibbles4(f32x4 q) const {
        if (hi <= 7.0f) return (uint32_t)__builtin_fmaf(q.w, 4096.0f, __builtin_fmaf(q.z, 256.0f, __builtin_fmaf(q.y, 16.0f, q.x + 34952.0f))) ^ 0x8888u;
        return ((uint32_t)(int)q.x & 0xfu) | (((uint32_t)(int)q.y & 0xfu) << 4) | (((uint32_t)(int)q.z & 0xfu) << 8) | (((uint32_t)(int)q.w & 0xfu) << 12);
    }
};

// max over the wave (order-free) in row moves and four lane reads
CAMX_DEV float wave_max64(float v) {
    v = fmaxf(v, lane_xor1(v)); v = fmaxf(v, lane_xor2(v)); v = fmaxf(v, lane_xor4(v)); v = fmaxf(v, lane_xor8(v));
    return fmaxf(fmaxf(lane_read(v, 0), lane_read(v, 16)), fmaxf(lane_read(v, 32), lane_read(v, 48)));
}
// row-wide max (order-free); lds: 4 floats
CAMX_DEV float row_max(float amax, float * lds) {
    const int tid = threadIdx.x;
    amax = wave_max64(amax);
    __syncthreads();
    if ((tid & 63) == 0) lds[tid >> 6] = amax;
    __syncthreads();
    return fmaxf(fmaxf(lds[0], lds[1]), fmaxf(lds[2], lds[3]));
}

template <int NR, typename Src>
CAMX_DEV void actq_fwd_row(Src src, int row, uint16_t * __restrict__ y, float * __restrict__ s_out, int K, float clip, int qmax,
                           uint16_t * __restrict__ codes, float * lds) {
    const int tid = threadIdx.x, l = slot_of(tid) & 31, hw = tid >> 5, nch = K / 128;
    f32x4 u[NR];
    const float amax = row_max(actq_rotate<NR, Src>(src, row, l, hw, nch, u), lds);
    const float s = fmaxf(amax * clip / (float)qmax, 1e-8f);
    const RowScale rs(s, amax, qmax);
    if (tid == 0 && s_out) s_out[row] = s;
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const int ch = hw + 8 * c;
        if (ch < nch) {
            const f32x4 q = rs.quant4(u[c]);
            if (y) { f32x4 d; d.x = q.x * s; d.y = q.y * s; d.z = q.z * s; d.w = q.w * s; *(u32x2 *)(y + (size_t)row * K + ch * 128 + 4 * l) = pack_f2bf_x4(d); }
            if (codes) codes[(size_t)row * (K / 4) + ch * 32 + l] = (uint16_t)rs.nibbles4(q);
        }
    }
}

template <int NR, typename Src>
__global__ void __launch_bounds__(256) actq_fwd_k(Src src, uint16_t * y, float * s, uint16_t * codes, int K, float clip, int qmax) {
    __shared__ float lds[4];
    actq_fwd_row<NR>(src, blockIdx.x, y, s, K, clip, qmax, codes, lds);
}

// ---- rows of at most 4096 values: one wave per row, two above 2048 ----------------------------------------------------------
// Lane (g = lane >> 4, slot s of its 16) holds elements 8 s .. 8 s + 7 of one chunk per round: round j of part p of W is chunk
// 4 W j + 4 p + g, so a wave's round is 512 consecutive values and all chunks of one residue mod 8, whose dL/ds terms the backward adds
// in chunk order, sit in one lane. Butterfly stages 1, 2, 4 pair registers, 8 .. 64 pair slots s ^ 1, 2, 4, 8: the same pairs in the same
// order as above. What a value costs is counted in issue cycles, measured on the card: an add, subtract, multiply, bit operation or
// multiply-add that reads at most two vector registers takes 2.3 per wave and SIMD, everything else (shifts, converts, maxima,
// compares, row moves, an operand in a scalar register) 4.2. Hence rounds of eight values that live as packed bf16 words between the
// passes, and maxima of packed words. bf16 rows, forward / backward, against four lanes a chunk with 32 values each (up to 2048) and a
// workgroup per row, buffers cold: 32768 x 512 40.3 -> 17.0 / 66.1 -> 27.0 us, 32768 x 1024 43.5 -> 27.1 / 69.4 -> 43.0, 16384 x 2048 35.7 ->
// 28.4 / 44.5 -> 39.0 (floor 20.6 / 31.0: bytes at 6.5 TB/s), 32768 x 2048 64.6 -> 48.6 / 81.2 -> 77.0, 8192 x 4096 35.3 -> 27.8 / 51.7 ->
// 38.7; the SiLU-fused pair at 16384 x 2048 47.2 -> 42.3 / 92.1 -> 77.2 (floor 34 / 52).
CAMX_DEV void bfly(float & a, float & b) { const float s = a + b, d = a - b; a = s; b = d; }
CAMX_DEV float bf_lo(uint32_t v) { return __builtin_bit_cast(float, v << 16); }
CAMX_DEV float bf_hi(uint32_t v) { return __builtin_bit_cast(float, v & 0xffff0000u); }
CAMX_DEV void unpack8(u32x4 w, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 4; i++) { const uint32_t p = w[i]; v[2 * i] = bf_lo(p); v[2 * i + 1] = bf_hi(p); }
}
// the same words, unknown to the compiler: it would hold their unpacked values from one pass to the next (two registers for one)
CAMX_DEV u32x4 unknown_words(u32x4 w) {
    uint32_t a = w.x, b = w.y, c = w.z, d = w.w;
    asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
    return (u32x4){a, b, c, d};
}
// eight values to packed bf16 by the hardware convert: a NaN stays one (see rbf4_any)
CAMX_DEV u32x4 pack8_any(const float (&v)[8]) { return (u32x4){hw_pk_bf16(v[0], v[1]), hw_pk_bf16(v[2], v[3]), hw_pk_bf16(v[4], v[5]), hw_pk_bf16(v[6], v[7])}; }
// A batch of 2^20 values or more streams: its bf16 outputs leave past the caches as whole lines (the wave's round is 1 KiB without a gap:
// 16384 x 2048 forward 31.4 -> 26.3 us, backward 40.1 -> 36.3 with g read past them too, buffers warm). fp32 gradients stay plain: a lane's eight values
// are two half lines, which only the cache puts together (61 -> 85 us).
typedef u32x4 u32x4_a8 __attribute__((aligned(8)));                      // (the block entry's operands are 8-byte aligned, its codes 2)
typedef uint32_t u32_a2 __attribute__((aligned(2)));
CAMX_DEV void store8(u32x2 v, void * p, bool stream) {
    if (stream) { asm volatile("" ::: "memory"); __builtin_nontemporal_store(v, (u32x2 *)p); asm volatile("" ::: "memory"); }
    else *(u32x2 *)p = v;
}
CAMX_DEV void store16(u32x4 v, void * p, bool stream) {
    if (stream) {                                        // (between two empty asm statements: the compiler makes one plain store of the two otherwise)
        asm volatile("" ::: "memory");
        __builtin_nontemporal_store(v, (u32x4_a8 *)p);
        asm volatile("" ::: "memory");
    }
    else *(u32x4_a8 *)p = v;
}
CAMX_DEV u32x4 pack8_canon(const float (&v)[8]) {                     // f2bf of eight values (NaN -> 0x7fc0)
    const u32x2 a = pack_f2bf_x4((f32x4){v[0], v[1], v[2], v[3]}), b = pack_f2bf_x4((f32x4){v[4], v[5], v[6], v[7]});
    return (u32x4){a.x, a.y, b.x, b.y};
}
// A cross-lane stage gives own + partner in the lower lane and partner - own in the upper one: a sign flip and an add per value. Here the
// upper lane keeps own - partner, the negative of its value: one multiply-add by +1 or -1 whose first operand comes from the partner
// (v_fmac_f32 with a row move; the compiler does not fold the move into a multiply-add, and the s_nop gives the first move the two wait
// states it needs behind the instructions before). Negation commutes with every later sum and difference and its rounding, so after
// all stages a lane's values carry the sign of its slot's parity, which the factor HSCALE takes along. Only a zero's sign is lost:
// sums that cancel are +0 in either form, so the last multiply adds +0; a sum is -0 only if the chunk's first element is -0 and its
// second a zero, and a wave that holds such a chunk runs the plain form.
struct Lanes16 {
    float s1, s2, s4, s8, h;                             // a stage's factor of the partner, HSCALE with the parity's sign
    bool first;                                          // the lane holds its chunk's first elements
    CAMX_DEV explicit Lanes16(int s) {
        s1 = s & 1 ? -1.0f : 1.0f; s2 = s & 2 ? -1.0f : 1.0f; s4 = s & 4 ? -1.0f : 1.0f; s8 = s & 8 ? -1.0f : 1.0f;
        h = (__builtin_popcount(s) & 1) ? -HSCALE : HSCALE;
        first = s == 0;
    }
    CAMX_DEV bool plain(uint32_t w0) const { return first && (w0 & 0x7fffffffu) == 0x00008000u; }          // elements 0 and 1: -0 and a zero
};
template <int CTRL>
CAMX_DEV void lane_stage8(float (&u)[8], float sg) {      // (own + partner) in the lower lane, (partner - own) in the upper one
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const float own = u[k];
        const float p = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, own), CTRL, 0xf, 0xf, true));
        u[k] = p + __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, own) ^ (__builtin_bit_cast(uint32_t, sg) & 0x80000000u));
    }
}
#define CAMX_FMAC8(CTRL, SG) \
    "v_fmac_f32_dpp %0, %0, " SG " " CTRL " row_mask:0xf bank_mask:0xf\n\tv_fmac_f32_dpp %1, %1, " SG " " CTRL " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f32_dpp %2, %2, " SG " " CTRL " row_mask:0xf bank_mask:0xf\n\tv_fmac_f32_dpp %3, %3, " SG " " CTRL " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f32_dpp %4, %4, " SG " " CTRL " row_mask:0xf bank_mask:0xf\n\tv_fmac_f32_dpp %5, %5, " SG " " CTRL " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f32_dpp %6, %6, " SG " " CTRL " row_mask:0xf bank_mask:0xf\n\tv_fmac_f32_dpp %7, %7, " SG " " CTRL " row_mask:0xf bank_mask:0xf\n\t"
// v = HSCALE . H128 of the chunk's packed bf16 values; plain: wave-uniform
CAMX_DEV void rotate128_w16(u32x4 w, float (&v)[8], const Lanes16 & ln, bool plain) {
    unpack8(w, v);
#pragma unroll
    for (int k = 0; k < 8; k += 2) bfly(v[k], v[k + 1]);
#pragma unroll
    for (int k = 0; k < 8; k += 4) { bfly(v[k], v[k + 2]); bfly(v[k + 1], v[k + 3]); }
#pragma unroll
    for (int k = 0; k < 4; k++) bfly(v[k], v[k + 4]);
    if (__builtin_expect(plain, 0)) {
        lane_stage8<0xB1>(v, ln.s1); lane_stage8<0x4E>(v, ln.s2); lane_stage8<0x141>(v, ln.s4); lane_stage8<0x128>(v, ln.s8);
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] *= HSCALE;
    } else {
        asm("s_nop 1\n\t" CAMX_FMAC8("quad_perm:[1,0,3,2]", "%8") CAMX_FMAC8("quad_perm:[2,3,0,1]", "%9") CAMX_FMAC8("row_half_mirror", "%10") CAMX_FMAC8("row_ror:8", "%11")
            : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]) : "v"(ln.s1), "v"(ln.s2), "v"(ln.s4), "v"(ln.s8));
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = __builtin_fmaf(v[k], ln.h, 0.0f);
    }
}
// the larger magnitude of two packed bf16 pairs, per half (a NaN's is the largest of all)
CAMX_DEV u16x2 absmax_pk(u16x2 m, uint32_t w) { return __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, w & 0x7fff7fffu)); }
CAMX_DEV u16x2 absmax_pk8(u32x4 w) { return absmax_pk(absmax_pk(absmax_pk(__builtin_bit_cast(u16x2, w.x & 0x7fff7fffu), w.y), w.z), w.w); }
CAMX_DEV float absmax_of(u16x2 m) { const uint32_t a = m.x, b = m.y; return __builtin_bit_cast(float, (a > b ? a : b) << 16); }
// max |u| of a row's packed words without its NaNs, and whether it holds one (wave-uniform)
template <int R>
CAMX_DEV float row_absmax_w(const u32x4 (&uw)[R], u16x2 most, bool & nan) {
    float m = absmax_of(most);
    nan = __builtin_amdgcn_ballot_w64(m != m) != 0;
    if (__builtin_expect(nan, 0)) {
        m = 0.0f;
#pragma unroll
        for (int j = 0; j < R; j++) {
            float v[8];
            unpack8(unknown_words(uw[j]), v);
#pragma unroll
            for (int k = 0; k < 8; k++) m = fmaxf(m, fabsf(v[k]));
        }
    }
    return wave_max64(m);
}
// the same over the two waves of a row, whose signs carry the NaNs; xch: four floats
template <int W>
CAMX_DEV float share_absmax(float amax, bool & nan, float * xch, int wave) {
    if (W == 1) return amax;
    if ((threadIdx.x & 63) == 0) xch[wave] = nan ? -amax : amax;         // (-0 for a row of NaNs)
    __syncthreads();
    const float a = xch[wave & ~1], b = xch[wave | 1];
    nan = __builtin_signbit(a) || __builtin_signbit(b);
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, fmaxf(fabsf(a), fabsf(b)))));
}
// u = bf16(H128 . bf16(source)) of the lane's rounds as packed words, from the fetched words; returns the lane's largest magnitudes
template <int R, typename Src>
CAMX_DEV u16x2 actq_rotate_w(const Src & src, const u32x4 (&raw)[R][Src::NW], const Lanes16 & ln, u32x4 (&uw)[R], u32x4 (&keep)[R]) {
    u16x2 most = {0, 0};
    bool zero = false;
#pragma unroll
    for (int j = 0; j < R; j++) { uw[j] = src.packed8(raw[j], keep[j]); zero |= ln.plain(uw[j].x); }
    const bool plain = __builtin_amdgcn_ballot_w64(zero) != 0;
#pragma unroll
    for (int j = 0; j < R; j++) {
        float v[8];
        rotate128_w16(uw[j], v, ln, plain);
        uw[j] = pack8_any(v);
        uw[j] = unknown_words(uw[j]);
        const u16x2 m = absmax_pk8(uw[j]);               // (an absent chunk holds zeros)
        most = __builtin_elementwise_max(most, m);
        __builtin_amdgcn_sched_barrier(0);               // (round by round: side by side they cost a wave per SIMD in registers)
    }
    return most;
}
// A chunk behind the row reads the row's first one and is replaced afterwards: a load under a condition ends in a copy of its result, and so in a wait for
// everything requested so far, before the next request goes out.
template <int R, int W, typename Src>
CAMX_DEV void fetch_row_w(const Src & src, int row, int e0, bool last_on, u32x4 (&raw)[R][Src::NW]) {
#pragma unroll
    for (int j = 0; j < R; j++) src.fetch(row, j < R - 1 || last_on ? e0 + 512 * W * j : e0 & 127, raw[j]);
}
template <int R, typename Src>
CAMX_DEV void absent_chunk_w(const Src &, bool last_on, u32x4 (&raw)[R][Src::NW]) {
#pragma unroll
    for (int w = 0; w < Src::NW; w++) {
        const u32x4 none = Src::absent(w);
        raw[R - 1][w] = (u32x4){last_on ? raw[R - 1][w].x : none.x, last_on ? raw[R - 1][w].y : none.y, last_on ? raw[R - 1][w].z : none.z, last_on ? raw[R - 1][w].w : none.w};
    }
}

// a table into LDS, 16 bytes per lane straight from device memory
CAMX_DEV void lds_table_copy(const void * src, void * dst, int bytes) {          // bytes % 1024 == 0; all four waves
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int j = wave; j < bytes / 1024; j += 4)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)((const uint8_t *)src + 1024 * j + 16 * lane),
                                         (__attribute__((address_space(3))) void *)((uint8_t *)dst + 1024 * j), 16, 0, 0);
}
// the values and codes of a row (or a wave's part of it) from its packed rotated words; y, codes: the row's, or null
template <int R, int W>
CAMX_DEV void quantize_row_w(const u32x4 (&uw)[R], float amax, float s, int qmax, int e0, bool last_on, uint16_t * y, uint16_t * codes, bool stream) {
    const RowScale rs(s, amax, qmax);
#pragma unroll
    for (int j = 0; j < R; j++) {
        if (j == R - 1 && !last_on) break;
        float q[8];
        unpack8(uw[j], q);
        const f32x4 a = rs.quant4((f32x4){q[0], q[1], q[2], q[3]}), b = rs.quant4((f32x4){q[4], q[5], q[6], q[7]});
        const int e = e0 + 512 * W * j;
        if (codes) *(u32_a2 *)(codes + (e >> 2)) = rs.nibbles4(a) | (rs.nibbles4(b) << 16);
        if (y) {
            const float v[8] = {a.x * s, a.y * s, a.z * s, a.w * s, b.x * s, b.y * s, b.z * s, b.w * s};
            store16(pack8_canon(v), y + e, stream);
        }
    }
}
// The kernel's time at 8192 rows and more is the larger of its arithmetic and its bytes, plus the launch's ramp; a wave that walks several
// rows with the next row's loads in flight measured 5 to 15 % slower.
template <typename Src, int R, int W>
__global__ void __launch_bounds__(256) actq_fwd_wave_k(Src src, uint16_t * __restrict__ y, float * __restrict__ s_out, uint16_t * __restrict__ codes,
                                                       int K, float clip, int qmax, int M, bool stream, const uint16_t * small_g = nullptr) {
    const int lane = threadIdx.x & 63, slot = slot_of(lane) & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), part = wave % W;
    const int c0 = 4 * part + (lane >> 4), e0 = 128 * c0 + 8 * slot;     // round j: + 512 W j
    const bool last_on = c0 + 4 * W * (R - 1) < K / 128;
    const int row = blockIdx.x * (4 / W) + wave / W;
    if (!Src::lds_tables && W == 1 && row >= M) return;
    u32x4 raw[R][Src::NW];
    fetch_row_w<R, W>(src, min(row, M - 1), e0, last_on, raw);
    if (Src::lds_tables) {                               // the gates' table, shared by the workgroup's rows
        __shared__ __attribute__((aligned(16))) uint16_t small[SWS_TAB];
        lds_table_copy(small_g, small, 2 * SWS_TAB);
        __builtin_amdgcn_s_waitcnt(0x0f70);              // vmcnt(0): this wave's part of the table (and its row)
        __syncthreads();
        src.set_small(small);
        if (W == 1 && row >= M) return;
    }
    __shared__ float xch[4];
    absent_chunk_w<R>(src, last_on, raw);
    const Lanes16 ln(slot);
    u32x4 uw[R], keep[R];                                // (keep: only the backward uses it)
    const u16x2 most = actq_rotate_w<R>(src, raw, ln, uw, keep);
    bool nan;
    float amax = row_absmax_w<R>(uw, most, nan);
    amax = share_absmax<W>(amax, nan, xch, wave);
    if (W > 1 && row >= M) return;
    const float s = fmaxf(amax * clip / (float)qmax, 1e-8f);
    if (lane == 0 && part == 0 && s_out) s_out[row] = s;
    quantize_row_w<R, W>(uw, amax, s, qmax, e0, last_on, y ? y + (size_t)row * K : nullptr, codes ? codes + (size_t)row * (K / 4) : nullptr, stream);
}

// ---- backward ----------------------------------------------------------------------------------------------------------------
// sum over the 32 lanes of a half-wave by xor 16, 8, 4, 2, 1 (slot space), then the eight half-wave sums in order
CAMX_DEV float half32_sum(float v) {
    v += lane_xor16(v); v += lane_xor8(v); v += lane_xor4(v); v += lane_xor2(v); v += lane_xor1(v);
    return v;
}
CAMX_DEV void block8_sum2(float & a, float & b, float * lds16) {
    const int tid = threadIdx.x;
    a = half32_sum(a); b = half32_sum(b);
    __syncthreads();
    if ((tid & 31) == 0) { lds16[tid >> 5] = a; lds16[8 + (tid >> 5)] = b; }
    __syncthreads();
    a = lds16[0]; b = lds16[8];
#pragma unroll
    for (int w = 1; w < 8; w++) { a += lds16[w]; b += lds16[8 + w]; }
}

// u / s for a row's values (bf16 numbers), s the row's scale (>= 1e-8): with r1 = 1 / s correctly rounded, t0 = u r1, its residual
// u - s t0 (exact) and t0 + residual r1 is the correctly rounded quotient for every pair of a bf16 and an fp32 significand (all 2^30
// checked on a CPU). Taken when s and max |u| / s are at most 2^60 and the lane's four t0 are at least 2^-60 in magnitude, so that
// nothing is out of range and no residual loses bits; other lanes divide (a zero among them: its quotient is the zero).
struct RowDiv {
    float s, r1; bool row_ok;
    CAMX_DEV RowDiv(float s_, float amax) : s(s_), r1(1.0f / s_) { row_ok = s_ >= 0x1p-60f && s_ <= 0x1p60f && amax * r1 <= 0x1p60f; }
    CAMX_DEV f32x4 div4(f32x4 u, bool needed = true) const {       // needed: false in a lane whose values are padding
        f32x4 t, t0 = {u.x * r1, u.y * r1, u.z * r1, u.w * r1};
#define T_(e) t.e = __builtin_fmaf(__builtin_fmaf(-s, t0.e, u.e), r1, t0.e);
        CAMX_EACH4(T_)
#undef T_
        const float least = fminf(fminf(fabsf(t0.x), fabsf(t0.y)), fminf(fabsf(t0.z), fabsf(t0.w)));     // (a NaN quotient is a NaN either way)
        if (needed && !(row_ok && least >= 0x1p-60f)) { t.x = u.x / s; t.y = u.y / s; t.z = u.z / s; t.w = u.w / s; }
        return t;
    }
    // the same of eight values, but for the sign of a zero quotient, which u = 0 does not ask to be divided for
    CAMX_DEV void div8(const float (&u)[8], float (&t)[8], bool needed) const {
        float least = 0x1p60f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float t0 = u[k] * r1;
            t[k] = __builtin_fmaf(__builtin_fmaf(-s, t0, u[k]), r1, t0);
            least = fminf(least, fabsf(t0));
        }
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(needed && !(row_ok && least >= 0x1p-60f)) != 0, 0)) {
            bool divide = !row_ok;
#pragma unroll
            for (int k = 0; k < 8; k++) divide |= u[k] != 0.0f && fabsf(u[k] * r1) < 0x1p-60f;
            if (__builtin_amdgcn_ballot_w64(needed && divide) != 0) {
#pragma unroll
                for (int k = 0; k < 8; k++) { const float d = u[k] / s; t[k] = divide ? d : t[k]; }
            }
        }
    }
};
// The straight-through step of one value: r = rintf(t), q its clamp to [lo, hi], m: r lies strictly inside. Gives the factor of g in
// dL/ds, m ? q - t : q, and m as 1 or 0.
struct Ste {
    float lo, hi, lo1, hi1;
    CAMX_DEV Ste(int qmax) : lo((float)(-qmax - 1)), hi((float)qmax), lo1((float)-qmax), hi1((float)(qmax - 1)) {}
    CAMX_DEV float operator()(float t, float & m) const {
        const float r = rintf(t), q = __builtin_amdgcn_fmed3f(r, lo, hi);              // (a NaN: lo, as fminf(fmaxf(NaN, lo), hi))
        const bool in = __builtin_amdgcn_fmed3f(r, lo1, hi1) == r;                      // lo < r < hi of an integer; false for a NaN
        m = in ? 1.0f : 0.0f;
        return q - (in ? t : 0.0f);
    }
};

// st8: eight values before their rounding to bf16, the wave-per-row kernel's form
struct SinkF32 {
    float * dx; int K;
    CAMX_DEV void operator()(int row, int k, f32x4 v, u32x2) const { *(f32x4 *)(dx + (size_t)row * K + k) = v; }
    CAMX_DEV void st8(int row, int k, const float (&v)[8], u32x4, bool) const {
        f32x4 * p = (f32x4 *)(dx + (size_t)row * K + k);
        p[0] = rbf4_canon((f32x4){v[0], v[1], v[2], v[3]}); p[1] = rbf4_canon((f32x4){v[4], v[5], v[6], v[7]});
    }
    CAMX_DEV void set_small(const float *) {}
};
struct SinkBF16 {
    uint16_t * dx; int K;
    CAMX_DEV void operator()(int row, int k, f32x4 v, u32x2) const { *(u32x2 *)(dx + (size_t)row * K + k) = pack_f2bf_x4(v); }
    CAMX_DEV void st8(int row, int k, const float (&v)[8], u32x4, bool stream) const { store16(pack8_canon(v), dx + (size_t)row * K + k, stream); }
    CAMX_DEV void set_small(const float *) {}
};
struct SinkLds { float * buf; CAMX_DEV void operator()(int, int k, f32x4 v, u32x2) const { *(f32x4 *)(buf + k) = v; } };
// dact back through act = bf16(bf16(silu g) * u): each product rounded to bf16, then silu's derivative
// ds * sig * fma(g, 1 - sig, 1), into dgu = [dg | du] rows of 2F. g is a bf16 value, so sig = 1 / (1 + expf(-g))
// is read from a table of all 65536 of them (filled on first use from the correctly rounded expf): one 4-byte load in place of an
// exponential and a division per value; the wave-per-row kernel holds the table's small form in LDS. (A table in device memory
// that also holds the fma doubles the entry, and the values in use no longer stay in the first-level cache: 15 % slower than
// no table at all.)
__device__ __attribute__((aligned(16))) float g_dsilu_lut[65536];
__device__ __attribute__((aligned(16))) float g_dsilu_small[SWS_TAB];            // the small form, for LDS
__global__ void __launch_bounds__(256) dsilu_lut_fill() {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    const float g = bf2f((uint16_t)i), ex = (float)exp(-(double)g), sig = 1.0f / (1.0f + ex);
    g_dsilu_lut[i] = sig;
}
__global__ void __launch_bounds__(256) dsilu_small_fill() {              // after dsilu_lut_fill, on the same stream
    const uint32_t e = blockIdx.x * 256 + threadIdx.x;
    if (e >= SWS_TAB) return;
    const uint32_t sign = e >> 12, i = e & SWS_SPAN;
    g_dsilu_small[e] = g_dsilu_lut[i == SWS_SPAN ? sign << 15 : (sign << 15) | (SWS_A0 + i)];
}
struct SinkSiluMul {
    const uint16_t * gu; int ld, F; uint16_t * dgu; const float * dlut;
    const float * dsmall;                          // the small sigmoid table in LDS, or null
    CAMX_DEV void set_small(const float * p) { dsmall = p; }
    CAMX_DEV void operator()(int row, int k, f32x4 dact, u32x2 keep) const {      // keep: the source's four bf16(silu g)
        const uint16_t * r = gu + (size_t)row * ld;
        u32x2 dgp, dup;
        grads4(*(const u32x2 *)(r + k), *(const u32x2 *)(r + F + k), keep, dact, dgp, dup);
        uint16_t * o = dgu + (size_t)row * (2 * F);
        *(u32x2 *)(o + k) = dgp;
        *(u32x2 *)(o + F + k) = dup;
    }
    // four values' dg and du from their gates, multipliers, bf16(silu g) and dact
    CAMX_DEV void grads4(u32x2 gw, u32x2 uw, u32x2 keep, f32x4 dact, u32x2 & dgp, u32x2 & dup) const { grads4(gw, uw, keep, dact, sigmoids4(gw), dgp, dup); }
    CAMX_DEV f32x4 sigmoids4(u32x2 gw) const { return (f32x4){dlut[gw.x & 0xffffu], dlut[gw.x >> 16], dlut[gw.y & 0xffffu], dlut[gw.y >> 16]}; }
    CAMX_DEV float small_at(uint32_t o) const { return *(const float *)((const uint8_t *)dsmall + o); }
    CAMX_DEV f32x4 small4(uint32_t o0, uint32_t o1) const {               // from the byte offsets into the 16-bit table
        const uint32_t a = o0 << 1, b = o1 << 1;                          // (the offsets use 14 bits of each half)
        return (f32x4){small_at(a & 0xffffu), small_at(a >> 16), small_at(b & 0xffffu), small_at(b >> 16)};
    }
    CAMX_DEV void grads4(u32x2 gw, u32x2 uw, u32x2 keep, f32x4 dact, f32x4 sig, u32x2 & dgp, u32x2 & dup) const {
        const f32x4 g = unpack_bf16x4(gw), u = unpack_bf16x4(uw), sl4 = unpack_bf16x4(keep);
        const f32x4 ds = rbf4_any((f32x4){dact.x * u.x, dact.y * u.y, dact.z * u.z, dact.w * u.w});       // (a NaN's bits are settled by the store's rounding)
        f32x4 dg, du;
#define S_(e) { du.e = dact.e * sl4.e; dg.e = ds.e * sig.e * __builtin_fmaf(g.e, 1.0f - sig.e, 1.0f); }
        CAMX_EACH4(S_)
#undef S_
        dgp = pack_f2bf_x4(dg); dup = pack_f2bf_x4(du);
    }
    // (the gates and multipliers are read a second time here: held in registers since the source fetched them they cost 48 more,
    // two waves per SIMD instead of three: 8192 x 2048 65 us instead of 62 in the layout of four values a lane, 41.6 in this one)
    CAMX_DEV void st8(int row, int k, const float (&v)[8], u32x4 keep, bool stream) const {
        const f32x4 a = {v[0], v[1], v[2], v[3]}, b = {v[4], v[5], v[6], v[7]};
        const uint16_t * r = gu + (size_t)row * ld + k;
        const u32x4 gw = *(const u32x4 *)r, uw = *(const u32x4 *)(r + F);
        u32x2 dg0, du0, dg1, du1;
        u16x2 most = {0, 0};
        const uint32_t o0 = small_offset2(gw.x, most), o1 = small_offset2(gw.y, most), o2 = small_offset2(gw.z, most), o3 = small_offset2(gw.w, most);
        f32x4 s0 = small4(o0, o1), s1 = small4(o2, o3);
        if (__builtin_expect(most.x == SWS_LAST || most.y == SWS_LAST, 0) && small_outside8(gw)) { s0 = sigmoids4((u32x2){gw.x, gw.y}); s1 = sigmoids4((u32x2){gw.z, gw.w}); }
        grads4((u32x2){gw.x, gw.y}, (u32x2){uw.x, uw.y}, (u32x2){keep.x, keep.y}, rbf4_any(a), s0, dg0, du0);      // (a NaN's bits are settled by the stores' rounding)
        grads4((u32x2){gw.z, gw.w}, (u32x2){uw.z, uw.w}, (u32x2){keep.z, keep.w}, rbf4_any(b), s1, dg1, du1);
        uint16_t * o = dgu + (size_t)row * (2 * F) + k;
        store16((u32x4){dg0.x, dg0.y, dg1.x, dg1.y}, o, stream);
        store16((u32x4){du0.x, du0.y, du1.x, du1.y}, o + F, stream);
    }
};

// lds16: 16 floats. sink receives bf16-valued floats: the gradient of the bf16 source, before any widening store.
template <int NR, typename Src, typename Sink>
CAMX_DEV void actq_bwd_row(Src src, int row, const uint16_t * __restrict__ g, Sink sink, int K, float clip, int qmax, float * lds16) {
    const int tid = threadIdx.x, l = slot_of(tid) & 31, hw = tid >> 5, nch = K / 128;
    f32x4 u[NR], gv[NR];
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const int ch = hw + 8 * c;
        u32x2 raw = {0u, 0u};
        if (ch < nch) raw = *(const u32x2 *)(g + (size_t)row * K + ch * 128 + 4 * l);
        gv[c] = unpack_bf16x4(raw);
    }
    u32x2 keep[NR];                                      // what the source hands to the sink (the fused SiLU form only)
    const float amax = row_max(actq_rotate<NR, Src>(src, row, l, hw, nch, u, keep), lds16);
    const float s_raw = amax * clip / (float)qmax, s = fmaxf(s_raw, 1e-8f);
    const Ste ste(qmax);
    // dL/ds = sum g (q - m t) and the number of max-|u| elements; m: the rounded value lies strictly inside (lo, hi). The
    // straight-through part g m is formed here (g is not needed afterwards); the ties are counted from the compares' lane masks
    // on the scalar unit, one counter per half-wave (a count is exact in any order).
    const RowDiv rd(s, amax);
    float dlds = 0.0f;
    int ties_lo = 0, ties_hi = 0;
    uint32_t tied = 0;                                   // bit c: some lane of this wave holds a max-|u| element in round c
#pragma unroll
    for (int c = 0; c < NR; c++) {
        if (hw + 8 * c < nch) {
            const f32x4 t4 = rd.div4(u[c]);
#define D_(e) { float m; const float x = ste(t4.e, m); dlds = __builtin_fmaf(gv[c].e, x, dlds); gv[c].e = gv[c].e * m; }
            CAMX_EACH4(D_)
#undef D_
#define T_(e) { const uint64_t tie = __builtin_amdgcn_ballot_w64(fabsf(u[c].e) == amax); any |= tie; \
                ties_lo += __builtin_popcount((uint32_t)tie); ties_hi += __builtin_popcount((uint32_t)(tie >> 32)); }
            uint64_t any = 0;
            // (a look whether the round holds such an element at all costs up to five registers here, a wave per SIMD at several widths: 8192 rows
            // of 7168 bf16 values 102.6 us with it, 94.2 without, fused 8192 x 6144 186 and 173)
            CAMX_EACH4(T_)
#undef T_
            if (any) tied |= 1u << c;
        }
    }
    float ties = (tid & 31) == 0 ? (float)((tid & 32) ? ties_hi : ties_lo) : 0.0f;
    block8_sum2(dlds, ties, lds16);
    const float coef = s_raw >= 1e-8f ? dlds * clip / (float)qmax / ties : 0.0f;
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const int ch = hw + 8 * c;
        if (ch < nch) {
            f32x4 d = gv[c];
            if (tied & (1u << c)) {                      // wave-uniform: a row has few such elements, most rounds skip this
#define V_(e) if (fabsf(u[c].e) == amax && u[c].e != 0.0f) d.e += u[c].e > 0.0f ? coef : -coef;
                CAMX_EACH4(V_)
#undef V_
            }
            const f32x4 r = rbf4_canon(scaled4(hadamard128_l4(rbf4_any(d), l, false)));      // rbf4_any: the gradient of the bf16 tensor u
            sink(row, ch * 128 + 4 * l, r, keep[c]);
        }
    }
}

template <int NR, typename Src, typename Sink>
__global__ void __launch_bounds__(256) actq_bwd_k(Src src, const uint16_t * g, Sink sink, int K, float clip, int qmax) {
    __shared__ float lds[16];
    actq_bwd_row<NR>(src, blockIdx.x, g, sink, K, clip, qmax, lds);
}

// ---- backward of rows of at most 4096 values: a wave or two per row, in the layout of actq_fwd_wave_k --------------------------------
// The sum of dL/ds keeps the tree of the workgroup form. There, the lane of half-wave h with index l adds the terms of elements
// 4 l .. 4 l + 3 of chunks h, h + 8, .. in order; here those sit in one lane (slot l >> 1) as registers 4 (l & 1) .. + 3 of its rounds: of every
// second round in a row of one wave, whose other rounds are chunks h + 4, of every round in a row of two. The 32 sums of a half-wave
// then combine by l ^ 16, 8, 4, 2 (slots) and 1 (registers), and the eight half-wave sums are added in order.
// Eight values at a time, as packed words between the passes: a group in which no lane's quotient can round to qmax (or below -qmax) and no
// lane holds the row's maximum needs no clamp, no mask and no look for ties, and its part of the gradient is g itself.
struct PairShare { float amax[4], sums[4][4]; int counts[4]; };          // what the two waves of a row hand each other
// g (packed, the gradient of the quantized values) becomes the gradient of the rotated values u (packed); returns whether a chunk's rotation
// has to keep a negative zero (see Lanes16)
template <int R, int W>
CAMX_DEV bool quantize_bwd_w(const u32x4 (&uw)[R], u32x4 (&gw)[R], float amax, bool nan, float clip, int qmax, const Lanes16 & ln, bool last_on, int wave, PairShare & x) {
    const int lane = threadIdx.x & 63;
    const float s_raw = amax * clip / (float)qmax, s = fmaxf(s_raw, 1e-8f);
    const Ste ste(qmax);
    const RowDiv rd(s, amax);
    // a group's largest quotient that leaves it alone: below qmax - 1/2 by more than its rounding (qmax up to 1024); none in a row with a NaN
    const float calm = nan || qmax > 1024 ? -1.0f : ste.hi - 0.51f;
    constexpr int NC = W == 1 && R > 1 ? 2 : 1;          // chains of rounds
    float acc[NC][2];                                    // the reference lanes' sums of dL/ds terms
#pragma unroll
    for (int c = 0; c < NC; c++) acc[c][0] = acc[c][1] = 0.0f;
    int ties_n = 0;
    uint32_t tied = 0;                                   // bit j: group j holds a max-|u| element in some lane
#pragma unroll
    for (int j = 0; j < R; j++) {
        const bool on = j < R - 1 || last_on;
        float u[8], gv[8], t[8], v[8];
        unpack8(unknown_words(uw[j]), u); unpack8(unknown_words(gw[j]), gv);
        rd.div8(u, t, on);
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = rintf(t[k]) - t[k];
        const float gm = absmax_of(absmax_pk8(uw[j]));
        if (__builtin_amdgcn_ballot_w64(on && (!(gm * rd.r1 < calm) || gm == amax)) != 0) {
            float m[8];
#pragma unroll
            for (int k = 0; k < 8; k++) { v[k] = ste(t[k], m[k]); m[k] *= gv[k]; }
            gw[j] = pack8_any(m);                        // (the products are bf16 values)
            int n = 0;
#pragma unroll
            for (int k = 0; k < 8; k++) n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(on && fabsf(u[k]) == amax));
            ties_n += n;
            if (n) tied |= 1u << j;
        }
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            float a = acc[j % NC][kk];
#pragma unroll
            for (int e = 0; e < 4; e++) a = __builtin_fmaf(gv[4 * kk + e], v[4 * kk + e], a);
            a = on ? a : acc[j % NC][kk];
            asm volatile("" : "+v"(a));                  // (here, not behind the last group with every group's values kept until then)
            acc[j % NC][kk] = a;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    float dlds;
    {
        float d[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) {
            float a = acc[c][0], b = acc[c][1];
            a += lane_xor8(a); b += lane_xor8(b);                        // l ^ 16
            a += lane_xor4(a); b += lane_xor4(b);                        // l ^ 8
            a += lane_xor2(a); b += lane_xor2(b);                        // l ^ 4
            a += lane_xor1(a); b += lane_xor1(b);                        // l ^ 2
            d[c] = a + b;                                                // l ^ 1
        }
        if (W == 1) {                                    // half-wave h: chain h >> 2, lanes 16 (h & 3) .. + 15
            dlds = lane_read(d[0], 0);
#pragma unroll
            for (int h = 1; h < 4 * NC; h++) dlds += lane_read(d[h >> 2], 16 * (h & 3));
            if (NC == 1) dlds += 0.0f;                   // (the absent half-waves' sums)
        } else {                                         // half-wave h: part h >> 2
            if ((lane & 15) == 0) x.sums[wave][lane >> 4] = d[0];
            if (lane == 0) x.counts[wave] = ties_n;
            __syncthreads();
            const float * sp = x.sums[wave & ~1];
            dlds = sp[0];
#pragma unroll
            for (int h = 1; h < 8; h++) dlds += sp[h];
            ties_n = x.counts[wave & ~1] + x.counts[wave | 1];
        }
    }
    const float coef = s_raw >= 1e-8f ? dlds * clip / (float)qmax / (float)ties_n : 0.0f;
    bool zero = false;
#pragma unroll
    for (int j = 0; j < R; j++) {
        if (__builtin_expect(tied & (1u << j), 0)) {     // wave-uniform: a row has few such elements
            float u[8], d[8];
            unpack8(unknown_words(uw[j]), u); unpack8(unknown_words(gw[j]), d);
#pragma unroll
            for (int k = 0; k < 8; k++)
                if ((j < R - 1 || last_on) && fabsf(u[k]) == amax && u[k] != 0.0f) d[k] += u[k] > 0.0f ? coef : -coef;
            gw[j] = pack8_any(d);                        // the gradient of the bf16 tensor u
        }
        zero |= ln.plain(gw[j].x);
    }
    return __builtin_amdgcn_ballot_w64(zero) != 0;
}
template <typename Src, typename Sink, int R, int W>
__global__ void __launch_bounds__(256) actq_bwd_wave_k(Src src, const uint16_t * __restrict__ g, Sink sink, int K, float clip, int qmax, int M, bool stream,
                                                       const uint16_t * small_g = nullptr, const float * dsmall_g = nullptr) {
    const int lane = threadIdx.x & 63, slot = slot_of(lane) & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), part = wave % W;
    const int c0 = 4 * part + (lane >> 4), e0 = 128 * c0 + 8 * slot;     // round j: + 512 W j
    const bool last_on = c0 + 4 * W * (R - 1) < K / 128;
    const int row_raw = blockIdx.x * (4 / W) + wave / W;
    if (!Src::lds_tables && W == 1 && row_raw >= M) return;
    const int row = min(row_raw, M - 1);
    u32x4 raw[R][Src::NW], gw[R];
    fetch_row_w<R, W>(src, row, e0, last_on, raw);
#pragma unroll
    for (int j = 0; j < R; j++) gw[j] = __builtin_nontemporal_load((const u32x4 *)(g + (size_t)row * K + (j < R - 1 || last_on ? e0 + 512 * W * j : e0 & 127)));
    if (Src::lds_tables) {                               // the gates' tables, shared by the workgroup's rows
        __shared__ __attribute__((aligned(16))) uint16_t small[SWS_TAB];
        __shared__ __attribute__((aligned(16))) float dsmall[SWS_TAB];
        lds_table_copy(small_g, small, 2 * SWS_TAB);
        lds_table_copy(dsmall_g, dsmall, 4 * SWS_TAB);
        __builtin_amdgcn_s_waitcnt(0x0f70);              // vmcnt(0): this wave's part of the tables (and its row)
        __syncthreads();
        src.set_small(small); sink.set_small(dsmall);
        if (W == 1 && row_raw >= M) return;
    }
    __shared__ PairShare share;
    absent_chunk_w<R>(src, last_on, raw);
    gw[R - 1] = (u32x4){last_on ? gw[R - 1].x : 0u, last_on ? gw[R - 1].y : 0u, last_on ? gw[R - 1].z : 0u, last_on ? gw[R - 1].w : 0u};
    const Lanes16 ln(slot);
    u32x4 uw[R], keep[R];
    const u16x2 most = actq_rotate_w<R>(src, raw, ln, uw, keep);
    bool nan;
    float amax = row_absmax_w<R>(uw, most, nan);
    amax = share_absmax<W>(amax, nan, share.amax, wave);
    const bool plain = quantize_bwd_w<R, W>(uw, gw, amax, nan, clip, qmax, ln, last_on, wave, share);
    if (W > 1 && row_raw >= M) return;
#pragma unroll
    for (int j = 0; j < R; j++) {
        float d[8];
        rotate128_w16(gw[j], d, ln, plain);
        if (j == R - 1 && !last_on) break;
        sink.st8(row, e0 + 512 * W * j, d, keep[j], stream);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// ---- block entry: h = RMSNorm(x) never materialized ------------------------------------------------------------------------
// row sum under the 256-thread tree, computed by the first wave (elements 256 j + 4 lane + k), result to all threads
template <typename F>
CAMX_DEV float row_tree_sum(F term, int d, float * slot) {
    if (threadIdx.x < 64) {
        const int lane = slot_of(threadIdx.x);
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int base = 0; base < d; base += 256) {
            const int k = base + 4 * lane;
            if (k < d) { const f32x4 a = term(k), b = term.other(k); acc.x = __builtin_fmaf(a.x, b.x, acc.x); acc.y = __builtin_fmaf(a.y, b.y, acc.y);
                         acc.z = __builtin_fmaf(a.z, b.z, acc.z); acc.w = __builtin_fmaf(a.w, b.w, acc.w); }
        }
        const float tot = wave_groups_in_order(group32_sum(acc));
        if (lane == 0) *slot = tot;
    }
    __syncthreads();
    const float r = *slot;
    __syncthreads();
    return r;
}
struct SqTerm { const float * x; CAMX_DEV f32x4 operator()(int k) const { return *(const f32x4 *)(x + k); } CAMX_DEV f32x4 other(int k) const { return *(const f32x4 *)(x + k); } };
struct AbTerm {
    const float * x; const float * w; float rstd; const uint16_t * wab;
    CAMX_DEV f32x4 operator()(int k) const {
        const f32x4 xv = *(const f32x4 *)(x + k), wv = *(const f32x4 *)(w + k);
        f32x4 a; a.x = rbf(xv.x * rstd * wv.x); a.y = rbf(xv.y * rstd * wv.y); a.z = rbf(xv.z * rstd * wv.z); a.w = rbf(xv.w * rstd * wv.w);
        return a;
    }
    CAMX_DEV f32x4 other(int k) const { return unpack_bf16x4(*(const u32x2 *)(wab + k)); }
};

// ---- block entry, rows of at most 1024 values: a wave per row, four values a lane -----------------------------------------------------
// Round c of the lane is elements 256 c + 4 slot .. + 3: the elements (the logical threads 4 slot .. + 3) it holds in the RMSNorm's sums, in the
// quantizer and in the projections, so x and the norm weights are read once and nothing crosses lanes but the rotation. hb: bf16(h), packed,
// zeros behind the row.
// u = bf16(H128 . bf16(h)), the row's max |u| without its NaNs, and whether it holds one
template <int NR>
CAMX_DEV float entry_rotate(const u32x2 (&hb)[NR], int lane, f32x4 (&u)[NR], bool & nan) {
    u16x2 most = {0, 0};
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const f32x4 v = scaled4(hadamard128_l4(unpack_bf16x4(hb[c]), lane & 31, false));
        const u32x2 w = {hw_pk_bf16(v.x, v.y), hw_pk_bf16(v.z, v.w)};
        u[c] = unpack_bf16x4(w);
        most = absmax_pk(absmax_pk(most, w.x), w.y);
    }
    float m = absmax_of(most);
    nan = __builtin_amdgcn_ballot_w64(m != m) != 0;
    if (__builtin_expect(nan, 0)) {
        m = 0.0f;
#pragma unroll
        for (int c = 0; c < NR; c++) m = fmaxf(m, absmax4(u[c]));
    }
    return wave_max64(m);
}
// values, codes, scale and rstd of a row
template <int NR>
CAMX_DEV void entry_row_fwd(const u32x2 (&hb)[NR], int lane, int row, bool stored, uint16_t * y, float * s_out, uint16_t * codes, float rstd, float * rstd_out, int d, float clip, int qmax, bool stream) {
    f32x4 u[NR];
    bool nan;
    const float amax = entry_rotate<NR>(hb, lane, u, nan);
    const float s = fmaxf(amax * clip / (float)qmax, 1e-8f);
    const RowScale rs(s, amax, qmax);
    if (!stored) return;                                 // (wave-uniform)
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const int k = 256 * c + 4 * lane;
        u[c] = rs.quant4(u[c]);
        if (c < NR - 1 || k < d) {
            if (y) store8(pack_f2bf_x4((f32x4){u[c].x * s, u[c].y * s, u[c].z * s, u[c].w * s}), y + (size_t)row * d + k, stream);
            if (codes) codes[((size_t)row * d + k) >> 2] = (uint16_t)rs.nibbles4(u[c]);
        }
    }
    if (lane == 0) { if (s_out) s_out[row] = s; if (rstd_out) rstd_out[row] = rstd; }          // (last: a wait for later loads waits for these stores too)
}
// dh, the gradient of bf16(h), from the packed gradient of the quantized values. The sum of dL/ds keeps the tree of the workgroup form (each
// of its half-wave sums is one chunk's here: round c holds chunks 2 c and 2 c + 1); a round in which no lane's quotient can round to qmax or holds
// the row's maximum needs no clamp, no mask and no look for ties (see actq_bwd_wave_k).
template <int NR>
CAMX_DEV void entry_row_bwd(const u32x2 (&hb)[NR], const u32x2 (&gy)[NR], int lane, f32x4 (&dh)[NR], int d, float clip, int qmax) {
    f32x4 u[NR], gv[NR];
    bool nan;
    const float amax = entry_rotate<NR>(hb, lane, u, nan);
    const float s_raw = amax * clip / (float)qmax, s = fmaxf(s_raw, 1e-8f);
    const Ste ste(qmax);
    const RowDiv rd(s, amax);
    const float calm = nan || qmax > 1024 ? -1.0f : ste.hi - 0.51f;
    float part[NR];
    int ties_n = 0;
    uint32_t tied = 0;                                   // bit c: some lane holds a max-|u| element in round c
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const bool on = c < NR - 1 || 256 * c + 4 * lane < d;
        gv[c] = unpack_bf16x4((u32x2){on ? gy[c].x : 0u, on ? gy[c].y : 0u});
        const f32x4 t = rd.div4(u[c], on);
        f32x4 v = {rintf(t.x) - t.x, rintf(t.y) - t.y, rintf(t.z) - t.z, rintf(t.w) - t.w};
        const float most = fmaxf(fmaxf(fabsf(u[c].x), fabsf(u[c].y)), fmaxf(fabsf(u[c].z), fabsf(u[c].w)));
        f32x4 g = gv[c];
        if (__builtin_amdgcn_ballot_w64(on && (!(most * rd.r1 < calm) || most == amax)) != 0) {
            int n = 0;
#define D_(e) { float m; v.e = ste(t.e, m); g.e = gv[c].e * m; n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(on && fabsf(u[c].e) == amax)); }
            CAMX_EACH4(D_)
#undef D_
            ties_n += n;
            if (n) tied |= 1u << c;
        }
        float a = 0.0f;
        a = __builtin_fmaf(gv[c].x, v.x, a); a = __builtin_fmaf(gv[c].y, v.y, a); a = __builtin_fmaf(gv[c].z, v.z, a); a = __builtin_fmaf(gv[c].w, v.w, a);
        part[c] = on ? a : 0.0f;
        gv[c] = g;
    }
    float dlds = 0.0f;                                   // the eight chunk sums in order (absent chunks add +0, as idle half-waves do)
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const float hs = half32_sum(part[c]);
        const float even = lane_read(hs, 0), odd = lane_read(hs, 32);
        dlds = c == 0 ? even : dlds + even;
        dlds += odd;
    }
    if (2 * NR < 8) dlds += 0.0f;
    const float coef = s_raw >= 1e-8f ? dlds * clip / (float)qmax / (float)ties_n : 0.0f;
#pragma unroll
    for (int c = 0; c < NR; c++) {
        f32x4 e = gv[c];
        if (__builtin_expect(tied & (1u << c), 0)) {     // wave-uniform: a row has few such elements, most rounds skip this
#define V_(x) if ((c < NR - 1 || 256 * c + 4 * lane < d) && fabsf(u[c].x) == amax && u[c].x != 0.0f) e.x += u[c].x > 0.0f ? coef : -coef;
            CAMX_EACH4(V_)
#undef V_
        }
        dh[c] = rbf4_canon(scaled4(hadamard128_l4(rbf4_any(e), lane & 31, false)));      // rbf4_any: the gradient of the bf16 tensor u
    }
}
// bf16(h) of four values, packed
CAMX_DEV u32x2 rms_pack4(f32x4 v, float rstd, f32x4 w) { return (u32x2){hw_pk_bf16(v.x * rstd * w.x, v.y * rstd * w.y), hw_pk_bf16(v.z * rstd * w.z, v.w * rstd * w.w)}; }
// sum of squares of the row under the 256-thread tree, from the lane's rounds (padding adds +0)
template <int NR>
CAMX_DEV float entry_rstd(const f32x4 (&xk)[NR], int d, float eps) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const f32x4 v = xk[c];
        acc.x = __builtin_fmaf(v.x, v.x, acc.x); acc.y = __builtin_fmaf(v.y, v.y, acc.y); acc.z = __builtin_fmaf(v.z, v.z, acc.z); acc.w = __builtin_fmaf(v.w, v.w, acc.w);
    }
    return rsqrt_exact(wave_groups_in_order(group32_sum(acc)) / (float)d + eps);
}
// A lane's rounds of an fp32 row. Behind the row it reads the row's first values, which entry_zero replaces once they are there (see fetch_row_w). NT: past the
// caches (of two loads chosen by a run-time flag the compiler makes a plain one).
template <bool NT, int NR>
CAMX_DEV void entry_load(const float * row, int d, int lane, f32x4 (&v)[NR]) {
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const int k = c < NR - 1 || 256 * c + 4 * lane < d ? 256 * c + 4 * lane : 0;
        if constexpr (NT) v[c] = __builtin_nontemporal_load((const f32x4 *)(row + k));
        else v[c] = *(const f32x4 *)(row + k);
    }
}
template <int NR>
CAMX_DEV void entry_zero(f32x4 (&v)[NR], int d, int lane) {
    const bool on = 256 * (NR - 1) + 4 * lane < d;
    f32x4 & e = v[NR - 1];
    e = (f32x4){on ? e.x : 0.0f, on ? e.y : 0.0f, on ? e.z : 0.0f, on ? e.w : 0.0f};
}
template <int NR>
CAMX_DEV void entry_pack(const f32x4 (&xk)[NR], const f32x4 (&wk)[NR], float rstd, int d, int lane, u32x2 (&hb)[NR]) {
#pragma unroll
    for (int c = 0; c < NR; c++) {
        hb[c] = rms_pack4(xk[c], rstd, wk[c]);
        if (c == NR - 1 && 256 * c + 4 * lane >= d) hb[c] = (u32x2){0u, 0u};            // (0 x an infinite rstd is a NaN, and the projections add the padding's products)
    }
}
// without projections
template <int NR>
__global__ void __launch_bounds__(64) block_entry_fwd_wave(const float * x, const float * nw, float eps, uint16_t * y, float * s, uint16_t * codes, float * rstd_out,
                                                           int d, float clip, int qmax, bool stream) {
    const int row = blockIdx.x, lane = slot_of(threadIdx.x);
    f32x4 xk[NR], wk[NR];
    entry_load<true, NR>(x + (size_t)row * d, d, lane, xk);
    entry_load<false, NR>(nw, d, lane, wk);
    entry_zero<NR>(xk, d, lane);
    const float rstd = entry_rstd<NR>(xk, d, eps);
    u32x2 hb[NR];
    entry_pack<NR>(xk, wk, rstd, d, lane, hb);
    entry_row_fwd<NR>(hb, lane, row, true, y, s, codes, rstd, rstd_out, d, clip, qmax, stream);
}

// Longer rows: a 256-thread workgroup per row (NR rounds of 1024 values). The projections: wave w takes rows w, w + 4, ... of wab, up to
// two of them at a time so that their loads fly together, each under the 256-thread tree (a lane holds the logical threads 4 lane ..
// 4 lane + 3, which add their elements 256 apart in order); rows of at most 2048 values keep bf16(h) in registers.
template <int NR>
__global__ void __launch_bounds__(256) block_entry_fwd_k(const float * x, const float * nw, const uint16_t * wab, int nab, float eps, uint16_t * y,
                                                         float * s, uint16_t * codes, uint16_t * ab, float * rstd_out, int d, float clip, int qmax) {
    __shared__ float lds[4];
    __shared__ float slot;
    const int row = blockIdx.x;
    const float * xr = x + (size_t)row * d;
    constexpr int NW = 4, NA = 4 * NR;                   // waves per row; 256-element steps of a row
    constexpr bool KEEP = NA <= 8;
    const int lane = slot_of(threadIdx.x & 63), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    f32x4 hk[KEEP ? NA : 1];
    const float ss = row_tree_sum(SqTerm{xr}, d, &slot);
    const float rstd = rsqrt_exact(ss / (float)d + eps);
    if (threadIdx.x == 0 && rstd_out) rstd_out[row] = rstd;
    actq_fwd_row<NR, RmsSrc>(RmsSrc{x, nw, rstd, d}, row, y, s, d, clip, qmax, codes, lds);
    if (nab == 0) return;
    const AbTerm term{xr, nw, rstd, wab};
    if (KEEP) {
#pragma unroll
        for (int i = 0; i < NA; i++) { const int k = 256 * i + 4 * lane; hk[KEEP ? i : 0] = k < d ? term(k) : (f32x4){0.0f, 0.0f, 0.0f, 0.0f}; }
    }
    constexpr int JB = NA <= 8 ? 2 : 1;                  // rows of wab whose loads fly together
    for (int j0 = wave; j0 < nab; j0 += JB * NW) {
        u32x2 wv[JB][NA];
#pragma unroll
        for (int jj = 0; jj < JB; jj++) {
            const int j = j0 + NW * jj;
#pragma unroll
            for (int i = 0; i < NA; i++) {
                const int k = 256 * i + 4 * lane;
                wv[jj][i] = (u32x2){0u, 0u};
                if (j < nab && k < d) wv[jj][i] = *(const u32x2 *)(wab + (size_t)j * d + k);
            }
        }
#pragma unroll
        for (int jj = 0; jj < JB; jj++) {
            const int j = j0 + NW * jj;
            if (j >= nab) break;                         // (wave-uniform)
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < NA; i++) {
                const int k = 256 * i + 4 * lane;
                if (k < d) {
                    const f32x4 a = KEEP ? hk[KEEP ? i : 0] : term(k), b = unpack_bf16x4(wv[jj][i]);
                    acc.x = __builtin_fmaf(a.x, b.x, acc.x); acc.y = __builtin_fmaf(a.y, b.y, acc.y);
                    acc.z = __builtin_fmaf(a.z, b.z, acc.z); acc.w = __builtin_fmaf(a.w, b.w, acc.w);
                }
            }
            const float tot = wave_groups_in_order(group32_sum(acc));
            if ((threadIdx.x & 63) == 0) ab[(size_t)row * nab + j] = f2bf(tot);
        }
    }
}

// ---- block entry with projections, rows of at most 1024 values: a wave per row, four rows share the projections on the matrix cores ----
// Bound by instruction issue: with the projections as vector multiply-adds of a row's own wave, they, the conversions of wab and sixteen
// reductions of 256 logical threads were two thirds of a row's instructions (32768 rows x 1024 values, 16 projections: 117 us, this
// kernel 86; 512 rows: 12.0 and 7.7; large batches with more than four projections: block_entry_fwd_rows16). A K = 1 matrix instruction
// (v_mfma_f32_4x4x1: 16 blocks of 4 x 4 single multiply-adds, each rounded like fmaf) computes for 16 logical threads t the terms of
// 4 rows x 4 projections, so a thread's chain over its elements t, t + 256, .. is a chain of NR such instructions in the same order.
// A workgroup's four waves own a row each and hand bf16(h) on through LDS; then wave w takes projections 4 w .. 4 w + 3 of all four rows.
// Roles: block Q (lanes 4 Q .. 4 Q + 3) is the logical threads 16 Q + 4 n + k, for one (n, k) per instruction. A: lane 4 Q + i holds row
// i's value there. B: lane 4 Q + j holds projection j's, from the caches; odd blocks hold their four
// projections in reverse, so that the tree's first step (t ^ 16, the other block of a pair) is a row_half_mirror. The following steps
// (t ^ 8, 4, 2, 1) pair n and k: registers. The eight group sums of a (row, projection) meet in LDS, where one lane adds them in order.
CAMX_DEV f32x4 mirror4(f32x4 v) { return (f32x4){lane_xor4(v.x), lane_xor4(v.y), lane_xor4(v.z), lane_xor4(v.w)}; }      // row_half_mirror
template <int NR>
__global__ void __launch_bounds__(256, 4) block_entry_fwd_quad(const float * __restrict__ x, const float * __restrict__ nw, const uint16_t * __restrict__ wab, int nab, float eps,
                                                               uint16_t * __restrict__ y, float * __restrict__ s_out, uint16_t * __restrict__ codes, uint16_t * __restrict__ ab,
                                                               float * __restrict__ rstd_out, int d, float clip, int qmax, int M, bool stream) {
    constexpr int HS = 128 * NR + 4;                     // words of a row of packed pairs; + 4: the four rows of a read fall on different banks
    __shared__ __attribute__((aligned(16))) uint32_t hbuf[4][HS];
    __shared__ __attribute__((aligned(16))) float gsum[4][4 * 4 * 8];         // [wave][row][projection][group]
    const int lraw = threadIdx.x & 63, lane = slot_of(lraw), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int Q = lraw >> 2, odd = Q & 1, jp = odd ? 3 - (lraw & 3) : lraw & 3;      // the lane's block and its projection of the wave's four
    const int r0 = 4 * blockIdx.x, row = r0 + wave;
    f32x4 xk[NR], wk[NR];
    entry_load<true, NR>(x + (size_t)min(row, M - 1) * d, d, lane, xk);
    entry_load<false, NR>(nw, d, lane, wk);
    entry_zero<NR>(xk, d, lane);
    const float rstd = entry_rstd<NR>(xk, d, eps);
    u32x2 hb[NR];
    entry_pack<NR>(xk, wk, rstd, d, lane, hb);
#pragma unroll
    for (int c = 0; c < NR; c++) *(u32x2 *)&hbuf[wave][128 * c + 2 * lane] = hb[c];
    entry_row_fwd<NR>(hb, lane, row, row < M, y, s_out, codes, rstd, rstd_out, d, clip, qmax, stream);
    u32x2 B[NR][4];                                      // (from the caches: 32 KiB for a workgroup)
#pragma unroll
    for (int c = 0; c < NR; c++)
#pragma unroll
        for (int n = 0; n < 4; n++) {
            const int k = 256 * c + 16 * Q + 4 * n;
            B[c][n] = (u32x2){0u, 0u};
            if (4 * wave + jp < nab && (c < NR - 1 || k < d)) B[c][n] = *(const u32x2 *)(wab + (size_t)(4 * wave + jp) * d + k);
        }
    __syncthreads();
    if (4 * wave < nab) {                            // (uniform in a wave)
        u32x4 A[NR][2];                              // row (lane & 3): elements 256 c + 16 Q .. + 15, packed pairs
#pragma unroll
        for (int c = 0; c < NR; c++)
#pragma unroll
            for (int h = 0; h < 2; h++) A[c][h] = *(const u32x4 *)&hbuf[lraw & 3][128 * c + 8 * Q + 4 * h];
        f32x4 sum[2];                                // [k & 1]; a word per row
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            const int k = kk == 1 ? 2 : kk == 2 ? 1 : kk;        // 0, 2, 1, 3: the pairs of t ^ 2
            f32x4 a[4];
#pragma unroll
            for (int n = 0; n < 4; n++) a[n] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int c = 0; c < NR; c++)
#pragma unroll
                for (int n = 0; n < 4; n++) {
                    const uint32_t av = A[c][n >> 1][2 * (n & 1) + (k >> 1)], bv = k >> 1 ? B[c][n].y : B[c][n].x;
                    a[n] = __builtin_amdgcn_mfma_f32_4x4x1f32(k & 1 ? bf_hi(av) : bf_lo(av), k & 1 ? bf_hi(bv) : bf_lo(bv), a[n], 0, 0, 0);
                }
            const f32x4 t0 = a[0] + mirror4(a[0]), t1 = a[1] + mirror4(a[1]), t2 = a[2] + mirror4(a[2]), t3 = a[3] + mirror4(a[3]);      // t ^ 16
            const f32x4 m0 = t0 + t2, m1 = t1 + t3;  // t ^ 8
            const f32x4 w = m0 + m1;                 // t ^ 4
            sum[k & 1] = k >> 1 ? sum[k & 1] + w : w;            // t ^ 2
        }
        const f32x4 g = sum[0] + sum[1];             // t ^ 1; a pair's blocks hold the same sums: the even one hands on rows 0 and 1, the odd one 2 and 3
        float * o = gsum[wave] + ((odd ? 8 : 0) + jp) * 8 + (Q >> 1);
        o[0] = odd ? g.z : g.x;
        o[4 * 8] = odd ? g.w : g.y;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier();
        const int rr = r0 + (lraw >> 2), j = 4 * wave + (lraw & 3);
        if (lraw < 16 && j < nab && rr < M) {
            const f32x4 a = *(const f32x4 *)(gsum[wave] + 8 * lraw), b = *(const f32x4 *)(gsum[wave] + 8 * lraw + 4);
            float tot = 0.0f;
            tot += a.x; tot += a.y; tot += a.z; tot += a.w; tot += b.x; tot += b.y; tot += b.z; tot += b.w;
            ab[(size_t)rr * nab + j] = f2bf(tot);
        }
    }
}

// ---- block entry, rows of at most 1024 values: two rows a wave, sixteen a workgroup, the projections on the matrix cores ----------------
// Bound by instruction issue (see actq_fwd_wave_k). A wave reads its rows four values a lane (element 256 c + 4 slot + k: the logical
// threads of the RMSNorm's sum), hands bf16(h) through LDS to the 16-lane layout of the quantizer, and after a barrier computes one
// group of 32 logical threads of the projections for all sixteen rows. A K = 1 matrix instruction (v_mfma_f32_16x16x1: four blocks of
// 16 rows x 16 projections of single multiply-adds, each rounded like fmaf) adds one element of four logical threads, so a thread's chain
// over its elements t, t + 256, .. is a chain of NR such instructions in the same order: wave w, instruction e, block b is thread
// 32 w + 8 b + e. A lane's eight elements of a step are 16 bytes of LDS (rows) and of device memory (projections), converted once for
// sixteen rows. The tree's first steps (t ^ 16, 8) pair blocks, which are registers of the result, the others (t ^ 4, 2, 1) instructions;
// the eight group sums meet in LDS, where a thread adds them in order.
// 32768 x 1024 with 16 projections 53 us, with 8 52; as four rows and four projections a wave 86 and 65. A barrier for the whole
// workgroup costs more than the matrix instructions save where there are few projections (4096 x 1024 with 4: 11.9 us, four rows a
// workgroup 11.5) and few workgroups (512 rows with 16: 10.2 and 7.6).
CAMX_DEV float bf_half(uint32_t v, int odd) { return odd ? bf_hi(v) : bf_lo(v); }
typedef float f32x16 __attribute__((ext_vector_type(16)));
CAMX_DEV void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); __builtin_amdgcn_wave_barrier(); __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront"); }
// the packed words of a row's rounds of 512 from its words in LDS; chunks behind the row as zeros
template <int R>
CAMX_DEV void words_from_lds(const uint32_t * row, int lane, int slot, bool last_on, u32x4 (&w)[R][1]) {
#pragma unroll
    for (int j = 0; j < R; j++) {
        w[j][0] = (u32x4){0u, 0u, 0u, 0u};
        if (j < R - 1 || last_on) w[j][0] = *(const u32x4 *)(row + 256 * j + 64 * (lane >> 4) + 4 * slot);
    }
}
template <int NR>
__global__ void __launch_bounds__(512, 6) block_entry_fwd_rows16(const float * __restrict__ x, const float * __restrict__ nw, const uint16_t * __restrict__ wab, int nab, float eps,
                                                              uint16_t * __restrict__ y, float * __restrict__ s_out, uint16_t * __restrict__ codes, uint16_t * __restrict__ ab,
                                                              float * __restrict__ rstd_out, int d, float clip, int qmax, int M, bool stream) {
    constexpr int HS = 128 * NR + 4, R = (NR + 1) / 2;   // words of a row of packed pairs; + 4: the sixteen rows of a read fall on different banks
    __shared__ __attribute__((aligned(16))) uint32_t hbuf[16][HS];
    __shared__ float gsum[8][16][16];         // [group][row][projection]
    const int lraw = threadIdx.x & 63, la = slot_of(lraw), slot = la & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = 16 * blockIdx.x;
    f32x4 xk[2][NR], wk[NR];
#pragma unroll
    for (int i = 0; i < 2; i++) entry_load<true, NR>(x + (size_t)min(r0 + 2 * wave + i, M - 1) * d, d, la, xk[i]);
    entry_load<false, NR>(nw, d, la, wk);
    float rstd[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        entry_zero<NR>(xk[i], d, la);
        rstd[i] = entry_rstd<NR>(xk[i], d, eps);
        u32x2 hb[NR];
        entry_pack<NR>(xk[i], wk, rstd[i], d, la, hb);
#pragma unroll
        for (int c = 0; c < NR; c++) *(u32x2 *)&hbuf[2 * wave + i][128 * c + 2 * la] = hb[c];
    }
    wave_lds_fence();
    const Lanes16 ln(slot);
    const int e0 = 128 * (lraw >> 4) + 8 * slot;
    const bool last_on = e0 + 512 * (R - 1) < d;
#pragma unroll 1
    for (int i = 0; i < 2; i++) {
        const int row = r0 + 2 * wave + i;
        u32x4 raw[R][1], uw[R], keep[R];
        words_from_lds<R>(hbuf[2 * wave + i], lraw, slot, last_on, raw);
        const u16x2 most = actq_rotate_w<R>(PlainBF16{}, raw, ln, uw, keep);
        bool nan;
        const float amax = row_absmax_w<R>(uw, most, nan);
        const float s = fmaxf(amax * clip / (float)qmax, 1e-8f);
        if (row < M) {                                   // (wave-uniform)
            quantize_row_w<R, 1>(uw, amax, s, qmax, e0, last_on, y ? y + (size_t)row * d : nullptr, codes ? codes + (size_t)row * (d / 4) : nullptr, stream);
            if (lraw == 0) { if (s_out) s_out[row] = s; if (rstd_out) rstd_out[row] = i ? rstd[1] : rstd[0]; }
        }
    }
    const int i16 = lraw & 15, b = lraw >> 4;            // A: row, B: projection; block
    u32x4 A[NR], B[NR];
#pragma unroll
    for (int c = 0; c < NR; c++) {                       // (from the caches: 32 KiB for a workgroup)
        const int k = 256 * c + 32 * wave + 8 * b;
        B[c] = (u32x4){0u, 0u, 0u, 0u};
        if (i16 < nab && (c < NR - 1 || k < d)) B[c] = *(const u32x4_a8 *)(wab + (size_t)i16 * d + k);
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NR; c++) A[c] = *(const u32x4 *)&hbuf[i16][128 * c + 16 * wave + 4 * b];
    f32x4 t[8];                                          // of instruction e: rows 4 b .. 4 b + 3 of projection i16
#pragma unroll
    for (int ee = 0; ee < 8; ee++) {
        const int e = (ee & 1) * 4 + (ee >> 1 & 1) * 2 + (ee >> 2);          // 0, 4, 2, 6, 1, 5, 3, 7: the pairs of t ^ 4, then of t ^ 2
        f32x16 a = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < NR; c++) {
            const uint32_t av = A[c][e >> 1], bv = B[c][e >> 1];
            a = __builtin_amdgcn_mfma_f32_16x16x1f32(bf_half(av, e & 1), bf_half(bv, e & 1), a, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);           // (one chain at a time: 80 registers, six waves per SIMD)
        }
#pragma unroll
        for (int r = 0; r < 4; r++) t[e][r] = (a[r] + a[8 + r]) + (a[4 + r] + a[12 + r]);            // t ^ 16, t ^ 8
        if (ee & 1) t[e - 4] += t[e];                    // t ^ 4
        if ((ee & 3) == 3) t[e & 1] += t[(e & 1) + 2];   // t ^ 2
    }
    const f32x4 sum = t[0] + t[1];                       // t ^ 1
#pragma unroll
    for (int r = 0; r < 4; r++) gsum[wave][4 * b + r][i16] = sum[r];
    __syncthreads();
    const int rr = threadIdx.x >> 4, j = threadIdx.x & 15;
    if (rr < 16 && r0 + rr < M && j < nab) {
        float tot = 0.0f;
#pragma unroll
        for (int g = 0; g < 8; g++) tot += gsum[g][rr][j];
        ab[(size_t)(r0 + rr) * nab + j] = f2bf(tot);
    }
}

// dx = rstd (dh w - xhat mean(dh w xhat)) of one row from the lane's registers
template <int NR>
CAMX_DEV void rms_bwd_row(const f32x4 (&xk)[NR], const f32x4 (&wk)[NR], float rstd, const f32x4 (&dh)[NR], float * dx, int d, int la, bool stream) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f}, gw[NR], xh[NR];
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const int k = 256 * c + 4 * la;
        gw[c] = xh[c] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
        if (c < NR - 1 || k < d) {
            const f32x4 w = wk[c], xv = xk[c];
            gw[c] = (f32x4){dh[c].x * w.x, dh[c].y * w.y, dh[c].z * w.z, dh[c].w * w.w};
            xh[c] = (f32x4){xv.x * rstd, xv.y * rstd, xv.z * rstd, xv.w * rstd};
            acc.x = __builtin_fmaf(gw[c].x, xh[c].x, acc.x); acc.y = __builtin_fmaf(gw[c].y, xh[c].y, acc.y);
            acc.z = __builtin_fmaf(gw[c].z, xh[c].z, acc.z); acc.w = __builtin_fmaf(gw[c].w, xh[c].w, acc.w);
        }
    }
    const float gs = group32_sum(acc);                   // the 32 logical threads of a group, then the eight groups in order
    float dot = lane_read(gs, 0);
#pragma unroll
    for (int q = 1; q < 8; q++) dot += lane_read(gs, 8 * q);
    dot = dot / (float)d;
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const int k = 256 * c + 4 * la;
        if (c < NR - 1 || k < d) {
            f32x4 r;
            r.x = rstd * (gw[c].x - xh[c].x * dot); r.y = rstd * (gw[c].y - xh[c].y * dot);
            r.z = rstd * (gw[c].z - xh[c].z * dot); r.w = rstd * (gw[c].w - xh[c].w * dot);
            store16(__builtin_bit_cast(u32x4, r), dx + k, stream);
        }
    }
}
// a lane's rounds of a bf16 row; behind the row its first values, for which entry_row_bwd puts zeros
template <int NR>
CAMX_DEV void entry_load16(const uint16_t * row, int d, int lane, u32x2 (&v)[NR]) {
#pragma unroll
    for (int c = 0; c < NR; c++) v[c] = __builtin_nontemporal_load((const u32x2 *)(row + (c < NR - 1 || 256 * c + 4 * lane < d ? 256 * c + 4 * lane : 0)));
}
// dh = actq backward of dy, plus the two projection groups' input gradients (wab rows [0, nab / 2) and [nab / 2, nab), each
// group's sum rounded to bf16); then the RMSNorm backward. d <= 1024. One wave per row, NR = ceil(d / 256) rounds: the lane's elements are
// the logical threads 4 slot .. 4 slot + 3 of the 256-thread tree of the dot product. This kernel: no projections.
template <int NR>
__global__ void __launch_bounds__(64) block_entry_bwd_k(const float * x, const float * nw, const float * rstd_in, const uint16_t * dy, float * dx, int d, float clip, int qmax, bool stream) {
    const int row = blockIdx.x, la = slot_of(threadIdx.x);
    const float rstd = rstd_in[row];
    f32x4 xk[NR], wk[NR], dh[NR];
    u32x2 gy[NR], hb[NR];
    entry_load<true, NR>(x + (size_t)row * d, d, la, xk);
    entry_load<false, NR>(nw, d, la, wk);
    entry_load16<NR>(dy + (size_t)row * d, d, la, gy);
    __builtin_amdgcn_sched_barrier(0);
    entry_pack<NR>(xk, wk, rstd, d, la, hb);
    entry_row_bwd<NR>(hb, gy, la, dh, d, clip, qmax);
    rms_bwd_row<NR>(xk, wk, rstd, dh, dx + (size_t)row * d, d, la, stream);
}

// The same for nab > 0 with the projections' part on the matrix cores (as vector multiply-adds of the row's own wave 143 us at 32768 x
// 1024 with 16 projections, here 84): a workgroup's four waves own a row each and first compute a quarter
// of that part for all four rows, one of the two groups for half of the column blocks of 256 (32768 x 256 with 4 projections 31.8 us, as
// one wave per column block 36.4, with vector multiply-adds 34.3). A K = 1 instruction adds one j's term dab[row][j] wab[j][column]
// (rounded like fmaf) for 4 rows x 64 columns: block Q's four columns are its lanes' own, so with A = dab (lane 4 Q + i: row i) and B = a
// lane's column of wab, D holds a lane's column with a word per row. The two groups' sums, rounded to bf16, reach the rows' owners
// through LDS. Loads return in order: rows of more than 256 values ask for what the projections need first (it comes from the caches) and for
// the row and its gradient behind it, so that the projections run while those are on their way (16 projections, 32768 x 1024 87.8 -> 84.9 us,
// 32768 x 512 48.6 -> 47.8, 512 x 512 8 % less); shorter rows are as fast either way (2048 x 256 1 % slower) and ask for the row first.
template <int NR>
__global__ void __launch_bounds__(256, 4) block_entry_bwd_quad(const float * x, const float * __restrict__ nw, const float * __restrict__ rstd_in, const uint16_t * __restrict__ wab,
                                                               int nab, const uint16_t * __restrict__ dy, const uint16_t * __restrict__ dab, float * dx, int d, float clip, int qmax, int M, bool stream) {
    __shared__ __attribute__((aligned(16))) uint32_t pbuf[4][2][128 * NR];                // [row][group][pairs of columns]
    const int lraw = threadIdx.x & 63, la = slot_of(lraw), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = nab / 2;
    const int r0 = 4 * blockIdx.x;
    const int row = min(r0 + wave, M - 1);               // (a wave past the end repeats the last row and stores nothing)
    constexpr bool LATE = NR >= 2;
    f32x4 xk[NR], wk[NR];
    u32x2 gy[NR];
    if (!LATE) { entry_load<false, NR>(nw, d, la, wk); entry_load<true, NR>(x + (size_t)row * d, d, la, xk); }
    // wave w: group w & 1 of column blocks (w >> 1) and (w >> 1) + 2; of a single block words w >> 1 of each lane's two
    constexpr int NT = (2 * NR + 3) / 4, NP = NR == 1 ? 1 : 2;
    const int h = wave & 1, c0 = NR == 1 ? 0 : wave >> 1, p0 = NR == 1 ? wave >> 1 : 0;
    uint32_t B[NT][8][NP];
    float av[8];
    const uint16_t * ar = dab + (size_t)min(r0 + (lraw & 3), M - 1) * nab + h * half;
#pragma unroll
    for (int j = 0; j < 8; j++) av[j] = bf2f(ar[min(j, half - 1)]);       // (no condition: see fetch_row_w; the terms from half on are not added)
#pragma unroll
    for (int j = 0; j < 8; j++) {
        if (j > 0 && j >= half) break;                   // (uniform)
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int k = 256 * (c0 + 2 * t) + 4 * la;   // (a column behind the row takes the first one's: its result is not stored)
            const uint16_t * b = wab + (size_t)(h * half + j) * d + (k < d ? k : 0);
            if (NP == 1) B[t][j][0] = ((const uint32_t *)b)[p0];
            else { const u32x2 v = *(const u32x2 *)b; B[t][j][0] = v.x; B[t][j][NP - 1] = v.y; }
        }
    }
    if (LATE) { entry_load<true, NR>(x + (size_t)row * d, d, la, xk); entry_load<false, NR>(nw, d, la, wk); entry_load16<NR>(dy + (size_t)row * d, d, la, gy); }
    const float rstd = rstd_in[row];
    f32x4 acc[NT][2 * NP];                               // (half >= 1: the first term opens the sums)
#pragma unroll
    for (int j = 0; j < 8; j++) {
        if (j == 0 || j < half) {                        // (uniform)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int k = 0; k < 2 * NP; k++) {
                    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
                    acc[t][k] = __builtin_amdgcn_mfma_f32_4x4x1f32(av[j], k & 1 ? bf_hi(B[t][j][k >> 1]) : bf_lo(B[t][j][k >> 1]), j ? acc[t][k] : zero, 0, 0, 0);
                }
        }
    }
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int cb = c0 + 2 * t;
        if (cb >= NR) break;                             // (uniform)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if (NP == 1) pbuf[r][h][2 * la + p0] = pack_f2bf_x4((f32x4){acc[t][0][r], acc[t][1][r], 0.0f, 0.0f}).x;
            else *(u32x2 *)&pbuf[r][h][128 * cb + 2 * la] = pack_f2bf_x4((f32x4){acc[t][0][r], acc[t][1][r], acc[t][2 * NP - 2][r], acc[t][2 * NP - 1][r]});
        }
    }
    if (!LATE) entry_load16<NR>(dy + (size_t)row * d, d, la, gy);
    u32x2 hb[NR];
    entry_pack<NR>(xk, wk, rstd, d, la, hb);
    f32x4 dh[NR];
    entry_row_bwd<NR>(hb, gy, la, dh, d, clip, qmax);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NR; c++) {
        const f32x4 ra = unpack_bf16x4(*(const u32x2 *)&pbuf[wave][0][128 * c + 2 * la]), rb = unpack_bf16x4(*(const u32x2 *)&pbuf[wave][1][128 * c + 2 * la]);
        dh[c].x = (dh[c].x + ra.x) + rb.x; dh[c].y = (dh[c].y + ra.y) + rb.y; dh[c].z = (dh[c].z + ra.z) + rb.z; dh[c].w = (dh[c].w + ra.w) + rb.w;
    }
    if (r0 + wave < M) rms_bwd_row<NR>(xk, wk, rstd, dh, dx + (size_t)row * d, d, la, stream);
}

__attribute__((visibility("hidden"))) int silu_luts_get(hipStream_t st, const uint16_t ** lut, const uint16_t ** small);       // quant.hip

// the derivative table's device address, filled once per device in stream order before its first reader; callers on any host
// thread go through one lock
static std::mutex g_dlut_mu;
static struct { bool ready; const float * lut; const float * small; } g_dlut_dev[64];
static int dsilu_luts_get(hipStream_t st, const float ** lut, const float ** small) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return CAMX_EINVAL;
    std::lock_guard<std::mutex> lock(g_dlut_mu);
    if (!g_dlut_dev[dev].ready) {
        dsilu_lut_fill<<<dim3(256), dim3(256), 0, st>>>();
        dsilu_small_fill<<<dim3((SWS_TAB + 255) / 256), dim3(256), 0, st>>>();
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return (int)e;
        void * sym = nullptr, * sym_small = nullptr;
        if (hipGetSymbolAddress(&sym, HIP_SYMBOL(g_dsilu_lut)) != hipSuccess || !sym) return CAMX_EINVAL;
        if (hipGetSymbolAddress(&sym_small, HIP_SYMBOL(g_dsilu_small)) != hipSuccess || !sym_small) return CAMX_EINVAL;
        if (hipStreamSynchronize(st) != hipSuccess) return CAMX_EINVAL;     // later calls may come on other streams
        g_dlut_dev[dev].lut = (const float *)sym;
        g_dlut_dev[dev].small = (const float *)sym_small;
        g_dlut_dev[dev].ready = true;
    }
    *lut = g_dlut_dev[dev].lut;
    *small = g_dlut_dev[dev].small;
    return CAMX_OK;
}

__attribute__((visibility("hidden"))) int dsilu_luts_init(hipStream_t st) {       // camx_init's half of this file
    const float * lut = nullptr, * small = nullptr;
    return dsilu_luts_get(st, &lut, &small);
}

// the wave-per-row kernels: rows of at most 4096 values (longer ones would need more registers than a wave has, or sums handed from wave
// to wave), operands aligned for 16-byte loads and 16- / 4-byte stores
static bool actq_wave_ok(int K, uintptr_t x, uintptr_t y, uintptr_t codes) { return K <= 4096 && !((x | y) & 15) && !(codes & 3); }
// Two waves a row (above 2048 values) from the batch that fills the chip with them; smaller ones are a chain of latencies, which a workgroup a row halves.
// bf16 / fp32 / SiLU forward at 3072 values, in turn: 64 rows 3.9 / 4.0 / 5.1 us (two waves 4.3 / 4.7 / 5.7), 256 rows 4.7 / 4.4 / 5.5 (4.9 / 5.1 / 6.1), 1024
// rows 7.3 / 8.1 / 10.2 (6.4 / 7.7 / 9.1); backward fp32 / SiLU 1 row 4.6 / 6.6 (4.9 / 7.5), 256 rows 6.3 / 8.7 (6.4 / 9.2), 512 rows 8.4 / 10.5 (8.2 / 9.7);
// bf16 256 rows 6.8 (6.2).
static bool actq_fwd_waves(int K, int M, bool bf16_rows) { return K <= 2048 || M >= (bf16_rows ? 512 : 1024); }
static bool actq_bwd_waves(int K, int M, bool bf16_rows) { return K <= 2048 || bf16_rows || M >= 512; }
// one instance per number of rounds of 512 values, above 2048 values two waves a row
#define ACTQ_WAVES(K, M, CALL)                                                                                          \
    {                                                                                                                   \
        const bool stream = (long)(M) * (K) >= (1L << 20);                                                              \
        const dim3 grid((unsigned)((K) > 2048 ? ((long)(M) + 1) / 2 : ((long)(M) + 3) / 4)), block(256);                \
        switch (((K) + 511) / 512) {                                                                                    \
            case 1: { constexpr int R = 1, W = 1; CALL; } break; case 2: { constexpr int R = 2, W = 1; CALL; } break;   \
            case 3: { constexpr int R = 3, W = 1; CALL; } break; case 4: { constexpr int R = 4, W = 1; CALL; } break;   \
            case 5: case 6: { constexpr int R = 3, W = 2; CALL; } break; default: { constexpr int R = 4, W = 2; CALL; } break; \
        }                                                                                                               \
    }

static int actq_check(int K, int qmax, int M) { return (K < 128 || K % 128 || K > 8192 || qmax < 1 || M < 0) ? CAMX_EINVAL : CAMX_OK; }

// one instance per number of rounds
#define ACTQ_ROUNDS(K, CALL)                                                                                           \
    switch (((K) + 1023) / 1024) {                                                                                     \
        case 1: { constexpr int NR = 1; CALL; } break; case 2: { constexpr int NR = 2; CALL; } break;                   \
        case 3: { constexpr int NR = 3; CALL; } break; case 4: { constexpr int NR = 4; CALL; } break;                   \
        case 5: { constexpr int NR = 5; CALL; } break; case 6: { constexpr int NR = 6; CALL; } break;                   \
        case 7: { constexpr int NR = 7; CALL; } break; default: { constexpr int NR = 8; CALL; } break;                  \
    }

// Sixteen rows share the projections, whatever their number, or four rows in steps of four projections. A workgroup of sixteen rows takes a CU's time
// once for every 4096 rows or part of them (16 projections x 1024: 4096 rows 11.9 us, 5120 17.3, 8192 18.6, 9216 23.8), one of four rows a quarter of
// them (14.3, 18.1, 25.4, 29.2). r: a row's time with four rows a workgroup over one's with sixteen, in sixteenths, from 32768 rows: 5 to 8 projections 1.19
// at 1024 values, 1.10 at 768, 1.00 at 256; 13 to 16 1.62, 1.43, 1.22 (an odd number of rounds of 256 leaves half a round of 512 empty).
static bool entry_rows16(int M, int d, int nab) {
    const int groups = (nab + 3) / 4, nr = (d + 255) / 256, r = nr == 1 ? 2 * groups + 11 : nr == 3 ? 3 * groups + 11 : 3 * groups + 12;
    return nab > 4 && M >= 4096 && (long)M * r >= (((long)M + 4095) / 4096) << 16;
}

extern "C" {

// actq_fwd_{f32,bf16} and actq_fwd_codes_{f32,bf16}: y bf16 [M][K] (optional when codes are written), s [M] (optional),
// codes [M][K / 2] bytes (optional; needs qmax <= 7)
int camx_actq_fwd(const void * x, int is_bf16, uint16_t * y, float * s, uint16_t * codes, int K, float clip, int qmax, int M, hipStream_t st) {
    if (!x || (!y && !codes) || actq_check(K, qmax, M) || ((uintptr_t)x & (is_bf16 ? 7 : 15)) || ((uintptr_t)y & 7) || ((uintptr_t)codes & 1)) return CAMX_EINVAL;
    if (M == 0) return CAMX_OK;
    if (actq_wave_ok(K, (uintptr_t)x, (uintptr_t)y, (uintptr_t)codes) && actq_fwd_waves(K, M, is_bf16)) {
        if (is_bf16) ACTQ_WAVES(K, M, (actq_fwd_wave_k<PlainBF16, R, W><<<grid, block, 0, st>>>(PlainBF16{(const uint16_t *)x, K}, y, s, codes, K, clip, qmax, M, stream)))
        else ACTQ_WAVES(K, M, (actq_fwd_wave_k<PlainF32, R, W><<<grid, block, 0, st>>>(PlainF32{(const float *)x, K}, y, s, codes, K, clip, qmax, M, stream)))
        CAMX_LAUNCH_RET();
    }
    if (is_bf16) { ACTQ_ROUNDS(K, (actq_fwd_k<NR><<<dim3(M), dim3(256), 0, st>>>(PlainBF16{(const uint16_t *)x, K}, y, s, codes, K, clip, qmax))) }
    else { ACTQ_ROUNDS(K, (actq_fwd_k<NR><<<dim3(M), dim3(256), 0, st>>>(PlainF32{(const float *)x, K}, y, s, codes, K, clip, qmax))) }
    CAMX_LAUNCH_RET();
}
int camx_silu_mul_actq_fwd(const uint16_t * gu, int ld, int F, uint16_t * y, float * s, uint16_t * codes, float clip, int qmax, int M, hipStream_t st) {
    if (!gu || (!y && !codes) || actq_check(F, qmax, M) || ld < 2 * F || (ld & 3) || ((uintptr_t)gu & 7) || ((uintptr_t)y & 7) || ((uintptr_t)codes & 1)) return CAMX_EINVAL;
    if (M == 0) return CAMX_OK;
    const uint16_t * lut = nullptr, * small = nullptr;
    const int rc = silu_luts_get(st, &lut, &small);
    if (rc) return rc;
    if (!(ld & 7) && actq_wave_ok(F, (uintptr_t)gu, (uintptr_t)y, (uintptr_t)codes) && actq_fwd_waves(F, M, false)) {
        ACTQ_WAVES(F, M, (actq_fwd_wave_k<SiluMulSrc, R, W><<<grid, block, 0, st>>>(SiluMulSrc{gu, ld, F, lut, nullptr}, y, s, codes, F, clip, qmax, M, stream, small)))
        CAMX_LAUNCH_RET();
    }
    ACTQ_ROUNDS(F, (actq_fwd_k<NR><<<dim3(M), dim3(256), 0, st>>>(SiluMulSrc{gu, ld, F, lut, nullptr}, y, s, codes, F, clip, qmax)))
    CAMX_LAUNCH_RET();
}
int camx_block_entry_fwd(const float * x, const float * nw, const uint16_t * wab, int nab, float eps, uint16_t * y, float * s, uint16_t * codes,
                         uint16_t * ab, float * rstd_out, int d, float clip, int qmax, int M, hipStream_t st) {
    if (!x || !nw || (!y && !codes) || actq_check(d, qmax, M) || nab < 0 || nab > 16 || (nab && (!wab || !ab)) || ((uintptr_t)x & 15) ||
        ((uintptr_t)nw & 15) || ((uintptr_t)wab & 7) || ((uintptr_t)y & 7) || ((uintptr_t)codes & 1)) return CAMX_EINVAL;
    if (M == 0) return CAMX_OK;
    if (d <= 1024) {                                     // rounds of 256 values
        const bool stream = (long)M * d >= (1L << 20);
#define ENTRY_ROUNDS(KERNEL, GRID, BLOCK, ...)                                                                          \
        switch ((d + 255) / 256) {                                                                                      \
            case 1: KERNEL<1><<<dim3((unsigned)(GRID)), dim3(BLOCK), 0, st>>>(__VA_ARGS__); break;                      \
            case 2: KERNEL<2><<<dim3((unsigned)(GRID)), dim3(BLOCK), 0, st>>>(__VA_ARGS__); break;                      \
            case 3: KERNEL<3><<<dim3((unsigned)(GRID)), dim3(BLOCK), 0, st>>>(__VA_ARGS__); break;                      \
            default: KERNEL<4><<<dim3((unsigned)(GRID)), dim3(BLOCK), 0, st>>>(__VA_ARGS__); break;                     \
        }
        if (entry_rows16(M, d, nab)) { ENTRY_ROUNDS(block_entry_fwd_rows16, ((long)M + 15) / 16, 512, x, nw, wab, nab, eps, y, s, codes, ab, rstd_out, d, clip, qmax, M, stream) }
        else if (nab > 0) { ENTRY_ROUNDS(block_entry_fwd_quad, ((long)M + 3) / 4, 256, x, nw, wab, nab, eps, y, s, codes, ab, rstd_out, d, clip, qmax, M, stream) }
        else { ENTRY_ROUNDS(block_entry_fwd_wave, M, 64, x, nw, eps, y, s, codes, rstd_out, d, clip, qmax, stream) }
        CAMX_LAUNCH_RET();
    }
    ACTQ_ROUNDS(d, (block_entry_fwd_k<NR><<<dim3(M), dim3(256), 0, st>>>(x, nw, wab, nab, eps, y, s, codes, ab, rstd_out, d, clip, qmax)))
    CAMX_LAUNCH_RET();
}

// actq_bwd_{f32,bf16}: g bf16 [M][K] the gradient of y; dx [M][K] in x's type
int camx_actq_bwd(const void * x, int is_bf16, const uint16_t * g, void * dx, int K, float clip, int qmax, int M, hipStream_t st) {
    if (!x || !g || !dx || actq_check(K, qmax, M) || ((uintptr_t)x & (is_bf16 ? 7 : 15)) || ((uintptr_t)dx & (is_bf16 ? 7 : 15)) || ((uintptr_t)g & 7)) return CAMX_EINVAL;
    if (M == 0) return CAMX_OK;
    if (actq_wave_ok(K, (uintptr_t)x | (uintptr_t)g, (uintptr_t)dx, 0) && actq_bwd_waves(K, M, is_bf16)) {
        if (is_bf16) ACTQ_WAVES(K, M, (actq_bwd_wave_k<PlainBF16, SinkBF16, R, W><<<grid, block, 0, st>>>(PlainBF16{(const uint16_t *)x, K}, g, SinkBF16{(uint16_t *)dx, K}, K, clip, qmax, M, stream)))
        else ACTQ_WAVES(K, M, (actq_bwd_wave_k<PlainF32, SinkF32, R, W><<<grid, block, 0, st>>>(PlainF32{(const float *)x, K}, g, SinkF32{(float *)dx, K}, K, clip, qmax, M, stream)))
        CAMX_LAUNCH_RET();
    }
    if (is_bf16) { ACTQ_ROUNDS(K, (actq_bwd_k<NR><<<dim3(M), dim3(256), 0, st>>>(PlainBF16{(const uint16_t *)x, K}, g, SinkBF16{(uint16_t *)dx, K}, K, clip, qmax))) }
    else { ACTQ_ROUNDS(K, (actq_bwd_k<NR><<<dim3(M), dim3(256), 0, st>>>(PlainF32{(const float *)x, K}, g, SinkF32{(float *)dx, K}, K, clip, qmax))) }
    CAMX_LAUNCH_RET();
}
// silu_mul_actq_bwd: g bf16 [M][F] the gradient of y; dgu bf16 [M][2F] = [dg | du], contiguous
int camx_silu_mul_actq_bwd(const uint16_t * gu, int ld, int F, const uint16_t * g, uint16_t * dgu, float clip, int qmax, int M, hipStream_t st) {
    if (!gu || !g || !dgu || actq_check(F, qmax, M) || ld < 2 * F || (ld & 3) || ((uintptr_t)gu & 7) || ((uintptr_t)g & 7) || ((uintptr_t)dgu & 7)) return CAMX_EINVAL;
    if (M == 0) return CAMX_OK;
    const uint16_t * lut = nullptr, * small = nullptr;
    const float * dlut = nullptr, * dsmall = nullptr;
    int rc = silu_luts_get(st, &lut, &small);
    if (!rc) rc = dsilu_luts_get(st, &dlut, &dsmall);
    if (rc) return rc;
    if (!(ld & 7) && actq_wave_ok(F, (uintptr_t)gu | (uintptr_t)g, (uintptr_t)dgu, 0) && actq_bwd_waves(F, M, false)) {
        ACTQ_WAVES(F, M, (actq_bwd_wave_k<SiluMulSrc, SinkSiluMul, R, W><<<grid, block, 0, st>>>(SiluMulSrc{gu, ld, F, lut, nullptr}, g, SinkSiluMul{gu, ld, F, dgu, dlut, nullptr}, F, clip, qmax, M, stream, small, dsmall)))
        CAMX_LAUNCH_RET();
    }
    ACTQ_ROUNDS(F, (actq_bwd_k<NR><<<dim3(M), dim3(256), 0, st>>>(SiluMulSrc{gu, ld, F, lut, nullptr}, g, SinkSiluMul{gu, ld, F, dgu, dlut, nullptr}, F, clip, qmax)))
    CAMX_LAUNCH_RET();
}
// block_entry_bwd: dy bf16 [M][d], dab bf16 [M][nab] (needed when nab > 0), rstd [M] from the forward; dx fp32 [M][d]; d <= 1024
int camx_block_entry_bwd(const float * x, const float * nw, const float * rstd, const uint16_t * wab, int nab, const uint16_t * dy,
                         const uint16_t * dab, float * dx, int d, float clip, int qmax, int M, hipStream_t st) {
    if (!x || !nw || !rstd || !dy || !dx || actq_check(d, qmax, M) || d > 1024 || nab < 0 || nab > 16 || (nab & 1) || (nab && (!wab || !dab)) ||
        ((uintptr_t)x & 15) || ((uintptr_t)nw & 15) || ((uintptr_t)dy & 7) || ((uintptr_t)dx & 15) || ((uintptr_t)wab & 7)) return CAMX_EINVAL;
    if (M == 0) return CAMX_OK;
    const bool stream = (long)M * d >= (1L << 20);
    if (nab > 0) { ENTRY_ROUNDS(block_entry_bwd_quad, ((long)M + 3) / 4, 256, x, nw, rstd, wab, nab, dy, dab, dx, d, clip, qmax, M, stream) }       // four rows share the projections' part
    else { ENTRY_ROUNDS(block_entry_bwd_k, M, 64, x, nw, rstd, dy, dx, d, clip, qmax, stream) }
#undef ENTRY_ROUNDS
    CAMX_LAUNCH_RET();
}

}   // extern "C"
