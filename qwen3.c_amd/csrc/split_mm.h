// split_mm.h - the int4 x fp32 matrix product of the prefill kernels on f16 MFMA.
//
//   y[x][o] = sum_g s[o][g] (sum_{i in g} x_i n'_i - (z[o][g] - 8) sum_{i in g} x_i),  n' = n - 8
//
// over 128-column groups g of an fmt6 tensor in the lanes layout (c/qwen.c:211-229).
//
// Arithmetic.  x of a (row, group) is scaled by a power of two so that its largest value lies
// in [2^14, 2^15) and split into two f16 planes, hi = f16(v) and lo = f16(v - hi): together
// 22 significant bits of every element (rounded to nearest, so the error is at most 2^-23 of
// the element itself, 2^-35 of the group's largest value for elements too small for that).
// n' is exact in f16, so every product is exact, and v_mfma_f32_32x32x16_f16 sums them in
// fp32, the small plane first.  Per group the sum is folded in fp32: v = p t - (z - 8) xsum,
// acc += s v (p the power of two).  Against 64 bits the result is closer than three int8
// digit planes of 23 bits below the group's maximum were (relative error of unit normal
// columns with one channel in 100 eight times as large, O = 8192, I = 2048: 1.3e-7 against
// 6.8e-7), and the fold takes 2 vector instructions per output and group instead of 7 (the
// zero points of two groups are one v_mfma_f32_32x32x2_f32).
//
// What bounds it: on random data these products take 21 ns per SIMD with the whole chip busy
// (15 with an eighth of it: the clock falls under the load), 26 ns with an LDS read and four
// vector instructions each.  512 x 8192 x 2048 takes 43 us, 42 ns a product, the matrix cores
// busy 34% of the time: the waves of a block wait for each other once per group (30% of their
// cycles) and stand ready behind each other's reads and vector instructions (42%).
//
// Operands (v_mfma_f32_32x32x16_f16: lane l holds row / column l % 32 and 8 of 16 k in half
// l / 32; the result's register r of lane l is row 8 (r / 4) + 4 (l / 32) + r % 4, column
// l % 32).  A = 32 weight rows, B = 32 rows of x.  One 32-bit weight word (8 columns) makes
// one lane's A operand: columns in the order 0 4 1 5 2 6 3 7, the odd ones 16 times as large
// (their nibbles are taken where they stand in the word), which the x planes make up for by
// holding the odd columns divided by 16.
#pragma once

#include "fmt6_device.h"
#include "internal.h"

#include <type_traits>

namespace coli {

typedef _Float16 sm_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 sm_h2 __attribute__((ext_vector_type(2)));
typedef float sm_f16 __attribute__((ext_vector_type(16)));
typedef float sm_f4u __attribute__((ext_vector_type(4), aligned(8)));

constexpr int kSmGS = 128;                 // columns per group
constexpr int kSmMaxG = kLaneMaxI / kSmGS; // groups of a row
constexpr int kSmUnits = 32;               // 16-byte units of one row and group (two planes)

// Byte offset, within the 512 bytes of a (row, group), of the 16-byte unit of plane (0 hi,
// 1 lo) that holds columns 8 j .. 8 j + 7 (j = 0..15).  Lanes layout: half b of a wave reads
// the chunks (32 columns) c + 2 b, c = 0, 1; word i of a chunk is columns 8 i of it.  128-byte
// lines hold one (plane, c): a staging row reads whole lines.
__device__ __forceinline__ uint32_t sm_unit(int plane, int j) {
    const int ch = j >> 2, i = j & 3;
    return (uint32_t)((plane * 2 + (ch & 1)) * 128 + (i * 2 + (ch >> 1)) * 16);
}

// 8 consecutive columns of one row -> their hi and lo units; v is already scaled
__device__ __forceinline__ void sm_split8(const float (&v)[8], uint4 &hi, uint4 &lo) {
    union {
        _Float16 h[8];
        uint4 u;
    } a, b;
    constexpr int ord[8] = {0, 4, 1, 5, 2, 6, 3, 7};
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const float x = (ord[k] & 1) ? v[ord[k]] * 0.0625f : v[ord[k]];
        a.h[k] = (_Float16)x;
        b.h[k] = (_Float16)(x - (float)a.h[k]);
    }
    hi = a.u;
    lo = b.u;
}

// 8 values (already scaled) -> their hi and lo units, in order
__device__ __forceinline__ void sp_split8(const float (&v)[8], uint4 &hi, uint4 &lo) {
    union {
        _Float16 h[8];
        uint4 u;
    } a, b;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        a.h[k] = (_Float16)v[k];
        b.h[k] = (_Float16)(v[k] - (float)a.h[k]);
    }
    hi = a.u;
    lo = b.u;
}

// The power of two that brings a group with maximum m (>= 0) to [2^14, 2^15), as exponents:
// x = v 2^-e, v = x 2^e.  Groups that are all zero or not finite keep 0; below 2^-135 the
// exponent stops, so that 2^-e is still an fp32 number.
__device__ __forceinline__ int sm_exp(float m) {
    if (!(m > 0.f) || !(m < INFINITY)) return 0;
    return 14 - max(ilogbf(m), -135);
}

// Columns 8 j .. 8 j + 7 of one (row, group) -> the split planes at dst (512 bytes) and, from
// lane j = 0, (p, sum of the group) at *xp.  The 16 aligned consecutive lanes that hold a
// group agree on its maximum and sum (in double, rounded once) by shuffles; lanes with valid =
// false join them and write nothing.
__device__ __forceinline__ void sm_row8(const float (&v)[8], bool valid, int j, uint8_t *dst, float2 *xp) {
    float m = 0.f;
    double sum = 0.0;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        m = fmaxf(m, fabsf(v[c]));
        sum += (double)v[c];
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
        m = fmaxf(m, __shfl_xor(m, o));
        sum += __shfl_xor(sum, o);
    }
    const int e = sm_exp(m);
    float x[8];
#pragma unroll
    for (int c = 0; c < 8; c++) x[c] = ldexpf(v[c], e);
    uint4 hi, lo;
    sm_split8(x, hi, lo);
    if (valid) {
        *(uint4 *)(dst + sm_unit(0, j)) = hi;
        *(uint4 *)(dst + sm_unit(1, j)) = lo;
        if (j == 0) *xp = make_float2(ldexpf(1.f, -e), (float)sum);
    }
}

// Waves of a block: RW share the x rows and own 32 weight rows each, KW split the groups.
// NT x tiles of 32 rows.  LDS: x planes of one group per k part, two buffers; [scale, 8 -
// zero] of the block's rows for two groups, two buffers.
template <int RW, int KW, int NT>
struct SmLds {
    uint4 b[KW][2][NT * 32 * kSmUnits];
    float s[KW][2][2][RW * 32];    // scale
    float sz[KW][2][2][RW * 32];   // scale * (8 - zero)
    float2 p[kSmMaxG + 1][NT * 32];   // (p, sum) of the block's x rows; after the last group zeros
};

// What a wave and its threads bring.  wr / wo: weight descriptors and byte offsets of this
// lane's row l % 16 of rows 0-15 and 16-31 of the wave's tile (kOOB: rows that read as zero);
// half: bytes from a row's even chunks to its odd ones.  sz: [scale, zero] pairs of row
// (thread of the k part) % (RW * 32), by group.  xr / xo: x planes and the byte offsets of
// the rows this thread stages.  xp: (p, sum) pairs by group of the x rows of this lane, one
// pointer per tile.  ng groups.
template <int RW, int KW, int NT>
struct SmSrc {
    static constexpr int NRB = 4 * NT;                       // blocks of 8 x rows
    static constexpr int kRows = NRB > RW ? NRB / RW : 1;    // x rows staged per thread
    __amdgpu_buffer_rsrc_t wr[2], xr;
    uint32_t wo[2], half, xo[kRows];
    const float2 *sz, *xp[NT];
    int ng, slast;
    // sz of row r of a matrix of n >= r rows (two pairs are read at a time, never past its ends)
    __device__ __forceinline__ void scales(const float *m, int r) {
        sz = (const float2 *)m + (size_t)r * ng;
        slast = ng > 1 ? ng - 2 : r > 0 ? -1 : 0;
    }
};

// x row (of the block's NT * 32) that this thread stages as its k-th
template <int RW, int KW, int NT>
__device__ __forceinline__ int sm_stage_row(int k) {
    const int lane = threadIdx.x & 63, rw = (threadIdx.x >> 6) % RW;
    constexpr int NRB = 4 * NT;
    return (NRB > RW ? rw + RW * k : rw % NRB) * 8 + (lane >> 3);
}

// lane's slot of unit u of x row r within a 128-byte line: the 16 rows that one LDS cycle
// reads then fall on different banks
__device__ __forceinline__ int sm_swz(int r) { return (r ^ ((r >> 3) & 3)) & 7; }

// A operand of the 8 columns of one word (see above): the codes go into the mantissa of f16 1024 or
// 1024 + 16 n, and the offset is subtracted (the conversion of Kim et al., "Who Says Elephants Can't
// Run", 2022, here with codes stored XOR 8)
__device__ __forceinline__ sm_h8 sm_a8(uint32_t w) {
    const uint32_t v = w >> 8;
    union {
        uint32_t u[4];
        sm_h2 h[4];
    } a;
    a.u[0] = (w & 0x000F000Fu) ^ 0x64086408u;   // f16 1024 + n
    a.u[1] = (w & 0x00F000F0u) ^ 0x64806480u;   // f16 1024 + 16 n
    a.u[2] = (v & 0x000F000Fu) ^ 0x64086408u;
    a.u[3] = (v & 0x00F000F0u) ^ 0x64806480u;
    const sm_h2 c1 = {(_Float16)-1032.f, (_Float16)-1032.f}, c16 = {(_Float16)-1152.f, (_Float16)-1152.f};
    const sm_h2 p0 = a.h[0] + c1, p1 = a.h[1] + c16, p2 = a.h[2] + c1, p3 = a.h[3] + c16;
    return sm_h8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// Swap the odd 16-lane rows of a with the even ones of b
__device__ __forceinline__ void sm_swap16(uint4 &a, uint4 &b) {
    const auto x = __builtin_amdgcn_permlane16_swap(a.x, b.x, false, false);
    const auto y = __builtin_amdgcn_permlane16_swap(a.y, b.y, false, false);
    const auto z = __builtin_amdgcn_permlane16_swap(a.z, b.z, false, false);
    const auto w = __builtin_amdgcn_permlane16_swap(a.w, b.w, false, false);
    a = make_uint4(x[0], y[0], z[0], w[0]);
    b = make_uint4(x[1], y[1], z[1], w[1]);
}

// The product: acc[t][r] (result layout above) of the wave's 32 weight rows and x tile t,
// summed over the groups of the wave's k part.  With KW > 1 the parts are added in LDS and
// the waves of part 0 hold the result.  All threads of the block take part.
//
// Groups go in pairs: one weight load of 64 contiguous bytes per row covers two of them (lane
// (q, j) reads 16 bytes at 16 [0 2 1 3][q] of row j; swapping 16-lane rows between rows 0-15
// and 16-31 then leaves one group per register).  Loads run ahead: x planes two groups, weights
// and scales one pair.
template <int RW, int KW, int NT>
__device__ __forceinline__ void sm_product(SmLds<RW, KW, NT> &L, const SmSrc<RW, KW, NT> &src, sm_f16 (&acc)[NT]) {
    constexpr int NRB = 4 * NT, kXV = NT * 16 / RW;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rw = wave % RW, kw = wave / RW, half = lane >> 5;
    const int np = (src.ng + 1) / 2, npk = (np + KW - 1) / KW, s0 = kw * npk;
    const int send = min(s0 + npk, np), gend = min(2 * send, src.ng);   // may be empty: s0 >= np
    const int q = lane >> 4, sq = ((q & 1) << 1) | (q >> 1);

    // rows at kOOB stay out of range whatever is added; past the last group the last is loaded again
    auto w_load = [&](int S, int i, uint4 (&d)[4]) {   // i = 2 (chunk parity) + (rows 16-31)
        d[i] = buf_load16<kCached>(src.wr[i & 1], src.wo[i & 1] + 64u * min(S, np - 1) + 16u * sq + (i >> 1 ? src.half : 0u));
    };
    // x: wave rw of the part takes the 1 KB blocks (8 rows x one 128-byte line) (row block, line)
    const int line0 = NRB > RW ? 0 : (rw / NRB) * kXV;
    auto x_load = [&](int g, int k, uint4 (&d)[kXV]) {
        const int rk = NRB > RW ? k / 4 : 0, ln = NRB > RW ? k % 4 : line0 + k;
        d[k] = buf_load16<kCached>(src.xr, src.xo[rk] + 512u * min(g, src.ng - 1) + (uint32_t)(ln * 128 + (lane & 7) * 16));
    };
    auto x_store = [&](int buf, int k, const uint4 (&d)[kXV]) {
        const int rb = NRB > RW ? rw + RW * (k / 4) : rw % NRB, ln = NRB > RW ? k % 4 : line0 + k;
        L.b[kw][buf][(rb * 4 + ln) * 64 + (lane ^ sm_swz(rb * 8 + (lane >> 3)))] = d[k];
    };
    const int st = threadIdx.x - kw * RW * 64;   // thread of the part; the first RW * 32 carry scales
    // both groups of a pair in one load (slast: the last place it may start)
    auto s_load = [&](int S) {
        const sm_f4u v = *(const sm_f4u *)(src.sz + min(2 * S, src.slast));
        return make_float4(v.x, v.y, v.z, v.w);
    };
    auto s_store = [&](int buf, int S, const float4 &v) {   // groups past the part's end count nothing
        if (st < RW * 32) {
            const bool last = 2 * S > src.slast;
            const float2 d[2] = {last ? make_float2(v.z, v.w) : make_float2(v.x, v.y), make_float2(v.z, v.w)};
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float sc = 2 * S + h < gend ? d[h].x : 0.f;
                L.s[kw][buf][h][st] = sc;
                L.sz[kw][buf][h][st] = 2 * S + h < gend ? sc * (8.f - d[h].y) : 0.f;
            }
        }
    };
    const int xrow = lane & 31, sw = half ^ sm_swz(xrow);
    const int bbase = (xrow >> 3) * 256 + (xrow & 7) * 8;

    // Registers of the pipeline: C the pair's words (even chunks of its groups in C[0], C[1], odd
    // ones in C[2], C[3]), W the next pair's, a the A operands by chunk parity, t the sums of
    // the running unit (group, x tile) and of the one before it, fs / fp that one's scales and
    // power.
    uint4 C[4], W[4], xv[2][kXV];
    sm_h8 a[2][4];
    sm_f16 t[2];
    float4 sv, fs[4];
    float fp = 0.f;
#pragma unroll
    for (int i = 0; i < NT; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) t[1][r] = 0.f;
#pragma unroll
    for (int r = 0; r < 4; r++) fs[r] = make_float4(0.f, 0.f, 0.f, 0.f);
    auto fs_at = [&](int r) {
        const float4 v = fs[r >> 2];
        return (r & 3) == 0 ? v.x : (r & 3) == 1 ? v.y : (r & 3) == 2 ? v.z : v.w;
    };
    auto swap_words = [&]() {
#pragma unroll
        for (int i = 0; i < 4; i++) C[i] = W[i];
        sm_swap16(C[0], C[1]);
        sm_swap16(C[2], C[3]);
    };
    auto word = [](const uint4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; };

    // One group (h = 0, 1 of its pair) from x buffer h: 16 NT steps of one product each, in a
    // fixed order (sched_barrier).  Among them go the LDS reads of the x operands kAhead steps
    // on, the fold of the unit before (one output a step), the next words' A operands and the
    // memory work: a burst of loads at the group's start held each wave for ~1000 cycles (the
    // CU's waves share the address unit).
    constexpr int kAhead = 6, kSteps = 16 * NT;
    auto group = [&](auto hc, int S, int sbuf) {
        constexpr int h = decltype(hc)::value;
        const int g = 2 * S + h;
        uint4 B[kAhead + 1];
        auto b_read = [&](int f) {   // step f: tile f / 16, then chunk parity, plane (small first), word
            const int k = f & 15, line = (1 - ((k >> 2) & 1)) * 2 + (k >> 3);
            B[f % (kAhead + 1)] = L.b[kw][h][(f >> 4) * 1024 + bbase + line * 64 + (sw ^ (2 * (k & 3)))];
        };
#pragma unroll
        for (int f = 0; f < kAhead; f++) b_read(f);
        float pn = L.p[min(g, src.ng)][xrow].x;
        const float az = h ? L.sz[kw][sbuf][half][rw * 32 + xrow] : 0.f;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int f = 0; f < kSteps; f++) {
            const int tt = f >> 4, k = f & 15, u = h * NT + tt, pt = (tt + NT - 1) % NT;   // pt: the tile being folded
            if (f + kAhead < kSteps) b_read(f + kAhead);
            if ((f & 1) == 0 && (f >> 1) < kXV) x_load(g + 2, f >> 1, xv[h]);
            if ((f & 1) == 1 && f >= kSteps - 2 * kXV) x_store(1 - h, (f - kSteps + 2 * kXV) >> 1, xv[1 - h]);
            if (h == 0 && f >= kSteps / 2 && (f & 1) == 0 && f < kSteps / 2 + 8) w_load(S + 1, (f - kSteps / 2) >> 1, W);
            if (h == 0 && f == 7) sv = s_load(S + 1);
            if (h == 1 && f == kSteps - 9) swap_words();
            if (f < 8 && (f & 1) == 0) a[1][f >> 1] = sm_a8(word(C[2 + h], f >> 1));
            if (f >= kSteps - 8 && (f & 1) == 0) a[0][(f - kSteps + 8) >> 1] = sm_a8(word(C[h ? 0 : 1], (f - kSteps + 8) >> 1));
            const sm_h8 bv = __builtin_bit_cast(sm_h8, B[f % (kAhead + 1)]);
            if (k == 0) {
                sm_f16 z;
#pragma unroll
                for (int r = 0; r < 16; r++) z[r] = 0.f;
                t[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0][0], bv, z, 0, 0, 0);
            } else {
                t[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[k >> 3][k & 3], bv, t[u & 1], 0, 0, 0);
            }
            acc[pt][k] = fmaf(fs_at(k), t[(u & 1) ^ 1][k] * fp, acc[pt][k]);
            if (tt == 0 && (k & 3) == 3) fs[k >> 2] = *(const float4 *)&L.s[kw][sbuf][h][rw * 32 + 8 * (k >> 2) + 4 * half];
            if (k == 15) {
                fp = pn;
                if (tt + 1 < NT) pn = L.p[min(g, src.ng)][(tt + 1) * 32 + xrow].x;
            }
            // the zero points of the pair: acc += (s (8 - z)) xsum, one fp32 product of K = 2 groups
            // (lane: row or column l % 32, group l / 32 of the pair)
            if (h == 1 && k == (NT > 1 ? 4 : 15))
                acc[tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(az, L.p[min(2 * S + half, src.ng - 1)][tt * 32 + xrow].y,
                                                               acc[tt], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

#pragma unroll
    for (int k = 0; k < kXV; k++) x_load(2 * s0, k, xv[0]);
#pragma unroll
    for (int i = 0; i < 4; i++) w_load(s0, i, W);
    sv = s_load(s0);
#pragma unroll
    for (int k = 0; k < kXV; k++) x_load(2 * s0 + 1, k, xv[1]);
    // (p, sum) of every group of the block's x rows: read by each wave from global memory they
    // took as long as the x planes (one 8-byte word of 32 rows per load).  The half pair past an odd
    // count has the next row's codes, whose sums may be past the fp32 range: power 0, not scale
    // 0 alone, which times infinity is NaN
    for (int g = 2 * wave + half; g <= src.ng; g += 2 * RW * KW)
#pragma unroll
        for (int i = 0; i < NT; i++) L.p[g][i * 32 + xrow] = g < src.ng ? src.xp[i][g] : make_float2(0.f, 0.f);
#pragma unroll
    for (int k = 0; k < kXV; k++) x_store(0, k, xv[0]);
    s_store(0, s0, sv);
    swap_words();
#pragma unroll
    for (int i = 0; i < 4; i++) a[0][i] = sm_a8(word(C[0], i));
    lds_barrier();
    for (int it = 0; it < npk; it++) {
        const int S = s0 + it;
        group(std::integral_constant<int, 0>{}, S, it & 1);
        lds_barrier();
        group(std::integral_constant<int, 1>{}, S, it & 1);
        s_store((it + 1) & 1, S + 1, sv);
        lds_barrier();
    }
#pragma unroll
    for (int r = 0; r < 16; r++) acc[NT - 1][r] = fmaf(fs_at(r), t[1][r] * fp, acc[NT - 1][r]);
    if constexpr (KW > 1) {   // every wave is past its last read of L.b
        float *red = (float *)&L.b[0][0][0];
        if (kw > 0)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) red[((((kw - 1) * RW + rw) * NT + t) * 16 + r) * 64 + lane] = acc[t][r];
        lds_barrier();
        if (kw == 0)
#pragma unroll
            for (int k = 1; k < KW; k++)
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int r = 0; r < 16; r++) acc[t][r] += red[((((k - 1) * RW + rw) * NT + t) * 16 + r) * 64 + lane];
    }
}

}  // namespace coli
