// Per-row int8 quantisation of bf16 activations for gfx950: the role of the Triton `_quant_row` with PRE_NONE
// (enhancers/fused_kernels.py:137-174) and of kitchen's quantize_int8_rowwise_convrot64 (enhancers/fused_int8.py:
// 178-181).
//
// Per row r of K values x (bf16):
//   mode 1 (ConvRot): each 256-group goes through four radix-4 stages of stride 1, 4, 16, 64 -- (a, b, c, d) ->
//     (a+b+c-d, a+b-c+d, a-b+c+d, -a+b+c+d), every sum left to right in float32 -- then * 0.0625;
//   mode 0 (plain per-token): y = x.
//   amax = min(max |y|, 3.38953139e38); scale = max(amax / 127, 1e-30) (stored as float32);
//   q = clamp(rint(bf16(bf16(y) / bf16(scale))), -128, 127).
//
// A row is held in registers by one wave (rows up to 6144 values in ConvRot mode, 8192 plain; four rows per
// 256-thread workgroup) or by the four waves of a workgroup (wider rows, up to 32768 values; the waves' partial
// maxima meet in LDS -- the maximum does not depend on the order it is taken in, so the bits do not depend on the
// split). ConvRot: a lane loads 16 consecutive values of a 256-group (the two lowest radix-4 digits), runs stages 1
// and 4 on them, exchanges through LDS so that it then holds the 16 values that share its two lowest digits
// (stride 16), and runs stages 16 and 64. Groups are independent until the row maximum, so a wave may take any of
// them: pass p of wave w of a row takes groups 4 (p W + w) .. 4 (p W + w) + 3, W waves per row. The quotient y / s is computed with a
// correctly rounded reciprocal of s (one IEEE division per row) and one Markstein correction step -- mul, then two
// fma -- which is the correctly rounded IEEE quotient for every normal result (subnormal quotients round to 0 in the
// integer anyway). Built without contraction; the fma calls are explicit.
//
// ConvRot rows may first go through the operation the reference's quantiser applies before its rotation (PRE,
// enhancers/fused_kernels.py:14-18,143-163): GELU by table lookup (torch's GELU of every bf16 value), the
// scale-and-shift bf16(bf16(x * s1) + shift) of the row's group, or LayerNorm without affine, rounded to bf16, and
// then the scale-and-shift. The LayerNorm statistics follow the reference's Welford order (:97-136): 128 virtual
// threads, thread t updating (mean, sigma2, count) over the 4-value vectors t, t + 128, ... of the row, then
// shuffle-down merges within 32-thread warps (16, 8, 4, 2, 1) and across warps (2, 3 into 0, 1; 1 into 0). Lane l
// of the wave plays virtual threads l and l + 64. rstd = 1 / sqrt(var + eps) correctly rounded (the reference's
// rsqrt.approx.f32 is an NVIDIA approximation).

#include <algorithm>
#include <type_traits>

#include "wf_common.h"

namespace wf {

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

constexpr float kAmaxClamp = 3.38953139e38f;

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b16) { return __uint_as_float(b16 << 16); }

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// the two bf16 values of a word as float32
__device__ __forceinline__ float bf_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf_hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }

// LDS accesses of one wave run in the order they are issued, so a wave that exchanges values through its own LDS region
// needs no wait: these fences only keep the compiler from moving one side's accesses past the other's.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// RN(y / s) for the row's finite scale s, given ns = -s and rs = RN(1 / s). HUGE rows (values past the amax clamp): an
// infinite y (a rotation that overflowed) gives y * rs = +-inf, which is the IEEE quotient; the correction step would
// turn it into NaN (inf - inf).
template <bool HUGE_ROW>
__device__ __forceinline__ float div_rn(float y, float ns, float rs) {
    const float q = y * rs;
    const float rem = __builtin_fmaf(q, ns, y);
    const float r = __builtin_fmaf(rem, rs, q);
    if constexpr (HUGE_ROW) return __builtin_isinf(q) ? q : r;
    else return r;
}

// the int8 of a pair of bf16 values y (low byte of each word): rint(bf16(y / s)) clamped to [-128, 127], a NaN to -128.
// The integer is read off the sum with 1.5 * 2^23, which rounds to nearest even as rint does.
template <bool HUGE_ROW>
__device__ __forceinline__ void quant2(uint32_t y, float ns, float rs, uint32_t& q0, uint32_t& q1) {
    const uint32_t t = pack_bf16(div_rn<HUGE_ROW>(bf_lo(y), ns, rs), div_rn<HUGE_ROW>(bf_hi(y), ns, rs));
    q0 = __float_as_uint(fminf(fmaxf(bf_lo(t), -128.0f), 127.0f) + 12582912.0f);
    q1 = __float_as_uint(fminf(fmaxf(bf_hi(t), -128.0f), 127.0f) + 12582912.0f);
}

// the row's maximum over its W waves (W = 1: the wave's own); every lane of the W waves gets it. W > 1 needs the
// whole workgroup to be one row (no wave leaves early), since it takes a workgroup barrier.
// Calls in a loop alternate turn between 0 and 1: a wave may write its next maximum while another still reads these.
template <int W>
__device__ __forceinline__ float row_max(float wave_amax, int wave, int turn = 0) {
    if constexpr (W == 1) {
        return wave_amax;
    } else {
        __shared__ float part[2][W];
        if ((threadIdx.x & 63) == 0) part[turn][wave] = wave_amax;
        __syncthreads();
        float m = part[turn][0];
#pragma unroll
        for (int i = 1; i < W; i++) m = fmaxf(m, part[turn][i]);
        return m;
    }
}

struct RowScale {
    float scale, nsb, rsb;     // the row's scale; minus its bf16 rounding, and that rounding's reciprocal
    bool huge;                 // the row holds values past the amax clamp
};

__device__ __forceinline__ RowScale row_scale(float amax) {
    RowScale r;
    r.huge = amax > kAmaxClamp;
    amax = fminf(amax, kAmaxClamp);
    r.scale = fmaxf(amax / 127.0f, 1.0e-30f);
    const float sb = round_bf16(r.scale);
    r.nsb = -sb;
    r.rsb = 1.0f / sb;
    return r;
}

// ----------------------------------------------------------------------------------------- operations (PRE)
struct PreArgs {
    const uint16_t* s;        // GELU: bf16 table [65536]; MOD / LNMOD: bf16 s1 = 1 + scale, [groups, K]
    const uint16_t* h;        // MOD / LNMOD: bf16 shift, [groups, K]
    int64_t rows_per_group;
    float eps;                // LNMOD
};

// Welford state of one virtual thread; its count is the same in every virtual thread at every step (K / 128 values
// each, doubled by each merge), so the counts and what is derived from them are computed once, not per thread.
struct Welford {
    float m, s;
};

// PyTorch's cuWelfordCombine(dataB = own, dataA = other) as the reference restates it, with the contractions it
// makes explicit (enhancers/fused_kernels.py:84-94); both sides hold co values, nab = co * (1 / (2 co))
__device__ __forceinline__ void wcombine(Welford& w, float mo, float so, float co, float nab) {
    const float delta = w.m - mo;
    w.m = __builtin_fmaf(nab, mo, nab * w.m);
    w.s = __builtin_fmaf((delta * delta) * co, nab, so + w.s);
}

// lane i's value of x from lane i + O of its row of 16 (the lanes past the row's end get their own)
template <int O>
__device__ __forceinline__ float row_down(float x) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(__float_as_uint(x), __float_as_uint(x), 0x100 + O, 0xf, 0xf,
                                                       false));
}

// 1 / c, correctly rounded, for the counts a virtual thread can reach (rows of up to 32768 values)
struct Reciprocals {
    float r[256];
};
static constexpr Reciprocals reciprocals() {
    Reciprocals t{};
    for (int c = 1; c <= 256; c++) t.r[c - 1] = 1.0f / (float)c;
    return t;
}
__constant__ Reciprocals kRecip = reciprocals();

// mean and sigma2 / K of one row (K % 512 == 0), every lane gets the result. The chain of updates is short; what it
// costs is instructions, so the count's reciprocals come from a table (scalar loads) and the merges within rows of 16
// lanes are DPP moves.
__device__ __forceinline__ void ln_stats(const uint16_t* xr, int K, int lane, float& mu, float& var) {
    Welford w[2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};
    const int nj = K >> 9;
#pragma unroll 4
    for (int j = 0; j < nj; j++) {
        uint2 u[2];
#pragma unroll
        for (int vt = 0; vt < 2; vt++) u[vt] = *reinterpret_cast<const uint2*>(xr + 4 * (lane + 64 * vt + 128 * j));
#pragma unroll
        for (int ii = 0; ii < 4; ii++) {
            const float rc = kRecip.r[4 * j + ii];
#pragma unroll
            for (int vt = 0; vt < 2; vt++) {
                const uint32_t p = ii < 2 ? u[vt].x : u[vt].y;
                const float v = ii & 1 ? bf_hi(p) : bf_lo(p);
                const float delta = v - w[vt].m;
                w[vt].m = __builtin_fmaf(delta, rc, w[vt].m);
                w[vt].s = __builtin_fmaf(delta, v - w[vt].m, w[vt].s);
            }
        }
    }
    // within each 32-thread virtual warp lane i < o merges lane i + o, o = 16, 8, 4, 2, 1 (the other lanes' results
    // are not used)
    // (every merge doubles the count, and rounding commutes with powers of two: co * RN(1 / (2 co)) is the same at
    // each of them)
    float co = (float)(4 * nj);
    const float na = co * (0.5f * kRecip.r[4 * nj - 1]);
#pragma unroll
    for (int vt = 0; vt < 2; vt++)
        wcombine(w[vt], __shfl_down(w[vt].m, 16, 32), __shfl_down(w[vt].s, 16, 32), co, na);
    auto merge = [&](auto o) {
        constexpr int O = decltype(o)::value;
        co = co + co;
#pragma unroll
        for (int vt = 0; vt < 2; vt++) wcombine(w[vt], row_down<O>(w[vt].m), row_down<O>(w[vt].s), co, na);
    };
    merge(std::integral_constant<int, 8>{});
    merge(std::integral_constant<int, 4>{});
    merge(std::integral_constant<int, 2>{});
    merge(std::integral_constant<int, 1>{});
    // warps 2, 3 (lanes 0, 32 of the second virtual thread) into warps 0, 1; then warp 1 (lane 32) into warp 0
    co = co + co;
    wcombine(w[0], w[1].m, w[1].s, co, na);
    const float mo = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w[0].m), 32));
    const float so = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w[0].s), 32));
    co = co + co;
    wcombine(w[0], mo, so, co, na);
    mu = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(w[0].m)));
    var = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(w[0].s))) / (float)K;
}

// ------------------------------------------------------------------------------------------------ plain rows
// W waves per row, CPL chunks of 8 values per lane: chunk c = (i W + w) 64 + lane of the row for wave w, i < CPL.
// K <= 512 W CPL, K % 8 == 0. W = 1: four rows per workgroup; W = 4: one.
template <int CPL, int W>
__global__ __launch_bounds__(256) void quant_plain(const uint16_t* __restrict__ x, int64_t M, int K,
                                                   int8_t* __restrict__ xq, float* __restrict__ xs) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, w = wave % W;
    const int64_t row = (int64_t)blockIdx.x * (4 / W) + wave / W;
    if (W == 1 && row >= M) return;             // whole waves leave together; W = 1 takes no workgroup barrier
    const uint4* xr = reinterpret_cast<const uint4*>(x + row * K);
    const int nchunks = K >> 3;
    uint4 v[CPL];
    // the maximum of the magnitudes' bits, two 16-bit halves at a time; with a NaN or an infinity among them the wave
    // takes it in float32 instead (NaNs ignored), and the division that keeps infinite quotients
    u16x2 mag = {0, 0};
#pragma unroll
    for (int i = 0; i < CPL; i++) {
        const int c = (i * W + w) * 64 + lane;
        v[i] = c < nchunks ? xr[c] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < CPL; i++) {
        const uint32_t u[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
        for (int h = 0; h < 4; h++)
            mag = __builtin_elementwise_max(mag, __builtin_bit_cast(u16x2, u[h] & 0x7fff7fffu));
    }
    const uint32_t top = max((uint32_t)mag[0], (uint32_t)mag[1]);
    const bool special = __any(top >= 0x7f80u);
    float amax = __uint_as_float(top << 16);
    if (special) {
        amax = 0.0f;
#pragma unroll
        for (int i = 0; i < CPL; i++) {
            const uint32_t u[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
            for (int h = 0; h < 4; h++) amax = fmaxf(fmaxf(amax, fabsf(bf_lo(u[h]))), fabsf(bf_hi(u[h])));
        }
    }
    const RowScale rs = row_scale(row_max<W>(wave_max(amax), wave));
    if (lane == 0 && w == 0) xs[row] = rs.scale;
    uint2* qr = reinterpret_cast<uint2*>(xq + row * K);
    auto store = [&](auto huge) {
#pragma unroll
        for (int i = 0; i < CPL; i++) {
            const int c = (i * W + w) * 64 + lane;
            if (c >= nchunks) continue;
            const uint32_t u[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
            uint32_t b[4];
#pragma unroll
            for (int h = 0; h < 4; h++) {
                uint32_t lo, hi;
                quant2<decltype(huge)::value>(u[h], rs.nsb, rs.rsb, lo, hi);
                b[h] = __builtin_amdgcn_perm(hi, lo, 0x0c0c0400u);     // (lo, hi) low bytes
            }
            qr[c] = make_uint2(b[0] | (b[1] << 16), b[2] | (b[3] << 16));
        }
    };
    if (rs.huge || special) store(std::true_type{});
    else store(std::false_type{});
}

// --------------------------------------------------------------------------------------------- ConvRot rows
// radix-4 stage on 4 values (a, b, c, d) in place, sums left to right (enhancers/fused_kernels.py:65-81)
__device__ __forceinline__ void h4(float& a, float& b, float& c, float& d) {
    const float y0 = ((a + b) + c) - d;
    const float y1 = ((a + b) - c) + d;
    const float y2 = ((a - b) + c) + d;
    const float y3 = ((-a + b) + c) + d;
    a = y0; b = y1; c = y2; d = y3;
}

// A wave's LDS window of 4 groups: 16 consecutive values of a group lie 20 floats apart, groups 336 apart, so that the
// 16-byte writes of 16 consecutive values and the reads of 64 lanes' single values (value tl + 16 m of group gl) both
// spread over all banks, and the writes stay 16-byte aligned.
constexpr int kGroupFloats = 336, kRunFloats = 20;
// the quantised bytes of a window, read back in 16-byte runs: groups 272 bytes apart (256 would put the four groups'
// byte writes in the same banks)
constexpr int kGroupBytes = 272;

// GELU by table: the table's entries of the exponents [kGeluExp, kGeluExp + 24) -- magnitudes 2^-18 up to 64 -- are held
// in LDS, both signs interleaved: entry 2 (|bits| - 128 kGeluExp) + sign. The few values outside come from the table.
constexpr uint32_t kGeluExp = 109, kGeluEntries = 24 * 128, kGeluFirst = kGeluExp * 128;

// W waves per row, NP passes of 4 groups (1024 values) per wave: K <= 1024 W NP, K % 256 == 0. Lane t of pass p
// of wave w owns group 4 (p W + w) + t / 16, position tl = t % 16. W = 1: four rows per workgroup; W = 4: one.
//
// Bound by instruction issue, not by memory: about 20 vector instructions per value (10 of them the rotation's sums).
// So the row's raw words of all passes load up front (their latency passes once), a rotated pass is kept as packed bf16
// pairs (all the quotient uses; half the registers, more waves), the quotient's correction is two two-operand fmas, the
// rounding to an integer one addition, and the LDS exchange is 16-byte writes with no waits. Measured on MI355X, before
// and after, bit-identical: 16384 x 5120 67-69 and 51-53 us (4.9 TB/s), 4096 x 13824 53 and 39; GELU 5152 x 8192 48-49
// and 40-42 (its table read from LDS instead of the L2), LayerNorm 5152 x 2048 24.1 and 18.5, 4096 x 8192 96 and 51
// (its statistics had an IEEE division per value); scale-and-shift 4096 x 5120 24.8 and 24.2.
//
// PRE 4 is GELU with every value read from the whole table in memory, one turn per wave (gelu_in_lds says where).
template <int NP, int PRE, int W>
__global__ __launch_bounds__(256) void quant_convrot(const uint16_t* __restrict__ x, int64_t M, int K,
                                                     int8_t* __restrict__ xq, float* __restrict__ xs, PreArgs pa) {
    __shared__ __align__(16) float stage[4][4 * kGroupFloats];      // per wave: one 4-group window
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, w = wave % W;
    int64_t row = (int64_t)blockIdx.x * (4 / W) + wave / W;
    const int G = K >> 8;                        // groups in the row
    const int gl = lane >> 4, tl = lane & 15;
    const uint16_t* gelu = nullptr;
    if constexpr (PRE == 1) {
        __shared__ __align__(16) uint16_t tab[2 * kGeluEntries];
        if ((reinterpret_cast<uintptr_t>(pa.s) & 15) == 0) {
            for (int i = threadIdx.x; i < (int)kGeluEntries / 8; i += 256) {
                const uint4 a = reinterpret_cast<const uint4*>(pa.s + kGeluFirst)[i];
                const uint4 b = reinterpret_cast<const uint4*>(pa.s + 0x8000u + kGeluFirst)[i];
                uint4* t = reinterpret_cast<uint4*>(tab + 16 * i);
                auto even = [](uint32_t u, uint32_t v) { return __builtin_amdgcn_perm(v, u, 0x05040100u); };
                auto odd = [](uint32_t u, uint32_t v) { return __builtin_amdgcn_perm(v, u, 0x07060302u); };
                t[0] = make_uint4(even(a.x, b.x), odd(a.x, b.x), even(a.y, b.y), odd(a.y, b.y));
                t[1] = make_uint4(even(a.z, b.z), odd(a.z, b.z), even(a.w, b.w), odd(a.w, b.w));
            }
        } else {
            for (int i = threadIdx.x; i < (int)kGeluEntries; i += 256) {
                tab[2 * i] = pa.s[kGeluFirst + i];
                tab[2 * i + 1] = pa.s[0x8000u + kGeluFirst + i];
            }
        }
        gelu = tab;
        __syncthreads();
    }
    if (W == 1 && row >= M) return;              // whole waves leave together; W = 1 takes no further workgroup barrier
    float* st = stage[wave];
    // 16 consecutive values [16 tl, 16 tl + 16) of this lane's group of pass p
    auto at = [&](int p) { return 256 * (4 * (p * W + w) + gl) + 16 * tl; };
    auto live = [&](int p) { return 4 * (p * W + w) + gl < G; };
    uint4 raw[NP][2];
    auto load_row = [&](int64_t r) {
#pragma unroll
        for (int p = 0; p < NP; p++) {
            raw[p][0] = raw[p][1] = make_uint4(0, 0, 0, 0);
            if (live(p)) {
                const uint4* src = reinterpret_cast<const uint4*>(x + r * K + at(p));
                raw[p][0] = src[0];
                raw[p][1] = src[1];
            }
        }
    };
    // (with more passes the next row's words would cost waves)
    constexpr bool AHEAD = PRE == 1 && NP <= 3;
    load_row(row);
    // scale and shift of a pass, loaded a pass ahead
    uint4 sh[2][4];
    auto load_mod = [&](const uint16_t* s, const uint16_t* h, int p) {
        if (p < NP && live(p)) {
            const uint4* sp = reinterpret_cast<const uint4*>(s + at(p));
            const uint4* hp = reinterpret_cast<const uint4*>(h + at(p));
            sh[p & 1][0] = sp[0];
            sh[p & 1][1] = sp[1];
            sh[p & 1][2] = hp[0];
            sh[p & 1][3] = hp[1];
        }
    };
    // GELU: the grid holds a few workgroups per CU, each taking every gridDim.x-th row (or four rows), so that the table
    // is loaded that often only; the next row's words load while this one's are quantised. Otherwise one turn.
    for (int turn = 0;; turn ^= 1) {
        float mu = 0.0f, rstd = 0.0f;
        const uint16_t *sr = nullptr, *hr = nullptr;
        if constexpr (PRE == 2 || PRE == 3) {
            // (32-bit division where it fits: the 64-bit one is a long sequence)
            const int64_t grp = M < (1LL << 31) && pa.rows_per_group < (1LL << 31)
                                    ? (int64_t)((uint32_t)row / (uint32_t)pa.rows_per_group)
                                    : row / pa.rows_per_group;
            sr = pa.s + grp * K;
            hr = pa.h + grp * K;
            load_mod(sr, hr, 0);
        }
        if constexpr (PRE == 3) {
            float var;
            ln_stats(x + row * K, K, lane, mu, var);
            rstd = (float)(1.0 / __builtin_sqrt((double)(var + pa.eps)));
        }
        uint32_t y[NP][8];                           // the rotated values as bf16 pairs (values m, m + 1)
        float amax = 0.0f;
#pragma unroll
        for (int p = 0; p < NP; p++) {
            uint32_t u[8] = {raw[p][0].x, raw[p][0].y, raw[p][0].z, raw[p][0].w,
                             raw[p][1].x, raw[p][1].y, raw[p][1].z, raw[p][1].w};
            if constexpr (PRE == 4) {
                if (live(p)) {
#pragma unroll
                    for (int h = 0; h < 8; h++) u[h] = pa.s[u[h] & 0xffffu] | ((uint32_t)pa.s[u[h] >> 16] << 16);
                }
            } else if constexpr (PRE == 1) {
                if (live(p)) {
                    // |bits| of the pairs' members; all 16 in the LDS part of the table, or value by value
                    uint32_t lo = 0xffffffffu, hi = 0;
#pragma unroll
                    for (int h = 0; h < 8; h++) {
                        const uint32_t a = u[h] & 0x7fffu, b = (u[h] >> 16) & 0x7fffu;
                        lo = min(lo, min(a, b));
                        hi = max(hi, max(a, b));
                    }
                    auto slot = [&](uint32_t b) { return 2u * (b & 0x7fffu) + (b >> 15) - 2u * kGeluFirst; };
                    if (lo >= kGeluFirst && hi < kGeluFirst + kGeluEntries) {
#pragma unroll
                        for (int h = 0; h < 8; h++)
                            u[h] = gelu[slot(u[h] & 0xffffu)] | ((uint32_t)gelu[slot(u[h] >> 16)] << 16);
                    } else {
#pragma unroll
                        for (int h = 0; h < 8; h++)
                            u[h] = pa.s[u[h] & 0xffffu] | ((uint32_t)pa.s[u[h] >> 16] << 16);
                    }
                }
            } else if constexpr (PRE == 2 || PRE == 3) {
                load_mod(sr, hr, p + 1);
                if (live(p)) {
                    const uint4 s0 = sh[p & 1][0], s1 = sh[p & 1][1], h0 = sh[p & 1][2], h1 = sh[p & 1][3];
                    const uint32_t sw[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
                    const uint32_t hw[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
#pragma unroll
                    for (int h = 0; h < 8; h++) {
                        if constexpr (PRE == 3) u[h] = pack_bf16((bf_lo(u[h]) - mu) * rstd, (bf_hi(u[h]) - mu) * rstd);
                        u[h] = pack_bf16(bf_lo(u[h]) * bf_lo(sw[h]), bf_hi(u[h]) * bf_hi(sw[h]));
                        u[h] = pack_bf16(bf_lo(u[h]) + bf_lo(hw[h]), bf_hi(u[h]) + bf_hi(hw[h]));
                    }
                }
            }
            float v[16];
#pragma unroll
            for (int h = 0; h < 8; h++) {
                v[2 * h] = bf_lo(u[h]);
                v[2 * h + 1] = bf_hi(u[h]);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) h4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);   // stride 1
#pragma unroll
            for (int q = 0; q < 4; q++) h4(v[q], v[q + 4], v[q + 8], v[q + 12]);                  // stride 4
            wave_lds_order();
            float4* run = reinterpret_cast<float4*>(st + gl * kGroupFloats + tl * kRunFloats);
#pragma unroll
            for (int q = 0; q < 4; q++) run[q] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
            wave_lds_order();
            // now the 16 values i = tl + 16 m (m = k2 + 4 k3) of the group
#pragma unroll
            for (int m = 0; m < 16; m++) v[m] = st[gl * kGroupFloats + m * kRunFloats + tl];
#pragma unroll
            for (int q = 0; q < 4; q++) h4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);   // stride 16
#pragma unroll
            for (int q = 0; q < 4; q++) h4(v[q], v[q + 4], v[q + 8], v[q + 12]);                  // stride 64
#pragma unroll
            for (int h = 0; h < 8; h++) {
                const float a = v[2 * h] * 0.0625f, b = v[2 * h + 1] * 0.0625f;
                amax = fmaxf(fmaxf(amax, fabsf(a)), fabsf(b));      // (a lane past the row's end holds zeros)
                y[p][h] = pack_bf16(a, b);
            }
        }
        const int64_t next = row + (int64_t)gridDim.x * (4 / W);
        if constexpr (AHEAD) {
            if (next < M) load_row(next);
        }
        const RowScale rs = row_scale(row_max<W>(wave_max(amax), wave, turn));
        if (lane == 0 && w == 0) xs[row] = rs.scale;
        // per pass: quantise into the wave's LDS window at the bytes' row positions, then store the pass's 1024 bytes
        // (four whole groups, contiguous in the row) with one 16-byte store per lane
        uint8_t* qb = reinterpret_cast<uint8_t*>(st) + gl * kGroupBytes;
        uint8_t* dst = reinterpret_cast<uint8_t*>(xq + row * K);
        auto store = [&](auto huge) {
#pragma unroll
            for (int p = 0; p < NP; p++) {
                if (4 * (p * W + w) >= G) break;     // the same for the whole wave
                wave_lds_order();
#pragma unroll
                for (int h = 0; h < 8; h++) {
                    uint32_t q0, q1;
                    quant2<decltype(huge)::value>(y[p][h], rs.nsb, rs.rsb, q0, q1);
                    qb[tl + 32 * h] = (uint8_t)q0;
                    qb[tl + 32 * h + 16] = (uint8_t)q1;
                }
                wave_lds_order();
                if (live(p)) *reinterpret_cast<uint4*>(dst + at(p)) = *reinterpret_cast<const uint4*>(qb + 16 * tl);
            }
        };
        if (rs.huge) store(std::true_type{});
        else store(std::false_type{});
        if (PRE != 1 || next >= M) break;
        row = next;
        if constexpr (!AHEAD) load_row(row);
    }
}

// widest rows taken: 32768 values (one workgroup of four waves per row)
constexpr int kMaxRowK = 32768;

// Wide rows, many of them, are bound by memory, and more of them in flight than three workgroups a CU (two at the widest)
// slow it: LDS that is asked for and not used keeps to that. us without and with it (MI355X): 16384 x 13824 124.7 and 115.4,
// 4096 x 20480 42.7 and 39.8, 8192 x 32768 162.4 and 143.5; but 16384 x 8208 73.1 and 76.9, 1024 x 9216 6.7 and 7.1. (Before
// the maxima went over 16-bit halves the registers kept to it: 122.3, 41.5, 156.6, 75.0, 7.3.)
static size_t plain_lds(int64_t M, int K) {
    if (M < 4096 || K < 9216) return 0;
    return K <= 26624 ? 52 * 1024 : 63 * 1024;
}

template <int CPL, int W>
static void launch_plain(const uint16_t* x, int64_t M, int K, int8_t* xq, float* xs, hipStream_t s) {
    const size_t lds = W == 1 ? 0 : plain_lds(M, K);
    quant_plain<CPL, W><<<dim3((unsigned)((M + 4 / W - 1) / (4 / W))), 256, lds, s>>>(x, M, K, xq, xs);
}

static void launch_plain_rows(const uint16_t* x, int64_t M, int K, int8_t* xq, float* xs, hipStream_t s) {
    if (K <= 8192) {                                   // one wave per row
        const int cpl = (K + 511) / 512;
        if (cpl <= 2) launch_plain<2, 1>(x, M, K, xq, xs, s);
        else if (cpl <= 4) launch_plain<4, 1>(x, M, K, xq, xs, s);
        else if (cpl <= 8) launch_plain<8, 1>(x, M, K, xq, xs, s);
        else if (cpl <= 10) launch_plain<10, 1>(x, M, K, xq, xs, s);
        else launch_plain<16, 1>(x, M, K, xq, xs, s);
    } else {                                           // four waves per row: 2048 values per chunk step
        const int cpl = (K + 2047) / 2048;
        if (cpl <= 6) launch_plain<6, 4>(x, M, K, xq, xs, s);
        else if (cpl <= 8) launch_plain<8, 4>(x, M, K, xq, xs, s);
        else if (cpl <= 12) launch_plain<12, 4>(x, M, K, xq, xs, s);
        else launch_plain<16, 4>(x, M, K, xq, xs, s);
    }
}

template <int NP, int PRE, int W>
static void launch_convrot_pre(const uint16_t* x, int64_t M, int K, int8_t* xq, float* xs, const PreArgs& pa,
                               hipStream_t s) {
    int64_t grid = (M + 4 / W - 1) / (4 / W);
    if (PRE == 1) grid = std::min<int64_t>(grid, 4 * 256);      // four workgroups' LDS fit a CU
    quant_convrot<NP, PRE, W><<<dim3((unsigned)grid), 256, 0, s>>>(x, M, K, xq, xs, pa);
}

// GELU from the table in LDS, or from memory. Filling it costs every workgroup 12 KiB of loads and a barrier before its
// first row, which narrow rows do not earn back: (us, memory against LDS, MI355X) 256 values 64 rows 3.9 and 4.4, 8192
// rows 8.3 and 9.5; 512 values 1024 rows 4.0 and 4.4; 1024 values 512 rows 4.1 and 4.3, but 2048 rows 5.3 and 5.0; 1280
// values 65536 rows 97 and 105 (a turn of four rows is short), 16384 rows 30.5 and 29.6; from 1536 values on LDS wins at
// every row count (2048 values: 64 rows 6.1 and 5.6, 4096 rows 13.2 and 9.8).
static bool gelu_in_lds(int64_t M, int K) {
    return K >= 1536 || (K > 1024 && M <= 16384) || (K == 1024 && M > 1024);
}

template <int PRE>
static void launch_convrot(const uint16_t* x, int64_t M, int K, int8_t* xq, float* xs, const PreArgs& pa,
                           hipStream_t s) {
    if (K <= 6144) {                                   // one wave per row, 1024 values per pass
        const int np = (K + 1023) / 1024;
        if (np <= 1) launch_convrot_pre<1, PRE, 1>(x, M, K, xq, xs, pa, s);
        else if (np <= 2) launch_convrot_pre<2, PRE, 1>(x, M, K, xq, xs, pa, s);
        else if (np <= 3) launch_convrot_pre<3, PRE, 1>(x, M, K, xq, xs, pa, s);
        else if (np <= 4) launch_convrot_pre<4, PRE, 1>(x, M, K, xq, xs, pa, s);
        else if (np <= 5) launch_convrot_pre<5, PRE, 1>(x, M, K, xq, xs, pa, s);
        else launch_convrot_pre<6, PRE, 1>(x, M, K, xq, xs, pa, s);
    } else {                                           // four waves per row, 4096 values per pass
        const int np = (K + 4095) / 4096;
        if (np <= 2) launch_convrot_pre<2, PRE, 4>(x, M, K, xq, xs, pa, s);
        else if (np <= 3) launch_convrot_pre<3, PRE, 4>(x, M, K, xq, xs, pa, s);
        else if (np <= 4) launch_convrot_pre<4, PRE, 4>(x, M, K, xq, xs, pa, s);
        else if (np <= 5) launch_convrot_pre<5, PRE, 4>(x, M, K, xq, xs, pa, s);
        else if (np <= 6) launch_convrot_pre<6, PRE, 4>(x, M, K, xq, xs, pa, s);
        else launch_convrot_pre<8, PRE, 4>(x, M, K, xq, xs, pa, s);
    }
}

// the checks both entry points share
static int check_rows(const char* who, const void* x, int64_t M, int64_t K, const int8_t* xq, const float* xs) {
    if (M < 0 || K <= 0) { set_error("%s: M = %lld, K = %lld", who, (long long)M, (long long)K); return WF_EINVAL; }
    if (M == 0) return WF_OK;
    if (!x || !xq || !xs) { set_error("%s: null pointer", who); return WF_EINVAL; }
    if (!aligned(x, 16) || !aligned(xq, 16) || !aligned(xs, 4)) {
        set_error("%s: x and xq must be 16-byte aligned", who);
        return WF_EUNSUPPORTED;
    }
    if (M > ((int64_t)1 << 33)) { set_error("%s: M too large", who); return WF_EUNSUPPORTED; }
    return WF_OK;
}

}  // namespace wf

extern "C" int wf_quant_rows_i8(const void* x_bf16, int64_t M, int64_t K, int mode, int8_t* xq, float* xs,
                                void* stream) {
    using namespace wf;
    const int rc = check_rows("wf_quant_rows_i8", x_bf16, M, K, xq, xs);
    if (rc != WF_OK || M == 0) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint16_t* xp = static_cast<const uint16_t*>(x_bf16);
    const int k = (int)K;
    if (mode == 0) {
        if (K % 16 || K > kMaxRowK) {
            set_error("wf_quant_rows_i8: plain mode needs K %% 16 == 0 and K <= %d (K = %lld)", kMaxRowK,
                      (long long)K);
            return WF_EUNSUPPORTED;
        }
        launch_plain_rows(xp, M, k, xq, xs, s);
    } else if (mode == 1) {
        if (K % 256 || K > kMaxRowK) {
            set_error("wf_quant_rows_i8: ConvRot mode needs K %% 256 == 0 and K <= %d (K = %lld)", kMaxRowK,
                      (long long)K);
            return WF_EUNSUPPORTED;
        }
        launch_convrot<0>(xp, M, k, xq, xs, PreArgs{nullptr, nullptr, 1, 0.0f}, s);
    } else {
        set_error("wf_quant_rows_i8: mode %d", mode);
        return WF_EUNSUPPORTED;
    }
    WF_LAUNCH_CHECK("wf_quant_rows_i8 launch");
    return WF_OK;
}

extern "C" int wf_quant_rows_i8_pre(const void* x_bf16, int64_t M, int64_t K, int pre, const void* s_bf16,
                                    const void* shift_bf16, int64_t rows_per_group, float eps, int8_t* xq, float* xs,
                                    void* stream) {
    using namespace wf;
    const int rc = check_rows("wf_quant_rows_i8_pre", x_bf16, M, K, xq, xs);
    if (rc != WF_OK || M == 0) return rc;
    if (pre < 0 || pre > 3) { set_error("wf_quant_rows_i8_pre: operation %d", pre); return WF_EUNSUPPORTED; }
    if (K % 256 || K > kMaxRowK || (pre == 3 && K % 512)) {
        set_error("wf_quant_rows_i8_pre: K = %lld (K %% 256 == 0, K <= %d; LayerNorm K %% 512 == 0)", (long long)K,
                  kMaxRowK);
        return WF_EUNSUPPORTED;
    }
    if (pre >= 1 && !s_bf16) { set_error("wf_quant_rows_i8_pre: null pointer"); return WF_EINVAL; }
    if (pre >= 2) {
        if (!shift_bf16) { set_error("wf_quant_rows_i8_pre: null pointer"); return WF_EINVAL; }
        if (rows_per_group <= 0 || M % rows_per_group) {
            set_error("wf_quant_rows_i8_pre: M = %lld is not a whole number of %lld-row groups", (long long)M,
                      (long long)rows_per_group);
            return WF_EUNSUPPORTED;
        }
        if (!aligned(s_bf16, 16) || !aligned(shift_bf16, 16)) {
            set_error("wf_quant_rows_i8_pre: scale and shift must be 16-byte aligned");
            return WF_EUNSUPPORTED;
        }
    }
    if (pre == 1 && !aligned(s_bf16, 2)) { set_error("wf_quant_rows_i8_pre: table alignment"); return WF_EUNSUPPORTED; }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint16_t* xp = static_cast<const uint16_t*>(x_bf16);
    const PreArgs pa{static_cast<const uint16_t*>(s_bf16), static_cast<const uint16_t*>(shift_bf16),
                     rows_per_group > 0 ? rows_per_group : 1, eps};
    const int k = (int)K;
    if (pre == 0) launch_convrot<0>(xp, M, k, xq, xs, pa, s);
    else if (pre == 1 && gelu_in_lds(M, k)) launch_convrot<1>(xp, M, k, xq, xs, pa, s);
    else if (pre == 1 && k <= 1024) launch_convrot_pre<1, 4, 1>(xp, M, k, xq, xs, pa, s);
    else if (pre == 1) launch_convrot_pre<2, 4, 1>(xp, M, k, xq, xs, pa, s);      // (1280 values, many rows)
    else if (pre == 2) launch_convrot<2>(xp, M, k, xq, xs, pa, s);
    else launch_convrot<3>(xp, M, k, xq, xs, pa, s);
    WF_LAUNCH_CHECK("wf_quant_rows_i8_pre launch");
    return WF_OK;
}
