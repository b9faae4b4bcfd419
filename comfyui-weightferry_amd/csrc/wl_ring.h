// Main loop and epilogue store of the GEMMs whose operands stream in whole 128-byte lines (gemm_bf16.hip, the int8
// GEMM's wl forms in gemm_i8.hip): C[BM x BN] += A[BM rows, K] . B[BN rows, K]^T, both operands K-major, 16-byte
// MFMA fragments (v_mfma_f32_32x32x16_bf16 and v_mfma_i32_32x32x32_i8 both take 16 bytes of row l % 32 at byte
// 16 (l / 32) of a 32-byte K step).
//
// Each K stage is 128 bytes of every row of both operands, loaded global -> LDS by the load unit (buffer_load ...
// lds): one 1 KiB load covers 8 rows x one whole cache line, the swizzle applied on the global side (lane l loads
// the chunk that belongs in slot l). Two stage buffers: the loads of stage p + 1 fly while stage p is computed. The
// texture-data return path pays per cache line touched, so whole-line stages cost it half of what 64-byte half-line
// stages do; that path, not the MFMA, bounded the 64-byte form of these tilings.
//
// One barrier per stage, before the last K step's MFMAs: each wave has waited for its own loads of stage p + 1 and
// for its own fragment reads of stage p, so after the barrier stage p + 1 is whole and stage p's buffer is free; the
// loads of stage p + 2 go out into it and the first fragments of stage p + 1 are read, both between the MFMAs of stage
// p's last K step (scheduling barriers keep the compiler from sinking the loads towards the next wait).
#pragma once

#include "lds_ring.h"

namespace wf {

typedef int32_t wl_frag __attribute__((ext_vector_type(4)));   // one 16-byte MFMA operand fragment

template <int VM_, int VN_, int WM_, int WN_>
struct WlShape {
    static constexpr int VM = VM_, VN = VN_, WM = WM_, WN = WN_;
    static constexpr int NT = 64 * VM * VN, NW = NT / 64;
    static constexpr int BM = VM * WM * 32, BN = VN * WN * 32;
    static constexpr int AI = BM / 8, BI = BN / 8;            // 1 KiB loads per stage (8 rows of 128 bytes)
    static constexpr int IPW = (AI + BI + NW - 1) / NW;       // per wave; spare issues of the last waves fill pad slots
    static constexpr int SLOTS = NW * IPW * 64;               // 16-byte slots per stage buffer
    static_assert(2 * SLOTS * 16 <= 160 * 1024, "two stage buffers fit the LDS");
};

// acc[i][j] (MFMA tile i of the wave's rows, j of its columns) over nk stages from stage s0 of rows [0, BM) of ra and
// [0, BN) of rb, KB bytes a row. sb0 / sb1: the kernel's two __shared__ stage buffers of S::SLOTS fragments (separate
// arrays, so the compiler tracks the loads into each on its own). mma(acc, a, b) returns acc + a . b.
//
// The order of a K step is pinned: behind each MFMA the next K step's fragment reads that fall to it, and in the last
// step the next stage's loads, one by one, each followed by a scheduling barrier. Left to the compiler the reads come
// in a burst before the MFMAs and the loads in one behind them; spread, they pass under the matrix unit. Measured on
// MI355X, in turn on random operands (us): int8 5152 x 8192 x 2048 92.6 against 95.3, 4096 x 5120 x 5120 89.3 against 90.0;
// bf16 4096 x 5120 x 5120 159.3 against 161.7, 4096 x 13824 x 5120 454.1 against 458.6. At 16384 rows, under the power
// limit, the runs resolve no difference (int8 16384 x 5120 x 5120 362 against 364, 16384 x 13824 x 5120 982 against 982).
// What is left is the loads' and the reads' own cost: bf16 16384 x 5120 x 5120 takes 636, 551 without the loads, 529
// without the reads, 419 with neither.
template <typename S, typename Acc, typename Mma>
__device__ __forceinline__ void wl_mainloop(__amdgpu_buffer_rsrc_t ra, __amdgpu_buffer_rsrc_t rb, uint32_t KB, int s0,
                                            int nk, int wave, int lane, wl_frag* sb0, wl_frag* sb1,
                                            Acc (&acc)[S::WM][S::WN], Mma&& mma) {
    constexpr int WM = S::WM, WN = S::WN, AI = S::AI, BI = S::BI, IPW = S::IPW, BM = S::BM;
    constexpr int READS = WM + WN, MFMAS = WM * WN;
    const int wm = wave / S::VN, wn = wave % S::VN;
    // load gi covers rows 8 g .. 8 g + 7 of its operand (g = gi, or gi - AI for B); lane l takes row 8 g + l / 8,
    // chunk swz8(row, l % 8) = swz8(l / 8, l % 8) ^ 4 (g & 1): two per-lane offsets and a wave-uniform row term
    const uint32_t lo_even = (uint32_t)(lane / 8) * KB + 16u * (uint32_t)swz8(lane / 8, lane % 8);
    const uint32_t lo_odd = lo_even ^ 64u;
    auto issue = [&](wl_frag* st, int kt, int q) {             // load q of this wave's IPW of stage kt
        const uint32_t k0 = (uint32_t)kt * 128u;
        const int gi = wave * IPW + q;
        const int gc = min(gi, AI + BI - 1);                   // a pad issue repeats the last B run into its pad slot
        const int g = gc < AI ? gc : gc - AI;
        lds_dma16(gc < AI ? ra : rb, st + 64 * gi, ((g & 1) ? lo_odd : lo_even) + (uint32_t)(8 * g) * KB + k0);
    };
    // fragment of K step ks (this lane's 16-byte half lk) of row r sits at slot r * 8 + swz8(r, 2 ks + lk) =
    // (r * 8 + swz8(r, lk)) ^ 2 ks; the swizzle depends on r % 16 only, so the wave's MFMA tiles (32 rows apart) sit
    // at constant distances from its first: one base per operand, XORed per K step
    const int lr = lane & 31, lk = lane >> 5;
    const int arow = wm * WM * 32 + lr, brow = wn * WN * 32 + lr;
    const int abase = arow * 8 + swz8(arow, lk), bbase = BM * 8 + brow * 8 + swz8(brow, lk);
    wl_frag fa[2][WM], fb[2][WN];
    auto fread = [&](const wl_frag* st, int ks, int set, auto rc) {    // read rc of a K step: a0, the b's, the other a's
        constexpr int r = decltype(rc)::value;
        if constexpr (r == 0) fa[set][0] = st[abase ^ (2 * ks)];
        else if constexpr (r <= WN) fb[set][r - 1] = (st + (bbase ^ (2 * ks)))[(r - 1) * 256];
        else fa[set][r - WN] = (st + (abase ^ (2 * ks)))[(r - WN) * 256];
    };
    // the MFMAs of `set`, between them the reads of K step ks of st into the other set and, with `load`, the loads of
    // stage kt into `free_`
    auto kstep = [&](auto load, int set, const wl_frag* st, int ks, wl_frag* free_, int kt) {
        static_for<MFMAS>([&](auto mc) {
            constexpr int m = decltype(mc)::value;
            acc[m / WN][m % WN] = mma(acc[m / WN][m % WN], fa[set][m / WN], fb[set][m % WN]);
            constexpr int r0 = m * READS / MFMAS, r1 = (m + 1) * READS / MFMAS;
            static_for<r1 - r0>([&](auto x) {
                fread(st, ks, set ^ 1, std::integral_constant<int, r0 + decltype(x)::value>{});
            });
            if constexpr (decltype(load)::value) {
                constexpr int q0 = m * IPW / MFMAS, q1 = (m + 1) * IPW / MFMAS;
                static_for<q1 - q0>([&](auto x) { issue(free_, kt, q0 + decltype(x)::value); });
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // stages at or past the last read past the slice's or row's end (other rows' bytes, or zeros past the buffer) into
    // a buffer no later stage reads: the loads always issue, so the compiler's per-buffer load tracking stays exact
    static_for<IPW>([&](auto q) { issue(sb0, s0, decltype(q)::value); });
    static_for<IPW>([&](auto q) { issue(sb1, s0 + 1, decltype(q)::value); });
    wait_vm<IPW>();                                      // the first stage landed; the second may be in flight
    wave_barrier_sync();
    static_for<READS>([&](auto rc) { fread(sb0, 0, 0, rc); });
    // stage p in cur (its first fragments already in set 0), stage p + 1 flying into oth
    auto step = [&](int p, wl_frag* cur, wl_frag* oth) {
        kstep(std::false_type{}, 0, cur, 1, nullptr, 0);
        kstep(std::false_type{}, 1, cur, 2, nullptr, 0);
        kstep(std::false_type{}, 0, cur, 3, nullptr, 0);
        wait_vm<0>();                                    // stage p + 1 landed (this wave's loads)
        __builtin_amdgcn_s_waitcnt(0xc07f);              // lgkmcnt(0): this wave's reads of cur are done
        wave_barrier_sync();                             // ... and every wave's: cur is free, p + 1 is whole
        kstep(std::true_type{}, 1, oth, 0, cur, p + 2);
    };
    int p = 0;
    for (; p + 2 <= nk; p += 2) {
        step(s0 + p, sb0, sb1);
        step(s0 + p + 1, sb1, sb0);
    }
    if (p < nk) step(s0 + p, sb0, sb1);
    wait_vm<0>();                                        // the stage buffers are idle from here on
    __builtin_amdgcn_s_waitcnt(0xc07f);
    wave_barrier_sync();
}

// Region of wave w for the epilogue: 32 rows x WN * 32 values of 16 bits in the idle stage buffers.
template <typename S>
__device__ __forceinline__ uint16_t* wl_out_region(wl_frag* sb0, wl_frag* sb1, int wave) {
    constexpr int PER_BUF = S::SLOTS * 16 / (32 * S::WN * 32 * 2);
    static_assert(PER_BUF >= 1 && S::NW <= PER_BUF * 2, "the output rows fit in the stage buffers");
    return reinterpret_cast<uint16_t*>(wave / PER_BUF == 0 ? sb0 : sb1) + (wave % PER_BUF) * 32 * S::WN * 32;
}

// What wl_store_tile does to a finished run of 8 outputs before it is stored; this one leaves it as it is. prefetch(m,
// n) loads what the run at row m, column n needs (in range), run(v, f, m, n) combines it; one(v, m, n) does the same
// to a single value.
struct StoreAsIs {
    struct Fetched {};
    static constexpr bool vec_ok = true;
    __device__ __forceinline__ Fetched prefetch(int, int) const { return {}; }
    __device__ __forceinline__ uint4 run(uint4 v, const Fetched&, int, int) const { return v; }
    __device__ __forceinline__ uint16_t one(uint16_t v, int, int) const { return v; }
};

// Rows [m0, m0 + ROWS) x columns [n0, n0 + TC) of Y from the wave's finished 16-bit values in LDS (row-major, TC a row),
// for outputs whose rows are not whole aligned 16-byte runs: 64 consecutive values a store (a lane that stores 8 of its
// own writes 2 bytes in every 16). Rows past M are not walked, and eight stores' LDS reads, and what fin loads for them,
// are in flight together; one after another over every row they cost few rows more than the wider stores give. us, lane by
// lane / one after another / here: int8 4096 x 5119 x 5120 115 / 98 / 97, 8 x 2607 x 3136 17.5 / 20.2 / 17.4, 300 x 3001 x
// 704 11.5 / 12.8 / 11.3; with the residual 26 x 12332 x 2624 36.0 / 39.5 / 28.0, 1500 x 2047 x 4096 46.7 / 51.1 / 34.5;
// bf16 4096 x 5119 x 5120 184 / 166 / 165, 5 x 6297 x 8192 75.4 / 78.0 / 75.1.
template <int TC, int ROWS, typename Fin>
__device__ __forceinline__ void store_values(const uint16_t* ot, uint16_t* Y, int M, int N, int m0, int n0, int lane,
                                             const Fin& fin) {
    static_assert(ROWS * TC % 512 == 0, "whole groups of eight stores");
    const int stores = n0 < N ? (min(M - m0, ROWS) * TC + 63) / 64 : 0;
    for (int it = 0; it < stores; it += 8) {
        uint16_t v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = ot[(it + u) * 64 + lane];
#pragma unroll
        for (int u = 0; u < 8; u++) {                      // (whatever fin loads, before a store could hold it up)
            const int q = (it + u) * 64 + lane;
            v[u] = fin.one(v[u], min(m0 + q / TC, M - 1), min(n0 + q % TC, N - 1));
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int q = (it + u) * 64 + lane, m = m0 + q / TC, n = n0 + q % TC;
            if (m < M && n < N) Y[(int64_t)m * N + n] = v[u];
        }
    }
}

// Stores the wave's WM * 32 x WN * 32 output tile at rows mw.., columns nw.. of Y [M, N] (16-bit values), 32 rows at
// a time through its LDS region ot: bits(i, j, e) gives the output bits of accumulator element e of MFMA tile (i, j)
// (row mw + 32 i + 8 (e / 4) + 4 (lane / 32) + e % 4, column nw + 32 j + lane % 32), fin's run() or one() the value
// stored. Whole 16-byte row runs go out when N % 8 == 0 and Y is 16-byte aligned, single values otherwise. The wave
// reads back only its own region, and its LDS writes and reads execute in order.
template <int WM, int WN, typename Bits, typename Fin = StoreAsIs>
__device__ __forceinline__ void wl_store_tile(uint16_t* ot, uint16_t* Y, int M, int N, int mw, int nw, int lane,
                                              Bits&& bits, const Fin& fin = Fin{}) {
    constexpr int TC = WN * 32, RUNS = TC / 8, NIT = 32 * RUNS / 64;
    const int lr = lane & 31, lk = lane >> 5;
    const uint4* ov = reinterpret_cast<const uint4*>(ot);
    const bool vec = (N & 7) == 0 && (reinterpret_cast<uintptr_t>(Y) & 15) == 0 && fin.vec_ok;
#pragma unroll
    for (int i = 0; i < WM; i++) {
        const int mi = mw + i * 32;
        typename Fin::Fetched f[NIT];
        if (vec) {
#pragma unroll
            for (int it = 0; it < NIT; it++) {
                const int q = it * 64 + lane;
                f[it] = fin.prefetch(min(mi + q / RUNS, M - 1), min(nw + 8 * (q % RUNS), N - 8));
            }
        }
#pragma unroll
        for (int e = 0; e < 16; e++)
#pragma unroll
            for (int j = 0; j < WN; j++) ot[(8 * (e >> 2) + 4 * lk + (e & 3)) * TC + j * 32 + lr] = bits(i, j, e);
        if (vec) {
#pragma unroll
            for (int it = 0; it < NIT; it++) {
                const int q = it * 64 + lane, r = q / RUNS, c = q % RUNS;
                const int m = mi + r, n = nw + 8 * c;
                const uint4 v = ov[q];
                if (m < M && n < N) *reinterpret_cast<uint4*>(Y + (int64_t)m * N + n) = fin.run(v, f[it], m, n);
            }
        } else {
            store_values<TC, 32>(ot, Y, M, N, mi, nw, lane, fin);
        }
    }
}

}  // namespace wf
