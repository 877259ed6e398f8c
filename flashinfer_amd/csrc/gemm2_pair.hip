// Grouped GEMM2 (fp8 weights) from SwiGLU values held as e4m3 pairs: the LDS
// tile of prefill sizes whose two wave groups take turns at the matrix cores.
//
// Replaces solution/triton/kernel.py:221-280 (_grouped_gemm2_kernel) and the
// routing-weight multiply of :337-368 where GEMM1 wrote act as hi + lo / 16
// (Plan::act_sc). Each weight fragment meets the two halves in two fp8 MFMAs
// that chain into one accumulator; lo's 2^-4 is the scale of the weight
// operand, the 32-column blocks' exponents the scales of the activations. The
// weights need no conversion, their fragments half the registers, so a wave
// holds 128 x 64 outputs and the workgroup 256 x 256: a k-block copies 96 KB
// for what the bf16 tile (128 x 256) copies 128 KB for.
#include "tile_common.hpp"

namespace mimoe {

namespace {

// 256 rows x 256 columns, 8 waves: group wm = wave / 4 (one wave of each group
// per SIMD) owns rows 128wm .. 128wm+127, wave wn of a group 64 columns. A
// k-block is four quarters q of 32 rows per group, each an M phase (read the
// activations from LDS, with q = 0 the weights) and a C phase (16 MFMAs),
// group 1 one phase behind group 0, so that one wave of a SIMD multiplies
// while the other reads, copies and applies the last block scales.
//
// One stage: a quarter's region (or the weights') is free once group 1 has
// read it, one slot after group 0, and takes the next k-block's copy in the M
// phase after, six slots before group 0 reads it again. Waits are counted per
// wave as in GEMM1's tile (gemm1_tile_p_kernel): at most N copies younger than
// the ones that the next slot reads, at the end of C (group 0) or M (group 1).
//
// Measured on MI355X (GEMM2 alone, one process, medians) against the
// persistent bf16 tile: T=14000 with every token on 8 experts 3,126 -> 2,703 us
// (1.05 -> 1.22 PF), T=8192 399 -> 373 where the slots fill 70 % of the tiles'
// rows; slower where they fill half (pairs_pay decides). One workgroup per CU
// that walks its XCD's tiles, against one per tile: 2,703 against 2,755 us,
// 373 against 382. In a register-only loop random e4m3 pairs ran 14 % faster
// than bf16 with the weights widened at the same power. What is left: ~6 us of
// a tile's ~50 before its first and after its last MFMA, and the clock, which
// random data holds at 1.6-1.8 GHz.
struct G2P {
    static constexpr int THREADS = 512;
    static constexpr int BM = GEMM2_PAIR_BM, BN = 256, NT = H / BN;
    static constexpr int B_BYTES = BN * BLK;
    static constexpr int Q_HALF = 64 * BLK;        // 64 rows (32 per group) of hi or lo
    static constexpr int Q_BYTES = 2 * Q_HALF;
    static constexpr int STAGE = B_BYTES + 4 * Q_BYTES;
    static constexpr int STAGE2 = B_BYTES + 2 * Q_BYTES;  // tiles of at most 128 rows, two stages
    static constexpr int SMEM = STAGE > 2 * STAGE2 ? STAGE : 2 * STAGE2;
    static constexpr int ROW = 2 * I;              // bytes of an act row
    static_assert(H % BN == 0 && BN / BLK == 2, "two 128-column weight scales per tile");
    static_assert(IB <= 32 && IB >= 4 && IB % 4 == 0, "weight scales: one lane per k-block and column block");
    static_assert(STAGE + IB * BM * 4 <= SMEM, "the second half of a large tile's exponents");
    static_assert(SMEM + IB * BM * 4 + 2 * (BM + 2 * 32) * 4 <= 160 * 1024, "LDS budget");
    static_assert((long long)BM * ROW < (1LL << 31), "tile offsets fit 32 bits");
};

template <int GM>
__global__ __launch_bounds__(512) void gemm2_pair_kernel(Plan p, const uint8_t* __restrict__ w2,
                                                         const float* __restrict__ w2s) {
    using C = G2P;
    // the stages, then exponents [kb][row]
    __shared__ __attribute__((aligned(1024))) uint8_t smem[C::SMEM + IB * C::BM * 4];
    __shared__ __attribute__((aligned(16))) float s_w[2][C::BM];        // routing weights

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave & 3, wm = wave >> 2;
    // Lane terms, set per tile from an opaque lane index: held across the tile
    // loop, what the forms below derive from them spills.
    int lane, r, g;
    FragOff fo(0, 0);
    int ar;        // copies: row of the quarter, group ar / 32, row ar % 32 of its 32
    uint32_t ac;   // and byte of the row
    uint32_t b_off[2];
    auto opaque = [&]() __attribute__((always_inline)) {
        int l = lane;
        asm volatile("" : "+v"(l));
        return l;
    };
    auto set_lane = [&]() __attribute__((always_inline)) {
        lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        r = lane & 15;
        g = lane >> 4;
        fo = FragOff(r, g);
        ar = wave * 8 + (lane >> 3);
        ac = ((lane & 7) ^ swzq(ar)) * 16;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = 32 * wave + 8 * i + (lane >> 3);
            b_off[i] = (uint32_t)row * I + ((lane & 7) ^ swzq(row)) * 16;
        }
    };

    // Activation copies go through a resource over the tile's rows: rows past
    // the expert arrive as zeros without being read. A wave copies 8 of a
    // quarter's 64 rows, hi and lo.
    struct Tile {
        int e, row0, nrows, nt;
    };
    auto locate = [&](int t) __attribute__((always_inline)) {
        Tile x;
        tile_at<C::NT, GM>(p.meta, META_MTILE2B, C::BM, t, x.e, x.row0, x.nrows, x.nt);
        x.e = __builtin_amdgcn_readfirstlane(x.e);
        x.nt = __builtin_amdgcn_readfirstlane(x.nt);
        x.row0 = __builtin_amdgcn_readfirstlane(x.row0);
        x.nrows = __builtin_amdgcn_readfirstlane(x.nrows);
        return x;
    };
    // what the copies read: the tile's activation rows and weight rows
    v4i rows;
    const uint8_t* wb;
    auto aim = [&](const Tile& x) __attribute__((always_inline)) {
        const uint64_t a = (uint64_t)p.act + (uint64_t)x.row0 * C::ROW;
        rows = (v4i){(int)(uint32_t)a, (int)((uint32_t)(a >> 32) & 0xffffu), x.nrows * C::ROW, 0x00020000};
        wb = w2 + ((size_t)x.e * H + x.nt * C::BN) * I;
    };
    const int total = p.meta[META_MTILE2B + EL] * C::NT;
    const int per_xcd = (total + 7) >> 3;
    const int t_step = gridDim.x >> 3;
    const int t_first = (blockIdx.x & 7) * per_xcd;
    const int t_end = min(total, t_first + per_xcd);
    int t = t_first + (blockIdx.x >> 3);
    if (t >= t_end) return;

    auto issue_b = [&](uint8_t* dst, int kb) __attribute__((always_inline)) {
        const uint8_t* base = wb + kb * BLK;
#pragma unroll
        for (int i = 0; i < 4; ++i) g2l16s(base + (i >> 1) * 16 * I, b_off[i & 1], dst + (wave * 4 + i) * 1024);
    };
    // quarter q of k-block kb; av: this lane's offset in quarter 0
    auto issue_q = [&](uint8_t* dst, uint32_t av, int q, int kb) __attribute__((always_inline)) {
        const uint32_t so = q * 32 * C::ROW + kb * (2 * BLK);
        b2l16(rows, av, so, dst + wave * 1024);
        b2l16(rows, av, so + BLK, dst + C::Q_HALF + wave * 1024);
    };
    // The exponents of k-block kb of a tile's sr rows (256; 128 in tiles of at
    // most 128 rows; rows past the expert repeat its last): 64 rows a wave, the
    // waves past them repeat the same copy, so that all waves count alike.
    auto issue_ex = [&](uint32_t* dst, const Tile& x, int sr, int kb) __attribute__((always_inline)) {
        const int part = (wave & (sr / 64 - 1)) * 64;
        g2l4s(p.act_sc + (size_t)kb * ((size_t)TOPK * p.T) + x.row0, (uint32_t)min(part + opaque(), x.nrows - 1) * 4,
              dst + kb * sr + part);
    };
    // A tile's routing weights, read by its epilogue.
    auto issue_w = [&](int buf, const Tile& x) __attribute__((always_inline)) {
        if (wave < 4)
            g2l4s(p.sorted_w + x.row0, (uint32_t)min(wave * 64 + opaque(), x.nrows - 1) * 4, &s_w[buf][wave * 64]);
    };

    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    // A wave's operands; local to a tile, so that none is live across the loop.
    struct Regs {
        v8i bfr[4], afr[2][2];  // weight fragments of the k-block; [row tile][hi | lo] of the quarter
        int sc[2];              // exponents of this lane's rows (32-column block g)
        float sb, sb_last;      // weight scale of this k-block and of the one before
        v4f pr[8];
    };
    int wsc = 127 | (123 << 8);  // weight operand's scale bytes: 2^0 for hi, 2^-4 for lo
    asm volatile("" : "+v"(wsc));
    int buf = 0;  // half of the constants' buffers that holds this tile's
    auto load_b = [&](Regs& w, const uint8_t* s, const float* wsb, int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 4; ++n) w.bfr[n] = lds_frag(s + (wn * 64 + n * 16) * BLK, fo);
        w.sb_last = w.sb;
        w.sb = wsb[kb];  // uniform: a scalar load
    };
    // ex: the quarter's exponents of this group's 32 rows
    auto load_q = [&](Regs& w, const uint8_t* s, const uint32_t* ex) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const uint8_t* sr = s + (wm * 32 + m * 16) * BLK;
            w.afr[m][0] = lds_frag(sr, fo);
            w.afr[m][1] = lds_frag(sr + C::Q_HALF, fo);
            w.sc[m] = reinterpret_cast<const uint8_t*>(ex + m * 16 + r)[g];
        }
    };
    // C phase: 8 units of 16 x 16 outputs, hi and lo chained. A unit's scale
    // FMAs issue three MFMAs after its last one; the last two units' run in
    // the next M phase (finish). The empty asm keeps them on this side.
    auto multiply = [&](Regs& w, v4f (*acc)[4]) __attribute__((always_inline)) {
        auto hi = [&](int u) __attribute__((always_inline)) {
            w.pr[u] = mfma_mx_16x16x128<0>(w.bfr[u & 3], wsc, w.afr[u >> 2][0], w.sc[u >> 2], zero);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto lo = [&](int u) __attribute__((always_inline)) {
            w.pr[u] = mfma_mx_16x16x128<1>(w.bfr[u & 3], wsc, w.afr[u >> 2][1], w.sc[u >> 2], w.pr[u]);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto add = [&](int u) __attribute__((always_inline)) {
            if (u < 0) return;
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[u >> 2][u & 3][v] += w.pr[u][v] * w.sb;
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int u = 0; u < 8; u += 2) {
            hi(u);
            hi(u + 1);
            add(u - 2);
            lo(u);
            add(u - 1);
            lo(u + 1);
        }
        asm volatile("" : "+v"(w.pr[6]));
        asm volatile("" : "+v"(w.pr[7]));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto finish = [&](Regs& w, v4f (*acc)[4], float s) __attribute__((always_inline)) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            acc[1][2][v] += w.pr[6][v] * s;
            acc[1][3][v] += w.pr[7][v] * s;
        }
#pragma unroll
        for (int m = 0; m < 2; ++m)
            asm volatile("" : "+v"(acc[m][0]), "+v"(acc[m][1]), "+v"(acc[m][2]), "+v"(acc[m][3]));
    };
    // Epilogue: routing weight (kernel.py:364), bf16 row for the combine.
    auto store_row = [&](const Tile& x, int l, int row, const v4f (&a)[4]) __attribute__((always_inline)) {
        row += l & 15;
        if (row >= x.nrows) return;
        const float w = s_w[buf][row];
        uint16_t* o = p.part + (size_t)(x.row0 + row) * H + x.nt * C::BN + wn * 64 + 4 * (l >> 4);
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const uint32_t u = (uint32_t)f2bf(w * a[n][0]) | ((uint32_t)f2bf(w * a[n][1]) << 16);
            const uint32_t v = (uint32_t)f2bf(w * a[n][2]) | ((uint32_t)f2bf(w * a[n][3]) << 16);
            *reinterpret_cast<uint2*>(o + n * 16) = make_uint2(u, v);
        }
    };

    // Ends a pipeline: no copy in flight, no wave still reading LDS.
    auto drain = [&](int group) __attribute__((always_inline)) {
        wait_vmem();
        if (group == 0) phase_end();  // group 1's last phase
        phase_end();
    };

    // A tile's pipeline runs on into the next tile of the workgroup where that
    // one has the same form (more, or at most, 128 rows): in place of k-blocks
    // past the last, the copies are the next tile's first ones and its
    // constants go to the buffers' other half. `primed`: the tile before did
    // this for x. Otherwise those copies repeat k-block IB - 1 into regions no
    // wave reads again, and the next tile starts a pipeline after this one
    // has drained.
    //
    // A tile of more than 128 rows. G: the wave's group; NQ: its quarters with
    // rows (4; 2 when its rows past 64 lie beyond the expert).
    auto large_tile = [&](auto g_c, auto nq_c, const Tile& x, const Tile& y, bool primed, bool on)
        __attribute__((always_inline)) {
        constexpr int G = decltype(g_c)::value;
        constexpr int NQ = decltype(nq_c)::value;
        uint8_t* const sB = smem;
        uint8_t* const sA = smem + C::B_BYTES;
        const uint32_t av = (uint32_t)((ar >> 5) * 128 + (ar & 31)) * C::ROW + ac;
        // exponents: after the stages, or in the bytes past this form's one stage
        auto exps = [&](int b) __attribute__((always_inline)) {
            return reinterpret_cast<uint32_t*>(smem + (b ? C::STAGE : C::SMEM));
        };
        const int last = on ? 0 : IB - 1;  // k-block copied in place of IB
        auto issue_a = [&](int q, int kb) __attribute__((always_inline)) {
            issue_q(sA + q * C::Q_BYTES, av, q, kb == IB ? last : kb);
        };
        if (!primed) {
            aim(x);
#pragma unroll 1
            for (int kb = 0; kb < IB; ++kb) issue_ex(exps(buf), x, C::BM, kb);
            issue_b(sB, 0);
            issue_a(0, 0);
            issue_a(1, 0);
            issue_a(2, 0);
            phase_end<4>();
            if constexpr (G == 1) phase_end();
        }
        issue_w(buf, x);
        Regs w;
        w.sb = 0.f;
        w.pr[6] = zero;
        w.pr[7] = zero;
        const float* const wsb = w2s + ((size_t)x.e * HB + x.nt * 2 + (wn >> 1)) * IB;
        v4f acc[2 * NQ][4];
#pragma unroll
        for (int m = 0; m < 2 * NQ; ++m)
#pragma unroll
            for (int n = 0; n < 4; ++n) acc[m][n] = zero;
        const uint32_t* const ex = exps(buf) + wm * 128;
#pragma unroll 1
        for (int kb = 0; kb < IB; ++kb) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                // M
                if (q < NQ) {
                    if (q == 0) load_b(w, sB, wsb, kb);
                    load_q(w, sA + q * C::Q_BYTES, ex + kb * C::BM + q * 32);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (q == 0) issue_a(3, kb);
                if (q == 1) {
                    if (on && kb == IB - 1) aim(y);
                    issue_b(sB, kb == IB - 1 ? last : kb + 1);
                }
                if (q == 2) issue_ex(exps(buf ^ 1), y, C::BM, kb);
                if (q >= 1) issue_a(q - 1, kb + 1);
                __builtin_amdgcn_sched_barrier(0);
                if (q >= 1 && q <= NQ) finish(w, acc + 2 * (q - 1), w.sb);
                if (q == 0 && NQ == 4) finish(w, acc + 2 * NQ - 2, w.sb_last);
                __builtin_amdgcn_sched_barrier(0);
                // what the next slot reads: quarter q + 1 (after 3, the next
                // k-block's weights and quarter 0)
                auto landed = [&]() __attribute__((always_inline)) {
                    if (q == 0) phase_end<4>(); else if (q == 1) phase_end<8>(); else if (q == 2) phase_end<9>(); else phase_end<5>();
                };
                if (G == 1) landed(); else phase_end();
                // C
                if (q < NQ) {
                    __builtin_amdgcn_sched_barrier(0);
                    multiply(w, acc + 2 * q);
                }
                if (G == 0) landed(); else phase_end();
            }
        }
        if constexpr (NQ == 4) finish(w, acc + 6, w.sb);
        if (!on) drain(G);
        const int l = opaque();
#pragma unroll
        for (int m = 0; m < 2 * NQ; ++m) store_row(x, l, wm * 128 + m * 16, acc[m]);
    };

    // A tile of at most 128 rows: group wm takes rows 64wm .. 64wm+63 as two
    // quarters; two stages, copied as in GEMM1's tile. NQ 0: copies only.
    auto small_tile = [&](auto g_c, auto nq_c, const Tile& x, const Tile& y, bool primed, bool on)
        __attribute__((always_inline)) {
        constexpr int G = decltype(g_c)::value;
        constexpr int NQ = decltype(nq_c)::value;
        constexpr int SR = 128;
        const uint32_t av = (uint32_t)((ar >> 5) * 64 + (ar & 31)) * C::ROW + ac;
        auto exps = [&](int b) __attribute__((always_inline)) { 
            return reinterpret_cast<uint32_t*>(smem + C::SMEM + b * (IB * SR * 4));
        };
        auto issue_a = [&](int q, int kb) __attribute__((always_inline)) {
            issue_q(smem + (kb & 1) * C::STAGE2 + C::B_BYTES + q * C::Q_BYTES, av, q, kb < IB ? kb : on ? kb - IB : IB - 1);
        };
        auto issue_ba = [&](int kb) __attribute__((always_inline)) {
            if (on && kb == IB) aim(y);
            issue_b(smem + (kb & 1) * C::STAGE2, kb < IB ? kb : on ? kb - IB : IB - 1);
            issue_a(0, kb);
        };
        if (!primed) {
            aim(x);
#pragma unroll 1
            for (int kb = 0; kb < IB; ++kb) issue_ex(exps(buf), x, SR, kb);
            issue_ba(0);
            issue_a(1, 0);
            issue_ba(1);
            phase_end<8>();
            if constexpr (G == 1) phase_end();
        }
        issue_w(buf, x);
        Regs w;
        w.sb = 0.f;
        w.pr[6] = zero;
        w.pr[7] = zero;
        const float* const wsb = w2s + ((size_t)x.e * HB + x.nt * 2 + (wn >> 1)) * IB;
        v4f acc[4][4];
#pragma unroll
        for (int m = 0; m < 2 * NQ; ++m)
#pragma unroll
            for (int n = 0; n < 4; ++n) acc[m][n] = zero;
        const uint32_t* const ex = exps(buf) + wm * 64;
#pragma unroll 1
        for (int kb = 0; kb < IB; ++kb) {
            const uint8_t* st = smem + (kb & 1) * C::STAGE2;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                // M
                if (q < NQ) {
                    if (q == 0) load_b(w, st, wsb, kb);
                    load_q(w, st + C::B_BYTES + q * C::Q_BYTES, ex + kb * SR + q * 32);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (q == 0) {
                    issue_ex(exps(buf ^ 1), y, SR, kb);
                    issue_a(1, kb + 1);
                } else {
                    issue_ba(kb + 2);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (q == 1 && NQ > 0) finish(w, acc, w.sb);
                if (q == 0 && NQ == 2) finish(w, acc + 2, w.sb_last);
                __builtin_amdgcn_sched_barrier(0);
                if (G == 1) phase_end<9>(); else phase_end();
                // C
                if (q < NQ) {
                    __builtin_amdgcn_sched_barrier(0);
                    multiply(w, acc + 2 * q);
                }
                if (G == 0) phase_end<9>(); else phase_end();
            }
        }
        if constexpr (NQ == 2) finish(w, acc + 2, w.sb);
        if (!on) drain(G);
        const int l = opaque();
#pragma unroll
        for (int m = 0; m < 2 * NQ; ++m) store_row(x, l, wm * 64 + m * 16, acc[m]);
    };

    Tile x = locate(t);
    bool primed = false;
    for (;;) {
        set_lane();
        const bool more = t + t_step < t_end;
        Tile y = x;
        if (more) y = locate(t + t_step);
        const bool on = more && (x.nrows <= 128) == (y.nrows <= 128);
        if (x.nrows <= 128) {
            const int mine = x.nrows - wm * 64;
            if (wm == 0) {
                if (mine > 32) small_tile(IntC<0>{}, IntC<2>{}, x, y, primed, on);
                else small_tile(IntC<0>{}, IntC<1>{}, x, y, primed, on);
            } else {
                if (mine > 32) small_tile(IntC<1>{}, IntC<2>{}, x, y, primed, on);
                else if (mine > 0) small_tile(IntC<1>{}, IntC<1>{}, x, y, primed, on);
                else small_tile(IntC<1>{}, IntC<0>{}, x, y, primed, on);
            }
        } else if (wm == 0) {
            large_tile(IntC<0>{}, IntC<4>{}, x, y, primed, on);
        } else if (x.nrows > 192) {
            large_tile(IntC<1>{}, IntC<4>{}, x, y, primed, on);
        } else {
            large_tile(IntC<1>{}, IntC<2>{}, x, y, primed, on);
        }
        if (!more) break;
        t += t_step;
        x = y;
        buf ^= 1;
        primed = on;
    }
}

}  // namespace

hipError_t launch_gemm2_pair(const Plan& p, const uint8_t* w2, const float* w2s, hipStream_t s) {
    const int tiles = (max_mtiles(p.T, G2P::BM) * G2P::NT + 7) / 8 * 8;
    const int cus = persistent_grid();
    hipLaunchKernelGGL((gemm2_pair_kernel<4>), dim3(tiles < cus ? tiles : cus), dim3(G2P::THREADS), 0, s, p, w2, w2s);
    return hipGetLastError();
}

}  // namespace mimoe
