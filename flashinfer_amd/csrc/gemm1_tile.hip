// Grouped FP8 GEMM1 + SwiGLU, LDS-tiled variant for many rows per expert.
//
// Same contract as gemm1_stream_kernel (solution/triton/kernel.py:69-186 and
// :301-330): act[s, j] = silu(G[s, I+j]) * G[s, j] with
//   G[s, n] = sum_kb sa[kb, tok(s)] * sb1[e, n/128, kb] * (A8[tok(s), kb-block] . W1[e, n, kb-block]).
//
// A workgroup of WM x WN waves computes a tile of BM = 64*WM rows (slots of
// one expert) by BG = 64*WN gate columns plus the BG matching up columns.
// Per 128-wide k-block (one scale block) the A rows (gathered by token), the
// 2*BG weight rows and the BM activation scales are copied global -> LDS
// with global_load_lds_dwordx4 into one of two stages, so the copy of
// k-block kb+1 overlaps the MFMAs on kb; one barrier per k-block.
// Each wave owns 64 rows x (64 gate + 64 up) columns: 4 x 8 MFMA tiles of
// v_mfma_scale_f32_16x16x128_f8f6f4, each scaled by sa*sb in fp32 as it is
// accumulated. The SwiGLU epilogue pairs gate and up columns in registers.
//
// LDS rows are 128 bytes; 16-byte chunk c of row r sits at position
// c ^ swz8(r), so the 16 rows read by lanes 0..15 hit distinct banks.
#include "tile_common.hpp"

namespace mimoe {

template <int WM, int WN>
struct G1Tile {
    static constexpr int NW = WM * WN;
    static constexpr int THREADS = 64 * NW;
    static constexpr int BM = 64 * WM;
    static constexpr int BG = 64 * WN;
    static constexpr int NT = I / BG;
    static constexpr int A_BYTES = BM * BLK;
    static constexpr int B_BYTES = 2 * BG * BLK;
    static constexpr int SA_BYTES = BM * 4;
    static constexpr int STAGE = A_BYTES + B_BYTES + SA_BYTES;
    static constexpr int A_LD = A_BYTES / 1024 / NW;  // 1 KB copies per wave per stage
    static constexpr int B_LD = B_BYTES / 1024 / NW;
    static constexpr int SA_WAVES = BM / 64;          // waves copying one scale each per lane
    static_assert(A_BYTES % (1024 * NW) == 0 && B_BYTES % (1024 * NW) == 0, "loader split");
    static_assert(SA_WAVES <= NW, "scale loader");
    static_assert(2 * STAGE <= 160 * 1024, "LDS budget");
};

template <int WM, int WN, int GM>
__global__ __launch_bounds__(64 * WM * WN) void gemm1_tile_kernel(
    Plan p, const uint8_t* __restrict__ hs, const float* __restrict__ hs_scale,
    const uint8_t* __restrict__ w1, const float* __restrict__ w1s) {
    using C = G1Tile<WM, WN>;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * C::STAGE];

    int e, row0, nrows, nt;
    if (!tile_coords<C::NT, GM>(p.meta, META_MTILE1, C::BM, e, row0, nrows, nt)) return;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int jb = nt * C::BG;

    // Loader: in its i-th copy, wave w fills LDS rows 8*(w*LD + i) .. +7;
    // lane l takes row +l/8, chunk position l%8.
    uint32_t a_off[C::A_LD], b_off[C::B_LD];
#pragma unroll
    for (int i = 0; i < C::A_LD; ++i) {
        const int row = 8 * (wave * C::A_LD + i) + (lane >> 3);
        const int c = (lane & 7) ^ swz8(row);
        const int tok = p.sorted_tok[row0 + min(row, nrows - 1)];
        a_off[i] = (uint32_t)tok * H + c * 16;
    }
#pragma unroll
    for (int i = 0; i < C::B_LD; ++i) {
        const int row = 8 * (wave * C::B_LD + i) + (lane >> 3);
        const int c = (lane & 7) ^ swz8(row);
        const int wrow = row < C::BG ? jb + row : I + jb + (row - C::BG);
        b_off[i] = (uint32_t)((e * N1 + wrow) * H + c * 16);
    }
    uint32_t sa_off = 0;
    if (wave < C::SA_WAVES) {
        const int row = 64 * wave + lane;
        sa_off = (uint32_t)p.sorted_tok[row0 + min(row, nrows - 1)];
    }

    // Copies whose 8 rows all lie past the expert's last row are skipped
    // (wave-uniform): those LDS rows only feed MFMA rows that are never
    // stored, and at medium T most of a 256-row tile is such rows.
    auto issue = [&](int stage, int kb) __attribute__((always_inline)) {
        uint8_t* s = smem + stage * C::STAGE;
#pragma unroll
        for (int i = 0; i < C::A_LD; ++i)
            if (8 * (wave * C::A_LD + i) < nrows)
                g2l16(hs + a_off[i] + kb * BLK, s + (wave * C::A_LD + i) * 1024);
#pragma unroll
        for (int i = 0; i < C::B_LD; ++i)
            g2l16(w1 + b_off[i] + kb * BLK, s + C::A_BYTES + (wave * C::B_LD + i) * 1024);
        if (wave < C::SA_WAVES)
            g2l4(hs_scale + (size_t)kb * p.T + sa_off, s + C::A_BYTES + C::B_BYTES + wave * 256);
    };

    const int wm = wave % WM, wn = wave / WM;
    const int r = lane & 15, g = lane >> 4;
    const float* sbg_p = w1s + ((size_t)e * N1B + jb / BLK) * HB;
    const float* sbu_p = w1s + ((size_t)e * N1B + (I + jb) / BLK) * HB;

    v4f acc[4][8];
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int n = 0; n < 8; ++n) acc[m][n] = zero;

    issue(0, 0);
    wait_vmem();
    __syncthreads();

#pragma unroll 1
    for (int kb = 0; kb < HB; ++kb) {
        const int cur = kb & 1;
        const uint8_t* sA = smem + cur * C::STAGE;
        const uint8_t* sB = sA + C::A_BYTES;
        const float* sSA = reinterpret_cast<const float*>(sB + C::B_BYTES);

        // Waves whose 64 rows lie past the expert's last row (partial row
        // tiles) only copy; the branch is wave-uniform.
        const bool active = wm * 64 < nrows;
        v8i a[4];
        if (active) {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const int row = wm * 64 + m * 16 + r;
                const uint8_t* base = sA + row * BLK;
                const int sw = swz8(row);
                const v4i lo = lds16(base + ((g ^ sw) << 4));
                const v4i hi = lds16(base + (((g + 4) ^ sw) << 4));
                a[m] = (v8i){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            }
        }
        // The copy of k-block kb+1 goes out after this wave's A reads, so its
        // LDS writes do not compete with them.
        if (kb + 1 < HB) issue(cur ^ 1, kb + 1);
        if (!active) {
            wait_vmem();
            __syncthreads();
            continue;
        }
        // Per-row scale products sa*sb for the gate half, then (re-read from
        // LDS) for the up half: one set of 16 registers instead of two.
        float cs[4][4];
        auto set_scales = [&](float sb) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const float4 s4 = *reinterpret_cast<const float4*>(sSA + wm * 64 + m * 16 + g * 4);
                cs[m][0] = s4.x * sb; cs[m][1] = s4.y * sb; cs[m][2] = s4.z * sb; cs[m][3] = s4.w * sb;
            }
        };
        // B fragments are read one column tile ahead so the LDS latency of
        // tile n+1 overlaps the MFMAs of tile n.
        auto read_b = [&](int n) __attribute__((always_inline)) {
            const int brow = (n < 4) ? (wn * 64 + n * 16 + r) : (C::BG + wn * 64 + (n - 4) * 16 + r);
            const uint8_t* base = sB + brow * BLK;
            const int sw = swz8(brow);
            const v4i lo = lds16(base + ((g ^ sw) << 4));
            const v4i hi = lds16(base + (((g + 4) ^ sw) << 4));
            return (v8i){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        };
        set_scales(sbg_p[kb]);
        v8i bnext = read_b(0);
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            if (n == 4) set_scales(sbu_p[kb]);
            const v8i b = bnext;
            if (n < 7) bnext = read_b(n + 1);
            // four independent MFMAs, then their scale-and-accumulate
            v4f pr[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) pr[m] = mfma_f8_16x16x128(a[m], b, zero);
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                acc[m][n][0] += pr[m][0] * cs[m][0];
                acc[m][n][1] += pr[m][1] * cs[m][1];
                acc[m][n][2] += pr[m][2] * cs[m][2];
                acc[m][n][3] += pr[m][3] * cs[m][3];
            }
        }
        wait_vmem();
        __syncthreads();
    }

#pragma unroll
    for (int m = 0; m < 4; ++m) {
#pragma unroll
        for (int n = 0; n < 4; ++n) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = wm * 64 + m * 16 + g * 4 + i;
                if (row < nrows) {
                    const float v = silu(acc[m][n + 4][i]) * acc[m][n][i];
                    store_act(p, (size_t)(row0 + row) * I + jb + wn * 64 + n * 16 + r, v);
                }
            }
        }
    }
}

// The same tile with the MFMA operands swapped and the MFMAs software-
// pipelined against their scale FMAs (variant 18).
//
// Weight rows are the MFMA's A operand and gathered activation rows its B
// operand, so lane l receives D[4g+v][l%16]: four output columns 4g..4g+3 of
// one row (r = l%16) of a 16x16 tile. The per-(row, k-block) activation
// scale and the per-(128 columns, k-block) weight scale then combine into a
// single factor u per lane and tile: 8 products per k-block per lane instead
// of 32, and the SwiGLU epilogue stores 4 adjacent bf16 (8 bytes) per lane.
// The activation scales sit in LDS as [row group][r][m], so one 16-byte read
// gives a lane the scales of its rows m*16 + r (m = 0..3).
//
// Inside a k-block the 32 MFMAs of a wave (8 column tiles x 4 row tiles) run
// as one sequence; the four scale-and-accumulate FMAs of MFMA t issue after
// MFMA t+2, so they execute while the matrix core works on later tiles
// rather than waiting on the result just issued. The last two MFMAs' FMAs
// carry into the next k-block. Weight fragments are read from LDS one column
// tile ahead.
template <int WM, int WN, int GM>
__global__ __launch_bounds__(64 * WM * WN) void gemm1_tile_t_kernel(
    Plan p, const uint8_t* __restrict__ hs, const float* __restrict__ hs_scale,
    const uint8_t* __restrict__ w1, const float* __restrict__ w1s) {
    using C = G1Tile<WM, WN>;
    static_assert(WN * 64 * 2 == 2 * C::BG && C::BG == 64 * WN, "column tiling");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * C::STAGE];

    int e, row0, nrows, nt;
    if (!tile_coords<C::NT, GM>(p.meta, META_MTILE1, C::BM, e, row0, nrows, nt)) return;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int jb = nt * C::BG;

    uint32_t a_off[C::A_LD], b_off[C::B_LD];
#pragma unroll
    for (int i = 0; i < C::A_LD; ++i) {
        const int row = 8 * (wave * C::A_LD + i) + (lane >> 3);
        const int c = (lane & 7) ^ swzq(row);
        const int tok = p.sorted_tok[row0 + min(row, nrows - 1)];
        a_off[i] = (uint32_t)tok * H + c * 16;
    }
#pragma unroll
    for (int i = 0; i < C::B_LD; ++i) {
        const int row = 8 * (wave * C::B_LD + i) + (lane >> 3);
        const int c = (lane & 7) ^ swzq(row);
        const int wrow = row < C::BG ? jb + row : I + jb + (row - C::BG);
        b_off[i] = (uint32_t)((e * N1 + wrow) * H + c * 16);
    }
    // scale loader: wave w < WM copies the 64 scales of rows 64w.., lane l
    // to LDS position 64w + l, which holds row 64w + (l % 4) * 16 + l / 4
    uint32_t sa_off = 0;
    if (wave < C::SA_WAVES) {
        const int row = 64 * wave + (lane & 3) * 16 + (lane >> 2);
        sa_off = (uint32_t)p.sorted_tok[row0 + min(row, nrows - 1)];
    }

    auto issue = [&](int stage, int kb) __attribute__((always_inline)) {
        uint8_t* s = smem + stage * C::STAGE;
#pragma unroll
        for (int i = 0; i < C::A_LD; ++i)
            if (8 * (wave * C::A_LD + i) < nrows)
                g2l16(hs + a_off[i] + kb * BLK, s + (wave * C::A_LD + i) * 1024);
#pragma unroll
        for (int i = 0; i < C::B_LD; ++i)
            g2l16(w1 + b_off[i] + kb * BLK, s + C::A_BYTES + (wave * C::B_LD + i) * 1024);
        if (wave < C::SA_WAVES)
            g2l4(hs_scale + (size_t)kb * p.T + sa_off, s + C::A_BYTES + C::B_BYTES + wave * 256);
    };

    const int wm = wave % WM, wn = wave / WM;
    const int r = lane & 15, g = lane >> 4;
    const float* sbg_p = w1s + ((size_t)e * N1B + jb / BLK) * HB;
    const float* sbu_p = w1s + ((size_t)e * N1B + (I + jb) / BLK) * HB;

    // acc[n][m]: column tile n (0..3 gate, 4..7 up) x row tile m
    v4f acc[8][4];
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
        for (int m = 0; m < 4; ++m) acc[n][m] = zero;

    issue(0, 0);
    wait_vmem();
    __syncthreads();

    const bool active = wm * 64 < nrows;  // wave-uniform: rows past the expert only copy
    // MFMA results of the last two tiles of the previous k-block and their
    // scale factors, applied early in the next one
    v4f carry0 = zero, carry1 = zero;
    float cu0 = 0.f, cu1 = 0.f;

#pragma unroll 1
    for (int kb = 0; kb < HB; ++kb) {
        const int cur = kb & 1;
        const uint8_t* sA = smem + cur * C::STAGE;
        const uint8_t* sB = sA + C::A_BYTES;
        const float* sSA = reinterpret_cast<const float*>(sB + C::B_BYTES);

        v8i a[4];
        float4 s4 = {0.f, 0.f, 0.f, 0.f};
        auto read_b = [&](int n) __attribute__((always_inline)) {
            const int brow = (n < 4) ? (wn * 64 + n * 16 + r) : (C::BG + wn * 64 + (n - 4) * 16 + r);
            const uint8_t* base = sB + brow * BLK;
            const int sw = swzq(brow);
            const v4i lo = lds16(base + ((g ^ sw) << 4));
            const v4i hi = lds16(base + (((g + 4) ^ sw) << 4));
            return (v8i){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        };
        v8i bcur = {0, 0, 0, 0, 0, 0, 0, 0};
        if (active) {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const int row = wm * 64 + m * 16 + r;
                const uint8_t* base = sA + row * BLK;
                const int sw = swzq(row);
                const v4i lo = lds16(base + ((g ^ sw) << 4));
                const v4i hi = lds16(base + (((g + 4) ^ sw) << 4));
                a[m] = (v8i){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            }
            s4 = *reinterpret_cast<const float4*>(sSA + wm * 64 + r * 4);
            bcur = read_b(0);
        }
        // The copy of k-block kb+1 goes out after this wave's fragment reads.
        if (kb + 1 < HB) issue(cur ^ 1, kb + 1);
        if (!active) {
            wait_vmem();
            __syncthreads();
            continue;
        }
        const float sbg = sbg_p[kb], sbu = sbu_p[kb];
        const float sam[4] = {s4.x, s4.y, s4.z, s4.w};
        float ug[4], uu[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) { ug[m] = sam[m] * sbg; uu[m] = sam[m] * sbu; }

        v4f pr[32];
        v8i bnext = bcur;
#pragma unroll
        for (int t = 0; t < 32; ++t) {
            const int n = t >> 2, m = t & 3;
            if (m == 0 && n + 1 < 8) bnext = read_b(n + 1);
            pr[t] = mfma_f8_16x16x128(bcur, a[m], zero);
            if (m == 3) bcur = bnext;
            if (t >= 2) {
                const int tn = (t - 2) >> 2, tm = (t - 2) & 3;
                const float u = tn < 4 ? ug[tm] : uu[tm];
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[tn][tm][v] += pr[t - 2][v] * u;
            } else if (t == 0) {
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[7][2][v] += carry0[v] * cu0;
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[7][3][v] += carry1[v] * cu1;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        carry0 = pr[30];
        carry1 = pr[31];
        cu0 = uu[2];
        cu1 = uu[3];
        wait_vmem();
        __syncthreads();
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        acc[7][2][v] += carry0[v] * cu0;
        acc[7][3][v] += carry1[v] * cu1;
    }

    if (!active) return;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int row = wm * 64 + m * 16 + r;
        if (row < nrows) {
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                uint32_t w[2], wl[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const float v0 = silu(acc[n + 4][m][2 * h]) * acc[n][m][2 * h];
                    const float v1 = silu(acc[n + 4][m][2 * h + 1]) * acc[n][m][2 * h + 1];
                    const uint16_t h0 = f2bf(v0), h1 = f2bf(v1);
                    w[h] = (uint32_t)h0 | ((uint32_t)h1 << 16);
                    wl[h] = (uint32_t)f2bf(v0 - bf2f(h0)) | ((uint32_t)f2bf(v1 - bf2f(h1)) << 16);
                }
                const size_t idx = (size_t)(row0 + row) * I + jb + wn * 64 + n * 16 + 4 * g;
                *reinterpret_cast<uint2*>(p.act + idx) = make_uint2(w[0], w[1]);
                if (p.act_lo) *reinterpret_cast<uint2*>(p.act_lo + idx) = make_uint2(wl[0], wl[1]);
            }
        }
    }
}

// The same 256 x (128 + 128) tile with its waves in two groups that take turns
// at the matrix cores (variant 19).
//
// Waves 0-3 (group 0: rows 0-127) and 4-7 (group 1: rows 128-255) share the
// four SIMDs, one wave of each group per SIMD; wave wn of a group owns 32
// gate columns and the matching 32 up columns. A k-block is four phases per
// wave, a barrier after each, and group 1 runs one phase behind group 0:
//   M0: read the weight fragments and row tiles 0-3 from LDS
//   C0: their 16 MFMAs
//   M1: read row tiles 4-7
//   C1: their 16 MFMAs
// so in every slot one wave of a SIMD multiplies from registers while the
// other one reads LDS, issues copies and applies the last scale factors. What
// bounded the one-group pipeline this replaces was LDS reads and barriers
// with an empty matrix core queue (all waves read their fragments at the same
// time): 2,657 cycles a k-block now against about 4,450 before, 2,048 of
// them MFMA. The rest is power: with random data the clock falls to 1.6-1.8
// GHz in this loop (2.1-2.2 in the same loop without its copies), so bytes
// and operations saved count as much as cycles. GEMM1 by events, alternating
// processes: T=14000 with every token on 8 experts 2,925 -> 2,585 us, T=8192
// 416 -> 372, T=2048 192 -> 185, T=1024 with 1,966 slots 202 -> 194.
//
// Copies (two stages): the weights and row tiles 0-3 of k-block kb + 2 go out
// in M1 of kb, after both groups have read theirs of kb (group 1 in the slot
// before); row tiles 4-7 of kb + 1 go out in M0 of kb. Either has six slots
// (1.5 k-blocks) to land. The copies that the next slot's readers need are
// waited for by the wave that issued them (vmcnt of the NV copies issued
// since) before the barrier that ends the slot: for group 0 that is the end
// of C0 / C1, for group 1, one slot behind, the end of M0 / M1.
//
// A tile of at most 128 rows gives each group 64 of them (M, C; two phases a
// k-block, half the activation copies) and uses the LDS for three stages. An
// expert's last row tile is often one.
//
// MFMA operands are swapped as in variant 18 (weights are the A operand, so a
// lane holds four output columns of one row and one scale factor per tile),
// and each MFMA's four scale FMAs issue LAG MFMAs later; the last ones of a
// phase run in the M phase after it. Same products and order of sums as
// variants 3 and 18, bitwise.
struct G1P {
    static constexpr int NW = 8;
    static constexpr int THREADS = 64 * NW;
    static constexpr int BM = 256;
    static constexpr int BG = 128;
    static constexpr int NT = I / BG;
    static constexpr int B_BYTES = 2 * BG * BLK;
    // stage: activation rows | weight rows | row scales
    static constexpr int A_BYTES = BM * BLK;
    static constexpr int STAGE = A_BYTES + B_BYTES + BM * 4;
    static constexpr int A2_BYTES = 128 * BLK;  // tiles of at most 128 rows
    static constexpr int STAGE2 = A2_BYTES + B_BYTES + 128 * 4;
    static constexpr int SMEM = 2 * STAGE > 3 * STAGE2 ? 2 * STAGE : 3 * STAGE2;
    static constexpr int LAG = 3;
    static_assert(SMEM + 2 * 64 * 4 <= 160 * 1024, "LDS budget");
    static_assert(HB <= 64 && HB >= 2, "weight scales: one lane per k-block");
};

// End of a phase: this wave's LDS reads are done and at most N of its copies
// are outstanding; then the workgroup's barrier.
template <int N>
__device__ __forceinline__ void phase_end() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
__device__ __forceinline__ void phase_end() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int GM>
__global__ __launch_bounds__(512) void gemm1_tile_p_kernel(
    Plan p, const uint8_t* __restrict__ hs, const float* __restrict__ hs_scale,
    const uint8_t* __restrict__ w1, const float* __restrict__ w1s) {
    using C = G1P;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[C::SMEM];
    __shared__ __attribute__((aligned(16))) float s_sb[2 * 64];  // [gate | up][kb] weight scales

    int e, row0, nrows, nt;
    if (!tile_coords<C::NT, GM>(p.meta, p.g1_mtile, C::BM, e, row0, nrows, nt)) return;
    // wave-uniform by construction; kept in SGPRs for the copies' scalar bases
    e = __builtin_amdgcn_readfirstlane(e);
    nt = __builtin_amdgcn_readfirstlane(nt);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 3, wm = wave >> 2;
    const int r = lane & 15, g = lane >> 4;
    const int jb = nt * C::BG;
    const bool small = nrows <= 128;

    auto token = [&](int row) __attribute__((always_inline)) {
        return (uint32_t)p.sorted_tok[row0 + min(row, nrows - 1)];
    };
    uint32_t b_off[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = 8 * (wave * 4 + i) + (lane >> 3);
        const int c = (lane & 7) ^ swzq(row);
        const int wrow = row < C::BG ? jb + row : I + jb + (row - C::BG);
        b_off[i] = (uint32_t)((e * N1 + wrow) * H + c * 16);
    }
    // copies address their rows as a k-block base (SGPRs) + a 32-bit offset
    auto issue_b = [&](uint8_t* dst, int k) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) g2l16s(w1 + k * BLK, b_off[i], dst + (wave * 4 + i) * 1024);
    };
    // The tile's weight scales (one 128-column block of gate, one of up, for
    // every k-block) are copied once by waves 4 and 5.
    if (wave == 4 || wave == 5) {
        const int nb = wave == 4 ? jb / BLK : (I + jb) / BLK;
        if (lane < HB) g2l4s(w1s + ((size_t)e * N1B + nb) * HB, lane * 4, s_sb + (wave - 4) * 64);
    }

    // fragment of 16 rows at s: this lane's row r, 16-byte chunks g and g + 4
    const int lo_off = r * BLK + ((g ^ swzq(r)) << 4), hi_off = r * BLK + (((g + 4) ^ swzq(r)) << 4);
    auto frag = [&](const uint8_t* s) __attribute__((always_inline)) {
        const v4i lo = lds16(s + lo_off);
        const v4i hi = lds16(s + hi_off);
        return (v8i){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    };
    // weight rows of column tile n (0, 1 gate; 2, 3 up) in a stage's weight region
    auto bcol = [&](int n) __attribute__((always_inline)) {
        return (n < 2 ? 32 * wn + 16 * n : C::BG + 32 * wn + 16 * (n - 2)) * BLK;
    };
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    v8i bfr[4], afr[4];   // fragments of the phase: weights, four row tiles
    float ug[4], uu[4];   // sa * sb of this lane's rows for the gate and up columns
    v4f pr[16];
    auto scale4 = [&](v4f& a, int t) __attribute__((always_inline)) {
        const float u = (t & 3) < 2 ? ug[t >> 2] : uu[t >> 2];
#pragma unroll
        for (int v = 0; v < 4; ++v) a[v] += pr[t][v] * u;
    };
    auto factors = [&](const float4& sa, float sbg, float sbu) __attribute__((always_inline)) {
        const float s4[4] = {sa.x, sa.y, sa.z, sa.w};
#pragma unroll
        for (int m = 0; m < 4; ++m) { ug[m] = s4[m] * sbg; uu[m] = s4[m] * sbu; }
    };
    // C phase: 16 MFMAs into acc[0..3] and the scale FMAs of all but the last
    // LAG. Empty asm statements keep the compiler from sinking those MFMAs
    // below the barrier.
    auto multiply = [&](v4f (*acc)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            pr[t] = mfma_f8_16x16x128(bfr[t & 3], afr[t >> 2], zero);
            if (t >= C::LAG) scale4(acc[(t - C::LAG) >> 2][(t - C::LAG) & 3], t - C::LAG);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int t = 16 - C::LAG; t < 16; ++t) asm volatile("" : "+v"(pr[t]));
        __builtin_amdgcn_sched_barrier(0);
    };
    // the last LAG scale FMAs of the phase before
    auto finish = [&](v4f (*acc)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 16 - C::LAG; t < 16; ++t) scale4(acc[t >> 2][t & 3], t);
#pragma unroll
        for (int m = 0; m < 4; ++m)
            asm volatile("" : "+v"(acc[m][0]), "+v"(acc[m][1]), "+v"(acc[m][2]), "+v"(acc[m][3]));
    };
    auto store_row = [&](int row, const v4f (&a)[4]) __attribute__((always_inline)) {
        if (row >= nrows) return;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            uint32_t w[2], wl[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float v0 = silu(a[n + 2][2 * h]) * a[n][2 * h];
                const float v1 = silu(a[n + 2][2 * h + 1]) * a[n][2 * h + 1];
                const uint16_t h0 = f2bf(v0), h1 = f2bf(v1);
                w[h] = (uint32_t)h0 | ((uint32_t)h1 << 16);
                wl[h] = (uint32_t)f2bf(v0 - bf2f(h0)) | ((uint32_t)f2bf(v1 - bf2f(h1)) << 16);
            }
            const size_t idx = (size_t)(row0 + row) * I + jb + wn * 32 + n * 16 + 4 * g;
            *reinterpret_cast<uint2*>(p.act + idx) = make_uint2(w[0], w[1]);
            if (p.act_lo) *reinterpret_cast<uint2*>(p.act_lo + idx) = make_uint2(wl[0], wl[1]);
        }
    };

    // A tile of more than 128 rows. G: the wave's group; MT: its row tiles
    // that are multiplied (8; 4 when its rows past 64 lie beyond the expert).
    auto large_tile = [&](auto g_c, auto mt_c) __attribute__((always_inline)) {
        constexpr int G = decltype(g_c)::value;
        constexpr int MT = decltype(mt_c)::value;
        constexpr int NV = 4 + 2 + (G == 0) + 2;  // weights, rows, group 0's row scales, rows
        // activation halves: rows 0-63 and 128-191 (row tiles 0-3 of both
        // groups), rows 64-127 and 192-255
        uint32_t a_off[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int j = wave * 2 + (i & 1);
            const int row = (i >> 1) * 64 + (j >> 3) * 128 + (j & 7) * 8 + (lane >> 3);
            a_off[i] = token(row) * H + ((lane & 7) ^ swzq(row)) * 16;
        }
        // row scales sit in LDS as [row group][r][m] (row 128wm + 16m + r), so
        // a lane reads those of its 8 rows as two 16-byte vectors; wave w of
        // group 0 copies 64 of them
        uint32_t sa_off = 0;
        if constexpr (G == 0) {
            const int idx = 64 * wave + lane;
            sa_off = token(128 * (idx >> 7) + 16 * (idx & 7) + ((idx & 127) >> 3)) * 4;
        }
        auto issue_a = [&](int half, int kb) __attribute__((always_inline)) {
            uint8_t* s = smem + (kb & 1) * C::STAGE;
            const uint8_t* base = hs + min(kb, HB - 1) * BLK;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int j = wave * 2 + i;
                g2l16s(base, a_off[half * 2 + i], s + (half * 64 + (j >> 3) * 128 + (j & 7) * 8) * BLK);
            }
        };
        auto issue_ba = [&](int kb) __attribute__((always_inline)) {
            uint8_t* s = smem + (kb & 1) * C::STAGE + C::A_BYTES;
            const int k = min(kb, HB - 1);
            issue_b(s, k);
            issue_a(0, kb);
            if constexpr (G == 0) g2l4s(hs_scale + (size_t)k * p.T, sa_off, s + C::B_BYTES + wave * 256);
        };
        issue_ba(0);
        issue_a(1, 0);
        issue_ba(1);
        phase_end<NV>();
        if constexpr (G == 1) phase_end();

        v4f acc[8][4];
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < 4; ++n) acc[m][n] = zero;
        // The copies of k-blocks past the last repeat it into regions that no
        // wave reads again.
#pragma unroll 1
        for (int kb = 0; kb < HB; ++kb) {
            const uint8_t* st = smem + (kb & 1) * C::STAGE;
            const uint8_t* sA = st + wm * 128 * BLK;
            const float* sSA = reinterpret_cast<const float*>(st + C::A_BYTES + C::B_BYTES) + wm * 128 + r * 8;
            // M0
#pragma unroll
            for (int n = 0; n < 4; ++n) bfr[n] = frag(st + C::A_BYTES + bcol(n));
#pragma unroll
            for (int m = 0; m < 4; ++m) afr[m] = frag(sA + m * 16 * BLK);
            const float4 sa0 = *reinterpret_cast<const float4*>(sSA);
            // read here, not in M1: group 0 copies kb + 2's scales over them there
            float4 sa1 = sa0;
            if constexpr (MT > 4) sa1 = *reinterpret_cast<const float4*>(sSA + 4);
            const float sbg = s_sb[kb], sbu = s_sb[64 + kb];
            __builtin_amdgcn_sched_barrier(0);
            issue_a(1, kb + 1);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (MT > 4) {
                if (kb) finish(acc + 4);
            }
            factors(sa0, sbg, sbu);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (G == 1) phase_end<NV>(); else phase_end();
            // C0
            __builtin_amdgcn_sched_barrier(0);
            multiply(acc);
            if constexpr (G == 0) phase_end<NV>(); else phase_end();
            // M1
            if constexpr (MT > 4) {
#pragma unroll
                for (int m = 0; m < 4; ++m) afr[m] = frag(sA + (64 + m * 16) * BLK);
                __builtin_amdgcn_sched_barrier(0);
            }
            issue_ba(kb + 2);
            __builtin_amdgcn_sched_barrier(0);
            finish(acc);
            if constexpr (MT > 4) factors(sa1, sbg, sbu);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (G == 1) phase_end<NV>(); else phase_end();
            // C1
            if constexpr (MT > 4) {
                __builtin_amdgcn_sched_barrier(0);
                multiply(acc + 4);
            }
            if constexpr (G == 0) phase_end<NV>(); else phase_end();
        }
        if constexpr (MT > 4) finish(acc + 4);
        if constexpr (G == 0) phase_end();
        wait_vmem();  // no copy into LDS may be pending when the workgroup ends
#pragma unroll
        for (int m = 0; m < MT; ++m) store_row(wm * 128 + m * 16 + r, acc[m]);
    };

    // A tile of at most 128 rows: group wm takes rows 64wm .. 64wm+63, two
    // phases a k-block, three stages. Rows past the expert (ACTIVE false) only
    // copy, in step with the others.
    auto small_tile = [&](auto g_c, auto active_c) __attribute__((always_inline)) {
        constexpr int G = decltype(g_c)::value;
        constexpr bool ACTIVE = decltype(active_c)::value;
        constexpr int NV = 4 + 2 + (G == 0);
        uint32_t a_off[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = (wave * 2 + i) * 8 + (lane >> 3);
            a_off[i] = token(row) * H + ((lane & 7) ^ swzq(row)) * 16;
        }
        // row scales as [row group][r][m] (row 64wm + 16m + r); waves 2 and 3
        // repeat the copies of waves 0 and 1, so that a group's waves count alike
        uint32_t sa_off = 0;
        if constexpr (G == 0) {
            const int idx = 64 * (wave & 1) + lane;
            sa_off = token(64 * (idx >> 6) + 16 * (idx & 3) + ((idx & 63) >> 2)) * 4;
        }
        auto issue = [&](int so, int kb) __attribute__((always_inline)) {
            uint8_t* s = smem + so;
            const int k = min(kb, HB - 1);
            issue_b(s + C::A2_BYTES, k);
#pragma unroll
            for (int i = 0; i < 2; ++i) g2l16s(hs + k * BLK, a_off[i], s + (wave * 2 + i) * 1024);
            if constexpr (G == 0)
                g2l4s(hs_scale + (size_t)k * p.T, sa_off, s + C::A2_BYTES + C::B_BYTES + (wave & 1) * 256);
        };
        issue(0, 0);
        issue(C::STAGE2, 1);
        phase_end<NV>();
        if constexpr (G == 1) phase_end();

        v4f acc[4][4];
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int n = 0; n < 4; ++n) acc[m][n] = zero;
        int s0 = 0, s2 = 2 * C::STAGE2;  // stages of kb and kb + 2
#pragma unroll 1
        for (int kb = 0; kb < HB; ++kb) {
            const uint8_t* st = smem + s0;
            // M
            float4 sa;
            float sbg, sbu;
            if constexpr (ACTIVE) {
#pragma unroll
                for (int n = 0; n < 4; ++n) bfr[n] = frag(st + C::A2_BYTES + bcol(n));
#pragma unroll
                for (int m = 0; m < 4; ++m) afr[m] = frag(st + (wm * 64 + m * 16) * BLK);
                sa = *reinterpret_cast<const float4*>(
                    reinterpret_cast<const float*>(st + C::A2_BYTES + C::B_BYTES) + wm * 64 + r * 4);
                sbg = s_sb[kb];
                sbu = s_sb[64 + kb];
                __builtin_amdgcn_sched_barrier(0);
            }
            issue(s2, kb + 2);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (ACTIVE) {
                if (kb) finish(acc);
                factors(sa, sbg, sbu);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (G == 1) phase_end<NV>(); else phase_end();
            // C
            if constexpr (ACTIVE) {
                __builtin_amdgcn_sched_barrier(0);
                multiply(acc);
            }
            if constexpr (G == 0) phase_end<NV>(); else phase_end();
            s0 = s0 == 2 * C::STAGE2 ? 0 : s0 + C::STAGE2;
            s2 = s2 == 2 * C::STAGE2 ? 0 : s2 + C::STAGE2;
        }
        if constexpr (ACTIVE) finish(acc);
        if constexpr (G == 0) phase_end();
        wait_vmem();  // no copy into LDS may be pending when the workgroup ends
        if constexpr (ACTIVE) {
#pragma unroll
            for (int m = 0; m < 4; ++m) store_row(wm * 64 + m * 16 + r, acc[m]);
        }
    };

    if (small) {
        if (wm == 0)
            small_tile(IntC<0>{}, BoolC<true>{});
        else if (nrows > 64)
            small_tile(IntC<1>{}, BoolC<true>{});
        else
            small_tile(IntC<1>{}, BoolC<false>{});
    } else if (wm == 0) {
        large_tile(IntC<0>{}, IntC<8>{});
    } else if (nrows > 192) {
        large_tile(IntC<1>{}, IntC<8>{});
    } else {
        large_tile(IntC<1>{}, IntC<4>{});
    }
}

hipError_t launch_gemm1_tile(const Plan& p, const uint8_t* hs, const float* hs_scale,
                             const uint8_t* w1, const float* w1s, int variant, hipStream_t s) {
    if (variant == 19) {
        // 8 row tiles per XCD walk: with 16, 2 columns x 16 rows of tiles run at
        // a time and copy 1.5x the distinct lines of 4 x 8 (T=14000 with every
        // token on 8 experts 2,755 against 2,705 us; T=8192 level).
        const int tiles = max_mtiles(p.T, G1P::BM) * G1P::NT;
        hipLaunchKernelGGL((gemm1_tile_p_kernel<8>), dim3((tiles + 7) / 8 * 8), dim3(G1P::THREADS), 0,
                           s, p, hs, hs_scale, w1, w1s);
    } else if (variant == 18) {
        using C = G1Tile<4, 2>;
        const int tiles = max_mtiles(p.T, C::BM) * C::NT;
        hipLaunchKernelGGL((gemm1_tile_t_kernel<4, 2, 16>), dim3((tiles + 7) / 8 * 8),
                           dim3(C::THREADS), 0, s, p, hs, hs_scale, w1, w1s);
    } else if (variant == 3) {
        using C = G1Tile<4, 2>;
        const int tiles = max_mtiles(p.T, C::BM) * C::NT;
        dim3 grid((tiles + 7) / 8 * 8);
        hipLaunchKernelGGL((gemm1_tile_kernel<4, 2, 16>), grid, dim3(C::THREADS), 0, s, p, hs,
                           hs_scale, w1, w1s);
    } else {
        using C = G1Tile<2, 2>;
        const int tiles = max_mtiles(p.T, C::BM) * C::NT;
        dim3 grid((tiles + 7) / 8 * 8);
        hipLaunchKernelGGL((gemm1_tile_kernel<2, 2, 4>), grid, dim3(C::THREADS), 0, s, p, hs,
                           hs_scale, w1, w1s);
    }
    return hipGetLastError();
}

}  // namespace mimoe
