// Dequant-fused matmul for mid-sized M (17 .. a few hundred rows, a few thousand of a narrow matrix) on gfx950.
//
// With so few rows there is one row tile (or a handful), so the tiled kernel's tile count
// - N / 256 - leaves most CUs idle unless K is split across workgroups, and every split
// costs a round trip of fp32 partial sums through memory.  Here the split along K happens
// inside the workgroup: a workgroup owns a strip of only 64 output columns (128 for a
// rotary head), and its four or eight waves each run the tiled kernel's wave loop over their own
// contiguous part of K.  The waves share nothing while they stream: each has its own
// double-buffered activation tile in LDS, filled by its own LDS-direct loads, so the loop
// has no barrier at all.  At the end the accumulator sets meet in LDS, where the waves share the
// row blocks among them.
//
// Wave tile: (32*MT) rows x NB blocks of 64 columns.
//   plain   : NB = 1, one 64-column strip; or (WIDE, long K and many rows) NB = 2, two adjacent strips.
//   SiLU*mul: NB = 2, the same 64 columns of the gate and of the up matrix.
//   rotary  : NB = 2, columns [0, 64) and [64, 128) of one head, so the wave that finishes
//             a row block holds d and d + 64 itself; or (PAIRED, few rows) NB = 1: 32 columns of a head and their
//             32 rotation partners, the two columns of a lane being d and d + 64.
// With NB = 2 every activation fragment read from LDS feeds twice as many MFMAs.
//
// Weights are decoded exactly once per row tile.  K can still be split across workgroups
// on top (last-arriver protocol of the other kernels) when the strips do not fill the
// chip; the partial sums exchanged are the workgroup's already reduced tile.
#include "gptq4_internal.h"

#include <type_traits>

// Development aid, compiled out of the product build: per-workgroup stamps of the 100 MHz clock at the
// phase boundaries of the kernel, written 32 MiB into the workspace (size it so).
#ifdef GPTQ4_PHASE_TIMERS
#define KS_STAMP(i)                                                                                             \
    do {                                                                                                        \
        if (threadIdx.x == 0 && p.counters != nullptr)                                                          \
            reinterpret_cast<unsigned long long *>(reinterpret_cast<char *>(p.counters) + (32 << 20))[(blockIdx.y * gridDim.x + blockIdx.x) * 8 + (i)] = \
                wall_clock64();                                                                                 \
    } while (0)
#else
#define KS_STAMP(i)
#endif

namespace {

constexpr int BK = 64;

// WIDE (plain epilogue only): two adjacent 64-column blocks per wave tile, like a rotary head.
// KS: waves of the workgroup, each with its own slice of K (4 or 8).  A wave spends about half of its life
// waiting (first loads, the exchanges at the end) and the other half issuing ~20 instructions per MFMA, one wave
// per SIMD; the matrix cores are busy 15 % of the time (SQ counters at 128 rows, 4096 x 4096).  A second wave
// per SIMD overlaps the two.  8 waves with 64-row tiles are 128 KiB of LDS: one workgroup per CU.
// PAIRED (rotary epilogue only): the workgroup owns 32 columns of a head and their 32 rotation partners (d, d + 64)
// instead of the whole head.  The two columns of a lane are then d and d + 64 - two 4-byte loads per row instead of one
// 8-byte load of adjacent columns - so the wave tile has ONE column block, like a plain strip, twice as many workgroups
// share the projection without splitting K, and the lane that finishes a value holds its rotation partner itself.
// SB: the packed words are in streaming order and w[].qzeros holds the {scale, zero} words, as in the tiled kernel's
// variant of the same name: per column one 8-byte load of rows 2 * lhi, 2 * lhi + 1 of a four-row chunk, K step ks
// multiplies packed row 4 * (ks / 2) + 2 * lhi + ks % 2 of the tile.
template <int EPI, int MT, bool WIDE, int KS, bool PAIRED = false, bool SB = false>
// (eight waves: one workgroup per CU - all its registers - wherever the wave tile has two column blocks or two row blocks)
__global__ __launch_bounds__(64 * KS, MT > 2 || (KS == 8 && (MT == 2 || (EPI != EPI_PLAIN && !PAIRED) || WIDE)) ? 1 : 2) void gptq4_kslice_kernel(MatmulArgs p) {
    static_assert(KS == 4 || KS == 8, "four or eight waves");
    static_assert(MT <= 3 && (MT <= 2 || KS == 4), "the activation tiles of eight waves of 96 rows do not fit the LDS");
    static_assert(!WIDE || EPI == EPI_PLAIN, "the other epilogues have two blocks already");
    static_assert(!PAIRED || EPI == EPI_ROPE, "paired columns are a rotary head's");
    constexpr bool ADJ = (EPI == EPI_ROPE && !PAIRED) || WIDE;  // the second block is columns + 64 of the same matrix
    constexpr int BM = 32 * MT;
    constexpr int NB = ((EPI == EPI_PLAIN && !WIDE) || PAIRED) ? 1 : 2;  // 64-column blocks of the wave tile
    constexpr int BN = ADJ ? 128 : 64;                  // output columns of the workgroup
    constexpr int NSET = NB;                            // value sets the finishing wave combines
    constexpr int A_HALVES = BM * BK;                   // one wave's K tile of activations
    constexpr int A_UNITS = BM / 8;                     // LDS-direct loads per wave and K tile (8 rows each)

    // Per-wave activation tiles (two objects, so that the compiler can tell the loads into one
    // from the reads of the other).  Afterwards the same memory is MT * 4 exchange regions of
    // 8 KiB: region (mt, w) = accumulators of row block mt from wave w.
    __shared__ __attribute__((aligned(16))) half_t As0[KS * A_HALVES];
    __shared__ __attribute__((aligned(16))) half_t As1[KS * A_HALVES];
    static_assert(2 * KS * A_HALVES * sizeof(half_t) >= (size_t)MT * KS * 32 * 64 * sizeof(float), "exchange regions do not fit");
    auto region = [&](int mt, int w) -> float * {
        const int r = mt * KS + w;
        constexpr int HALF = MT * KS / 2;
        return reinterpret_cast<float *>(r < HALF ? As0 : As1) + (r < HALF ? r : r - HALF) * (32 * 64);
    };

    KS_STAMP(0);
    GPTQ4_FETCH_MATMUL_ARGS(p);
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ksl = wave;
    const int l32 = lane & 31;
    const int lhi = lane >> 5;

    const int M = p.M, K = p.K, N = p.N;
    const int tiles_m = (M + BM - 1) / BM;

    // XCD-contiguous logical tile index, row tiles fastest; the workgroup's K tiles [wg_begin, wg_begin + wg_len), its
    // rank `split` among the `nsplit` workgroups that share the tile, and the tile's index `xtile` among those that
    // exchange partial sums
    int logical, split, nsplit, wg_begin, wg_len, xtile;
    {
        const bool tail = p.tail_split > 1;  // one-dimensional grid: whole tiles first, then the parts of the shared ones
        const int total = tail ? p.tail_first : (int)gridDim.x;
        const int per = total >> 3, rem = total & 7;
        const int xcd = blockIdx.x & 7;
        logical = xcd * per + (xcd < rem ? xcd : rem) + (blockIdx.x >> 3);
        if (!tail) {
            split = blockIdx.y;
            nsplit = p.splitk;
            wg_begin = split * p.slot_q + min(split, p.slot_rem);
            wg_len = p.slot_q + (split < p.slot_rem ? 1 : 0);
            xtile = logical;
        } else if ((int)blockIdx.x < total) {
            split = 0, nsplit = 1, wg_begin = 0, wg_len = p.K / BK, xtile = 0;
        } else {
            // (ahead of the whole tile of an older workgroup beside it while it multiplies, so that its sums are exchanged while
            // that one still works: the waves of the older one are served first otherwise.  383 x 3840 x 3840 21.7 -> 19.8 us,
            // 185 x 2560 x 7680 17.9 -> 16.4)
            __builtin_amdgcn_s_setprio(1);
            const int s = p.tail_split, w = (int)blockIdx.x - total;
            xtile = w / s;
            split = w - xtile * s;
            logical = total + xtile;
            nsplit = s;
            const int nkt = p.K / BK, q = nkt / s, r = nkt - q * s;
            wg_begin = split * q + min(split, r);
            wg_len = q + (split < r ? 1 : 0);
        }
    }
    const int tile_n = logical / tiles_m;
    const int tile_m = logical - tile_n * tiles_m;
    const int m0 = tile_m * BM;
    // the launch covers columns [n_begin, n_begin + n_count) of the N; PAIRED: tile_n counts quarter heads,
    // n0 = the first of the tile's 32 low columns
    const int n0 = PAIRED ? p.n_begin + (tile_n >> 1) * 128 + (tile_n & 1) * 32 : p.n_begin + tile_n * BN;

    // block j of the wave tile: matrix j at the strip's columns (SiLU*mul), or columns
    // 64*j .. 64*j + 63 of the head (rotary); the lane's 2 columns of it (PAIRED: ncol and ncol + 64)
    const int ncol = PAIRED ? n0 + l32 : n0 + 2 * l32;

    f16_t acc[NB][MT][2];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[j][mt][t][i] = 0.f;

    // K tiles of the workgroup (split across workgroups), then of this wave
    const int wq = wg_len / KS, wr = wg_len % KS;
    const int k_begin = wg_begin + ksl * wq + min(ksl, wr);
    const int nk = k_begin + wq + (ksl < wr ? 1 : 0);

    if (nk > k_begin) {
        half_t *const buf0 = As0 + wave * A_HALVES;
        half_t *const buf1 = As1 + wave * A_HALVES;
        // Activations global -> LDS directly.  One instruction fills 8 rows x 8 chunks of 16
        // bytes; the chunk that lands at position c of row r is global chunk c ^ ((r >> 1) & 7),
        // which makes the 128-bit fragment reads conflict-free without padding.
        // Four units share an LDS base and the lane's four offsets: their distance is the instruction's own offset, which moves both addresses, so the
        // lane's is that much smaller (8 rows are 4096 bytes at least).  Rows from M on are not read: an offset out of the
        // buffer's range loads zeros, and a tile that does not exist is one of an empty buffer - no memory is touched for what
        // is requested ahead of a wave's last tile.
        uint32_t a_off[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int row = 8 * u + (lane >> 3);
            const int c = (lane & 7) ^ ((row >> 1) & 7);
            a_off[u] = (uint32_t)row * (uint32_t)K * 2u + 16u * c - 1024u * u;
        }
        auto dma_a = [&](half_t *dst, int tile, int u) {
            const int rows = tile < nk ? min(32, max(M - m0 - 8 * (u & ~3), 0)) : 0;
            const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(p.x + (size_t)(m0 + 8 * (u & ~3)) * K), 0, (int)((uint32_t)rows * (uint32_t)K * 2u), 0x00020000);
            auto *const lds = (__attribute__((address_space(3))) void *)(dst + (u & ~3) * 512);
            switch (u & 3) {
                case 0: __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, lds, 16, (int)a_off[0], tile * (BK * 2), 0, 0); break;
                case 1: __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, lds, 16, (int)a_off[1], tile * (BK * 2), 1024, 0); break;
                case 2: __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, lds, 16, (int)a_off[2], tile * (BK * 2), 2048, 0); break;
                default: __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, lds, 16, (int)a_off[3], tile * (BK * 2), 3072, 0); break;
            }
            if (u == A_UNITS - 1) asm volatile("" ::: "memory");  // the loads that follow stay behind these
        };
        const int sw = (l32 >> 1) & 7;  // (row >> 1) & 7 for every row this lane reads (rows = 32*j + l32)

        // Packed words of two K tiles: slot [par][ks] holds step ks of a tile of parity par.  It
        // is decoded during step ks - 1 and refilled during step ks - once its old contents
        // are dead, so the load can land in place - with the same step two tiles on.
        // (SB: slot [par][2 * m + t] holds, for column t, the words of steps 2 * m and 2 * m + 1; both are refilled during step
        // 2 * m + 1)
        // Addresses are scalars of the wave plus offsets of the lane that never change, as in the tiled kernel.
        uint2 b2[NB][2][4];
        constexpr int NMAT = (EPI == EPI_SILU_MUL) ? 2 : 1;
        const int strip_bytes = (K >> 7) * 1024, groups = K / p.groupsize;
        // SB: the strips of the wave's columns from its first one on; columns 64 further are four strips further
        const int sb_lane = PAIRED ? (l32 >> 4) * strip_bytes + (l32 & 15) * 16 + 8 * lhi : (l32 >> 3) * strip_bytes + (2 * l32 & 15) * 16 + 8 * lhi;
        const int sb_meta_lane = PAIRED ? (l32 >> 4) * groups * 64 + (l32 & 15) * 4 : (l32 >> 3) * groups * 64 + (2 * l32 & 15) * 4;
        constexpr int STRIPS = PAIRED ? 6 : ADJ ? 8 : 4;
        const uint32_t *sb_words[NMAT];
        __amdgpu_buffer_rsrc_t sb_meta_rsrc[NMAT];
        if constexpr (SB) {
#pragma unroll
            for (int j = 0; j < NMAT; ++j) {
                sb_words[j] = p.w[j].qweight + (size_t)(n0 >> 4) * (size_t)(K >> 7) * 256;
                sb_meta_rsrc[j] = __builtin_amdgcn_make_buffer_rsrc((void *)(p.w[j].qzeros + (size_t)(n0 >> 4) * (size_t)groups * 16), 0, STRIPS * groups * 64, 0x00020000);
            }
        }
        // checkpoint order: the lane's offset behind the first row of a step, its scales and its word of zero points
        const int wlane = PAIRED ? (lhi * N + l32) * 4 : (lhi * N + 2 * l32) * 4;
        const int slane = PAIRED ? 2 * l32 : 4 * l32, zlane = PAIRED ? (l32 >> 3) * 4 : (l32 >> 2) * 4;
        auto load_b2 = [&](int par, int tile, int ks) {
            if constexpr (SB) {
                if (ks & 1) {
#pragma unroll
                    for (int j = 0; j < NB; ++j) {
                        const int at = tile * 512 + ((ADJ && j) ? 4 * strip_bytes : 0), m = 256 * (ks >> 1);
                        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)sb_words[j < NMAT ? j : 0], 0, tile < nk ? STRIPS * strip_bytes : 0, 0x00020000);
                        b2[j][par][ks - 1] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, sb_lane + m, at, 0));
                        b2[j][par][ks] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, sb_lane + m + (PAIRED ? 0 : 16), at + (PAIRED ? 4 * strip_bytes : 0), 0));
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    // (the tile's eight rows, whose first is found in 64 bits)
                    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc((void *)(p.w[j < NMAT ? j : 0].qweight + n0 + (uint64_t)(uint32_t)tile * (uint32_t)(8 * N)), 0, tile < nk ? (8 * N - n0) * 4 : 0, 0x00020000);
                    if constexpr (PAIRED) {
                        b2[j][par][ks].x = __builtin_amdgcn_raw_buffer_load_b32(rows, wlane, 2 * ks * N * 4, 0);
                        b2[j][par][ks].y = __builtin_amdgcn_raw_buffer_load_b32(rows, wlane + 256, 2 * ks * N * 4, 0);
                    } else {
                        b2[j][par][ks] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rows, wlane + ((ADJ && j) ? 256 : 0), 2 * ks * N * 4, 0));
                    }
                }
            }
        };
        auto word_of = [&](int j, int par, int step, int t) -> uint32_t {
            if constexpr (SB) {
                const uint2 w = b2[j][par][(step & ~1) + t];
                return (step & 1) ? w.y : w.x;
            } else {
                return t ? b2[j][par][step].y : b2[j][par][step].x;
            }
        };
        // Scale and zero words run two tiles ahead as well: slot [par] is loaded in the first step of a tile of parity par and
        // made into the decode constants of the tile two on during the last step of the tile in between.
        uint32_t g_s[NB][2], g_z[NB][2];
        uint32_t g_z_hi[2];              // PAIRED: the zero word of the lane's second column,
        uint16_t g_s16[2], g_s16_hi[2];  // and, checkpoint order, the scales of its two columns (widened at their use)
        const uint32_t group_magic = p.tile_group_magic;  // (group = tile / (groupsize / 64): exact for every tile)
        const int group_shift = p.tile_group_shift;
        auto load_group2 = [&](int par, int tile) {
            const uint32_t g = __umulhi((uint32_t)min(tile, nk - 1), group_magic) >> group_shift;
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                const int mat = j < NMAT ? j : 0;
                if constexpr (SB) {
                    // {scale | zero << 16} of the lane's two columns of each block, in g_s and g_z
                    const int at = (int)g * 64 + ((ADJ && j) ? 4 * groups * 64 : 0);
                    if constexpr (PAIRED) {
                        g_s[j][par] = __builtin_amdgcn_raw_buffer_load_b32(sb_meta_rsrc[mat], sb_meta_lane, at, 0);
                        g_z[j][par] = __builtin_amdgcn_raw_buffer_load_b32(sb_meta_rsrc[mat], sb_meta_lane, at + 4 * groups * 64, 0);
                    } else {
                        const uint2 m2 = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(sb_meta_rsrc[mat], sb_meta_lane, at, 0));
                        g_s[j][par] = m2.x;
                        g_z[j][par] = m2.y;
                    }
                } else {
                    const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc((void *)(p.w[mat].scales + n0 + (uint64_t)g * (uint32_t)N), 0, (N - n0) * 2, 0x00020000);
                    const __amdgpu_buffer_rsrc_t zr = __builtin_amdgcn_make_buffer_rsrc((void *)(p.w[mat].qzeros + (n0 >> 3) + (uint64_t)g * (uint32_t)(N >> 3)), 0, (N - n0) >> 1, 0x00020000);
                    if constexpr (PAIRED) {
                        g_s16[par] = __builtin_amdgcn_raw_buffer_load_b16(sr, slane, 0, 0);
                        g_s16_hi[par] = __builtin_amdgcn_raw_buffer_load_b16(sr, slane + 128, 0, 0);
                        g_z[j][par] = __builtin_amdgcn_raw_buffer_load_b32(zr, zlane, 0, 0);
                        g_z_hi[par] = __builtin_amdgcn_raw_buffer_load_b32(zr, zlane + 32, 0, 0);
                    } else {
                        g_s[j][par] = __builtin_amdgcn_raw_buffer_load_b32(sr, slane + ((ADJ && j) ? 128 : 0), 0, 0);
                        g_z[j][par] = __builtin_amdgcn_raw_buffer_load_b32(zr, zlane + ((ADJ && j) ? 32 : 0), 0, 0);
                    }
                }
            }
        };
        ColDecodeNat cn[NB][2];
        auto make_cn = [&](int par, int j, int t) {
            // (the empty asm statements keep the arithmetic here: the compiler otherwise does it, and waits for the words, where they
            // are loaded, a tile earlier)
            uint32_t scale;
            if constexpr (PAIRED && !SB) {
                uint16_t half = t ? g_s16_hi[par] : g_s16[par];
                asm volatile("" : "+v"(half));
                scale = half;
            } else {
                scale = (SB && t) ? g_z[j][par] : g_s[j][par];
                asm volatile("" : "+v"(scale));
            }
            if constexpr (SB) {
                cn[j][t] = make_col_decode_nat((scale >> 16) & 0xFu, scale);
            } else {
                uint32_t zeros = (t && PAIRED) ? g_z_hi[par] : g_z[j][par];
                asm volatile("" : "+v"(zeros));
                cn[j][t] = PAIRED ? make_col_decode_nat((zeros >> ((l32 & 7) * 4)) & 0xFu, scale)
                                  : make_col_decode_nat((zeros >> (((2 * l32) & 7) * 4 + 4 * t)) & 0xFu, t ? scale >> 16 : scale);
            }
        };

        // The second tile's rows are asked for when the first one's words are there: with 128 KiB of rows in front of them (eight
        // waves, 64 rows) a wave waited 1.6 us for its first product instead of 1.2, which calls of two K tiles a wave do not make
        // up for (833 x 1024 x 1024 7.86 -> 7.57 us, 170 x 1024 x 2816 7.92 -> 7.63).
        const int second = k_begin + 1;
#pragma unroll
        for (int u = 0; u < A_UNITS; ++u) dma_a(buf0, k_begin, u);
        load_group2(0, k_begin);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) load_b2(0, k_begin, ks);
        constexpr int FIRST_STEPS = SB ? 2 : 4;  // (SB: the other two stand behind the rows, among the loads that the first wait in the loop counts)
#pragma unroll
        for (int ks = 0; ks < FIRST_STEPS; ++ks) load_b2(1, second, ks);
        h8_t bf[NB][2];
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                make_cn(0, j, t);
                bf[j][t] = decode_word_natural(word_of(j, 0, 0, t), cn[j][t]);
            }
        asm volatile("" : "+v"(bf[0][0])::"memory");
#pragma unroll
        for (int u = 0; u < A_UNITS; ++u) dma_a(buf1, second, u);
        load_group2(1, second);  // made into constants at the end of tile k_begin
#pragma unroll
        for (int ks = FIRST_STEPS; ks < 4; ++ks) load_b2(1, second, ks);
        // fragment mt of K step ks of the tile in `src`
        auto read_a = [&](const half_t *src, int ks, int mt) {
            return *reinterpret_cast<const h8_t *>(src + (mt * 32 + l32) * BK + 8 * ((SB ? 4 * (ks >> 1) + 2 * lhi + (ks & 1) : 2 * ks + lhi) ^ sw));
        };
        // (the first tile's packed words and the whole second tile's loads follow the first tile's; it is this wave's own tile: no barrier)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 * NB + A_UNITS) : "memory");
        h8_t ahead[MT];  // fragments of the step to come
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) ahead[mt] = read_a(buf0, 0, mt);

        // One K tile (of parity `par` counted from k_begin) out of buffer `cur`: four steps of 2 * NB * MT slots, each an MFMA
        // with its share of what has to be done for the step to come, as in the tiled kernel.  With the wait, the requests and
        // the fragment reads of a tile in front of its products and addresses of 64 bits per lane, a K tile of 64 rows x 64
        // columns took four waves 0.88 us on 64 CUs and 1.04 on all 256, eight waves (twice the work) 1.57 and 1.96; now 0.70 and
        // 0.86, 1.34 and 1.78, and 1.10 -> 0.95 for 96 rows: what is left is the rows' way through the CU (some 60 GB/s each, four
        // waves or eight) beside ~190 instructions a wave.  Graph replays over rotating weights: 4096 x 4096 at 320 rows
        // 23.3 -> 19.4 us, 5120 x 5120 at 200 rows 26.8 -> 21.6 (both of four waves), 11008 x 4096 at 700 rows 76.8 -> 71.5; slower by 2 - 4 %
        // with K = 5120 at some row counts from 32 to 125, where either loop waits for the weights from HBM (with warm ones 12 % faster).
        // (final: a last tile that nothing follows, where the loop ends on one - the tiles go in pairs)
        auto k_tile = [&](half_t *cur, const half_t *nxt, int kt, int par, auto final) {
            constexpr bool FINAL = decltype(final)::value;
            constexpr int SLOTS = 2 * NB * MT;
            constexpr int ROW_SLOTS = (SLOTS + 3) / 4;  // slots of the last step in which rows are asked for
            // packed words of four steps and scale/zero words: the loads behind those of a tile's rows
            constexpr int BEHIND = SB ? (PAIRED ? 6 : 5 * NB) : 6 * NB * (PAIRED ? 2 : 1);
            const int tile2 = kt + 2;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                const bool next = ks < 3 || !FINAL;  // a step follows
                h8_t af[MT], bnext[NB][2];
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) af[mt] = ahead[mt];
                DecodeNat dec;
                if (ks < 3 || FINAL) __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), once for the step's fragments
                __builtin_amdgcn_sched_barrier(0);
                // Loads complete in order, and behind the LDS-direct loads of the next tile this wave issued the packed words of
                // four K steps and scale/zero words: at most that many outstanding means the tile has landed.
                // (tests/test_wait_counts.py counts the loads behind the tile's in the compiled code of every variant.)
                if (ks == 3 && !FINAL) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BEHIND) : "memory");
#pragma unroll
                for (int i = 0; i < SLOTS; ++i) {
                    const int j = i / (2 * MT), t = (i / MT) & 1, mt = i % MT;
                    acc[j][mt][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[mt], bf[j][t], acc[j][mt][t], 0, 0, 0);
                    if (i < MT && next) ahead[i] = ks < 3 ? read_a(cur, ks + 1, i) : read_a(nxt, 0, i);
                    if (ks == 3 && !FINAL) {
                        // (all of this wave's reads of `cur` are done.  Asked for early: over the whole step, 65 rows of gate/up
                        // 5120 x 13824 in checkpoint order took 37.1 us instead of 34.9)
#pragma unroll
                        for (int u = i * A_UNITS / ROW_SLOTS; u < (i + 1) * A_UNITS / ROW_SLOTS && u < A_UNITS; ++u) dma_a(cur, tile2, u);
                    }
                    // (this step's words were decoded during the previous step, the scale/zero slot made into constants in the tile
                    // before; the last step's words stand behind the rows)
                    if (i == (ks == 3 ? SLOTS - 1 : 0) && !FINAL) load_b2(par, tile2, ks);
                    if (ks == 0 && i == 1 && !FINAL) load_group2(par, tile2);
                    if (next) {
                        // words of the next step (step 0 of the next tile when ks == 3), a stage of four instructions at a time
#pragma unroll
                        for (int st = 4 * mt / MT; st < 4 * (mt + 1) / MT; ++st) {
                            if (ks == 3 && st == 0) make_cn(par ^ 1, j, t);
                            dec.stage(st, ks < 3 ? word_of(j, par, ks + 1, t) : word_of(j, par ^ 1, 0, t), cn[j][t]);
                            if (ks == 3 && st >= 2) dec.pin(st);
                            if (st == 3) bnext[j][t] = dec.value();
                        }
                    }
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // the MFMA first
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (next) {
#pragma unroll
                    for (int j = 0; j < NB; ++j) bf[j][0] = bnext[j][0], bf[j][1] = bnext[j][1];
                }
            }
        };
        KS_STAMP(1);
        // pairs of tiles without a branch between them (a join there would make the compiler move packed words that are still
        // in flight, and wait for them), then the odd one
        int kt = k_begin;
        for (; kt + 1 < nk; kt += 2) {
            k_tile(buf0, buf1, kt, 0, std::false_type{});
            k_tile(buf1, buf0, kt + 1, 1, std::false_type{});
        }
        if (kt < nk) k_tile(buf0, buf1, kt, 0, std::true_type{});
    }
    // every LDS-direct load has landed and every wave is done reading before the tiles are
    // reused for the exchange
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    KS_STAMP(3);
    __syncthreads();
    KS_STAMP(2);

    // ---- the KS accumulator sets meet, one column block at a time.  Row block mt is finished by PARTS waves
    // (one with four waves, two with eight): wave mt * PARTS + part takes registers i = part * IW .. + IW - 1.
    // acc[j][mt][t][i]: row = 32*mt + 8*(i/4) + 4*lhi + i%4 of the tile, column = 2*l32 + t of block j.
    // vals[j][t][ii], i = part * IW + ii: the sums the epilogue combines - plain: the strip; SiLU*mul: gate and
    // up; rotary: columns d < 64 and d >= 64 of the head.  Only waves < MT * PARTS hold any.
    constexpr int PARTS = KS / 4;
    constexpr int IW = 16 / PARTS;
    float vals[NSET][2][IW];
    const bool owner = wave < MT * PARTS;
    const int own_mt = wave / PARTS, part = wave % PARTS;
    const int i0 = part * IW;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        if (j > 0) __syncthreads();  // the owners are done reading the previous block
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            float *const dst = region(mt, wave);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) dst[(t * 16 + i) * 64 + lane] = acc[j][mt][t][i];
        }
        __syncthreads();
#ifdef GPTQ4_PHASE_TIMERS
        if (j == 0 && nsplit == 1) KS_STAMP(6);
#endif
        if (owner) {
            const float *src[KS];
#pragma unroll
            for (int w = 0; w < KS; ++w) src[w] = region(own_mt, w) + i0 * 64 + lane;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int ii = 0; ii < IW; ++ii) {
                    float v[KS];
#pragma unroll
                    for (int w = 0; w < KS; ++w) v[w] = src[w][(t * 16 + ii) * 64];
                    float sum = v[0];
#pragma unroll
                    for (int w = 1; w < KS; ++w) sum += v[w];
                    vals[j][t][ii] = sum;
                }
        }
    }

    KS_STAMP(4);
    constexpr int NREG = NSET * 2 * IW;  // values per lane of an owner wave
    if (nsplit > 1) {
        __builtin_amdgcn_s_setprio(0);  // (parts beside whole tiles, see above)
        // K split across workgroups as well: each publishes its reduced tile (agent-scope
        // atomics, no cache maintenance), the last one to arrive sums them in split order.
        __shared__ int s_is_last;
        const int tile = xtile;
        const size_t per_split = (size_t)MT * PARTS * NREG * 64;
        float *const mine = p.partials + ((size_t)tile * nsplit + split) * per_split + (size_t)wave * NREG * 64 + lane;
        if (owner) {
#pragma unroll
            for (int s = 0; s < NSET; ++s)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int ii = 0; ii < IW; ++ii)
                        __hip_atomic_store(mine + ((s * 2 + t) * IW + ii) * 64, vals[s][t][ii], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        KS_STAMP(5);
        __syncthreads();
        if (tid == 0) {
            const int old = __hip_atomic_fetch_add(&p.counters[tile * COUNTER_STRIDE], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_is_last = (old == nsplit - 1);
        }
        __syncthreads();
        KS_STAMP(6);
        if (!s_is_last) return;
        if (owner) {
            // E of the lane's values from SPR splits per round, 32 loads in flight per lane: a round is one round trip
            constexpr int E = NREG < 32 ? NREG : 32;
            constexpr int SPR = 32 / E;
            const float *const all = p.partials + (size_t)tile * nsplit * per_split + (size_t)wave * NREG * 64 + lane;
#pragma unroll
            for (int e0 = 0; e0 < NREG; e0 += E) {
                float sum[E];
#pragma unroll
                for (int e = 0; e < E; ++e) sum[e] = 0.f;
#pragma unroll 1
                for (int c0 = 0; c0 < nsplit; c0 += SPR) {
                    float got[SPR][E];
#pragma unroll
                    for (int k = 0; k < SPR; ++k)
#pragma unroll
                        for (int e = 0; e < E; ++e)  // (past the last split: the last one again, not added)
                            got[k][e] = __hip_atomic_load(all + (size_t)min(c0 + k, nsplit - 1) * per_split + (e0 + e) * 64, __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                    for (int k = 0; k < SPR; ++k)
#pragma unroll
                        for (int e = 0; e < E; ++e) sum[e] += (c0 + k < nsplit) ? got[k][e] : 0.f;
                }
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const int f = e0 + e;  // = (s * 2 + t) * IW + ii
                    vals[f / (2 * IW)][(f / IW) & 1][f % IW] = sum[e];
                }
            }
        }
        if (tid == 0) __hip_atomic_store(&p.counters[tile * COUNTER_STRIDE], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!owner) return;

    // ---- epilogue of registers i0 .. i0 + IW - 1 of row block own_mt
    const int row0 = m0 + own_mt * 32 + 4 * lhi;
    auto row_of = [&](int ii) { return row0 + 8 * ((i0 + ii) >> 2) + ((i0 + ii) & 3); };
    if (EPI == EPI_PLAIN) {
        // Stores go out 16 bytes per lane (store_block_rows), turned through the part of this wave's exchange region
        // that only this wave read: its own registers' slots of the first column, 64 floats per register.
        uint32_t *const tr = reinterpret_cast<uint32_t *>(region(own_mt, wave)) + i0 * 64;
        const int block_row0 = m0 + own_mt * 32 + 2 * i0;  // first row of the 2 * IW rows this wave finishes
#pragma unroll
        for (int j = 0; j < NSET; ++j) {
            h2_t bias2 = {(half_t)0.f, (half_t)0.f};
            if (p.bias != nullptr) bias2 = as_h2(*reinterpret_cast<const uint32_t *>(p.bias + ncol + 64 * j));
            uint32_t w[IW];
#pragma unroll
            for (int ii = 0; ii < IW; ++ii) {
                h2_t o = {(half_t)vals[j][0][ii], (half_t)vals[j][1][ii]};
                if (p.bias != nullptr) o = o + bias2;
                w[ii] = as_u32(o);
            }
            store_block_rows<IW>(tr, w, lane, [&](int, int rr) -> half_t * {
                const int row = block_row0 + rr;
                return row < M ? p.y + (size_t)row * N + n0 + 64 * j : nullptr;
            });
        }
    } else if (EPI == EPI_SILU_MUL) {
        // (4 bytes per lane: the output is half as wide as the tile, the wider stores gain nothing here and their
        // registers cost the loop of the 64-row variants five more spilled values)
#pragma unroll
        for (int ii = 0; ii < IW; ++ii) {
            const int row = row_of(ii);
            if (row < M) {
                const h2_t o = {(half_t)(silu_f32(vals[0][0][ii]) * vals[NSET - 1][0][ii]),
                                (half_t)(silu_f32(vals[0][1][ii]) * vals[NSET - 1][1][ii])};
                *reinterpret_cast<uint32_t *>(p.y + (size_t)row * N + n0 + 2 * l32) = as_u32(o);
            }
        }
    } else {
        // the workgroup's 128 columns are one head of q, k or v
        const RopeArgs &r = p.rope;
        const int head_col = n0 >> 7;
        const int which = head_col / r.H;
        const int head = head_col - which * r.H;
        const int cap = (which == 0) ? r.S : r.kv_capacity;
        half_t *const dst = ((which == 0) ? r.q : (which == 1) ? r.k : r.v) + (size_t)head * cap * 128 + 2 * l32;
        const size_t seq_stride = (size_t)r.H * cap * 128;
        const bool at_position = (which != 0) && r.kv_offset < 0;  // cache row = the token's position
        const int row_shift = (which == 0 || r.kv_offset < 0) ? 0 : r.kv_offset;
        int pos[IW];
        if (which < 2 || at_position) {
#pragma unroll
            for (int ii = 0; ii < IW; ++ii) pos[ii] = max(r.position_ids[min(row_of(ii), M - 1)], 0);
        }
        if constexpr (PAIRED) {
            // the lane's two values are columns d and d + 64 of the head: the same products and sums as below
            const int d = (n0 & 127) + l32;
            float c1[IW], s1[IW];
            if (which < 2) {
#pragma unroll
                for (int ii = 0; ii < IW; ++ii) {
                    const int tp = min(pos[ii], r.max_pos - 1);
                    c1[ii] = r.cos_table[(size_t)tp * 64 + d];
                    s1[ii] = r.sin_table[(size_t)tp * 64 + d];
                }
            }
#pragma unroll
            for (int ii = 0; ii < IW; ++ii) {
                const int row = row_of(ii);
                float lo = vals[0][0][ii], hi = vals[0][1][ii];
                if (which < 2) {
                    const float a = lo * c1[ii] - hi * s1[ii];
                    const float b = hi * c1[ii] + lo * s1[ii];
                    lo = a, hi = b;
                }
                if (row < M) {
                    int bb, srow;
                    split_row(r, row, bb, srow);
                    const int crow = at_position ? min(pos[ii], r.kv_capacity - 1) : srow + row_shift;
                    half_t *const at = dst - 2 * l32 + d + (size_t)bb * seq_stride + (size_t)crow * 128;
                    at[0] = (half_t)lo;
                    at[64] = (half_t)hi;
                }
            }
            KS_STAMP(7);
            return;
        }
        float2 cs[IW], sn[IW];
        if (which < 2) {
#pragma unroll
            for (int ii = 0; ii < IW; ++ii) {
                const int tp = min(pos[ii], r.max_pos - 1);
                cs[ii] = *reinterpret_cast<const float2 *>(r.cos_table + (size_t)tp * 64 + 2 * l32);
                sn[ii] = *reinterpret_cast<const float2 *>(r.sin_table + (size_t)tp * 64 + 2 * l32);
            }
        }
#pragma unroll
        for (int ii = 0; ii < IW; ++ii) {
            const int row = row_of(ii);
            float lo0 = vals[0][0][ii], lo1 = vals[0][1][ii], hi0 = vals[NSET - 1][0][ii], hi1 = vals[NSET - 1][1][ii];
            if (which < 2) {
                const float a0 = lo0 * cs[ii].x - hi0 * sn[ii].x, a1 = lo1 * cs[ii].y - hi1 * sn[ii].y;
                const float b0 = hi0 * cs[ii].x + lo0 * sn[ii].x, b1 = hi1 * cs[ii].y + lo1 * sn[ii].y;
                lo0 = a0, lo1 = a1, hi0 = b0, hi1 = b1;
            }
            // (4 bytes per lane, as for gate/up: with 16-byte stores this epilogue was 2 - 6 % slower at 256 and 512 rows
            // with the weights from HBM, and the 64-row variants spilled two more values)
            if (row < M) {
                int bb, srow;
                split_row(r, row, bb, srow);
                const int crow = at_position ? min(pos[ii], r.kv_capacity - 1) : srow + row_shift;
                half_t *const at = dst + (size_t)bb * seq_stride + (size_t)crow * 128;
                const h2_t olo = {(half_t)lo0, (half_t)lo1}, ohi = {(half_t)hi0, (half_t)hi1};
                *reinterpret_cast<uint32_t *>(at) = as_u32(olo);
                *reinterpret_cast<uint32_t *>(at + 64) = as_u32(ohi);
            }
        }
    }
    KS_STAMP(7);
}

template <int EPI, int MT, bool WIDE, int KS, bool PAIRED = false>
int launch_one(const MatmulArgs &a, int tiles, hipStream_t stream) {
    dim3 grid((unsigned)tiles, (unsigned)a.splitk), block(64 * KS);
    if (a.tail_split > 1) grid = dim3((unsigned)(a.tail_first + (tiles - a.tail_first) * a.tail_split), 1u);
    if (a.stream_b)
        hipLaunchKernelGGL((gptq4_kslice_kernel<EPI, MT, WIDE, KS, PAIRED, true>), grid, block, 0, stream, a);
    else
        hipLaunchKernelGGL((gptq4_kslice_kernel<EPI, MT, WIDE, KS, PAIRED>), grid, block, 0, stream, a);
    return (int)hipGetLastError();
}

// 96-row tiles: four waves, one workgroup per CU
template <int EPI, int MT>
int launch_tall(const MatmulArgs &a, const KslicePlan &pl, hipStream_t stream) {
    if constexpr (EPI == EPI_ROPE) {
        if (pl.paired) return launch_one<EPI_ROPE, MT, false, 4, true>(a, pl.tiles, stream);
    }
    if constexpr (EPI == EPI_PLAIN) {
        if (pl.wide) return launch_one<EPI_PLAIN, MT, true, 4>(a, pl.tiles, stream);
    }
    return launch_one<EPI, MT, false, 4>(a, pl.tiles, stream);
}

template <int EPI, int KS>
int launch_waves(const MatmulArgs &a, const KslicePlan &pl, hipStream_t stream) {
    if constexpr (EPI == EPI_ROPE) {
        if (pl.paired)
            return pl.mt == 1 ? launch_one<EPI_ROPE, 1, false, KS, true>(a, pl.tiles, stream)
                              : launch_one<EPI_ROPE, 2, false, KS, true>(a, pl.tiles, stream);
    }
    if constexpr (KS == 8) {
        if (EPI == EPI_PLAIN && !pl.wide)
            return pl.mt == 1 ? launch_one<EPI_PLAIN, 1, false, 8>(a, pl.tiles, stream) : launch_one<EPI_PLAIN, 2, false, 8>(a, pl.tiles, stream);
        // (128-column strips of a plain projection on 32-row tiles are not built for eight waves; neither plan asks for them)
        if (EPI == EPI_PLAIN) return pl.mt == 1 ? (int)hipErrorInvalidValue : launch_one<EPI_PLAIN, 2, true, 8>(a, pl.tiles, stream);
        return pl.mt == 1 ? launch_one<EPI, 1, false, 8>(a, pl.tiles, stream) : launch_one<EPI, 2, false, 8>(a, pl.tiles, stream);
    } else {
        if (EPI == EPI_PLAIN && pl.wide)
            return pl.mt == 1 ? launch_one<EPI_PLAIN, 1, true, KS>(a, pl.tiles, stream) : launch_one<EPI_PLAIN, 2, true, KS>(a, pl.tiles, stream);
        return pl.mt == 1 ? launch_one<EPI, 1, false, KS>(a, pl.tiles, stream) : launch_one<EPI, 2, false, KS>(a, pl.tiles, stream);
    }
}

template <int EPI>
int launch_epi(const MatmulArgs &a, const KslicePlan &pl, hipStream_t stream) {
    if (pl.mt == 3) return launch_tall<EPI, 3>(a, pl, stream);
    return pl.waves == 8 ? launch_waves<EPI, 8>(a, pl, stream) : launch_waves<EPI, 4>(a, pl, stream);
}

}  // namespace

KsliceTuning g_kslice_tuning = {1, 0, 0, 0, 0, 0};

// The plan by scores, for launches of more than one round, forced shapes, and calls outside one_round_margin's range.
// Row tile: 32 rows up to M = 32, else 64 - or 32 for plain projections where that scores higher, see below.  (Four
// activation tiles per wave instead of two - the tile three K tiles on requested while one is multiplied - gained nothing
// that eight waves do not gain as well.)  How far K is split across workgroups on top is scored below.
// One variant of it: the rotary epilogue on whole heads or on paired quarter heads.  *score: that of the split it
// chose (0 with a forced split).
static KslicePlan plan_variant(int epi, int M, int N, int K, bool has_perm, bool paired, double *score) {
    KslicePlan pl = {};
    // eight waves for plain projections wherever they fit (checked below): ahead of four waves by 4 - 18 % at
    // LLaMA-7B / 30B shapes from 17 to 256 rows with the same tiles, level at 512; the gate/up pair and the rotary epilogue
    // take eight up to 32 rows (one workgroup per CU then: two column blocks per wave tile need the registers of a whole SIMD; 7B QKV
    // 16.9 -> 15.6 us, gate/up 19.6 -> 18.6, 13B QKV 19.3 -> 18.0) and stay at four beyond (level or 3 % behind)
    // (paired quarter heads: one column block per wave tile like a plain strip, so eight waves fit as they do there)
    pl.paired = paired;
    pl.waves = g_kslice_tuning.waves ? g_kslice_tuning.waves : ((epi == EPI_PLAIN || pl.paired || M <= 32) ? 8 : 4);
    int ks = pl.waves;
    // plain projections: 128-column strips (half the activation traffic per weight byte, half the tiles) pay
    // from 256 rows on when K is long (LLaMA-7B down_proj: 39.8 -> 37.3 us at 256 rows, 66.2 -> 61.1 at 512;
    // o_proj with K = 4096 loses below 512 rows)
    pl.wide = epi == EPI_PLAIN && (g_kslice_tuning.wide > 0 || (g_kslice_tuning.wide == 0 && M >= 256 && K >= 8192));
    const int bn = ((epi == EPI_ROPE && !pl.paired) || pl.wide) ? 128 : 64;
    const int nk = K / 64;
    pl.mt = g_kslice_tuning.mt ? g_kslice_tuning.mt : (M <= 32 ? 1 : 2);
    if (pl.mt > 2) pl.waves = ks = 4;
    int bm = 32 * pl.mt;
    pl.tiles = ((M + bm - 1) / bm) * (N / bn);
    const long cus = device_shape().cus;  // 256 on MI355X
    double split_score = 0.0;  // of the split choose_split returned last (automatic choice only)
    auto choose_split = [&](int ks) {
        int s = 1;
        split_score = 0.0;
        if (g_kslice_tuning.splitk > 0) {
            s = g_kslice_tuning.splitk;
        } else {
            // Score 1..8 splits by how evenly tiles * s workgroups fill 256 CUs holding two each (w / 256 up to 256,
            // else w / (512 * ceil(w / 512)), never below 0.8 from 512 workgroups on: with several rounds the
            // scheduler evens things out), every extra split at 4 % + 15 / (K tiles) of the time, at least 4 K
            // tiles per wave.  Fitted to sweeps at LLaMA-7B / 13B / 30B shapes, 32..256 rows: on average 1 % off
            // the best split (a fixed target of 512 workgroups: 2.3 %, worst case 17 %).
            const double pen = 0.04 + 15.0 / (double)nk;
            double best = -1.0;
            for (int c = 1; c <= 8 && c <= nk / (4 * ks); ++c) {
                const long w = (long)pl.tiles * c;
                double e = (w <= cus) ? (double)w / (double)cus : (double)w / ((double)(2 * cus) * (double)((w + 2 * cus - 1) / (2 * cus)));
                if (w >= 2 * cus && e < 0.8) e = 0.8;
                const double score = e / (1.0 + pen * (c - 1));
                if (score > best + 1e-9) {
                    best = score;
                    s = c;
                }
            }
            split_score = best;
        }
        if (s > GEMM_MAX_SPLITK) s = GEMM_MAX_SPLITK;
        if (s < 1 || pl.tiles > SKINNY_MAX_TILES) s = 1;
        return s;
    };
    int s = choose_split(ks);
    // Plain projections on 64-column strips, 33 rows and more: 32-row tiles as well, where twice as many tiles fill
    // the chip without a split across workgroups (or with a smaller one) - each weight is then decoded once per 32
    // rows instead of once per 64, priced at 0.85 of the rate, but the exchange through memory goes.  Same score as
    // for the splits.  4096 x 4096 at 128 rows: 256 tiles of 32 rows, 12.8 -> 11.5 us; 5120 x 5120 at 96 rows 16.2 ->
    // 12.9, 13824 x 5120 at 96 rows 32.3 -> 28.8; 64-row tiles stay where they score higher (11008 x 4096 at 128
    // rows, 5120 x 5120 at 128 rows: 320 tiles of 32 rows would not fit one round).
    if (epi == EPI_PLAIN && !pl.wide && M > 32 && g_kslice_tuning.mt == 0 && g_kslice_tuning.splitk == 0) {
        const double score2 = split_score;
        const int tiles2 = pl.tiles;
        pl.tiles = ((M + 31) / 32) * (N / bn);
        const int s1 = choose_split(ks);
        if (score2 > 0.0 && 0.85 * split_score > score2 + 1e-9 && pl.tiles <= SKINNY_MAX_TILES) {
            pl.mt = 1;
            bm = 32;
            s = s1;
        } else {
            pl.tiles = tiles2;
        }
    }
    // eight waves: 128 KiB of LDS with 64-row tiles, so only in launches of at most one workgroup per CU; with 32-row
    // tiles two workgroups share a CU and four waves a SIMD, which leaves each 128 registers - enough for one
    // column block per wave tile only, so two blocks also need the CU to themselves; and every wave needs a K tile
    // or two
    if (pl.waves == 8) {
        const int nb = ((epi == EPI_PLAIN && !pl.wide) || pl.paired) ? 1 : 2;
        if (((pl.mt == 2 || nb == 2) && (long)pl.tiles * s > cus) || (pl.mt == 1 && nb == 2 && epi == EPI_PLAIN) || nk / s < 16) {
            pl.waves = ks = 4;
            s = choose_split(ks);
        }
    }
    pl.splitk = s;
    // Unsplit tiles past a whole number of rounds (one per CU and round; two workgroups of four waves are resident
    // per CU, and two that share a CU take 1.6 times what one takes alone): up to half a round of them - whole column
    // strips, every row tile, so that a row's summation order does not depend on its place in the batch - are cut along
    // K into as many parts as spread them over the chip, and the parts run beside the whole tiles.  LLaMA-7B gate/up
    // at 128 rows: 344 tiles, 88 of them in two parts each.
    pl.tail_first = 0;
    pl.tail_split = 1;
    if (s == 1 && pl.waves == 4 && g_kslice_tuning.splitk == 0 && g_gemm_tuning.tail != 1 && pl.tiles > cus && pl.tiles <= SKINNY_MAX_TILES) {
        const long tiles_m = (M + bm - 1) / bm, strips = N / bn;
        const long rest = pl.tiles % cus;
        const long cut_strips = (rest + tiles_m - 1) / tiles_m, cut = cut_strips * tiles_m;
        if (rest > 0 && 2 * cut <= cus && cut_strips < strips) {
            long parts = cus / cut;
            if (parts > nk / (4 * ks)) parts = nk / (4 * ks);  // at least 4 K tiles per wave
            if (parts > GEMM_MAX_SPLITK) parts = GEMM_MAX_SPLITK;
            if (parts >= 2) {
                pl.tail_first = (int)(pl.tiles - cut);
                pl.tail_split = (int)parts;
            }
        }
    }
    // the wave loop needs the activations unpermuted and at least one K tile per wave
    pl.ok = !has_perm && (N % bn) == 0 && nk / s >= ks;
    *score = split_score;
    return pl;
}

// Rotary epilogue: whole heads (tiles of 128 columns) or tiles of 32 columns of a head and their 32 rotation partners -
// twice as many tiles, so that few rows fill the chip without splitting K across workgroups (an exchange of partial
// sums through memory, 3 us), at the price of two 4-byte loads per row and lane instead of one 8-byte load and half as
// many MFMAs per activation fragment (priced at 0.85 of the rate).  Each variant is planned by itself and the better
// split score wins (never with a larger split than whole heads take).  LLaMA-7B QKV: 15.7 -> 13.0 us at 17 rows, 16.2 -> 13.4 at 32 (16 rows: 12.4), 21.1 -> 16.9 at 64,
// 42.4 -> 37.0 at 192; 13B 18.7 -> 16.2 at 32, 24.6 -> 20.6 at 64; 30B 60 -> 54 at 96 rows and whole heads below that
// (312 paired tiles do not fit one round of 256 CUs).  The plan for launches of more than one round (and for forced shapes).
static KslicePlan rounds_plan(int epi, int M, int N, int K, bool has_perm) {
    double score = 0.0;
    if (epi != EPI_ROPE || g_kslice_tuning.paired == 2) return plan_variant(epi, M, N, K, has_perm, false, &score);
    if (g_kslice_tuning.paired == 1) return plan_variant(epi, M, N, K, has_perm, true, &score);
    double score_p = 0.0;
    const KslicePlan heads = plan_variant(epi, M, N, K, has_perm, false, &score);
    const KslicePlan pairs = plan_variant(epi, M, N, K, has_perm, true, &score_p);
    // (only where whole heads leave the chip short of two workgroups per CU: beyond that the score's steps at whole
    // rounds say nothing about twice as many, smaller tiles - 7B QKV at 512 rows: 768 whole heads 72.6 us, 1536 paired
    // tiles 87.8)
    const bool few = (long)heads.tiles < 2 * device_shape().cus;
    return (pairs.ok && few && score > 0.0 && pairs.splitk <= heads.splitk && 0.85 * score_p > score + 1e-9) ? pairs : heads;
}

// ---- launches of at most one round: every workgroup resident at once, so that the time is that of one workgroup:
//   t0 + steps * (step + load * workgroups / CUs) + exchange
// with steps = K tiles of the longest wave, `step` that of one workgroup or of two to a CU, `load` what the others' traffic
// adds to a step, and the cost of splitting K across workgroups (the first split, then every further one).  One line per
// kernel variant, in us, fitted to 3500 timings over 20 projections (K and N from 2048 to 19968) at 24 to 768 rows with the
// weights from HBM - of the loop before its instructions were dealt to its MFMAs.  Against 5000 timings of the present one (31 projections,
// K from 1024 to 17920, 17 to 768 rows, streaming order): 5 - 11 % off per variant, on average 8 % low (32-row tiles, eight waves) to 2 %
// high (96-row tiles).  (Where it may decide: one_round_margin.)
struct RoundCost {
    float t0, one, two, load, split, more;  // two = 0: one workgroup to a CU
};
static const RoundCost round_cost[3][2][2] = {
    // [row tile / 32 - 1][eight waves][two column blocks]
    {{{4.2f, 0.480f, 0.751f, 0.065f, 1.98f, 0.40f}, {6.1f, 0.665f, 1.265f, 0.178f, 2.59f, 0.67f}},
     {{4.8f, 0.632f, 1.375f, 0.168f, 1.62f, 0.40f}, {5.7f, 1.327f, 0.f, 0.364f, 3.00f, 0.50f}}},
    {{{5.2f, 0.579f, 0.890f, 0.215f, 2.22f, 0.43f}, {8.1f, 0.681f, 1.432f, 0.404f, 3.18f, 0.64f}},
     {{5.6f, 0.823f, 0.f, 0.458f, 1.65f, 0.47f}, {9.1f, 1.210f, 0.f, 0.903f, 1.81f, 0.55f}}},
    {{{5.0f, 0.760f, 0.f, 0.279f, 2.27f, 0.49f}, {8.2f, 1.024f, 0.f, 0.491f, 3.44f, 0.85f}}, {}}};

// us, or 0 for a launch of more than one round
static double one_round_estimate(int epi, int K, const KslicePlan &pl, long cus) {
    const bool two_blocks = !((epi == EPI_PLAIN && !pl.wide) || pl.paired);
    const RoundCost &c = round_cost[pl.mt - 1][pl.waves == 8][two_blocks];
    const long wgs = (long)pl.tiles * pl.splitk;
    if (wgs > (c.two > 0.f ? 2 : 1) * cus) return 0.0;
    const int steps = ((K / 64 + pl.splitk - 1) / pl.splitk + pl.waves - 1) / pl.waves;
    return c.t0 + steps * ((wgs <= cus ? c.one : c.two) + c.load * (double)wgs / (double)cus) +
           (pl.splitk > 1 ? c.split + c.more * (pl.splitk - 2) : 0.0);
}

// What the tiled kernel takes, whatever plan it chooses (us; fitted to its loop before, too; against the present one 10 - 11 % off, on
// average right for plain calls and 3 - 5 % high for the others; see one_round_margin).
static double tiled_estimate(int epi, int M, int N, int K) {
    const double tiles = (double)((M + 127) / 128) * (N / (epi == EPI_SILU_MUL ? 128 : 256)) / device_shape().cus, nk = K / 64;
    const double t0 = epi == EPI_PLAIN ? 12.9 : epi == EPI_SILU_MUL ? 8.5 : 19.0;
    const double flat = epi == EPI_PLAIN ? 0.122 : epi == EPI_SILU_MUL ? 0.568 : 0.155;
    const double knee = epi == EPI_PLAIN ? 0.028 : epi == EPI_SILU_MUL ? 0.44 : 0.078;
    return t0 + nk * (flat + (tiles > knee ? 0.86 * (tiles - knee) : 0.0));
}

// How far a launch of one round has to be ahead of the tiled kernel's estimate to be planned (0: never), so that the two
// estimates' errors do not choose the slower one.  Both were fitted at 24 to 768 rows; against the plan by scores and the tiled
// kernel they were then timed on 1800 calls outside the fit (17 to 8192 rows, K from 512 to 32768, N from 256 to 32000), with the
// loops of that time (with the present ones the plan taken is 2.4 % behind the fastest of all timed, on average over 558 calls of 17 to
// 768 rows, and more than 5 % behind for 92 of them, 25 % at most):
//   up to 768 rows, 5 % ahead:     on average 11 % (plain, gate/up) and 20 % (rotary) faster; 11 of 871 calls slower, by 5 - 11 %
//   769 .. 2048 rows, 15 % ahead:  on average 27 % and 29 % faster, 3 of 405 slower (12 % at most); at 5 % ahead 21 were, up to 24 %
//   2049 .. 8192 rows, 30 % ahead: 40 of 99 calls still go there, 17 % faster, 1 slower; at 5 % ahead 17 were, up to 38 %
//   K below 1024, over 64 rows:    the tiled kernel takes half of what its line says (512 x 6144 at 512 rows 8.9 us, estimated
//                                  16.3): 98 of 291 plain and gate/up calls were slower, up to 79 %; no rotary call was
static double one_round_margin(int epi, int M, int K) {
    if (K < 1024 && M > 64 && epi != EPI_ROPE) return 0.0;
    return M <= 768 ? 0.95 : M <= 2048 ? 0.85 : M <= 8192 ? 0.70 : 0.0;
}

// The fastest launch of at most one round by that estimate, if it is ahead of the tiled kernel by that margin (ok = false otherwise).
// 96-row tiles exist for this: one row tile for 65 .. 96 rows, two for 129 .. 192, where 64- and 128-row tiles pad a third
// to a half, each weight decoded once per 96 rows: LLaMA-7B gate/up at 96 rows 35.3 -> 30.1 us, 13B 47.9 -> 38.2; QKV
// (plain) at 192 rows 37.2 -> 29.5; 4096 x 4096 at 640 rows 37.7 -> 31.0.  (128-row tiles never were the fastest: with two
// column blocks they spill, with one they halve the workgroups of 64-row tiles.)
static KslicePlan one_round_plan(int epi, int M, int N, int K) {
    KslicePlan best = {};
    const int cus = device_shape().cus, nk = K / 64;
    double best_us = one_round_margin(epi, M, K) * tiled_estimate(epi, M, N, K);
    for (int mt = 1; mt <= 3; ++mt)
        for (int waves = 4; waves <= 8; waves += 4)
            for (int form = 0; form < (epi == EPI_SILU_MUL ? 1 : 2); ++form) {
                KslicePlan pl = {};
                pl.mt = mt;
                pl.waves = waves;
                pl.wide = epi == EPI_PLAIN && form == 1;
                pl.paired = epi == EPI_ROPE && form == 1;
                pl.tail_split = 1;
                pl.ok = pl.one_round = true;
                const int bn = (pl.wide || (epi == EPI_ROPE && !pl.paired)) ? 128 : 64;
                // (variants that are not built: the activation tiles do not fit, or were never the faster ones)
                if ((N % bn) != 0 || (waves == 8 && (mt == 3 || (mt == 1 && pl.wide)))) continue;
                pl.tiles = ((M + 32 * mt - 1) / (32 * mt)) * (N / bn);
                for (pl.splitk = 1; pl.splitk <= 8; ++pl.splitk) {
                    // (two K tiles a wave at least; below a quarter of the CUs the estimate was not fitted)
                    if (nk / pl.splitk < 2 * waves) break;
                    const double us = one_round_estimate(epi, K, pl, cus);
                    if (us <= 0.0) break;
                    if (4L * pl.tiles * pl.splitk < cus) continue;
                    if (us < best_us) {
                        best_us = us;
                        best = pl;
                    }
                }
            }
    return best;
}

KslicePlan kslice_plan(int epi, int M, int N, int K, bool has_perm, bool allow_one_round) {
    const KsliceTuning &t = g_kslice_tuning;
    KslicePlan pl = rounds_plan(epi, M, N, K, has_perm);
    if (t.mode != 1 || t.mt != 0 || t.splitk != 0 || t.wide != 0 || t.waves != 0 || t.paired != 0 || has_perm || !allow_one_round) return pl;
    const KslicePlan one = one_round_plan(epi, M, N, K);
    if (!one.ok) return pl;
    // the plan by scores stays where the estimates do not tell the two apart (7 %: it may then be level with the tiled kernel's
    // estimate instead of ahead of it); with its last strips shared along K it takes some 6 % less than the estimate for whole tiles
    const int cus = device_shape().cus;
    const double us = (pl.ok ? one_round_estimate(epi, K, pl, cus) : 0.0) * (pl.tail_split > 1 ? 0.94 : 1.0);
    if (us > 0.0 && us <= 1.07 * one_round_estimate(epi, K, one, cus)) {
        pl.one_round = true;
        return pl;
    }
    return one;
}

size_t kslice_partial_bytes(int epi, const KslicePlan &pl) {
    // (the same with four or eight waves: eight split the 32 values per lane and block over two owner waves)
    const int nset = ((epi == EPI_PLAIN && !pl.wide) || pl.paired) ? 1 : 2;
    if (pl.tail_split > 1) return (size_t)(pl.tiles - pl.tail_first) * pl.tail_split * pl.mt * nset * 32 * 64 * sizeof(float);
    return pl.splitk > 1 ? (size_t)pl.tiles * pl.splitk * pl.mt * nset * 32 * 64 * sizeof(float) : 0;
}

int launch_kslice(int epi, MatmulArgs &a, const KslicePlan &pl, hipStream_t stream) {
    set_tile_group(a);
    switch (epi) {
        case EPI_PLAIN: return launch_epi<EPI_PLAIN>(a, pl, stream);
        case EPI_SILU_MUL: return launch_epi<EPI_SILU_MUL>(a, pl, stream);
        default: return launch_epi<EPI_ROPE>(a, pl, stream);
    }
}
