// The last step of a greedy decode token: logits = x . W^T with the fp16 lm_head weight W [V, K] and the index of the
// largest logit per row, in one launch - and, for a decoding loop, what the next step starts from: the token and its place in
// the sequence, the position, and on request the token's embedding row.  (The reference's scripts call the model's lm_head - a dense
// fp16 linear - and take the argmax of its output, generate.py.)
//
// A memory-bound stream over V x K x 2 bytes.  The rows of W are dealt to the workgroups in contiguous ranges and inside a
// workgroup to its eight waves; a wave takes four rows at a time, 256 contiguous bytes of each per load, as the A operand of
// v_mfma_f32_4x4x4_16b_f16: sixteen independent products of four rows by four columns, block b on the sixteenth b of the load's
// values, whose sums meet across the lanes at the end of the four rows.  The x rows, four to a product, are B out of LDS.  4 KiB
// of W per wave are in flight while the 4 KiB before are multiplied (8 KiB: the same from 5120 columns on, 49.9 against 47.0 us at
// 4096; 2 KiB: 58).  With sixteen rows to a product (v_mfma_f32_16x16x32_f16) a load touched 64 bytes of sixteen rows - half
// lines, which the streaming hint then fetched twice (58.8 us with it, 53.6 without).  With four, us, W from HBM, the sixteen's
// time first (argmax): 32000 x 4096 at 1 / 8 / 16 rows 59.6 / 60.9 / 66.1 -> 48.0 / 48.9 / 51.3 (5.5 TB/s; a plain read of as many
// bytes takes 40), x 1024 19.7 / 21.4 / 24.4 -> 16.5 / 18.3 / 20.5, x 256 11.5 / 12.5 / 15.4 -> 10.3 / 11.5 / 13.7, and at the most rows
// that fit the LDS x 5120 (15) 70.4 -> 60.6, x 6656 (12) 87.6 -> 73.1, x 8192 (9) 109.9 -> 89.0.  Rows of 256 values leave half of a
// wave's loads empty, which shows where the vocabulary is long: 128256 x 256 19.1 / 20.0 / 23.0 -> 19.5 / 20.7 / 23.8.
// Rows are dealt evenly, not in fours: lanes past a tile's rows load nothing.  Sums are rounded to fp16 as the linear layer's
// output would be.  They are the result (LOGITS), or the best (value, index) per x row is kept in registers - torch.argmax's
// choice among equal values and NaN -, the workgroups' bests go through the workspace, one 8-byte value each, and the last
// workgroup to arrive picks the winners, one wave per x row (2 - 4 us of the launch).
#include "../../include/gptq4.h"
#include "gptq4_internal.h"
#include "gptq4_norm.h"

namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
constexpr int HEAD_WAVES = 8;
constexpr int HEAD_MAX_B = 16;
constexpr int HEAD_STEPS = 4;  // loads of 256 bytes of four rows per group

// torch.argmax's order: NaN above every number, the lower index among equal values.  No branches: a wave's lanes differ in the outcome.
__device__ __forceinline__ bool better(float v, int i, float bv, int bi) {
    return (v > bv) | ((v == bv) & (i < bi)) | ((v != v) & ((bv == bv) | (i < bi)));
}

// Sums over the sixteen lanes of a wave that are equal modulo 4, of four values at a time: lane l gets that of v[l / 16], always
// summed in the same order.  Each exchange halves what is left to sum instead of giving every lane everything: eight
// vector instructions where four sums in every lane take sixteen and eight reads through the LDS (argmax of 16 rows
// through 128256 x 256 30.1 -> 23.8 us, 50304 x 1024 28.7 -> 27.3, 32000 x 4096 51.9 -> 51.3).
__device__ __forceinline__ float blocks_sum(f4_t v) {
    auto half = [](float a) { return __builtin_bit_cast(uint32_t, a); };
    auto both = [](auto pair) { return __builtin_bit_cast(float, (uint32_t)pair[0]) + __builtin_bit_cast(float, (uint32_t)pair[1]); };
    // (the upper half of the one against the lower half of the other, then the odd sixteens against the even ones)
    const float s02 = both(__builtin_amdgcn_permlane32_swap(half(v[0]), half(v[2]), false, false));
    const float s13 = both(__builtin_amdgcn_permlane32_swap(half(v[1]), half(v[3]), false, false));
    float s = both(__builtin_amdgcn_permlane16_swap(half(s02), half(s13), false, false));
    s += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, s), 0x128, 0xF, 0xF, true));        // row_ror:8
    return s + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, s), 0x124, 0xF, 0xF, true));  // row_ror:4
}

// NORM: 0 x as it is, 1 its RMSNorm, 2 the RMSNorm of x + delta; NB: groups of four x rows; LOGITS: the sums themselves are
// the result
template <int NORM, int NB, bool LOGITS>
__global__ __launch_bounds__(64 * HEAD_WAVES) void gptq4_head_kernel(HeadArgs p) {
    // [B][p.pitch] chunks of 16 bytes.  Rows four chunks apart beyond their length: the sixteen lanes of a pass read 64 bytes of
    // each of four rows, all banks once.
    extern __shared__ uint4 head_xs[];
    __shared__ float s_val[HEAD_WAVES][HEAD_MAX_B];
    __shared__ int s_idx[HEAD_WAVES][HEAD_MAX_B];
    __shared__ float s_part[4];
    __shared__ int s_last;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int blk = lane >> 2, c = lane & 3;
    const int B = p.B, K = p.K, chunks = K >> 3, pitch = p.pitch;

    // this wave's rows, in ntile tiles of `step` rows (four at most)
    const int wg0 = blockIdx.x * p.rows_per_wg, wg1 = min(wg0 + p.rows_per_wg, p.V);
    const int per_wave = (p.rows_per_wg + HEAD_WAVES - 1) / HEAD_WAVES;
    const int r0 = wg0 + wave * per_wave, r1 = min(r0 + per_wave, wg1);
    const int ntile = (per_wave + 3) / 4, step = (per_wave + ntile - 1) / ntile;
    const int loads = K >> 7;  // of 256 bytes of every row
    const int groups = (loads + HEAD_STEPS - 1) / HEAD_STEPS;
    // (rows of 4096 or 8192 values are a power of two apart: waves that all started at the beginning of their rows would ask
    // the same few memory channels at a time, so every wave starts at a group of its own and goes round; where the groups are a
    // multiple of seven the waves share one or two starting points: 3584 and 7168 columns, level with wave number % groups)
    const int g_first = (int)((blockIdx.x * HEAD_WAVES + wave) * 7u % (unsigned)groups);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(p.w), 0, (int)0x7FFFFFF0, 0x00020000);
    u32x4_t cur[HEAD_STEPS], nxt[HEAD_STEPS];
    auto fetch = [&](u32x4_t (&dst)[HEAD_STEPS], int row0, int g) {
        const int row = row0 + c;
        // (a row past the tile, and what is past the row in its last group: an offset the buffer rejects - zeros, no memory touched)
        const uint32_t off = (c < step && row < r1) ? (uint32_t)row * (uint32_t)(K * 2) + 16u * blk : 0x80000000u;
#pragma unroll
        for (int j = 0; j < HEAD_STEPS; ++j)
            dst[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, g * HEAD_STEPS + j < loads ? off : 0x80000000u, (uint32_t)(g * HEAD_STEPS + j) * 256u, 2);  // (streamed once)
    };
    if constexpr (NORM == 0) {
        fetch(cur, r0, g_first);
        for (int i = tid; i < B * chunks; i += 64 * HEAD_WAVES) {
            const int b = i / chunks;
            head_xs[i + b * (pitch - chunks)] = reinterpret_cast<const uint4 *>(p.x)[i];
        }
    } else {
        NormLoads<NORM_KEEP> row;
        norm_issue_row0<NORM == 2, NORM_KEEP>(p.x, p.delta, p.nrm_weight, K, tid & 255, row);
        fetch(cur, r0, g_first);
        norm_rows_put<NORM == 2, NORM_KEEP>(p.x, p.delta, p.nrm_weight, nullptr, [&](int, int at, uint4 v) { head_xs[at] = v; }, s_part, 1, K,
                                            p.eps, tid & 255, row, tid < 256);
    }
    __syncthreads();

    const uint4 *xb[NB];
    float bv[NB];
    int bi[NB];
    f4_t acc[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) {
        xb[n] = head_xs + min(4 * n + c, B - 1) * pitch + blk;
        bv[n] = -INFINITY;
        bi[n] = 0x7fffffff;
        acc[n] = f4_t{0.f, 0.f, 0.f, 0.f};
    }
    int row0 = r0, g = g_first, left = groups;
    for (int t = ntile * groups; t > 0; --t) {
        const bool tile_ends = left == 1;
        const int row_n = tile_ends ? row0 + step : row0, g_n = g + 1 == groups ? 0 : g + 1;
        left = tile_ends ? groups : left - 1;
        fetch(nxt, t > 1 ? row_n : r1, g_n);
#pragma unroll
        for (int j = 0; j < HEAD_STEPS; ++j) {
            if (g * HEAD_STEPS + j >= loads) break;  // (nothing of x is there either)
            const uint2 w[2] = {make_uint2(cur[j].x, cur[j].y), make_uint2(cur[j].z, cur[j].w)};
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                const uint4 xv = xb[n][16 * (g * HEAD_STEPS + j)];
                acc[n] = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(h4_t, w[0]), __builtin_bit_cast(h4_t, make_uint2(xv.x, xv.y)), acc[n], 0, 0, 0);
                acc[n] = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(h4_t, w[1]), __builtin_bit_cast(h4_t, make_uint2(xv.z, xv.w)), acc[n], 0, 0, 0);
            }
        }
        if (tile_ends) {
            // Every sixteen lanes go on with a row of the tile: one comparison per x row, without branches.  (Four comparisons one
            // after the other, each behind its sum's way across the lanes and behind branches, took 3.7 us of the launch for every
            // four x rows at 32000 rows of W, whatever their length: x 1024 at 16 rows 29.9 us.)
            const int at = lane >> 4, row = row0 + at;
            const bool mine = (at < step) & (row < r1);
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                const half_t h = (half_t)blocks_sum(acc[n]);  // the linear layer's fp16 output
                if constexpr (LOGITS) {
                    if (mine & ((lane & 12) == 0) & (4 * n + c < B)) p.logits[(size_t)(4 * n + c) * p.V + row] = h;
                } else {
                    const bool up = mine & better((float)h, row, bv[n], bi[n]);
                    bv[n] = up ? (float)h : bv[n];
                    bi[n] = up ? row : bi[n];
                }
                acc[n] = f4_t{0.f, 0.f, 0.f, 0.f};
            }
        }
        row0 = row_n, g = g_n;
#pragma unroll
        for (int j = 0; j < HEAD_STEPS; ++j) cur[j] = nxt[j];
    }
    if constexpr (LOGITS) return;
    // lanes c, c + 16, c + 32, c + 48 hold the bests of four rows of every tile
#pragma unroll
    for (int n = 0; n < NB; ++n) {
#pragma unroll
        for (int o = 16; o <= 32; o <<= 1) {
            const float ov = __shfl_xor(bv[n], o);
            const int oi = __shfl_xor(bi[n], o);
            const bool up = better(ov, oi, bv[n], bi[n]);
            bv[n] = up ? ov : bv[n];
            bi[n] = up ? oi : bi[n];
        }
        if (lane < 4) {
            s_val[wave][4 * n + lane] = bv[n];
            s_idx[wave][4 * n + lane] = bi[n];
        }
    }
    __syncthreads();

    // ---- the workgroup's best per x row -> workspace; the last workgroup to arrive reduces them
    const int nwg = gridDim.x;
    if (tid < B) {
        float bv = -INFINITY;
        int bi = 0x7fffffff;
#pragma unroll
        for (int wv = 0; wv < HEAD_WAVES; ++wv)
            if (better(s_val[wv][tid], s_idx[wv][tid], bv, bi)) bv = s_val[wv][tid], bi = s_idx[wv][tid];
        __hip_atomic_store(p.best + (size_t)blockIdx.x * HEAD_MAX_B + tid, (uint64_t)__float_as_uint(bv) | (uint64_t)(uint32_t)bi << 32, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
        const int old = __hip_atomic_fetch_add(&p.counters[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = (old == nwg - 1);
    }
    __syncthreads();
    if (!s_last) return;
    if (tid == 0) __hip_atomic_store(&p.counters[0], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int b = wave; b < B; b += HEAD_WAVES) {
        float bv = -INFINITY;
        int bi = 0x7fffffff;
        for (int i = lane; i < nwg; i += 256) {
            uint64_t got[4];  // (together: a round trip each costs more than everything else here; past the last workgroup the last one again)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                got[k] = __hip_atomic_load(p.best + (size_t)min(i + 64 * k, nwg - 1) * HEAD_MAX_B + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float v = __uint_as_float((uint32_t)got[k]);
                const int at = (int)(got[k] >> 32);
                if (better(v, at, bv, bi)) bv = v, bi = at;
            }
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            const float ov = __shfl_xor(bv, o);
            const int oi = __shfl_xor(bi, o);
            if (better(ov, oi, bv, bi)) bv = ov, bi = oi;
        }
        const int token = __builtin_amdgcn_readfirstlane(min(bi, p.V - 1));  // (whatever happens, a row of the table)
        if (lane == 0) p.tokens[b] = (long long)token;
        if (p.positions != nullptr) {
            if (lane == 0) {
                const int at = p.positions[b] + 1;
                p.positions[b] = at;
                if (at >= 0 && at < p.history_capacity) p.history[(size_t)b * p.history_capacity + at] = (long long)token;
            }
            if (p.embed == nullptr) continue;
            const uint4 *src = reinterpret_cast<const uint4 *>(p.embed + (size_t)token * K);
            uint4 *dst = reinterpret_cast<uint4 *>(p.next_hidden + (size_t)b * K);
            for (int i = lane; i < chunks; i += 64) dst[i] = src[i];
        }
    }
}

template <int NORM, int NB, bool LOGITS>
int launch_kernel(HeadArgs &a, hipStream_t stream) {
    const int cus = device_shape().cus;
    const int nwg = a.V < cus ? a.V : cus;
    a.rows_per_wg = (a.V + nwg - 1) / nwg;
    const int grid = (a.V + a.rows_per_wg - 1) / a.rows_per_wg;
    a.pitch = a.K / 8 + 4;
    if ((size_t)a.B * a.pitch * 16 > (size_t)HEAD_LDS_BYTES) a.pitch = a.K / 8 + 1;
    const size_t lds = (size_t)a.B * a.pitch * 16;
    if (lds > 48 * 1024) {
        static LdsGrant grant;
        if (const int rc = allow_lds(grant, reinterpret_cast<const void *>(&gptq4_head_kernel<NORM, NB, LOGITS>), HEAD_LDS_BYTES)) return rc;
    }
    hipLaunchKernelGGL((gptq4_head_kernel<NORM, NB, LOGITS>), dim3((unsigned)grid), dim3(64 * HEAD_WAVES), lds, stream, a);
    return (int)hipGetLastError();
}

template <bool LOGITS>
int launch_rows(HeadArgs &a, hipStream_t stream) {
    switch ((a.B + 3) / 4) {
        case 1: return launch_kernel<0, 1, LOGITS>(a, stream);
        case 2: return launch_kernel<0, 2, LOGITS>(a, stream);
        case 3: return launch_kernel<0, 3, LOGITS>(a, stream);
        default: return launch_kernel<0, 4, LOGITS>(a, stream);
    }
}

}  // namespace

size_t head_argmax_partial_bytes() { return (size_t)device_shape().cus * HEAD_MAX_B * sizeof(uint64_t); }

bool head_argmax_fits(int B, int K, int V) {
    return B >= 1 && B <= HEAD_MAX_B && V >= 1 && K >= 256 && (K % 256) == 0 && (size_t)V * K * 2 < 0x7FFFFFF0ull &&
           (size_t)B * (K / 8 + 1) * 16 <= (size_t)HEAD_LDS_BYTES;
}

int launch_head_argmax(HeadArgs &a, hipStream_t stream) {
    if (a.nrm_weight == nullptr) return launch_rows<false>(a, stream);
    return a.delta == nullptr ? launch_kernel<1, 1, false>(a, stream) : launch_kernel<2, 1, false>(a, stream);
}

int launch_head_logits(HeadArgs &a, hipStream_t stream) { return launch_rows<true>(a, stream); }
