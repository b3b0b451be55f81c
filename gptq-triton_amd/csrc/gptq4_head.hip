// The last step of a greedy decode token: logits = x . W^T with the fp16 lm_head weight W [V, K] and the index of the
// largest logit per row, in one launch - and, for a decoding loop, what the next step starts from: the token and its place in
// the sequence, the position, and on request the token's embedding row.  (The reference's scripts call the model's lm_head - a dense
// fp16 linear - and take the argmax of its output, generate.py.)
//
// A memory-bound stream over V x K x 2 bytes.  The rows of W are dealt to the workgroups in contiguous ranges and inside a
// workgroup to its eight waves; a wave multiplies up to 16 of its rows at a time, as the A operand of
// v_mfma_f32_16x16x32_f16 (lane (r, c): 16 bytes of row c), with the x rows as B out of LDS, so that one to sixteen
// sequences cost the same: 8 KiB of W per wave are in flight while the 8 KiB before are multiplied.  Rows are dealt evenly,
// not in sixteens: lanes past a tile's rows load nothing.  Sums are rounded to fp16 as the linear layer's output would be;
// the best (value, index) per x row is kept in registers - torch.argmax's choice among equal values and NaN -, the
// workgroups' bests go through the workspace and the last workgroup to arrive picks the winners, one wave per x row.
#include "../../include/gptq4.h"
#include "gptq4_internal.h"
#include "gptq4_norm.h"

namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
constexpr int HEAD_WAVES = 8;
constexpr int HEAD_MAX_B = 16;
constexpr int HEAD_STEPS = 8;  // matrix steps (32 values of every row) per group of loads

// torch.argmax's order: NaN above every number, the lower index among equal values.
__device__ __forceinline__ bool better(float v, int i, float bv, int bi) {
    if (v != v || bv != bv) return v != v && (bv == bv || i < bi);
    return v > bv || (v == bv && i < bi);
}

// NORM: 0 x as it is, 1 its RMSNorm, 2 the RMSNorm of x + delta
template <int NORM>
__global__ __launch_bounds__(64 * HEAD_WAVES) void gptq4_head_argmax_kernel(HeadArgs p) {
    // [B][K / 8 + 1] chunks of 16 bytes: rows a chunk apart cost 4 conflict cycles a read at 8 and at 16 rows (SQ_LDS_BANK_CONFLICT:
    // 4096 of a CU's 95 k cycles for 32000 x 4096), rows a power of two apart would meet in one bank
    extern __shared__ uint4 head_xs[];
    __shared__ float s_val[HEAD_WAVES][HEAD_MAX_B];
    __shared__ int s_idx[HEAD_WAVES][HEAD_MAX_B];
    __shared__ float s_part[4];
    __shared__ int s_last;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane >> 4, c = lane & 15;
    const int B = p.B, K = p.K, chunks = K >> 3, pitch = chunks + 1;

    // this wave's rows, in ntile tiles of `step` rows (16 at most)
    const int wg0 = blockIdx.x * p.rows_per_wg, wg1 = min(wg0 + p.rows_per_wg, p.V);
    const int per_wave = (p.rows_per_wg + HEAD_WAVES - 1) / HEAD_WAVES;
    const int r0 = wg0 + wave * per_wave, r1 = min(r0 + per_wave, wg1);
    const int ntile = (per_wave + 15) / 16, step = (per_wave + ntile - 1) / ntile;
    const int groups = K / (32 * HEAD_STEPS);
    // (rows of 4096 or 8192 values are a power of two apart: waves that all started at the beginning of their rows would ask
    // the same few memory channels at a time, so every wave starts at a group of its own and goes round)
    const int g_first = (int)((blockIdx.x * HEAD_WAVES + wave) * 7u % (unsigned)groups);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(p.w), 0, (int)0x7FFFFFF0, 0x00020000);
    u32x4_t cur[HEAD_STEPS], nxt[HEAD_STEPS];
    auto fetch = [&](u32x4_t (&dst)[HEAD_STEPS], int row0, int g) {
        const int row = row0 + c;
        // (a row past the tile: an offset the buffer rejects - zeros, no memory touched)
        const uint32_t off = (c < step && row < r1) ? (uint32_t)row * (uint32_t)(K * 2) + 16u * r : 0x80000000u;
#pragma unroll
        for (int j = 0; j < HEAD_STEPS; ++j) dst[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, off, (uint32_t)(g * HEAD_STEPS + j) * 64u, 0);
    };
    if constexpr (NORM == 0) {
        fetch(cur, r0, g_first);
        for (int i = tid; i < B * chunks; i += 64 * HEAD_WAVES) {
            const int b = i / chunks;
            head_xs[i + b] = reinterpret_cast<const uint4 *>(p.x)[i];
        }
    } else {
        NormLoads<NORM_KEEP> row;
        norm_issue_row0<NORM == 2, NORM_KEEP>(p.x, p.delta, p.nrm_weight, K, tid & 255, row);
        fetch(cur, r0, g_first);
        norm_rows_put<NORM == 2, NORM_KEEP>(p.x, p.delta, p.nrm_weight, nullptr, [&](int, int at, uint4 v) { head_xs[at] = v; }, s_part, 1, K,
                                            p.eps, tid & 255, row, tid < 256);
    }
    __syncthreads();

    const uint4 *const xb = head_xs + min(c, B - 1) * pitch + r;
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    f4_t acc = {0.f, 0.f, 0.f, 0.f};
    int row0 = r0, g = g_first, left = groups;
    for (int t = ntile * groups; t > 0; --t) {
        const bool tile_ends = left == 1;
        const int row_n = tile_ends ? row0 + step : row0, g_n = g + 1 == groups ? 0 : g + 1;
        left = tile_ends ? groups : left - 1;
        fetch(nxt, t > 1 ? row_n : r1, g_n);
#pragma unroll
        for (int j = 0; j < HEAD_STEPS; ++j)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, cur[j]), __builtin_bit_cast(h8_t, xb[4 * (g * HEAD_STEPS + j)]), acc,
                                                         0, 0, 0);
        if (tile_ends) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int at = 4 * r + i, row = row0 + at;
                const float v = (float)(half_t)acc[i];  // the linear layer's fp16 output
                if (at < step && row < r1 && better(v, row, bv, bi)) bv = v, bi = row;
            }
            acc = f4_t{0.f, 0.f, 0.f, 0.f};
        }
        row0 = row_n, g = g_n;
#pragma unroll
        for (int j = 0; j < HEAD_STEPS; ++j) cur[j] = nxt[j];
    }
    // lanes c, c + 16, c + 32, c + 48 hold bests of x row c
#pragma unroll
    for (int o = 16; o <= 32; o <<= 1) {
        const float ov = __shfl_xor(bv, o);
        const int oi = __shfl_xor(bi, o);
        if (better(ov, oi, bv, bi)) bv = ov, bi = oi;
    }
    if (lane < HEAD_MAX_B) {
        s_val[wave][lane] = bv;
        s_idx[wave][lane] = bi;
    }
    __syncthreads();

    // ---- the workgroup's best per x row -> workspace; the last workgroup to arrive reduces them
    const int nwg = gridDim.x;
    if (tid < B) {
        bv = -INFINITY;
        bi = 0x7fffffff;
#pragma unroll
        for (int wv = 0; wv < HEAD_WAVES; ++wv)
            if (better(s_val[wv][tid], s_idx[wv][tid], bv, bi)) bv = s_val[wv][tid], bi = s_idx[wv][tid];
        float *dst = p.part + ((size_t)blockIdx.x * HEAD_MAX_B + tid) * 2;
        __hip_atomic_store(dst, bv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(reinterpret_cast<int *>(dst) + 1, bi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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
        bv = -INFINITY;
        bi = 0x7fffffff;
        for (int i = lane; i < nwg; i += 64) {
            const float *src = p.part + ((size_t)i * HEAD_MAX_B + b) * 2;
            const float v = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const int at = __hip_atomic_load(reinterpret_cast<const int *>(src) + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (better(v, at, bv, bi)) bv = v, bi = at;
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

template <int NORM>
int launch_norm(HeadArgs &a, hipStream_t stream) {
    const int cus = device_shape().cus;
    const int nwg = a.V < cus ? a.V : cus;
    a.rows_per_wg = (a.V + nwg - 1) / nwg;
    const int grid = (a.V + a.rows_per_wg - 1) / a.rows_per_wg;
    const size_t lds = (size_t)a.B * (a.K / 8 + 1) * 16;
    if (lds > 48 * 1024) {
        static LdsGrant grant;
        if (const int rc = allow_lds(grant, reinterpret_cast<const void *>(&gptq4_head_argmax_kernel<NORM>), HEAD_LDS_BYTES)) return rc;
    }
    hipLaunchKernelGGL((gptq4_head_argmax_kernel<NORM>), dim3((unsigned)grid), dim3(64 * HEAD_WAVES), lds, stream, a);
    return (int)hipGetLastError();
}

}  // namespace

size_t head_argmax_partial_bytes() { return (size_t)device_shape().cus * HEAD_MAX_B * 2 * sizeof(float); }

bool head_argmax_fits(int B, int K, int V) {
    return B >= 1 && B <= HEAD_MAX_B && V >= 1 && K >= 256 && (K % 256) == 0 && (size_t)V * K * 2 < 0x7FFFFFF0ull &&
           (size_t)B * (K / 8 + 1) * 16 <= (size_t)HEAD_LDS_BYTES;
}

int launch_head_argmax(HeadArgs &a, hipStream_t stream) {
    if (a.nrm_weight == nullptr) return launch_norm<0>(a, stream);
    return a.delta == nullptr ? launch_norm<1>(a, stream) : launch_norm<2>(a, stream);
}
