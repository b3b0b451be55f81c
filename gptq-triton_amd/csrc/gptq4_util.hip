// Format kernels: weight materialisation (bit-exact decode), act-order row sort,
// rotary table.  None of them is on the per-token path.
#include "gptq4_internal.h"

namespace {

// One thread per packed word: 8 rows of one column.  Uses the same decode_word as the
// matmul kernels, so a bit-exact check of this kernel checks their decode too.
__global__ __launch_bounds__(256) void gptq4_dequant_kernel(const uint32_t *__restrict__ qweight,
                                                            const uint32_t *__restrict__ qzeros,
                                                            const half_t *__restrict__ scales,
                                                            const int32_t *__restrict__ g_idx,
                                                            half_t *__restrict__ out, int K, int N,
                                                            int groupsize) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    const int r = blockIdx.y;
    if (n >= N) return;
    const uint32_t w = qweight[(size_t)r * N + n];
    const int zshift = (n & 7) * 4;
    half_t vals[8];
    if (g_idx == nullptr) {
        const int g = (8 * r) / groupsize;
        const uint32_t z = (qzeros[(size_t)g * (N >> 3) + (n >> 3)] >> zshift) & 0xFu;
        const ColDecode c = make_col_decode(z, reinterpret_cast<const uint16_t *>(scales)[(size_t)g * N + n]);
        h2_t p[4];
        decode_word(w, c, p);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            vals[jj] = p[jj].x;
            vals[jj + 4] = p[jj].y;
        }
    } else {
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int g = g_idx[8 * r + t];
            const uint32_t z = (qzeros[(size_t)g * (N >> 3) + (n >> 3)] >> zshift) & 0xFu;
            const ColDecode c = make_col_decode(z, reinterpret_cast<const uint16_t *>(scales)[(size_t)g * N + n]);
            h2_t p[4];
            decode_word(w, c, p);
            vals[t] = (t < 4) ? p[t & 3].x : p[t & 3].y;
        }
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) out[(size_t)(8 * r + t) * N + n] = vals[t];
}

// out nibble-row j = in nibble-row perm[j]
__global__ __launch_bounds__(256) void gptq4_sort_rows_kernel(const uint32_t *__restrict__ qweight,
                                                              const int32_t *__restrict__ perm,
                                                              uint32_t *__restrict__ out, int K, int N) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    const int r = blockIdx.y;
    if (n >= N) return;
    uint32_t w = 0;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const int src = perm[8 * r + t];
        const uint32_t sw = qweight[(size_t)(src >> 3) * N + n];
        w |= ((sw >> ((src & 7) * 4)) & 0xFu) << (4 * t);
    }
    out[(size_t)r * N + n] = w;
}

// out[m][j] = x[m][perm[j]]: the activations in the order of the sorted weight rows.  One thread
// makes 8 neighbouring outputs of one row (K % 8 == 0, perm 16-byte aligned).
__global__ __launch_bounds__(256) void gptq4_gather_cols_kernel(const half_t *__restrict__ x,
                                                                const int32_t *__restrict__ perm,
                                                                half_t *__restrict__ out, int K) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (8 * c >= K) return;
    const int4 i0 = *reinterpret_cast<const int4 *>(perm + 8 * c);
    const int4 i1 = *reinterpret_cast<const int4 *>(perm + 8 * c + 4);
    const uint16_t *row = reinterpret_cast<const uint16_t *>(x) + (size_t)blockIdx.y * K;
    uint4 o;
    o.x = (uint32_t)row[i0.x] | ((uint32_t)row[i0.y] << 16);
    o.y = (uint32_t)row[i0.z] | ((uint32_t)row[i0.w] << 16);
    o.z = (uint32_t)row[i1.x] | ((uint32_t)row[i1.y] << 16);
    o.w = (uint32_t)row[i1.z] | ((uint32_t)row[i1.w] << 16);
    *reinterpret_cast<uint4 *>(out + (size_t)blockIdx.y * K + 8 * c) = o;
}

// The same through LDS, for rows that fit: one workgroup per row copies the row there in whole 16-byte chunks and gathers
// from it - single 2-byte reads of global memory cost a cache line each.  KEEP: chunks a thread holds (longer rows loop), with
// the permutation asked for together with the row - one round trip to memory instead of two, which is what few long rows
// wait for.  With the streaming-order projection behind it (us, KEEP 0 in 256 threads / 4 in 512): 13824 x 5120 at 20 rows
// 25.9 / 23.5, 100 rows 41.5 / 39.6, 17920 x 6656 at 20 rows 34.8 / 32.0; short rows and many rows lose by the larger
// workgroups: 1024 x 1024 at 20 rows 7.9 / 8.0, 13824 x 5120 at 400 rows 91.7 / 93.3.
template <int NT, int KEEP>
__global__ __launch_bounds__(NT) void gptq4_gather_cols_lds_kernel(const half_t *__restrict__ x,
                                                                   const int32_t *__restrict__ perm,
                                                                   half_t *__restrict__ out, int K) {
    extern __shared__ uint4 row_chunks[];  // K / 8
    const int chunks = K >> 3, tid = threadIdx.x;
    const uint4 *src = reinterpret_cast<const uint4 *>(x + (size_t)blockIdx.x * K);
    const int4 *order = reinterpret_cast<const int4 *>(perm);
    uint4 held[KEEP ? KEEP : 1];
    int4 idx[KEEP ? KEEP : 1][2];
#pragma unroll
    for (int n = 0; n < KEEP; ++n) {
        const int c = tid + NT * n;
        if (c < chunks) {
            held[n] = src[c];
            idx[n][0] = order[2 * c];
            idx[n][1] = order[2 * c + 1];
        }
    }
#pragma unroll
    for (int n = 0; n < KEEP; ++n)
        if (tid + NT * n < chunks) row_chunks[tid + NT * n] = held[n];
    for (int c = tid + NT * KEEP; c < chunks; c += NT) row_chunks[c] = src[c];
    __syncthreads();
    const uint16_t *row = reinterpret_cast<const uint16_t *>(row_chunks);
    uint4 *dst = reinterpret_cast<uint4 *>(out + (size_t)blockIdx.x * K);
    auto put = [&](int c, int4 i0, int4 i1) {
        uint4 o;
        o.x = (uint32_t)row[i0.x] | ((uint32_t)row[i0.y] << 16);
        o.y = (uint32_t)row[i0.z] | ((uint32_t)row[i0.w] << 16);
        o.z = (uint32_t)row[i1.x] | ((uint32_t)row[i1.y] << 16);
        o.w = (uint32_t)row[i1.z] | ((uint32_t)row[i1.w] << 16);
        dst[c] = o;
    };
#pragma unroll
    for (int n = 0; n < KEEP; ++n)
        if (tid + NT * n < chunks) put(tid + NT * n, idx[n][0], idx[n][1]);
    for (int c = tid + NT * KEEP; c < chunks; c += NT) put(c, order[2 * c], order[2 * c + 1]);
}

__global__ __launch_bounds__(256) void gptq4_rope_table_kernel(float *__restrict__ cos_out,
                                                               float *__restrict__ sin_out, int max_pos,
                                                               int half_dim, float base) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= max_pos * half_dim) return;
    const int pos = idx / half_dim;
    const int i = idx - pos * half_dim;
    // inv_freq = float32 nearest to base^(-2i/D) (evaluated in double, rounded once);
    // angle = float(pos) * inv_freq as a float32 product
    const double expo = (double)(2 * i) / (double)(2 * half_dim);
    const float inv_freq = (float)(1.0 / pow((double)base, expo));
    const float theta = (float)pos * inv_freq;
    // evaluate in double on the float32 angle: exact-to-rounding table values
    cos_out[idx] = (float)cos((double)theta);
    sin_out[idx] = (float)sin((double)theta);
}

}  // namespace

DeviceShape device_shape() {
    enum { MAX_DEVICES = 64 };
    static DeviceShape known[MAX_DEVICES];  // cus == 0: not asked yet
    const DeviceShape fallback = {256, 8};
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
        (void)hipGetLastError();
        return fallback;
    }
    if (known[dev].cus == 0) {  // (a race between two first callers writes the same values twice)
        DeviceShape d = fallback;
        int v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) d.cus = v;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeNumberOfXccs, dev) == hipSuccess && v > 0) d.xcds = v;
        (void)hipGetLastError();
        known[dev] = d;
    }
    return known[dev];
}

int launch_dequant(const uint32_t *qweight, const uint32_t *qzeros, const half_t *scales,
                   const int32_t *g_idx, half_t *out, int K, int N, int groupsize, hipStream_t stream) {
    dim3 grid((unsigned)((N + 255) / 256), (unsigned)(K / 8)), block(256);
    hipLaunchKernelGGL(gptq4_dequant_kernel, grid, block, 0, stream, qweight, qzeros, scales, g_idx, out, K,
                       N, groupsize);
    return (int)hipGetLastError();
}

int launch_sort_rows(const uint32_t *qweight, const int32_t *perm, uint32_t *out, int K, int N,
                     hipStream_t stream) {
    dim3 grid((unsigned)((N + 255) / 256), (unsigned)(K / 8)), block(256);
    hipLaunchKernelGGL(gptq4_sort_rows_kernel, grid, block, 0, stream, qweight, perm, out, K, N);
    return (int)hipGetLastError();
}

int launch_gather_cols(const half_t *x, const int32_t *perm, half_t *out, int M, int K, hipStream_t stream) {
    if (M > 16 && (size_t)K * sizeof(half_t) <= 65536) {
        const size_t lds = (size_t)K * sizeof(half_t);
        if (M <= 128 && K > 4096)
            hipLaunchKernelGGL((gptq4_gather_cols_lds_kernel<512, 4>), dim3((unsigned)M), dim3(512), lds, stream, x, perm, out, K);
        else
            hipLaunchKernelGGL((gptq4_gather_cols_lds_kernel<256, 0>), dim3((unsigned)M), dim3(256), lds, stream, x, perm, out, K);
        return (int)hipGetLastError();
    }
    const int threads = (K / 8 >= 256) ? 256 : 64;
    if (M > 65535) return (int)hipErrorInvalidConfiguration;  // rows ride in grid.y here; callers reject this on the host first
    dim3 grid((unsigned)((K / 8 + threads - 1) / threads), (unsigned)M), block(threads);
    hipLaunchKernelGGL(gptq4_gather_cols_kernel, grid, block, 0, stream, x, perm, out, K);
    return (int)hipGetLastError();
}

int launch_rope_table(float *cos_out, float *sin_out, int max_pos, int D, float base, hipStream_t stream) {
    const int total = max_pos * (D / 2);
    dim3 grid((unsigned)((total + 255) / 256)), block(256);
    hipLaunchKernelGGL(gptq4_rope_table_kernel, grid, block, 0, stream, cos_out, sin_out, max_pos, D / 2,
                       base);
    return (int)hipGetLastError();
}
