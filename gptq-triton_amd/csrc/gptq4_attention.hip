// Causal attention over a prompt for gfx950 (head dimension 128): the pass between the fused QKV + rotary projection,
// whose q and KV-cache rows it reads where they lie, and o_proj, whose input [B, S, H * 128] it writes directly.
// (The reference hands this step to torch's scaled_dot_product_attention and transposes the result,
// fused_attention.py:117-141; with a 2048-token prompt it is a sixth of the prompt pass.)
//
// One workgroup of four waves per 128 queries of one head, a wave per 32 queries; the keys come in blocks of 64
// through LDS, shared by the four waves.  Both products run on v_mfma_f32_32x32x16_f16 in their TRANSPOSED form, so
// that what one produces is what the next consumes without leaving the lane:
//   S^T = K Q^T   A = 32 keys x 16 dims out of LDS (rows of 256 bytes, 272 apart),
//                 B = the wave's queries, in registers for the whole kernel; lane (h, q) then holds, for its query
//                 column q, the scores of keys 8 * i + 4 * h + j of each half block (register 4 * i + j);
//   O^T = V^T P^T A = 32 dims x 16 keys, B = 16 keys x 32 queries: the lane's own probabilities, registers 8 * u .. 8 * u + 7
//                 of a half block for step u.  That fixes which key sits in which of the 16 contraction slots of a
//                 step - slot 8 * h + t is key 4 * h + t (t < 4) or 8 + 4 * h + t - 4 - and V^T is written to LDS with
//                 its keys in that order (the two middle groups of four swapped), rows of 64 keys = 128 bytes, 144 apart.
// The softmax runs per lane on its own query column (one exchange per block with the other half-wave for the running
// maximum; the row sums meet once, at the end), in base 2 with the scale folded in.  Blocks beyond a wave's last
// visible key are skipped by that wave; heavy and light query blocks are paired up by workgroup id (see the kernel).
#include "../../include/gptq4.h"
#include "gptq4_internal.h"

#include <type_traits>

namespace {

typedef float f16x_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
constexpr int FA_K_BUF = 64 * 17, FA_V_BUF = 128 * 9;                      // 16-byte chunks per buffer
constexpr size_t FA_LDS_BYTES = (size_t)2 * (FA_K_BUF + FA_V_BUF) * 16;  // 71,680
constexpr int FA_GROUP = 4;  // heads of an XCD worked on together when it has many (1 MiB of keys and values each at 2048 tokens; 4 MiB of L2)

// (fmaxf makes the compiler quiet possible signalling NaNs first, one more instruction per operand; the scores are
// matrix-core outputs or -inf.  Not on results of a matrix product that nothing has waited for: the compiler does not count
// the cycles between a product and an asm statement that reads its result, and the hardware does not wait.  Every chain of
// them begins with the fmaxf of a result of each product, in front of which the compiler puts the cycles they still need.)
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// The larger of the lane's value and that of the lane 32 on, in both.
__device__ __forceinline__ float max_of_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    const uint32_t own = r[0], other = r[1];  // (variables: of the vector's elements themselves the compiler casts the first one twice)
    return fmaxf(__builtin_bit_cast(float, own), __builtin_bit_cast(float, other));
}

// a * b, rounded by itself: not made one instruction with an addition that takes it.
__device__ __forceinline__ float product(float a, float b) {
#pragma clang fp contract(off)
    return a * b;
}

__device__ __forceinline__ int key_slot(int key) {  // position of a key of a 64-key block in V^T's row
    const int o = key & 15;
    return (key & ~15) | (o < 4 ? o : o < 8 ? o + 4 : o < 12 ? o - 4 : o);
}

__global__ __launch_bounds__(256, 2) void gptq4_attn_prefill_kernel(const half_t *__restrict__ q, const half_t *__restrict__ kc,
                                                                    const half_t *__restrict__ vc, half_t *__restrict__ out, int H,
                                                                    int S, int capacity, int past, float scale_log2e, int nq, int nbh) {
    // Two buffers of K [64 keys][16 chunks of 8 dims] and V^T [128 dims][8 chunks of 8 key slots], every row one chunk longer
    // than its data (17 and 9 chunks): the LDS serves a 16-byte read of 16 lanes at a time from 64 banks, and rows 272 /
    // 144 bytes apart put the 16 chunks into 16 different 16-byte slots of 256 - with plain strides, so that every address
    // below is a lane constant plus an immediate.
    extern __shared__ uint4 fa_smem[];
    uint4 *const k_s = fa_smem;                  // 2 x 64 x 17 chunks
    uint4 *const v_s = fa_smem + 2 * FA_K_BUF;   // 2 x 128 x 9 chunks
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, c32 = lane & 31;
    // Workgroup id -> (head, query block).  Consecutive ids go to the eight XCDs in turn, each with an L2 of its own:
    // id % 8 picks the XCD and all query blocks of a head are given to one XCD (head % 8, for the heads up to the last
    // multiple of eight; the rest are dealt as if there were one XCD), so that a head's keys and values are fetched into
    // one L2 only.  Within an XCD the heavy halves of all its heads come first (a query block's work grows with its
    // index), then the light halves in the matching order: when the whole grid is resident at once, a CU's two workgroups
    // are blocks nq - 1 - j and j of one head and add up to the same work everywhere; when it is not, long work goes first.
    int qb, bh;
    {
        const int nb8 = nbh & ~7, cut = nb8 * nq;
        int y = blockIdx.x, heads = nbh, head_step = 1, head0 = 0;
        if (y < cut) {
            head0 = y & 7, head_step = 8, heads = nb8 >> 3, y >>= 3;
        } else {
            y -= cut, heads = nbh - nb8, head0 = nb8;
        }
        // (more than eight heads to an XCD: in groups of FA_GROUP heads, each group in the order above, so that the keys and
        // values in use stay within the L2)
        int group0 = 0;
        if (heads > 8) {
            const int per = FA_GROUP * nq, g = y / per;
            group0 = g * FA_GROUP, y -= g * per, heads = min(FA_GROUP, heads - group0);
        }
        const int half = (nq + 1) >> 1, first = heads * half;
        int hl;
        if (y < first) {
            hl = y / half;
            qb = nq - 1 - (y - hl * half);
        } else {
            const int k = y - first, low = nq - half;
            hl = k / low;
            qb = k - hl * low;
        }
        hl += group0;
        bh = head0 + hl * head_step;
    }
    const int q0 = qb * 128 + wave * 32;  // first query of the wave
    const int kv_len = past + S;

    // ---- the wave's queries: B operand of S^T, lane (h, q): dims 16 * ks + 8 * h .. + 7
    h8_t qf[8];
    {
        const int row = min(q0 + c32, S - 1);
        const uint4 *qp = reinterpret_cast<const uint4 *>(q + ((size_t)bh * S + row) * 128);
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) qf[ks] = __builtin_bit_cast(h8_t, qp[2 * ks + h]);
    }
    f16x_t o[4];
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
    float m = -INFINITY, l = 0.f;

    const int kmax = min(kv_len, past + (qb + 1) * 128);  // keys any query of the workgroup sees
    const int nblk = (kmax + 63) >> 6;
    const int my_last = past + min(q0 + 31, S - 1);      // last key the wave's last query sees
    const int my_first = past + q0;                      // last key its first query sees
    const half_t *kb = kc + (size_t)bh * capacity * 128;
    const half_t *vb = vc + (size_t)bh * capacity * 128;

    // ---- staging, two LDS buffers: while block i is multiplied, block i + 1 goes from registers into the other buffer
    //      and block i + 2 is on its way from memory; one barrier per block.
    //      K chunk id = tid + 256 * n -> (key id / 16, chunk id % 16): whole rows per 16 lanes.
    //      V: thread (pair p = tid % 32, dc = tid / 32 + 8 * n) holds chunk dc of keys 2p and 2p + 1 - neighbours in V^T's
    //      slot order too - and writes, per dimension, one dword {key 2p, key 2p + 1}: half a wave fills 128 bytes of a row.
    // (buffer loads: rows from kv_len on come back as zeros - they are masked.  The block's offset is part of the lane
    // offset: the range check does not see a scalar offset)
    const int kv_bytes = (int)((uint32_t)kv_len * 256u);
    const uint32_t k_voff = (uint32_t)(tid >> 4) * 256u + (uint32_t)(tid & 15) * 16u;  // + 16 keys per n
    const uint32_t v_voff = (uint32_t)(2 * (tid & 31)) * 256u + (uint32_t)(tid >> 5) * 16u;  // + 1 key per kk, + 8 chunks per n
    u32x4_t kr[4], vr[2][2];
    // (a block beyond the last one is asked of an empty buffer: zeros without a trip to memory)
    auto fetch_k = [&](int blk, int n) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(kb), 0, blk < nblk ? kv_bytes : 0, 0x00020000);
        return __builtin_amdgcn_raw_buffer_load_b128(rs, k_voff + 16u * 256u * n + (uint32_t)blk * (64u * 256u), 0, 0);
    };
    auto fetch_v = [&](int blk, int n, int kk) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(vb), 0, blk < nblk ? kv_bytes : 0, 0x00020000);
        return __builtin_amdgcn_raw_buffer_load_b128(rs, v_voff + 256u * kk + 128u * n + (uint32_t)blk * (64u * 256u), 0, 0);
    };
#define FETCH_K(blk) _Pragma("unroll") for (int n = 0; n < 4; ++n) kr[n] = fetch_k(blk, n);
#define FETCH_V(blk) \
    _Pragma("unroll") for (int n = 0; n < 2; ++n) _Pragma("unroll") for (int kk = 0; kk < 2; ++kk) vr[n][kk] = fetch_v(blk, n, kk);
    const int vslot = key_slot(2 * (tid & 31));  // even: the pair's dword
    uint4 *const k_put = k_s + (tid >> 4) * 17 + (tid & 15);                                          // + 16 rows per n
    uint32_t *const v_put = reinterpret_cast<uint32_t *>(v_s) + (8 * (tid >> 5)) * 36 + (vslot >> 1);  // + 36 dwords per dim
    auto stage_k = [&](int buf, int n) { k_put[buf * FA_K_BUF + n * (16 * 17)] = __builtin_bit_cast(uint4, kr[n]); };
    auto stage_v = [&](int buf, int part) {  // an eighth of it: word part % 4 of chunk part / 4
        const int n = part >> 2, w = part & 3;
        const uint32_t lo = vr[n][0][w], hi = vr[n][1][w];
        // halves 2 * w and 2 * w + 1 of the two keys
        uint32_t *const at = v_put + buf * (FA_V_BUF * 4) + (64 * n + 2 * w) * 36;
        at[0] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
        at[36] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
    };
    // ---- The order of work.  A wave issues an instruction every five cycles and a product takes 32, so a step's some 330
    //      instructions (32 products, 32 LDS reads, 32 exponentials) bound a wave that is alone on its SIMD, and what it waits
    //      for in between comes on top: they are dealt to the products one by one.  Left to the compiler (fragments read one
    //      product ahead, exponentials in front of the products that take them, the accumulators rescaled behind a branch) a
    //      block of 64 keys took 1.45 us, now 1.2: 32 heads x 2000 tokens 60 -> 53 us, 8 x 2048 45 -> 39.5, 52 x 2000 103 -> 94,
    //      8 x 52 x 2048 629 -> 590, 32 x 128 behind 1000 28.2 -> 25.3.
    //      K is staged two blocks ahead of the block whose probabilities are being made and V one, in
    //      two buffers each, with one barrier per block: step i issues the products for the scores of block i + 1 with the
    //      probabilities of block i between them, then O^T += V^T P^T for block i with the maximum of block i + 1's scores and
    //      the staging between those.  Step i writes K block i + 2 over block i (last read in step i - 1) and V block
    //      i + 1 over block i - 1, and asks for K block i + 3 and V block i + 2 (beyond the last block: of an empty buffer).
    {
        FETCH_K(0)
        FETCH_V(0)
        u32x4_t k1[4];  // (block 1 of K asked for together with block 0: one round trip to memory before the first product)
        if (nblk > 1) {
#pragma unroll
            for (int n = 0; n < 4; ++n) k1[n] = fetch_k(1, n);
        }
#pragma unroll
        for (int n = 0; n < 4; ++n) stage_k(0, n);
#pragma unroll
        for (int n = 0; n < 8; ++n) stage_v(0, n);
        if (nblk > 1) {
#pragma unroll
            for (int n = 0; n < 4; ++n) k_put[FA_K_BUF + n * (16 * 17)] = __builtin_bit_cast(uint4, k1[n]);
            FETCH_K(2)
            FETCH_V(1)
        }
    }
    const uint4 *const k_get = k_s + c32 * 17 + h;  // the lane's key row of a half block, chunk h
    const uint4 *const v_get = v_s + c32 * 9 + h;   // the lane's dim row of a block of 32, chunk h
    // operand A of product n of a step: K block i + 1 (0 .. 15, the two half blocks of 32 keys in turn), V block i (16 .. 31,
    // four blocks of 32 dims to a step of 16 keys)
    auto fragment = [&](int buf, int n) {
        return __builtin_bit_cast(h8_t, n < 16 ? k_get[(buf ^ 1) * FA_K_BUF + (n & 1) * (32 * 17) + 2 * (n >> 1)]
                                               : v_get[buf * FA_V_BUF + (n & 3) * (32 * 9) + 2 * ((n - 16) >> 2)]);
    };
    f16x_t sa[2], sb[2];
    auto block_max = [&](const f16x_t(&s)[2]) {
        float mx = fmaxf(s[0][0], s[1][0]);
#pragma unroll
        for (int i = 1; i < 16; ++i) mx = max3(mx, s[0][i], s[1][i]);
        return mx;
    };
    __syncthreads();
#pragma unroll
    for (int n = 0; n < 16; ++n) {
        if (n < 2) {
#pragma unroll
            for (int i = 0; i < 16; ++i) sa[n & 1][i] = 0.f;
        }
        sa[n & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fragment(1, n), qf[n >> 1], sa[n & 1], 0, 0, 0);
    }
    float mx = block_max(sa);  // of the lane's scores of the block to come
    constexpr int AHEAD = 4;   // LDS reads in flight ahead of the products
    // (last: the workgroup's last block, which no other's scores and no staging follow)
    auto step = [&](int blk, auto parity, auto last, f16x_t(&s)[2], f16x_t(&sn)[2]) {
        constexpr int buf = decltype(parity)::value;
        constexpr bool LAST = decltype(last)::value;
        __syncthreads();  // K block blk + 1 and V block blk are in their buffers; the buffers written below have been read
        const int key0 = blk * 64;
        h8_t ring[AHEAD];
#pragma unroll
        for (int n = 0; n < AHEAD; ++n) ring[n] = fragment(buf, LAST ? 16 + n : n);
        // ---- masking (only a block that reaches past the wave's first query's last key)
        if (key0 + 63 > my_first) {
            asm volatile("" ::: "memory");  // (keeps this a branch: turned into selects the masking would run for every block)
            const int limit = past + q0 + c32 - key0 - 4 * h;  // last visible key of this lane's query, in the lane's numbering
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (32 * rb + 8 * (i >> 2) + (i & 3) > limit) s[rb][i] = -INFINITY;
            mx = block_max(s);
        }
        const float m_new = fmaxf(m, max_of_halves(mx) * scale_log2e);  // (the scale is positive: the maximum commutes with it)
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;  // (a query beyond S in a clamped row: nothing visible yet)
        const float corr = __builtin_amdgcn_exp2f(m - m_use);
        m = m_new;
        float sum = 0.f;
        const h2_t ones = {(_Float16)1.0f, (_Float16)1.0f};
        uint32_t pf[4][4];
        // Probabilities 2 * p and 2 * p + 1 of the lane's 32 in three stages, a slot apart so that none waits for the one before
        // (the row sum takes them as the product takes them: rounded to fp16, two per instruction).  The empty asm statements
        // keep them where they stand: the compiler sinks arithmetic towards its use, past the scheduling barriers.
        auto probability = [&](int p, int stage) {
            if (p < 0 || p > 15) return;
            const int rb = p >> 3, i = 2 * (p & 7);
            float x = s[rb][i], y = s[rb][i + 1];
            if (stage == 0) x = __builtin_fmaf(x, scale_log2e, -m_use), y = __builtin_fmaf(y, scale_log2e, -m_use);
            if (stage == 1) x = __builtin_amdgcn_exp2f(x), y = __builtin_amdgcn_exp2f(y);
            if (stage == 2) {
                const h2_t pp = {(_Float16)x, (_Float16)y};
                sum = __builtin_amdgcn_fdot2(pp, ones, sum, false);
                pf[p >> 2][p & 3] = as_u32(pp);
                asm volatile("" : "+v"(pf[p >> 2][p & 3]), "+v"(sum));
                return;
            }
            asm volatile("" : "+v"(x), "+v"(y));
            s[rb][i] = x, s[rb][i + 1] = y;
        };
        // slot n of the step's 32: pair p's stages in slots 3 * p / 2, + 1 and + 2 (the products of its 16 keys are in slots
        // 16 + 4 * (p / 4) and on)
        auto probabilities = [&](int n) {
#pragma unroll
            for (int stage = 0; stage < 3; ++stage) {
                const int at = n - stage;
                if (at >= 0 && at % 3 != 2) probability(2 * (at / 3) + at % 3, stage);
            }
        };
        // (ahead of the other workgroup's wave on this SIMD while that one is staging or waiting at its barrier: 656 -> 622 us
        // at 416 heads, 84.6 -> 80.1 at 40)
        __builtin_amdgcn_s_setprio(1);
        l = product(l, corr);  // (`sum` is added behind it: with one rounding for both, a result in some 10^4 is another fp16 value)
        // The next block's scores, and the accumulators brought to the new maximum on the way.  (Some lane's maximum moves in
        // most blocks of a sequence: behind a branch these 64 instructions took 380 of 2700 cycles a block on average.  An
        // older maximum kept until it is 2^8 too small saves most of them too, but the largest probability is then no longer an
        // exact 1: 2 - 6 % further from 64 bits.)
#pragma unroll
        for (int n = 0; n < 16; ++n) {
            if constexpr (!LAST) {
                if (n < 2) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) sn[n & 1][i] = 0.f;
                }
                sn[n & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ring[n % AHEAD], qf[n >> 1], sn[n & 1], 0, 0, 0);
                ring[n % AHEAD] = fragment(buf, n + AHEAD);
            }
            probabilities(n);
#pragma unroll
            for (int i = 0; i < 4; ++i) o[n >> 2][4 * (n & 3) + i] *= corr;
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // the product first
            __builtin_amdgcn_sched_barrier(0);
        }
        float mx2 = -INFINITY;  // (two in turns: neither waits for the other)
#pragma unroll
        for (int n = 0; n < 16; ++n) {
            const h8_t pv = __builtin_bit_cast(h8_t, (u32x4_t){pf[n >> 2][0], pf[n >> 2][1], pf[n >> 2][2], pf[n >> 2][3]});
            o[n & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ring[n % AHEAD], pv, o[n & 3], 0, 0, 0);
            if (n + AHEAD < 16) ring[n % AHEAD] = fragment(buf, 16 + n + AHEAD);
            probabilities(16 + n);
            if (LAST) {
            } else if (n < 4) {
                stage_k(buf, n);
                kr[n] = fetch_k(blk + 3, n);
            } else if (n < 12) {
                stage_v(buf ^ 1, n - 4);
                if (n == 7 || n == 11) vr[n >> 3][0] = fetch_v(blk + 2, n >> 3, 0), vr[n >> 3][1] = fetch_v(blk + 2, n >> 3, 1);
            }
            if (!LAST && n == 8) {
                mx = fmaxf(sn[0][0], sn[1][0]);
                mx2 = max3(mx, sn[0][1], sn[1][1]);
            }
            if (!LAST && n > 8) {
                mx = max3(mx, sn[0][2 * n - 16], sn[1][2 * n - 16]);
                mx2 = max3(mx2, sn[0][2 * n - 15], sn[1][2 * n - 15]);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        mx = fmaxf(mx, mx2);
        l += sum;
        __builtin_amdgcn_s_setprio(0);
    };
    using even = std::integral_constant<int, 0>;
    using odd = std::integral_constant<int, 1>;
    const int mine = (my_last >> 6) + 1;  // blocks that the wave sees a key of
    const int followed = min(mine, nblk - 1);
    for (int blk = 0; blk < followed; blk += 2) {
        step(blk, even{}, std::false_type{}, sa, sb);
        if (blk + 1 < followed) step(blk + 1, odd{}, std::false_type{}, sb, sa);
    }
    if (mine == nblk) {
        if (followed & 1)
            step(followed, odd{}, std::true_type{}, sb, sa);
        else
            step(followed, even{}, std::true_type{}, sa, sb);
    }
    for (int blk = mine; blk < nblk; ++blk) {  // (the workgroup's others: the wave only takes part in the staging)
        __syncthreads();
        if (blk + 1 < nblk) {
#pragma unroll
            for (int n = 0; n < 4; ++n) stage_k(blk & 1, n);
#pragma unroll
            for (int n = 0; n < 8; ++n) stage_v((blk & 1) ^ 1, n);
            FETCH_K(blk + 3)
            FETCH_V(blk + 2)
        }
    }

    // ---- out[b, s, head * 128 + d] = O[s, d] / l: lane (h, q) holds dims 32 * db + 8 * i + 4 * h + j of its query
    l += __shfl_xor(l, 32);
    const int row = q0 + c32;
    if (row < S) {
        const float inv = 1.0f / l;
        const int b = bh / H, head = bh - b * H;
        half_t *dst = out + (((size_t)b * S + row) * H + head) * 128;
#pragma unroll
        for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                h2_t lo, hi;
                lo.x = (half_t)(o[db][4 * i] * inv);
                lo.y = (half_t)(o[db][4 * i + 1] * inv);
                hi.x = (half_t)(o[db][4 * i + 2] * inv);
                hi.y = (half_t)(o[db][4 * i + 3] * inv);
                uint2 w;
                w.x = __builtin_bit_cast(uint32_t, lo);
                w.y = __builtin_bit_cast(uint32_t, hi);
                *reinterpret_cast<uint2 *>(dst + 32 * db + 8 * i + 4 * h) = w;
            }
    }
}

#undef FETCH_K
#undef FETCH_V

}  // namespace

int launch_attn_prefill(const half_t *q, const half_t *kc, const half_t *vc, half_t *out, int B, int H, int S, int capacity, int past,
                        float scale, hipStream_t stream) {
    const int qblocks = (S + 127) / 128;
    static LdsGrant grant;
    if (const int rc = allow_lds(grant, reinterpret_cast<const void *>(&gptq4_attn_prefill_kernel), FA_LDS_BYTES)) return rc;
    hipLaunchKernelGGL(gptq4_attn_prefill_kernel, dim3((unsigned)(qblocks * B * H)), dim3(256), FA_LDS_BYTES, stream, q, kc, vc, out, H, S,
                       capacity, past, scale * 1.4426950408889634f, qblocks, B * H);
    return (int)hipGetLastError();
}
