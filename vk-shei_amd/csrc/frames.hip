// Portable-backend decode: one query token over exact K/V frames.
//
// Replaces GpuBackend::decode (gpu_backend.rs:149-377), whose OpenCL kernels
// mslim_qk / mslim_softmax / mslim_pv (gpu_attention.cl:5-82) take an f32
// query [q_heads][D], raw little-endian K/V frames [tokens][kv_heads][D] in
// BF16, F16 or F32 (key and value formats independent) and produce f32
// output [q_heads][D].  Everything here is computed in f32; formats are
// decoded exactly (BF16 and F16 widen to f32 without rounding).
//
// Two kernels.  frames_group_kernel takes head dimensions that are a multiple
// of 8 up to 256 with 16-byte aligned rows: a workgroup owns one kv head (up to
// eight of its query heads) and one split of the tokens, so each K and V byte
// is read once for the whole group, in 16-byte pieces of whole rows.
// frames_split_kernel takes every other shape: a workgroup owns one (query
// head, split) pair, one token per thread for the score, then P.V with the
// head dimension across threads.  Both carry an online softmax over the
// tokens of a split, and the splits are combined in fixed order (in the last
// workgroup of a kv head, or by a merge launch), so the result is
// deterministic for a given split count.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace mslim {

namespace {

constexpr int kThreads = 256;

template <int FMT>
struct Fmt;
template <>
struct Fmt<kFormatBf16> {
    __device__ static float at(const void *p, int64_t i) {
        return read_bf16(static_cast<const uint16_t *>(p)[i]);
    }
    __device__ static void widen8(const uint4 w, float *out) {
        const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            out[2 * j] = bf16_lo(u[j]);
            out[2 * j + 1] = bf16_hi(u[j]);
        }
    }
};
template <>
struct Fmt<kFormatF16> {
    __device__ static float at(const void *p, int64_t i) {
        return half_to_float(static_cast<const uint16_t *>(p)[i]);
    }
    __device__ static void widen8(const uint4 w, float *out) {
        const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            out[2 * j] = half_to_float((uint16_t)(u[j] & 0xffffu));
            out[2 * j + 1] = half_to_float((uint16_t)(u[j] >> 16));
        }
    }
};
template <>
struct Fmt<kFormatF32> {
    __device__ static float at(const void *p, int64_t i) { return static_cast<const float *>(p)[i]; }
};

struct FramesArgs {
    const float *q;
    const void *k, *v;
    float *out;
    float *partial_ml;   // [q_heads][splits][2]
    float *partial_acc;  // [q_heads][splits][D]
    int64_t tokens;
    int q_heads, kv_heads, head_dim;
    int split_tokens, splits;
    float scale;
    int *counters;  // frames_group_kernel: [kv_heads][head chunks], zero between launches
};

// Block-wide reductions of one float per thread (every thread gets the result).
__device__ float block_max(float v, float *red) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = wave_xor_max(v, m);
    const int wave = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[wave] = v;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}
__device__ float block_sum(float v, float *red) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = wave_xor_sum(v, m);
    const int wave = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[4 + wave] = v;
    __syncthreads();
    return (red[4] + red[5]) + (red[6] + red[7]);
}

// Dot product of the query (in LDS) with one key row.  VEC reads the row in
// 16-byte pieces; the caller guarantees 16-byte alignment of every row.
template <int KF, bool VEC>
__device__ float key_dot(const float *q_lds, const void *k, int64_t row, int d) {
    float dot = 0.0f;
    if constexpr (VEC && KF != kFormatF32) {
        const uint4 *p = reinterpret_cast<const uint4 *>(static_cast<const char *>(k) + row * 2);
        for (int j = 0; j < d; j += 8) {
            float e[8];
            Fmt<KF>::widen8(p[j / 8], e);
#pragma unroll
            for (int i = 0; i < 8; ++i) dot = fmaf(q_lds[j + i], e[i], dot);
        }
    } else if constexpr (VEC) {
        const float4 *p = reinterpret_cast<const float4 *>(static_cast<const float *>(k) + row);
        for (int j = 0; j < d; j += 4) {
            const float4 e = p[j / 4];
            dot = fmaf(q_lds[j], e.x, dot);
            dot = fmaf(q_lds[j + 1], e.y, dot);
            dot = fmaf(q_lds[j + 2], e.z, dot);
            dot = fmaf(q_lds[j + 3], e.w, dot);
        }
    } else {
        for (int j = 0; j < d; ++j) dot = fmaf(q_lds[j], Fmt<KF>::at(k, row + j), dot);
    }
    return dot;
}

// DG threads share one token's P.V row (DG = the head dimension rounded up to
// a power of two, at most 256); kThreads / DG groups take interleaved tokens.
template <int KF, int VF, bool VEC>
__global__ __launch_bounds__(kThreads) void frames_split_kernel(FramesArgs a) {
    __shared__ float q_lds[kFramesMaxDim];
    __shared__ float p_lds[kThreads];
    __shared__ float red[8];
    __shared__ float acc_lds[kThreads];

    const int tid = threadIdx.x;
    const int qh = blockIdx.y;
    const int split = blockIdx.x;
    const int d = a.head_dim;
    const int kvh = qh / (a.q_heads / a.kv_heads);
    for (int j = tid; j < d; j += kThreads) q_lds[j] = a.q[(int64_t)qh * d + j];

    int dg = 1;
    while (dg < d && dg < kThreads) dg <<= 1;
    const int groups = kThreads / dg;
    const int grp = tid / dg;
    const int lane_d = tid % dg;
    constexpr int kMaxPer = kFramesMaxDim / kThreads;  // dims per thread when D > 256
    float acc[kMaxPer];
#pragma unroll
    for (int i = 0; i < kMaxPer; ++i) acc[i] = 0.0f;

    const int64_t begin = (int64_t)split * a.split_tokens;
    const int64_t end = min(a.tokens, begin + a.split_tokens);
    const int64_t row_stride = (int64_t)a.kv_heads * d;
    float m_run = -INFINITY, l_run = 0.0f;
    __syncthreads();

    for (int64_t t0 = begin; t0 < end; t0 += kThreads) {
        const int64_t t = t0 + tid;
        float s = -INFINITY;
        if (t < end) s = key_dot<KF, VEC>(q_lds, a.k, t * row_stride + (int64_t)kvh * d, d) * a.scale;
        const float m_new = fmaxf(m_run, block_max(s, red));
        const float alpha = expf(m_run - m_new);
        const float p = t < end ? expf(s - m_new) : 0.0f;
        p_lds[tid] = p;
        l_run = l_run * alpha + block_sum(p, red);  // block_sum's barriers publish p_lds
        m_run = m_new;
#pragma unroll
        for (int i = 0; i < kMaxPer; ++i) acc[i] *= alpha;
        const int n = (int)min((int64_t)kThreads, end - t0);
        for (int j = grp; j < n; j += groups) {
            const float pj = p_lds[j];
            const int64_t vrow = (t0 + j) * row_stride + (int64_t)kvh * d;
#pragma unroll
            for (int i = 0; i < kMaxPer; ++i) {
                const int dim = lane_d + i * dg;
                if (dim < d) acc[i] = fmaf(pj, Fmt<VF>::at(a.v, vrow + dim), acc[i]);
            }
        }
        __syncthreads();  // p_lds is rewritten by the next tile
    }

    // Sum the token groups (only when several share the tile: then D <= 128
    // and each thread holds one dimension).
    if (groups > 1) {
        acc_lds[tid] = acc[0];
        __syncthreads();
        if (tid < dg) {
            float sum = 0.0f;
            for (int g = 0; g < groups; ++g) sum += acc_lds[g * dg + tid];
            acc[0] = sum;
        }
    }
    if (grp != 0) return;
    if (a.splits == 1) {
#pragma unroll
        for (int i = 0; i < kMaxPer; ++i) {
            const int dim = lane_d + i * dg;
            if (dim < d) a.out[(int64_t)qh * d + dim] = acc[i] / l_run;
        }
        return;
    }
    const int64_t slot = (int64_t)qh * a.splits + split;
    if (tid == 0) {
        a.partial_ml[slot * 2] = m_run;
        a.partial_ml[slot * 2 + 1] = l_run;
    }
#pragma unroll
    for (int i = 0; i < kMaxPer; ++i) {
        const int dim = lane_d + i * dg;
        if (dim < d) a.partial_acc[slot * d + dim] = acc[i];
    }
}

// Fixed-order log-sum-exp merge of the splits of one query head.
__global__ __launch_bounds__(kThreads) void frames_merge_kernel(FramesArgs a) {
    const int qh = blockIdx.x;
    const float *ml = a.partial_ml + (int64_t)qh * a.splits * 2;
    const float *acc = a.partial_acc + (int64_t)qh * a.splits * a.head_dim;
    float m = -INFINITY;
    for (int s = 0; s < a.splits; ++s) m = fmaxf(m, ml[2 * s]);
    float l = 0.0f;
    for (int s = 0; s < a.splits; ++s) l += expf(ml[2 * s] - m) * ml[2 * s + 1];
    for (int dim = threadIdx.x; dim < a.head_dim; dim += kThreads) {
        float o = 0.0f;
        for (int s = 0; s < a.splits; ++s) o += expf(ml[2 * s] - m) * acc[(int64_t)s * a.head_dim + dim];
        a.out[(int64_t)qh * a.head_dim + dim] = o / l;
    }
}

// Eight elements of a row as f32.
template <int FMT>
struct Row8 {
    uint4 w;
    __device__ __forceinline__ void load(const void *p, int64_t i) {
        w = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(p) + i);
    }
    __device__ __forceinline__ void widen(float *out) const { Fmt<FMT>::widen8(w, out); }
};
template <>
struct Row8<kFormatF32> {
    float4 lo, hi;
    __device__ __forceinline__ void load(const void *p, int64_t i) {
        const float4 *q = reinterpret_cast<const float4 *>(static_cast<const float *>(p) + i);
        lo = q[0];
        hi = q[1];
    }
    __device__ __forceinline__ void widen(float *out) const {
        out[0] = lo.x; out[1] = lo.y; out[2] = lo.z; out[3] = lo.w;
        out[4] = hi.x; out[5] = hi.y; out[6] = hi.z; out[7] = hi.w;
    }
};

// Sum over the LPR lanes (8, 16 or 32, aligned) that hold a row: cross-lane
// moves inside 16 lanes, one exchange beyond.  Every lane gets the sum.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
    return x + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
template <int LPR>
__device__ __forceinline__ float row_sum(float x) {
    x = dpp_add<0xB1>(x);   // quad_perm 1,0,3,2
    x = dpp_add<0x4E>(x);   // quad_perm 2,3,0,1
    x = dpp_add<0x141>(x);  // mirror of 8
    if (LPR >= 16) x = dpp_add<0x140>(x);  // mirror of 16
    if (LPR >= 32) x += __shfl_xor(x, 16, 64);
    return x;
}

// Relaxed agent-scope pairs: written through to, and read from, the point
// where the XCDs' L2 caches meet (the order of decode.hip's split merge).
__device__ __forceinline__ void put_pair(float *p, float x, float y) {
    const uint64_t w = (uint64_t)__float_as_uint(x) | ((uint64_t)__float_as_uint(y) << 32);
    __hip_atomic_store(reinterpret_cast<uint64_t *>(p), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 get_pair(const float *p) {
    const uint64_t w = __hip_atomic_load(reinterpret_cast<const uint64_t *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_float2(__uint_as_float((uint32_t)w), __uint_as_float((uint32_t)(w >> 32)));
}

// One (kv head, chunk of at most GT of its query heads, split) per workgroup.
// LPR lanes hold a row, 8 dimensions each (lanes past the head dimension hold
// zeros), so a load instruction covers 64 / LPR whole rows and a score is 8
// FMAs and a lane sum; the row's lanes then add p times their V piece.  Everything is
// f32, as in frames_split_kernel, with exp2 of scores in log2 units.  Bound by
// latency: the few loads each workgroup makes, then the count and the merge.  Against one workgroup per
// (query head, split), whose lanes each walked a row of their own: 4,096
// tokens of binary16, 32/8 heads of 128 (17 MB): 55.3 us (two launches) -> 12.8
// us; 300 tokens of 24/8 heads 8.0 us.
// Loads of K, and of V, in flight per wavefront: four, two where eight heads'
// queries and sums leave no registers for more.
constexpr int group_steps(int heads) { return heads == 8 ? 2 : 4; }
constexpr int kGroupWaves = kThreads / 64;

template <int KF, int VF, int LPR, int GT>
__global__ __launch_bounds__(kThreads) void frames_group_kernel(FramesArgs a) {
    constexpr int kSteps = group_steps(GT);
    constexpr int RPI = 64 / LPR;                       // rows per load instruction
    constexpr int ROWS = kGroupWaves * kSteps * RPI;    // tokens per iteration of the workgroup
    constexpr int PARTS = kGroupWaves * RPI;            // running softmaxes per query head
    constexpr int DMAX = LPR * 8;
    __shared__ __align__(16) float acc_lds[PARTS][GT][DMAX];
    __shared__ float ml_lds[PARTS][GT][2];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane / LPR, d0 = (lane % LPR) * 8;
    const int dim = a.head_dim;
    const int group = a.q_heads / a.kv_heads;
    const int chunks = (group + GT - 1) / GT;
    const int split = blockIdx.x;
    const int kvh = blockIdx.y / chunks, chunk = blockIdx.y % chunks;
    const int heads = min(GT, group - chunk * GT);  // of this workgroup
    const int qh0 = kvh * group + chunk * GT;
    const bool live = d0 < dim;
    const int dc = live ? d0 : 0;

    float q[GT][8], acc[GT][8], m[GT], l[GT];
#pragma unroll
    for (int g = 0; g < GT; ++g) {
        // (lanes past the head dimension hold zeros through their K pieces)
        const float4 *qp = reinterpret_cast<const float4 *>(a.q + (int64_t)(qh0 + min(g, heads - 1)) * dim + dc);
        const float4 lo = qp[0], hi = qp[1];
        q[g][0] = lo.x; q[g][1] = lo.y; q[g][2] = lo.z; q[g][3] = lo.w;
        q[g][4] = hi.x; q[g][5] = hi.y; q[g][6] = hi.z; q[g][7] = hi.w;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][e] = 0.0f;
        m[g] = -INFINITY;
        l[g] = 0.0f;
    }
    const float scale = a.scale * kLog2e;  // scores in log2 units
    const int64_t begin = (int64_t)split * a.split_tokens;
    const int64_t end = min(a.tokens, begin + a.split_tokens);
    const int64_t row_stride = (int64_t)a.kv_heads * dim;
    const int64_t head_off = (int64_t)kvh * dim + dc;

    // Rows past the split re-read its last row; their p is zero.  The next
    // iteration's K pieces load over this one's once its scores are taken, and
    // likewise V.
    Row8<KF> kr[kSteps];
    Row8<VF> vr[kSteps];
    auto load_k = [&](int64_t t0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kSteps; ++u)
            kr[u].load(a.k, min(t0 + u * RPI + lr, end - 1) * row_stride + head_off);
    };
    auto load_v = [&](int64_t t0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kSteps; ++u)
            vr[u].load(a.v, min(t0 + u * RPI + lr, end - 1) * row_stride + head_off);
    };
    const int64_t first = begin + wave * kSteps * RPI;
    load_k(first);
    load_v(first);
    for (int64_t t0 = first; t0 < end; t0 += ROWS) {
        float s[kSteps][GT];
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
            float kv[8];
            kr[u].widen(kv);
            if (!live) {
#pragma unroll
                for (int e = 0; e < 8; ++e) kv[e] = 0.0f;
            }
            const bool valid = t0 + u * RPI + lr < end;
#pragma unroll
            for (int g = 0; g < GT; ++g) {
                float dot = q[g][0] * kv[0];
#pragma unroll
                for (int e = 1; e < 8; ++e) dot = fmaf(q[g][e], kv[e], dot);
                const float score = row_sum<LPR>(dot) * scale;
                s[u][g] = valid ? score : -INFINITY;
            }
        }
        if (t0 + ROWS < end) load_k(t0 + ROWS);
#pragma unroll
        for (int g = 0; g < GT; ++g) {
            float m_new = m[g];
#pragma unroll
            for (int u = 0; u < kSteps; ++u) m_new = fmaxf(m_new, s[u][g]);
            // A row group that has met no score above -inf keeps m = -inf and
            // l = 0: a score of -inf (a row past the split, or a key's own)
            // weighs nothing whatever the base.
            const float alpha = m_new == m[g] ? 1.0f : __builtin_amdgcn_exp2f(m[g] - m_new);
            const float base = m_new == -INFINITY ? 0.0f : m_new;
            m[g] = m_new;
            l[g] *= alpha;
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[g][e] *= alpha;
#pragma unroll
            for (int u = 0; u < kSteps; ++u) {
                s[u][g] = t0 + u * RPI + lr < end ? __builtin_amdgcn_exp2f(s[u][g] - base) : 0.0f;
                l[g] += s[u][g];
            }
        }
#pragma unroll
        for (int u = 0; u < kSteps; ++u) {
            float vv[8];
            vr[u].widen(vv);
            // a repeated row adds nothing, whatever it holds
            if (t0 + u * RPI + lr >= end) {
#pragma unroll
                for (int e = 0; e < 8; ++e) vv[e] = 0.0f;
            }
#pragma unroll
            for (int g = 0; g < GT; ++g)
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[g][e] = fmaf(s[u][g], vv[e], acc[g][e]);
        }
        if (t0 + ROWS < end) load_v(t0 + ROWS);
    }

    const int part = wave * RPI + lr;
#pragma unroll
    for (int g = 0; g < GT; ++g) {
        *reinterpret_cast<float4 *>(&acc_lds[part][g][d0]) = make_float4(acc[g][0], acc[g][1], acc[g][2], acc[g][3]);
        *reinterpret_cast<float4 *>(&acc_lds[part][g][d0 + 4]) = make_float4(acc[g][4], acc[g][5], acc[g][6], acc[g][7]);
        if (d0 == 0) {
            ml_lds[part][g][0] = m[g];
            ml_lds[part][g][1] = l[g];
        }
    }
    __syncthreads();

    // The softmaxes of the workgroup, then (splits > 1) those of the splits,
    // in fixed order: thread -> (query head, 4 dimensions).
    const int items = heads * (dim / 4);
    for (int it = tid; it < items; it += kThreads) {
        const int g = it / (dim / 4), d = it % (dim / 4) * 4;
        float mx = -INFINITY, sum = 0.0f;
        float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int i = 0; i < PARTS; ++i) mx = fmaxf(mx, ml_lds[i][g][0]);
#pragma unroll
        for (int i = 0; i < PARTS; ++i) {
            // l = 0: every score of this part was -inf, or it had no token
            const float w = ml_lds[i][g][1] == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(ml_lds[i][g][0] - mx);
            sum = fmaf(w, ml_lds[i][g][1], sum);
            const float4 x = *reinterpret_cast<const float4 *>(&acc_lds[i][g][d]);
            o.x = fmaf(w, x.x, o.x); o.y = fmaf(w, x.y, o.y); o.z = fmaf(w, x.z, o.z); o.w = fmaf(w, x.w, o.w);
        }
        const int64_t slot = (int64_t)(qh0 + g) * a.splits + split;
        if (a.splits == 1) {
            *reinterpret_cast<float4 *>(a.out + (int64_t)(qh0 + g) * dim + d) =
                make_float4(o.x / sum, o.y / sum, o.z / sum, o.w / sum);
        } else {
            float *p = a.partial_acc + slot * dim + d;
            put_pair(p, o.x, o.y);
            put_pair(p + 2, o.z, o.w);
            if (d == 0) put_pair(a.partial_ml + slot * 2, mx, sum);
        }
    }
    if (a.splits == 1) return;
    // Every store of this workgroup has reached the coherence point before
    // thread 0 counts it; the workgroup that counts last merges.
    __builtin_amdgcn_s_waitcnt(0);
    __shared__ int last;
    __syncthreads();
    if (tid == 0) {
        int *ctr = a.counters + blockIdx.y;
        last = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.splits - 1;
        if (last) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last) return;
    // The threads beyond the items share the splits: lane group j takes splits
    // j, j + ways, ... and the groups meet in LDS, in order.
    const int ways = items >= kThreads ? 1 : min(kThreads / items, PARTS);
    const int way = tid / items;
    for (int it = ways > 1 ? tid % items : tid; it < items; it += kThreads) {
        const int g = it / (dim / 4), d = it % (dim / 4) * 4;
        const int64_t slot0 = (int64_t)(qh0 + g) * a.splits;
        float mx = -INFINITY, sum = 0.0f;
        float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        // one round trip per kBatch splits; indices past the last repeat it
        constexpr int kBatch = GT == 8 ? 8 : 16;
        for (int s0 = way; s0 < a.splits && way < ways; s0 += kBatch * ways) {
            float2 ml[kBatch], x0[kBatch], x1[kBatch];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const int64_t slot = slot0 + min(s0 + j * ways, a.splits - 1);
                ml[j] = get_pair(a.partial_ml + slot * 2);
                x0[j] = get_pair(a.partial_acc + slot * dim + d);
                x1[j] = get_pair(a.partial_acc + slot * dim + d + 2);
            }
            float m_new = mx;
#pragma unroll
            for (int j = 0; j < kBatch; ++j) m_new = fmaxf(m_new, ml[j].x);
            const float alpha = m_new == mx ? 1.0f : __builtin_amdgcn_exp2f(mx - m_new);
            mx = m_new;
            sum *= alpha;
            o.x *= alpha; o.y *= alpha; o.z *= alpha; o.w *= alpha;
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                if (s0 + j * ways < a.splits) {
                    const float w = ml[j].y == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(ml[j].x - mx);
                    sum = fmaf(w, ml[j].y, sum);
                    o.x = fmaf(w, x0[j].x, o.x); o.y = fmaf(w, x0[j].y, o.y);
                    o.z = fmaf(w, x1[j].x, o.z); o.w = fmaf(w, x1[j].y, o.w);
                }
            }
        }
        if (ways > 1) {
            __syncthreads();  // every thread is here: one pass, items < kThreads
            if (way < ways) {
                *reinterpret_cast<float4 *>(&acc_lds[way][g][d]) = o;
                if (d == 0) {
                    ml_lds[way][g][0] = mx;
                    ml_lds[way][g][1] = sum;
                }
            }
            __syncthreads();
            if (way > 0) return;
            mx = -INFINITY;
            for (int j = 0; j < ways; ++j) mx = fmaxf(mx, ml_lds[j][g][0]);
            sum = 0.0f;
            o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            for (int j = 0; j < ways; ++j) {
                const float w = ml_lds[j][g][1] == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(ml_lds[j][g][0] - mx);
                sum = fmaf(w, ml_lds[j][g][1], sum);
                const float4 x = *reinterpret_cast<const float4 *>(&acc_lds[j][g][d]);
                o.x = fmaf(w, x.x, o.x); o.y = fmaf(w, x.y, o.y); o.z = fmaf(w, x.z, o.z); o.w = fmaf(w, x.w, o.w);
            }
        }
        *reinterpret_cast<float4 *>(a.out + (int64_t)(qh0 + g) * dim + d) =
            make_float4(o.x / sum, o.y / sum, o.z / sum, o.w / sum);
    }
}

// Output of an empty cache (gpu_backend.rs:157-159); a kernel rather than a
// memset so that the call stays a plain kernel node under graph capture.
__global__ __launch_bounds__(kThreads) void frames_zero_kernel(float *out, int n) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n) out[i] = 0.0f;
}

// Query heads per workgroup of frames_group_kernel: the group, in chunks of at
// most eight.
int group_heads(int group) { return group >= 5 ? 8 : group >= 3 ? 4 : group; }

template <int KF, int VF, int LPR>
hipError_t launch_group(const FramesArgs &a, hipStream_t stream) {
    const int group = a.q_heads / a.kv_heads, gt = group_heads(group);
    const dim3 grid((unsigned)a.splits, (unsigned)(a.kv_heads * ((group + gt - 1) / gt)));
    if (gt == 8) hipLaunchKernelGGL((frames_group_kernel<KF, VF, LPR, 8>), grid, dim3(kThreads), 0, stream, a);
    else if (gt == 4) hipLaunchKernelGGL((frames_group_kernel<KF, VF, LPR, 4>), grid, dim3(kThreads), 0, stream, a);
    else if (gt == 2) hipLaunchKernelGGL((frames_group_kernel<KF, VF, LPR, 2>), grid, dim3(kThreads), 0, stream, a);
    else hipLaunchKernelGGL((frames_group_kernel<KF, VF, LPR, 1>), grid, dim3(kThreads), 0, stream, a);
    return hipGetLastError();
}

template <int KF, int VF>
hipError_t launch_formats(const FramesArgs &a, bool grouped, bool vec, hipStream_t stream) {
    if (grouped) {
        if (a.head_dim <= 64) return launch_group<KF, VF, 8>(a, stream);
        if (a.head_dim <= 128) return launch_group<KF, VF, 16>(a, stream);
        return launch_group<KF, VF, 32>(a, stream);
    }
    const dim3 grid((unsigned)a.splits, (unsigned)a.q_heads);
    if (vec)
        hipLaunchKernelGGL((frames_split_kernel<KF, VF, true>), grid, dim3(kThreads), 0, stream, a);
    else
        hipLaunchKernelGGL((frames_split_kernel<KF, VF, false>), grid, dim3(kThreads), 0, stream, a);
    return hipGetLastError();
}

template <int KF>
hipError_t launch_value_format(const FramesArgs &a, int vf, bool grouped, bool vec, hipStream_t stream) {
    if (vf == kFormatBf16) return launch_formats<KF, kFormatBf16>(a, grouped, vec, stream);
    if (vf == kFormatF16) return launch_formats<KF, kFormatF16>(a, grouped, vec, stream);
    return launch_formats<KF, kFormatF32>(a, grouped, vec, stream);
}

}  // namespace

// Whole 16-byte pieces of K, V, Q and output rows (V and K rows of 8 elements
// are 16 or 32 bytes) and a head dimension that 32 lanes hold.  Rows of one or
// two pieces leave most of their eight lanes idle, and over few tokens a token
// per thread is faster (2/1 heads of 8: 256 tokens 4.9 us against 8.6, 2,000
// tokens 8.7 and 9.7, 4,096 tokens 10.8 and 10.6; 16/1 heads of 16: 256 tokens
// 6.2 and 8.5, 600 tokens 9.2 and 8.9).
bool frames_grouped(const FramesLaunch &l) {
    if (l.head_dim <= 16 && l.tokens * l.head_dim * l.head_dim <= 131072) return false;
    const uintptr_t p = reinterpret_cast<uintptr_t>(l.k) | reinterpret_cast<uintptr_t>(l.v) |
                        reinterpret_cast<uintptr_t>(l.q) | reinterpret_cast<uintptr_t>(l.out);
    return l.head_dim % 8 == 0 && l.head_dim <= 256 && (p & 15) == 0 && (int64_t)l.kv_heads * l.q_heads <= 65535;
}

int frames_counters(const FramesLaunch &l) {
    const int group = l.q_heads / l.kv_heads, gt = group_heads(group);
    return l.kv_heads * ((group + gt - 1) / gt);
}

int frames_split_tokens(const FramesLaunch &l) {
    if (frames_grouped(l)) {
        // One workgroup per CU, at least one iteration each and at most 64
        // splits for the last workgroup to merge: every split is one more
        // count of the same counter and one more partial in the merge (4,096
        // tokens of 32/8 heads, 16 / 32 / 64 splits: 13.9 / 12.9 / 18.9 us).
        const int rows = kGroupWaves * group_steps(group_heads(l.q_heads / l.kv_heads)) * (64 / (l.head_dim <= 64 ? 8 : l.head_dim <= 128 ? 16 : 32));
        const int64_t most = std::max(1, std::min(64, 256 / frames_counters(l)));
        const int64_t per = (l.tokens + most - 1) / most;
        return (int)((std::max<int64_t>(per, rows) + rows - 1) / rows * rows);
    }
    // About 2,048 workgroups over the whole launch, at least one 256-token
    // tile per split.
    int64_t splits = (2048 + l.q_heads - 1) / l.q_heads;
    const int64_t tiles = (l.tokens + kThreads - 1) / kThreads;
    splits = std::max<int64_t>(1, std::min(splits, tiles));
    const int64_t per = (l.tokens + splits - 1) / splits;
    return (int)((per + kThreads - 1) / kThreads * kThreads);
}

hipError_t launch_frames_decode(const FramesLaunch &l, hipStream_t stream) {
    if (l.tokens == 0) {
        const int n = l.q_heads * l.head_dim;
        hipLaunchKernelGGL(frames_zero_kernel, dim3((unsigned)((n + kThreads - 1) / kThreads)), dim3(kThreads),
                           0, stream, l.out, n);
        return hipGetLastError();
    }
    FramesArgs a{};
    a.q = l.q; a.k = l.k; a.v = l.v; a.out = l.out;
    a.partial_ml = l.partial_ml; a.partial_acc = l.partial_acc;
    a.counters = l.counters;
    a.tokens = l.tokens;
    a.q_heads = l.q_heads; a.kv_heads = l.kv_heads; a.head_dim = l.head_dim;
    a.split_tokens = l.split_tokens;
    a.splits = (int)((l.tokens + l.split_tokens - 1) / l.split_tokens);
    a.scale = l.scale;
    const bool grouped = frames_grouped(l);
    // 16-byte row pieces when every row start is 16-byte aligned.
    const int kb = l.key_format == kFormatF32 ? 4 : 2;
    const bool vec = ((int64_t)l.head_dim * kb) % 16 == 0 && (reinterpret_cast<uintptr_t>(l.k) & 15) == 0;
    hipError_t e;
    if (l.key_format == kFormatBf16) e = launch_value_format<kFormatBf16>(a, l.value_format, grouped, vec, stream);
    else if (l.key_format == kFormatF16) e = launch_value_format<kFormatF16>(a, l.value_format, grouped, vec, stream);
    else e = launch_value_format<kFormatF32>(a, l.value_format, grouped, vec, stream);
    if (e != hipSuccess || a.splits == 1 || grouped) return e;
    hipLaunchKernelGGL(frames_merge_kernel, dim3((unsigned)a.q_heads), dim3(kThreads), 0, stream, a);
    return hipGetLastError();
}

}  // namespace mslim
