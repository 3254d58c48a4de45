// BF16 projections of prompt chunks on MFMA (more than 16 token rows):
//   out[t][r] = BF16(sum_k x[t][k] * w[r][k]),  fp32 accumulation, rounded once.
// The prefill products of the reference (llm_prefill_gemv_reuse8/16/32,
// llm_prefill_fused_qkv_reuse8 and llm_prefill_fused_swiglu_reuse8,
// gpu_llm.cl:553-683, :1253-1383, driven from gpu_llm/prefill.rs:132-290;
// tv_hip_matrix_multiply, hipblaslt_bridge.cpp:203-233, under its HIP
// backend) as one hand-written gfx950 kernel:
//   * a workgroup owns a tile of 64 or 128 weight rows x 64 to 256 token rows of
//     the output, its wavefronts 32 x 32 to 64 x 64 of it, as blocks of
//     v_mfma_f32_32x32x16_bf16 with the weights as A (rows = M) and the token
//     rows as B (N), so a lane ends up with 4 consecutive output rows of one
//     token per 4 accumulators;
//   * both operands are K-contiguous; 64-element k-steps of both move HBM ->
//     LDS with global_load_lds_dwordx4 into a ring of three or four stages
//     (128-byte rows, 16-byte slots XOR-swizzled by (row / 2) % 8, so every 16
//     rows of a fragment read fall in distinct banks), one barrier per k-step;
//   * fragment reads and copies are pinned between the MFMAs, and the last
//     sub-step's MFMAs of a k-step run after the next barrier, behind the next
//     stage's first fragment reads;
//   * the k range of a matrix is cut into segments, as many as its size alone
//     says, each summed from zero and the sums added in order.  A launch whose
//     tiles would leave CUs idle gives every segment a workgroup of its own
//     that writes its fp32 sum, and a second launch adds them; any other
//     launch adds them in registers, to the same bits;
//   * tiles are dealt to XCDs in contiguous slices with the token tiles of a
//     weight slice adjacent, so each weight row is read from HBM by one XCD;
//   * epilogues: plain, residual add (out = BF16(resid + BF16(acc)), llm_add
//     after the product), SwiGLU of a gate and an up product computed in the
//     same tile (llm_swiglu after both), and up to three matrices with their
//     own outputs in one launch (Q, K, V), each equal bit for bit to the
//     plain product followed by the elementwise kernel.
// Every segment is summed by one wavefront in fixed k order, so a token row's
// results do not depend on the tiling, on the rows that share its launch (17 to
// 512 of them) or on timing, and a fused launch equals the separate ones.
// What bounds it: up to about 100 token rows the weights' HBM stream, above
// them the latency of first reads (about 1.5 us against a ring of 64 to 96
// KiB; the pure MFMA loop takes two thirds of the time at 512 tokens).
// Against 128 x 128 / 128 x 64 tiles of four wavefronts split by inner alone
// (us, 4,096 hidden, 14,336 intermediate; O, Q-K-V, gate and up, down):
//   20 tokens   30 / 30 / 56 / 58   ->  12 / 16 / 43 / 26
//   128 tokens  33 / 32 / 60 / 76   ->  17 / 22 / 52 / 38
//   300 tokens  33 / 32 / 123 / 65  ->  25 / 33 / 109 / 58
//   512 tokens  34 / 39 / 131 / 80  ->  30 / 39 / 116 / 68
// Shapes outside the fast path (inner not a multiple of 64, unaligned
// pointers) run proj_generic_kernel: one wavefront per output, lane-strided
// partial sums and a fixed reduction tree.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>

namespace mslim {

namespace {

constexpr int kKAlign = 64;   // inner must be a multiple of this for the tiled kernel
constexpr int kXcds = 8;
constexpr int kMaxSeg = 3;

enum Epi { kPlain = 0, kAdd = 1, kSwiglu = 2 };

struct ProjArgs {
    const uint16_t *w[kMaxSeg];
    uint16_t *out[kMaxSeg];
    int rows[kMaxSeg];
    int segments;
    const uint16_t *w_up;   // SwiGLU: up weights beside w[0] (gate)
    const uint16_t *act_table;  // SwiGLU: swiglu_act_bf16 of every gate value
    const uint16_t *resid;  // add: [tokens][rows[0]], may equal out[0]
    const uint16_t *x;      // [tokens][inner]
    int inner, tokens;
    int n_tiles;            // token tiles
    // Work items (row tile, token tile, k split) before matrix s;
    // [segments] = all.
    int first_item[kMaxSeg + 1];
    // Matrix s is summed in ksegs[s] segments of its k-steps [i nk / ksegs,
    // (i + 1) nk / ksegs).  ksplit[s] is 1 (an item adds them all up) or
    // ksegs[s] (item (tile, i) writes segment i to partial + part_base[s], fp32
    // [ksegs][product][tokens][rows], product the gate (0) or up (1) sum of
    // SwiGLU; a second launch adds the partials in order and applies the
    // epilogue).
    int ksegs[kMaxSeg];
    int ksplit[kMaxSeg];
    int64_t part_base[kMaxSeg];
    float *partial;
};

// Swizzle of a row of NSL 16-byte slots: the slot XOR this.  The 64 banks of
// 4 bytes hold 16 slots, 16 / NSL rows; one LDS cycle of a fragment read
// serves 16 rows at one slot, and they fall in distinct banks when the rows
// that share a place modulo 16 / NSL take distinct slots.
template <int NSL>
__device__ __forceinline__ int proj_swz(int row) {
    return (row / (16 / NSL)) & (NSL - 1);
}

// A configuration: BM weight rows x BN token rows per workgroup, MI x NJ
// 32 x 32 MFMA blocks per wavefront, k-steps of BK inputs in a ring of ST LDS
// stages.
template <int BM_, int BN_, int MI_, int NJ_, int BK_, int ST_, int WAVES_ = 4>
struct Config {
    static constexpr int BM = BM_, BN = BN_, MI = MI_, NJ = NJ_, BK = BK_, ST = ST_, WAVES = WAVES_;
};

// LDS of a configuration: ST stages of the weight tile(s) and the token tile;
// the SwiGLU epilogue of the tiles with many outputs reuses it for the 128 KiB
// activation table (the others read the table from L2).
constexpr int kTableBytes = kSwigluTableEntries * 2;
template <class C>
constexpr bool table_in_lds(int epi) {
    return epi == kSwiglu && C::BM * C::BN >= 128 * 64;
}
template <class C>
constexpr int proj_lds_bytes(int epi) {
    const int stages = C::ST * ((epi == kSwiglu ? 2 : 1) * C::BM + C::BN) * C::BK * 2;
    return table_in_lds<C>(epi) && stages < kTableBytes ? kTableBytes : stages;
}

// SUM: some item adds up several segments.  The totals and the test per k-step
// would cost the launches without one 2% (gate and up of a 4,096 / 14,336 layer
// at 17 to 64 tokens: 50.1 us, with them 51.2).
template <class C, int EPI, bool SUM>
__global__ __launch_bounds__(C::WAVES * 64) __attribute__((amdgpu_waves_per_eu(C::WAVES / 4))) void proj_kernel(ProjArgs a) {
    constexpr int kStages = C::ST;
    constexpr int kBM = C::BM;
    constexpr int kBK = C::BK;
    constexpr int ROWB = kBK * 2;     // bytes of one row of a stage
    constexpr int NSL = kBK / 8;      // 16-byte slots per row
    constexpr int RPC = 1024 / ROWB;  // rows per 1 KiB copy chunk
    constexpr int SUB = kBK / 16;     // MFMA k-steps per stage
    constexpr int WAVES = C::WAVES;
    constexpr int MI = C::MI, NJ = C::NJ;
    constexpr int WM = 32 * MI, WT = 32 * NJ;  // rows and tokens of a wavefront
    constexpr int WR = kBM / WM;      // wavefronts along the rows
    constexpr int BN = C::BN;
    static_assert(WR * (BN / WT) == WAVES && kBM % WM == 0 && BN % WT == 0, "wavefronts tile the workgroup");
    constexpr int NA = EPI == kSwiglu ? 2 : 1;
    constexpr int A_BYTES = kBM * kBK * 2;  // one weight stage
    constexpr int B_BYTES = BN * kBK * 2;
    constexpr int A_CH = kBM / RPC / WAVES;   // 1 KiB copy chunks per wavefront
    constexpr int B_CH = BN / RPC / WAVES;
    constexpr int PER_STAGE = NA * A_CH + B_CH;  // copies per wavefront per k-step
    static_assert(A_CH >= 1 && B_CH >= 1 && PER_STAGE * (kStages - 2) <= 63, "copy plan");
    __shared__ __align__(16) unsigned char lds[proj_lds_bytes<C>(EPI)];
    unsigned char *const a_lds = lds;                                  // [kStages][A_BYTES]
    unsigned char *const u_lds = lds + kStages * A_BYTES;              // SwiGLU up: [kStages][A_BYTES]
    unsigned char *const b_lds = lds + kStages * NA * A_BYTES;         // [kStages][B_BYTES]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave % WR, wc = wave / WR;
    const int h = lane >> 5;

    // XCD-aware tile: workgroup L runs on XCD L % 8; each XCD takes a
    // contiguous slice of the items, ordered (row tile, token tile, k split).
    const int items = a.first_item[a.segments];
    const int per_xcd = (items + kXcds - 1) / kXcds;
    const int w_index = (int)(blockIdx.x % kXcds) * per_xcd + (int)(blockIdx.x / kXcds);
    if (w_index >= items) return;
    // The segment's matrix, by uniform selects (a dynamic index into the
    // kernel arguments would not stay scalar).
    const bool s1 = a.segments > 1 && w_index >= a.first_item[1], s2 = a.segments > 2 && w_index >= a.first_item[2];
    const int ksplit = s2 ? a.ksplit[2] : s1 ? a.ksplit[1] : a.ksplit[0];
    const int in_seg = w_index - (s2 ? a.first_item[2] : s1 ? a.first_item[1] : 0);
    const int t_index = in_seg / ksplit, split = in_seg % ksplit;
    const int mt = t_index / a.n_tiles, nt = t_index % a.n_tiles;
    const int rows = s2 ? a.rows[2] : s1 ? a.rows[1] : a.rows[0];
    const int m0 = mt * kBM;
    const uint16_t *const wseg = s2 ? a.w[2] : s1 ? a.w[1] : a.w[0];
    uint16_t *const out = s2 ? a.out[2] : s1 ? a.out[1] : a.out[0];
    const int n0 = nt * BN;
    const int inner = a.inner;
    const int nk_all = inner / kBK;
    const int kb = (int)((int64_t)split * nk_all / ksplit);
    const int nk = (int)((int64_t)(split + 1) * nk_all / ksplit) - kb;
    const int ksegs = !SUM || ksplit > 1 ? 1 : s2 ? a.ksegs[2] : s1 ? a.ksegs[1] : a.ksegs[0];  // of this item

    // Copy offsets: chunk c of a stage is RPC rows; lane l lands in row
    // RPC c + l / NSL, physical slot l % NSL, and fetches the logical slot
    // (l % NSL) ^ proj_swz(row) of that row.  Rows past the matrix re-read
    // its last row (their outputs are not written).
    const uint32_t row_bytes = (uint32_t)inner * 2;
    uint32_t aoff[A_CH], boff[B_CH];
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
        const int r = RPC * (wave + WAVES * i) + lane / NSL;
        aoff[i] = (uint32_t)(min(m0 + r, rows - 1) - m0) * row_bytes +
                  (uint32_t)(((lane % NSL) ^ proj_swz<NSL>(r)) * 16);
    }
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
        const int r = RPC * (wave + WAVES * i) + lane / NSL;
        boff[i] = (uint32_t)(min(n0 + r, a.tokens - 1) - n0) * row_bytes +
                  (uint32_t)(((lane % NSL) ^ proj_swz<NSL>(r)) * 16);
    }
    const int64_t k_first = (int64_t)kb * kBK;
    const char *const wbase = uniform_ptr(reinterpret_cast<const char *>(wseg + (int64_t)m0 * inner + k_first));
    const char *const ubase =
        EPI == kSwiglu ? uniform_ptr(reinterpret_cast<const char *>(a.w_up + (int64_t)m0 * inner + k_first))
                       : nullptr;
    const char *const xbase = uniform_ptr(reinterpret_cast<const char *>(a.x + (int64_t)n0 * inner + k_first));
    uint32_t a_dst[kStages], u_dst[kStages], b_dst[kStages];
#pragma unroll
    for (int st = 0; st < kStages; ++st) {
        a_dst[st] = lds_offset(a_lds + st * A_BYTES + wave * 1024);
        u_dst[st] = EPI == kSwiglu ? lds_offset(u_lds + st * A_BYTES + wave * 1024) : 0;
        b_dst[st] = lds_offset(b_lds + st * B_BYTES + wave * 1024);
    }
    // Copy c of a k-step into stage st, from byte offset k of its rows.
    auto copy_one = [&](int st, int64_t k, int c) __attribute__((always_inline)) {
        if (c < NA * A_CH) {
            const int i = c / NA;
            if (c % NA == 0) dma16_async(wbase + k, aoff[i], a_dst[st] + i * WAVES * 1024);
            else dma16_async(ubase + k, aoff[i], u_dst[st] + i * WAVES * 1024);
        } else {
            const int i = c - NA * A_CH;
            dma16_async(xbase + k, boff[i], b_dst[st] + i * WAVES * 1024);
        }
    };

    // Fragment addresses in stage 0: row WM wr + l % 32 (weights) or WT wc +
    // l % 32 (tokens), logical slot 2 s + l / 32 of sub-step s, physical slot
    // that ^ proj_swz(row) = (2 s + h) ^ proj_swz(l % 32).  A 32-row block and
    // a stage are immediate offsets (the swizzle depends on row % 32 only).
    uint32_t fa[SUB], fu[SUB], fb[SUB];
    {
        const uint32_t abase = lds_offset(a_lds), ubase_l = lds_offset(u_lds), bbase = lds_offset(b_lds);
#pragma unroll
        for (int s = 0; s < SUB; ++s) {
            const uint32_t sw = (uint32_t)(((2 * s + h) ^ proj_swz<NSL>(lane & 31)) * 16);
            fa[s] = abase + (uint32_t)(WM * wr + (lane & 31)) * ROWB + sw;
            fu[s] = ubase_l + (uint32_t)(WM * wr + (lane & 31)) * ROWB + sw;
            fb[s] = bbase + (uint32_t)(WT * wc + (lane & 31)) * ROWB + sw;
        }
    }

    floatx16_t acc[MI][NJ], accu[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] = 0.0f;
                if (EPI == kSwiglu) accu[i][j][r] = 0.0f;
            }

    // Sums of the segments that are complete.  -0 leaves the first one as it
    // is, whatever its sign of zero.
    floatx16_t total[MI][NJ], totalu[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                total[i][j][r] = -0.0f;
                if (EPI == kSwiglu) totalu[i][j][r] = -0.0f;
            }
    auto end_segment = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    total[i][j][r] = __fadd_rn(total[i][j][r], acc[i][j][r]);
                    acc[i][j][r] = 0.0f;
                    if (EPI == kSwiglu) {
                        totalu[i][j][r] = __fadd_rn(totalu[i][j][r], accu[i][j][r]);
                        accu[i][j][r] = 0.0f;
                    }
                }
    };
    int seg = 1, seg_end = nk / ksegs;  // the first k-step after the current segment

    // Fragments of one sub-step: NJ of the tokens, MI of each weight matrix.
    struct Frag {
        bf16x8_t a[NA * MI], b[NJ];
    };
    constexpr int READS = NA * MI + NJ;
    constexpr int MFMAS = NA * MI * NJ;
    auto read_one = [&](Frag &f, int st, int s, int r) __attribute__((always_inline)) {
        // the first MFMA needs a[0] and b[0]
        if (r == 0) f.b[0] = lds_read_b128(fb[s] + st * B_BYTES);
        else if (r <= NA * MI) {
            const int i = (r - 1) / NA;
            if ((r - 1) % NA == 0) f.a[NA * i] = lds_read_b128(fa[s] + st * A_BYTES + i * 32 * ROWB);
            else f.a[NA * i + 1] = lds_read_b128(fu[s] + st * A_BYTES + i * 32 * ROWB);
        } else {
            const int j = r - NA * MI;
            f.b[j] = lds_read_b128(fb[s] + st * B_BYTES + j * 32 * ROWB);
        }
    };
    auto mfma_one = [&](const Frag &f, int m) __attribute__((always_inline)) {
        const int j = m / (NA * MI), i = m % (NA * MI) / NA;
        if (m % NA == 0) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[NA * i], f.b[j], acc[i][j], 0, 0, 0);
        else accu[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[NA * i + 1], f.b[j], accu[i][j], 0, 0, 0);
    };
    // One phase: the MFMAs of `cur`, with the fragment reads of sub-step s of
    // stage st into `nxt` spread over the first half of them and part `part`
    // of SUB of the k-step's copies into stage sd over all of them.  The order is pinned: left to
    // itself the compiler sinks the reads below the MFMAs, and with one
    // wavefront per SIMD every phase then waits out their latency.
    auto phase = [&](const Frag &cur, Frag &nxt, int st, int s, auto mfma_tag, auto read_tag, int part, int sd,
                     int64_t k) __attribute__((always_inline)) {
        constexpr bool do_mfma = decltype(mfma_tag)::value, do_read = decltype(read_tag)::value;
        constexpr int HALF = MFMAS >= 2 ? MFMAS / 2 : 1;
#pragma unroll
        for (int m = 0; m < MFMAS; ++m) {
            if constexpr (do_read) {
#pragma unroll
                for (int r = 0; r < READS; ++r)
                    if (r * HALF / READS == m) read_one(nxt, st, s, r);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (do_mfma) mfma_one(cur, m);
#pragma unroll
            for (int c = 0; c < PER_STAGE; ++c)
                if (c * (SUB * MFMAS) / PER_STAGE == part * MFMAS + m) copy_one(sd, k, c);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // K loop.  Iteration kt: this wavefront's copy of k-step kt has landed
    // (later ones may be in flight), the barrier publishes it and frees the
    // stage of kt-1, which receives k-step kt + kStages - 1 (the last k-step
    // is repeated past the end so the wait counts stay exact).  The fragments
    // of kt-1's last sub-step were read before the barrier; their MFMAs run
    // while the first fragments of kt are in flight.  Sub-step s uses
    // fragment set s % 2.
    using Yes = std::true_type;
    using No = std::false_type;
    static_assert(SUB % 2 == 0, "sub-steps alternate two fragment sets");
    Frag f0, f1;
    auto k_bytes = [&](int kt) __attribute__((always_inline)) { return (int64_t)min(kt, nk - 1) * ROWB; };
#pragma unroll
    for (int st = 0; st < kStages - 1; ++st)
#pragma unroll
        for (int c = 0; c < PER_STAGE; ++c) copy_one(st, k_bytes(st), c);
    auto iteration = [&](int kt, int st, int sd, auto mfma_tag) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(vmcnt_lds_imm((kStages - 2) * PER_STAGE));
        raw_barrier();
        const int64_t k = k_bytes(kt + kStages - 1);
        phase(f1, f0, st, 0, mfma_tag, Yes{}, 0, sd, k);
        if (SUM && kt == seg_end) {
            end_segment();
            ++seg;
            seg_end = (int)((int64_t)seg * nk / ksegs);
        }
#pragma unroll
        for (int s = 0; s + 1 < SUB; ++s) {
            if (s % 2 == 0) phase(f0, f1, st, s + 1, Yes{}, Yes{}, s + 1, sd, k);
            else phase(f1, f0, st, s + 1, Yes{}, Yes{}, s + 1, sd, k);
        }
    };
    // Stage of k-step kt is kt % kStages; the loop is unrolled by kStages so
    // every stage index is a constant.
    iteration(0, 0, kStages - 1, No{});
    for (int kt = 1; kt < nk; kt += kStages) {
#pragma unroll
        for (int u = 0; u < kStages; ++u) {
            if (kt + u >= nk) break;
            iteration(kt + u, (1 + u) % kStages, u % kStages, Yes{});
        }
    }
    phase(f1, f0, 0, 0, Yes{}, No{}, SUB, 0, 0);
    if (SUM) end_segment();
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // no copy may still target LDS at exit

    // SwiGLU: the activation table replaces the stages in LDS (one 128 KiB
    // copy per workgroup, from L2), after every wavefront's last fragment
    // read.
    const uint16_t *table = a.act_table;
    if (table_in_lds<C>(EPI) && ksplit == 1) {
        __syncthreads();
        const char *tb = uniform_ptr(reinterpret_cast<const char *>(a.act_table));
        const uint32_t dst = lds_offset(lds + wave * 1024);
#pragma unroll
        for (int i = 0; i < kTableBytes / 1024 / WAVES; ++i)
            dma16_async(tb + (int64_t)(wave + WAVES * i) * 1024, (uint32_t)lane * 16, dst + i * WAVES * 1024);
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        __syncthreads();
        table = reinterpret_cast<const uint16_t *>(lds);
    }

    auto &sum = SUM ? total : acc;
    auto &su = SUM ? totalu : accu;
    // Epilogue: lane l holds token WT wc + 32 j + l % 32 and, per group g of
    // four accumulators, rows WM wr + 32 i + 8 g + 4 h .. +3.
    if (ksplit > 1) {
        const int64_t outs = (int64_t)a.tokens * rows;
        float *const part = a.partial + (s2 ? a.part_base[2] : s1 ? a.part_base[1] : a.part_base[0]) + split * NA * outs;
        float *const part_up = part + outs;
        const bool vecf = (rows & 3) == 0;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int t = n0 + WT * wc + 32 * j + (lane & 31);
            if (t >= a.tokens) continue;
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int r = m0 + WM * wr + 32 * i + 8 * g + 4 * h;
                    if (r >= rows) continue;
                    const int64_t o = (int64_t)t * rows + r;
                    if (vecf && r + 3 < rows) {
                        const floatx4_t v = {sum[i][j][4 * g], sum[i][j][4 * g + 1], sum[i][j][4 * g + 2],
                                             sum[i][j][4 * g + 3]};
                        *reinterpret_cast<floatx4_t *>(part + o) = v;
                        if (EPI == kSwiglu) {
                            const floatx4_t u = {su[i][j][4 * g], su[i][j][4 * g + 1], su[i][j][4 * g + 2],
                                                 su[i][j][4 * g + 3]};
                            *reinterpret_cast<floatx4_t *>(part_up + o) = u;
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            if (r + e >= rows) break;
                            part[o + e] = sum[i][j][4 * g + e];
                            if (EPI == kSwiglu) part_up[o + e] = su[i][j][4 * g + e];
                        }
                    }
                }
        }
        return;
    }
    const bool vec = (rows & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 7) == 0 &&
                     (EPI != kAdd || (reinterpret_cast<uintptr_t>(a.resid) & 7) == 0);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int t = n0 + WT * wc + 32 * j + (lane & 31);
        if (t >= a.tokens) continue;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int r = m0 + WM * wr + 32 * i + 8 * g + 4 * h;
                if (r >= rows) continue;
                uint16_t y[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint16_t p = write_bf16(sum[i][j][4 * g + e]);
                    if (EPI == kSwiglu) y[e] = swiglu_mul_bf16(table[p], write_bf16(su[i][j][4 * g + e]));
                    else y[e] = p;
                }
                const int64_t o = (int64_t)t * rows + r;
                if (vec && r + 3 < rows) {
                    if (EPI == kAdd) {
                        const uint2 rv = *reinterpret_cast<const uint2 *>(a.resid + o);
                        const uint16_t rs[4] = {(uint16_t)rv.x, (uint16_t)(rv.x >> 16), (uint16_t)rv.y,
                                                (uint16_t)(rv.y >> 16)};
#pragma unroll
                        for (int e = 0; e < 4; ++e) y[e] = write_bf16(__fadd_rn(read_bf16(rs[e]), read_bf16(y[e])));
                    }
                    uint2 w;
                    w.x = (uint32_t)y[0] | ((uint32_t)y[1] << 16);
                    w.y = (uint32_t)y[2] | ((uint32_t)y[3] << 16);
                    *reinterpret_cast<uint2 *>(out + o) = w;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (r + e >= rows) break;
                        uint16_t v = y[e];
                        if (EPI == kAdd) v = write_bf16(__fadd_rn(read_bf16(a.resid[o + e]), read_bf16(v)));
                        out[o + e] = v;
                    }
                }
            }
    }
}

// Split matrices (grid y): out = epilogue(BF16(partial[0] + partial[1] +
// ...)), the partials added in split order, four outputs per thread.
template <int EPI>
__global__ __launch_bounds__(256) void proj_merge_kernel(ProjArgs a) {
    constexpr int NA = EPI == kSwiglu ? 2 : 1;
    const int seg = blockIdx.y;
    const int ksplit = a.ksplit[seg];
    const int64_t n = (int64_t)a.tokens * a.rows[seg];
    const int64_t i0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (ksplit == 1 || i0 >= n) return;
    const float *const part = a.partial + a.part_base[seg];
    uint16_t *const out = a.out[seg];
    // Four outputs with 16-byte partials and 8-byte outputs (and residual):
    // one vector access each; otherwise element by element.  The arithmetic
    // per element is the same either way.
    const bool vec = (n & 3) == 0 && (reinterpret_cast<uintptr_t>(part) & 15) == 0 &&
                     ((reinterpret_cast<uintptr_t>(out) | (EPI == kAdd ? reinterpret_cast<uintptr_t>(a.resid) : 0)) & 7) == 0;
    if (vec) {
        float4 v = *reinterpret_cast<const float4 *>(part + i0);
        float4 vu = EPI == kSwiglu ? *reinterpret_cast<const float4 *>(part + n + i0) : float4{};
#pragma unroll 4
        for (int s = 1; s < ksplit; ++s) {
            const float4 w = *reinterpret_cast<const float4 *>(part + (int64_t)s * NA * n + i0);
            v = float4{__fadd_rn(v.x, w.x), __fadd_rn(v.y, w.y), __fadd_rn(v.z, w.z), __fadd_rn(v.w, w.w)};
            if (EPI == kSwiglu) {
                const float4 wu = *reinterpret_cast<const float4 *>(part + ((int64_t)s * NA + 1) * n + i0);
                vu = float4{__fadd_rn(vu.x, wu.x), __fadd_rn(vu.y, wu.y), __fadd_rn(vu.z, wu.z), __fadd_rn(vu.w, wu.w)};
            }
        }
        const float vs[4] = {v.x, v.y, v.z, v.w}, us[4] = {vu.x, vu.y, vu.z, vu.w};
        uint16_t rs[4] = {0, 0, 0, 0};
        if (EPI == kAdd) {
            const uint2 r = *reinterpret_cast<const uint2 *>(a.resid + i0);
            rs[0] = (uint16_t)r.x; rs[1] = (uint16_t)(r.x >> 16); rs[2] = (uint16_t)r.y; rs[3] = (uint16_t)(r.y >> 16);
        }
        uint16_t ys[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint16_t y = write_bf16(vs[e]);
            if (EPI == kSwiglu) y = swiglu_mul_bf16(a.act_table[y], write_bf16(us[e]));
            if (EPI == kAdd) y = write_bf16(__fadd_rn(read_bf16(rs[e]), read_bf16(y)));
            ys[e] = y;
        }
        *reinterpret_cast<uint2 *>(out + i0) =
            uint2{(uint32_t)ys[0] | ((uint32_t)ys[1] << 16), (uint32_t)ys[2] | ((uint32_t)ys[3] << 16)};
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int64_t i = i0 + e;
        if (i >= n) break;
        float v = part[i], vu = EPI == kSwiglu ? part[n + i] : 0.0f;
        for (int s = 1; s < ksplit; ++s) {
            v = __fadd_rn(v, part[(int64_t)s * NA * n + i]);
            if (EPI == kSwiglu) vu = __fadd_rn(vu, part[((int64_t)s * NA + 1) * n + i]);
        }
        uint16_t y = write_bf16(v);
        if (EPI == kSwiglu) y = swiglu_mul_bf16(a.act_table[y], write_bf16(vu));
        if (EPI == kAdd) y = write_bf16(__fadd_rn(read_bf16(a.resid[i]), read_bf16(y)));
        out[i] = y;
    }
}

// Any shape: one wavefront per output element.  Lane l sums k = l, l + 64,
// ... in order, then the 64 partial sums meet in a fixed butterfly, so the
// fp32 error stays near (K / 64 + 6) roundings of the magnitudes.
template <int EPI>
__global__ __launch_bounds__(256) void proj_generic_kernel(ProjArgs a) {
    const int lane = threadIdx.x & 63;
    const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    int64_t total = 0;
    for (int s = 0; s < a.segments; ++s) total += (int64_t)a.rows[s] * a.tokens;
    if (item >= total) return;
    int seg = 0;
    int64_t rest = item;
    while (rest >= (int64_t)a.rows[seg] * a.tokens) {
        rest -= (int64_t)a.rows[seg] * a.tokens;
        ++seg;
    }
    const int rows = a.rows[seg];
    const int t = (int)(rest / rows), r = (int)(rest % rows);
    const uint16_t *w = a.w[seg] + (int64_t)r * a.inner;
    const uint16_t *u = EPI == kSwiglu ? a.w_up + (int64_t)r * a.inner : nullptr;
    const uint16_t *x = a.x + (int64_t)t * a.inner;
    float s = 0.0f, su = 0.0f;
    for (int k = lane; k < a.inner; k += 64) {
        const float xv = read_bf16(x[k]);
        s = __fmaf_rn(read_bf16(w[k]), xv, s);
        if (EPI == kSwiglu) su = __fmaf_rn(read_bf16(u[k]), xv, su);
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
        s = __fadd_rn(s, __shfl_xor(s, m, 64));
        if (EPI == kSwiglu) su = __fadd_rn(su, __shfl_xor(su, m, 64));
    }
    if (lane != 0) return;
    const int64_t o = (int64_t)t * rows + r;
    uint16_t y = write_bf16(s);
    if (EPI == kSwiglu) y = swiglu_bf16(y, write_bf16(su));
    if (EPI == kAdd) y = write_bf16(__fadd_rn(read_bf16(a.resid[o]), read_bf16(y)));
    a.out[seg][o] = y;
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// The configurations, smallest tile first; a SwiGLU tile holds half the output
// rows (gate and up rows side by side).  Wavefront tiles of 32 x 32 to 64 x 64,
// two wavefronts per SIMD except in the smallest, which fits twice on a CU.
enum { kTile64x64, kTile64x128, kTile128x128, kTile128x256, kTiles };
template <int TILE, int EPI>
struct TileConfig;
template <int EPI>
struct TileConfig<kTile64x64, EPI> : Config<64, 64, 1, 1, 64, 4, 4> {};
template <int EPI>
struct TileConfig<kTile64x128, EPI> : Config<64, 128, 1, 1, 64, EPI == kSwiglu ? 3 : 4, 8> {};
template <int EPI>
struct TileConfig<kTile128x128, EPI> : Config<128, 128, 1, 2, 64, EPI == kSwiglu ? 3 : 4, 8> {};
template <int EPI>
struct TileConfig<kTile128x256, EPI>
    : Config<EPI == kSwiglu ? 64 : 128, 256, EPI == kSwiglu ? 1 : 2, 2, 64, 3, 8> {};

// What the choices below know of a configuration: its tile, and the measured
// time of a k-step of 64 inputs with one workgroup per CU and the weights in
// HBM (us; two resident 64 x 64 workgroups take twice that).
struct TileCost {
    int bm, bn;
    double step;
};
constexpr TileCost kPlainCost[kTiles] = {{64, 64, 0.27}, {64, 128, 0.36}, {128, 128, 0.50}, {128, 256, 0.71}};
constexpr TileCost kSwigluCost[kTiles] = {{64, 64, 0.62}, {64, 128, 0.55}, {128, 128, 1.00}, {64, 256, 0.80}};
constexpr int kCus = 256;
constexpr double kStreamBytesPerUs = 4.8e6;   // weights from HBM
constexpr double kMergeUs = 3.5;              // the merge launch, beside its traffic
constexpr double kMergeBytesPerUs = 6.0e6;
constexpr int kMinSplitSteps = 8;             // k-steps of a split, at least
constexpr int64_t kSplitBytes = 16ll << 20;   // partials of a launch, at most (inner < 8192; SwiGLU twice that)
constexpr double kGain = 0.5;                 // a larger tile or a split must save this (us)

int64_t tiles_of(const TileCost &c, int rows, int tokens) {
    return (int64_t)((rows + c.bm - 1) / c.bm) * ((tokens + c.bn - 1) / c.bn);
}

// Partials of a split matrix, in whole 16-byte pieces.
size_t split_floats(int ksplit, int products, int rows, int tokens) {
    return ((size_t)ksplit * products * rows * tokens + 3) & ~(size_t)3;
}

// Segments that a [rows][inner] matrix is summed in: as many as give every CU
// about one 64 x 64 tile's segment, a power of two, eight k-steps at least.
// From the matrix alone: a token row gets the same bits in every launch of more
// than 16 rows, and K and V beside their Q those of a launch of their own.
//   * 320 tiles' segments at most, since more queue behind one another (8,192
//     rows and inputs at 64 tokens: 33 us with two, 45 with four); 640 from
//     16,384 inputs, whose segments are long enough (28,672 inputs to 8,192
//     rows: 64 tokens 107 us with two, 98 with four, 150 tokens 165 and 123).
//   * One where there are more than twice as many rows as inputs (gate, up, the
//     LM head): the sums are too short for a merge, and adding segments in
//     registers is not free either (2,048 inputs to 8,192 rows at 300 tokens:
//     31.2 us with one, 32.1 with two).
//   * Eight only from 8,192 inputs and a quarter as many rows, the down
//     projections: K and V of fewer rows share a launch with Q, and their
//     eight splits put more items behind Q's (8,192 + 1,024 + 1,024 rows of
//     8,192 inputs at 128 tokens: 107 us, with four at most 55).
int k_segments(int inner, int rows) {
    const int most = inner >= 8192 && (int64_t)rows * 4 >= inner ? 8 : 4;
    const int64_t tiles = (rows + 63) / 64, limit = inner >= 16384 ? 640 : 320;
    int n = 1;
    if (rows > 2 * inner) return n;
    while (n < most && tiles * n * 2 <= limit && inner / kKAlign / (n * 2) >= kMinSplitSteps) n *= 2;
    return n;
}

}  // namespace

// The choice that finishes first when the launch's items are dealt to the
// resident workgroups and the merge, if any, is added.
ProjPlan plan_proj(const SkinnyMatrix *m, int count, const uint16_t *w_up, const uint16_t *x, int inner, int tokens,
                   bool may_split) {
    ProjPlan best{};
    bool fast = inner % kKAlign == 0 && aligned16(x) && (!w_up || aligned16(w_up));
    for (int s = 0; s < count; ++s) fast = fast && aligned16(m[s].w);
    best.tile = fast ? 0 : -1;
    if (!fast) return best;
    const int steps = inner / kKAlign, products = w_up ? 2 : 1;
    for (int s = 0; s < count; ++s) best.ksegs[s] = k_segments(inner, m[s].rows);
    // Unsplit, all matrices split, and of Q, K, V either Q or the others.
    const int masks[4] = {0, 7, 1, 6};
    double least = -1.0;
    for (int k = 0; k < (may_split ? count == 3 ? 4 : 2 : 1); ++k) {
        ProjPlan p = best;
        p.partial_floats = 0;
        double merge = 0.0;
        for (int s = 0; s < count; ++s) {
            p.ksplit[s] = masks[k] >> s & 1 ? p.ksegs[s] : 1;
            if (p.ksplit[s] == 1) continue;
            const size_t floats = split_floats(p.ksplit[s], products, m[s].rows, tokens);
            p.partial_floats += floats;
            merge += 2.0 * floats * sizeof(float) / kMergeBytesPerUs;
        }
        if (k && !p.partial_floats) continue;
        // the merge's model is fitted up to here; past it 300 tokens of 4,096
        // inputs and rows measured 30.1 us split, 25.1 unsplit
        if (inner < 8192 && (int64_t)(p.partial_floats * sizeof(float)) > kSplitBytes * products) continue;
        if (p.partial_floats) merge += kMergeUs;
        for (p.tile = 0; p.tile < kTiles; ++p.tile) {
            const TileCost &c = w_up ? kSwigluCost[p.tile] : kPlainCost[p.tile];
            int64_t items = 0;
            double work = 0.0, longest = 0.0, bytes = 0.0;  // work and longest in k-steps
            for (int s = 0; s < count; ++s) {
                const int64_t n = tiles_of(c, m[s].rows, tokens) * p.ksplit[s];
                const double each = (double)steps / p.ksplit[s];
                items += n;
                work += n * each;
                longest = std::max(longest, each);
                bytes += (double)m[s].rows * inner * 2 * products;
            }
            // equal items run in whole rounds; unequal ones leave about half
            // of the longest item behind the mean
            const double rounds = (double)((items + kCus - 1) / kCus);
            const bool equal = work == items * longest;
            const double span =
                equal ? rounds * longest : std::max(longest, work / kCus + (rounds > 1 ? longest / 2 : 0.0));
            const double us = std::max(span * c.step, bytes / kStreamBytesPerUs) + merge;
            if (least < 0.0 || us < least - kGain) {
                least = us;
                best = p;
            }
        }
    }
    return best;
}

namespace {

ProjArgs proj_args(const ProjPlan &plan, const SkinnyMatrix *m, int count, const uint16_t *x, int inner, int tokens) {
    ProjArgs a{};
    for (int s = 0; s < count; ++s) {
        a.w[s] = m[s].w;
        a.out[s] = m[s].out;
        a.rows[s] = m[s].rows;
        a.ksegs[s] = plan.ksegs[s];
        a.ksplit[s] = plan.ksplit[s];
    }
    a.segments = count;
    a.x = x;
    a.inner = inner;
    a.tokens = tokens;
    return a;
}

template <class C, int EPI>
hipError_t launch_config(ProjArgs &a, hipStream_t stream) {
    a.n_tiles = (a.tokens + C::BN - 1) / C::BN;
    a.first_item[0] = 0;
    for (int s = 0; s < a.segments; ++s)
        a.first_item[s + 1] = a.first_item[s] + (a.rows[s] + C::BM - 1) / C::BM * a.n_tiles * a.ksplit[s];
    for (int s = a.segments + 1; s <= kMaxSeg; ++s) a.first_item[s] = a.first_item[a.segments];
    const unsigned grid = (unsigned)((a.first_item[a.segments] + kXcds - 1) / kXcds * kXcds);
    bool sum = false;
    for (int s = 0; s < a.segments; ++s) sum |= a.ksplit[s] < a.ksegs[s];
    if (sum) hipLaunchKernelGGL((proj_kernel<C, EPI, true>), dim3(grid), dim3(C::WAVES * 64), 0, stream, a);
    else hipLaunchKernelGGL((proj_kernel<C, EPI, false>), dim3(grid), dim3(C::WAVES * 64), 0, stream, a);
    return hipGetLastError();
}

template <int EPI>
hipError_t launch(const ProjPlan &plan, ProjArgs &a, float *partial, hipStream_t stream) {
    if (plan.tile < 0) {
        int64_t total = 0;
        for (int s = 0; s < a.segments; ++s) total += (int64_t)a.rows[s] * a.tokens;
        hipLaunchKernelGGL((proj_generic_kernel<EPI>), dim3((unsigned)((total + 3) / 4)), dim3(256), 0, stream, a);
        return hipGetLastError();
    }
    if (plan.partial_floats && !partial) return hipErrorInvalidValue;
    a.partial = partial;
    int64_t base = 0, most = 0;
    for (int s = 0; s < a.segments; ++s) {
        a.part_base[s] = base;
        if (a.ksplit[s] == 1) continue;
        base += (int64_t)split_floats(a.ksplit[s], EPI == kSwiglu ? 2 : 1, a.rows[s], a.tokens);
        most = std::max(most, (int64_t)a.rows[s] * a.tokens);
    }
    hipError_t e;
    switch (plan.tile) {
        case kTile64x64: e = launch_config<TileConfig<kTile64x64, EPI>, EPI>(a, stream); break;
        case kTile64x128: e = launch_config<TileConfig<kTile64x128, EPI>, EPI>(a, stream); break;
        case kTile128x128: e = launch_config<TileConfig<kTile128x128, EPI>, EPI>(a, stream); break;
        default: e = launch_config<TileConfig<kTile128x256, EPI>, EPI>(a, stream); break;
    }
    if (e != hipSuccess || !most) return e;
    hipLaunchKernelGGL((proj_merge_kernel<EPI>), dim3((unsigned)((most + 1023) / 1024), (unsigned)a.segments), dim3(256),
                       0, stream, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_proj(const ProjPlan &plan, const SkinnyMatrix *m, int count, const uint16_t *x, int inner,
                       int tokens, float *partial, hipStream_t stream) {
    ProjArgs a = proj_args(plan, m, count, x, inner, tokens);
    return launch<kPlain>(plan, a, partial, stream);
}

hipError_t launch_proj_add(const ProjPlan &plan, const SkinnyMatrix &m, const uint16_t *resid, const uint16_t *x,
                           int inner, int tokens, float *partial, hipStream_t stream) {
    ProjArgs a = proj_args(plan, &m, 1, x, inner, tokens);
    a.resid = resid;
    return launch<kAdd>(plan, a, partial, stream);
}

hipError_t launch_proj_swiglu(const ProjPlan &plan, const SkinnyMatrix &gate, const uint16_t *w_up, const uint16_t *x,
                              int inner, int tokens, const uint16_t *act_table, float *partial, hipStream_t stream) {
    ProjArgs a = proj_args(plan, &gate, 1, x, inner, tokens);
    a.w_up = w_up;
    a.act_table = act_table;
    return launch<kSwiglu>(plan, a, partial, stream);
}

}  // namespace mslim
