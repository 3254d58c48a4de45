// ColdStore record codec for pages already resident in the device pool.
//
// A ColdStore record (cold_store.rs:269-349) is
//   header[104] | K token hashes[8*tokens] | V token hashes[8*tokens] |
//   K payload | V payload | footer[56]
// where the payloads are head-major [heads][tokens][row] byte images.  A
// pool page is exactly such a payload (page_tokens rows per head), so the
// bytes that make a record out of a pool page are the "frame": the header,
// both token-hash tables and the footer.  This file computes frames on the
// device; the host writes frame prefix | payloads | footer to the file (seal)
// or compares a stored record's frame with a recomputed one (verified
// restore).  Every value is byte-identical to the host codec.
//
// A record's tokens are rows first_row .. first_row + tokens - 1 of its pool
// page (a record can start inside a page when a turn ended there).  In staged
// mode the payloads are read instead from compacted staging slots (slot i of
// k_pool / v_pool holds record i as [heads][tokens][row], the layout
// record_payloads writes), so a stored record can be verified before any of
// its bytes reach the pool.
//
// Three launches:
//   * token_hashes_kernel: one lane per (record, K/V, token) computes the
//     FNV-1a-64 of that token's bytes over all heads (cold_store.rs:725-742).
//     These lanes are independent, so this launch streams the payloads at
//     close to HBM rate;
//   * payload_sums_kernel: the FNV-1a-64 checksums of the K and V payloads
//     (cold_store.rs:909-922), one wavefront per payload;
//   * frame_kernel: the hash-table checksums and the header, then the record
//     checksum and SHA-256 (FIPS 180-4) over header | hashes | K | V and the
//     footer, three wavefronts per 64 records.  SHA-256 is a sequential chain
//     over the record's bytes, so this launch is bounded by the longest chain,
//     not by bandwidth; it is meant for sealing or verifying many records at
//     once.
#include "common.hpp"
#include "kernels.hpp"

namespace mslim {

namespace {

constexpr uint64_t kFnvOffset = 0xcbf29ce484222325ull;
constexpr uint64_t kFnvPrime = 0x100000001b3ull;
constexpr int kHeaderWords = kRecordHeaderBytes / 4;   // 26
constexpr int kFooterWords = kRecordFooterBytes / 4;   // 14
constexpr int kKeySumWord = 18;                        // K payload checksum, V's follows

__device__ __forceinline__ uint64_t fnv_byte(uint64_t s, uint32_t b) { return (s ^ b) * kFnvPrime; }

// FNV-1a over the four little-endian bytes of a word.
__device__ __forceinline__ uint64_t fnv_word(uint64_t s, uint32_t w) {
    s = fnv_byte(s, w & 0xffu);
    s = fnv_byte(s, (w >> 8) & 0xffu);
    s = fnv_byte(s, (w >> 16) & 0xffu);
    return fnv_byte(s, w >> 24);
}

__device__ __forceinline__ uint64_t fnv_chunk(uint64_t s, const u32x4_t &c) {
    s = fnv_word(s, c[0]);
    s = fnv_word(s, c[1]);
    s = fnv_word(s, c[2]);
    return fnv_word(s, c[3]);
}

__device__ __forceinline__ bool record_valid(const RecordDesc &r, int page_tokens, int64_t pool_pages) {
    return r.tokens >= 1 && (uint64_t)r.first_row + r.tokens <= (uint64_t)page_tokens && r.pool_page >= 0 &&
           (int64_t)r.pool_page < pool_pages;
}

// A record the frame kernels can read: in staged mode its pool page and
// first row are not used.
__device__ __forceinline__ bool record_ok(const FramesCodecLaunch &a, const RecordDesc &r) {
    if (a.staged) return r.tokens >= 1 && r.tokens <= (uint32_t)a.page_tokens;
    return record_valid(r, a.page_tokens, a.pool_pages);
}

// Row 0 of head 0 of record `rec`'s payload and the byte distance between
// heads: inside its pool page, or in its compacted staging slot.
struct PayloadAt {
    const unsigned char *base;
    int64_t head_stride;
};
__device__ __forceinline__ PayloadAt payload_at(const FramesCodecLaunch &a, const void *src, const RecordDesc &r,
                                                int rec, int row_bytes) {
    const int64_t page_bytes = (int64_t)a.kv_heads * a.page_tokens * row_bytes;
    const unsigned char *s = static_cast<const unsigned char *>(src);
    if (a.staged) return {s + (int64_t)rec * page_bytes, (int64_t)r.tokens * row_bytes};
    return {s + (int64_t)r.pool_page * page_bytes + (int64_t)r.first_row * row_bytes,
            (int64_t)a.page_tokens * row_bytes};
}

// Iterates the 16-byte chunks of one token's bytes over all heads (or of a
// whole head-major payload when `rows_per_head` rows are taken per head):
// heads outer, rows, then 16-byte columns.
struct ChunkWalk {
    const unsigned char *head_base;  // row 0 of the current head
    const unsigned char *row;        // current row
    int64_t head_stride;             // bytes between heads in the pool page
    int row_bytes;
    int col;
    int rows_left;                   // rows left in this head after `row`
    int rows_per_head;

    __device__ __forceinline__ const u32x4_t *ptr() const {
        return reinterpret_cast<const u32x4_t *>(row + col);
    }
    __device__ __forceinline__ void advance() {
        col += 16;
        if (col == row_bytes) {
            col = 0;
            if (rows_left > 0) {
                row += row_bytes;
                --rows_left;
            } else {
                head_base += head_stride;
                row = head_base;
                rows_left = rows_per_head - 1;
            }
        }
    }
};

// One lane per (record, part, token).  Chunks are loaded kPrefetch ahead of
// the FNV chain so every lane keeps several 16-byte loads in flight.
constexpr int kPrefetch = 8;

__global__ __launch_bounds__(256) void token_hashes_kernel(FramesCodecLaunch a) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t per_record = 2 * (int64_t)a.page_tokens;
    if (gid >= (int64_t)a.count * per_record) return;
    const int rec = (int)(gid / per_record);
    const int rem = (int)(gid - (int64_t)rec * per_record);
    const int part = rem / a.page_tokens;  // 0 = K, 1 = V
    const int token = rem - part * a.page_tokens;
    const RecordDesc r = a.records[rec];
    if (!record_ok(a, r) || token >= (int)r.tokens) return;

    const int row_bytes = a.head_dim * 2;
    const PayloadAt at = payload_at(a, part ? a.v_pool : a.k_pool, r, rec, row_bytes);
    ChunkWalk w;
    w.head_base = at.base + (int64_t)token * row_bytes;
    w.row = w.head_base;
    w.head_stride = at.head_stride;
    w.row_bytes = row_bytes;
    w.col = 0;
    w.rows_left = 0;
    w.rows_per_head = 1;
    const int chunks = a.kv_heads * (row_bytes / 16);

    u32x4_t buf[kPrefetch];
    ChunkWalk ld = w;
#pragma unroll
    for (int i = 0; i < kPrefetch; ++i) {
        if (i < chunks) {
            buf[i] = *ld.ptr();
            ld.advance();
        }
    }
    uint64_t s = kFnvOffset;
    int c = 0;
    for (; c + kPrefetch <= chunks; c += kPrefetch) {
#pragma unroll
        for (int i = 0; i < kPrefetch; ++i) {
            const u32x4_t cur = buf[i];
            if (c + kPrefetch + i < chunks) {
                buf[i] = *ld.ptr();
                ld.advance();
            }
            s = fnv_chunk(s, cur);
        }
    }
#pragma unroll
    for (int i = 0; i < kPrefetch; ++i)
        if (c + i < chunks) s = fnv_chunk(s, buf[i]);

    unsigned char *frame = static_cast<unsigned char *>(a.frames) + (int64_t)rec * a.frame_bytes;
    uint64_t *table = reinterpret_cast<uint64_t *>(frame + kRecordHeaderBytes);
    table[part * (int)r.tokens + token] = s;
}

// FNV-1a over the little-endian bytes of a payload by one wavefront, each lane
// on a segment of up to 512 bytes of a 32 KiB tile.  One step is
// s' = (s ^ b) P mod 2^64, and s ^ b = s + d with d set by b and the low byte of
// s alone.  So once the low byte l at the start of a segment is known, the
// segment maps any state s with that low byte to (s - l) P^n + C, where C is
// the segment's own chain started from l, and the lanes' results combine in 64
// multiply-adds.
//
// The low byte runs by itself: l' = (l ^ b) 0xb3 mod 256.  Bit j of it depends
// on bits 0..j only, and flipping bit j of the start flips just bit j of the
// end (0xb3 is odd).  So with bits 0..j-1 of every start known and bit j taken
// as zero, the parity of the end bits of the segments before one is its true
// bit j.  A pass runs the byte chain twice, packed in 16-bit halves, with bit
// j zero and one, which settles bits j and j + 1.  Four such passes of three
// cheap instructions per byte and one pass of the full chain, over segments
// held in registers, replace one full chain over the whole payload.  For 2,016
// records of two 32 KiB payloads: 0.6 ms as the first part of the frame
// kernel's chain; 223 us with 32 lanes re-reading their segments for eight
// passes; 94 us here.
constexpr int kSumLanes = 64;
constexpr int kSumChunks = 32;  // of a segment, in registers
typedef unsigned short ushort2_t __attribute__((ext_vector_type(2)));

constexpr uint64_t fnv_prime_power(int n) {
    uint64_t p = 1;
    for (int i = 0; i < n; ++i) p *= kFnvPrime;
    return p;
}

__global__ __launch_bounds__(256) void payload_sums_kernel(FramesCodecLaunch a) {
    const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + threadIdx.x / 64));
    const int lane = threadIdx.x & 63;
    const int rec = wave / 2, part = wave % 2;  // one wavefront per (record, K or V)
    if (rec >= a.count) return;
    const RecordDesc r = a.records[rec];
    if (!record_ok(a, r)) return;
    const int tokens = (int)r.tokens;
    const int row_bytes = a.head_dim * 2, row_chunks = row_bytes / 16;
    const int chunks = a.kv_heads * tokens * row_chunks;  // of the payload
    const PayloadAt at = payload_at(a, part ? a.v_pool : a.k_pool, r, rec, row_bytes);
    const uint64_t below = ((uint64_t)1 << lane) - 1;

    uint64_t sum = kFnvOffset;
    for (int t0 = 0; t0 < chunks; t0 += kSumLanes * kSumChunks) {
        const int here = min(chunks - t0, kSumLanes * kSumChunks);
        const int per = (here + kSumLanes - 1) / kSumLanes;
        const int c0 = min(lane * per, here), n = min(c0 + per, here) - c0;
        // The segment: chunk t0 + c0 lies in row (t0 + c0) / row_chunks of the
        // head-major rows.
        const int row = (t0 + c0) / row_chunks, head = row / tokens;
        ChunkWalk walk;
        walk.head_base = at.base + (int64_t)head * at.head_stride;
        walk.row = walk.head_base + (int64_t)(row - head * tokens) * row_bytes;
        walk.head_stride = at.head_stride;
        walk.row_bytes = row_bytes;
        walk.col = (t0 + c0) % row_chunks * 16;
        walk.rows_left = tokens - 1 - (row - head * tokens);
        walk.rows_per_head = tokens;
        u32x4_t c[kSumChunks];
#pragma unroll
        for (int i = 0; i < kSumChunks; ++i) {
            if (i < n) {
                c[i] = *walk.ptr();
                walk.advance();
            }
        }
        uint32_t start = 0;
#pragma unroll 1
        for (int j = 0; j < 8; j += 2) {
            ushort2_t l = {(unsigned short)start, (unsigned short)(start | (1u << j))};
            const ushort2_t prime = {(unsigned short)(kFnvPrime & 0xff), (unsigned short)(kFnvPrime & 0xff)};
#pragma unroll
            for (int i = 0; i < kSumChunks; ++i) {
                if (i >= n) continue;
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        // byte e of the word in both halves (0x0c: zero)
                        const uint32_t b = __builtin_amdgcn_perm(0, c[i][k], 0x0c000c00u + 0x00010001u * e);
                        l = (l ^ __builtin_bit_cast(ushort2_t, b)) * prime;
                    }
            }
            auto settle = [&](uint32_t end, int bit) __attribute__((always_inline)) {
                const uint64_t ends = __builtin_amdgcn_ballot_w64(((end >> bit) & 1u) != 0);
                return ((uint32_t)(sum >> bit) ^ (uint32_t)__popcll(ends & below)) & 1u;
            };
            const uint32_t low = settle(l[0], j);
            const uint32_t high = settle(low ? l[1] : l[0], j + 1);
            start |= low << j | high << (j + 1);
        }
        uint64_t chain = start, power = 1;
#pragma unroll
        for (int i = 0; i < kSumChunks; ++i)
            if (i < n) chain = fnv_chunk(chain, c[i]);
        uint64_t square = fnv_prime_power(16);  // of one chunk
        for (int e = n; e; e >>= 1, square *= square)
            if (e & 1) power *= square;
#pragma unroll 1
        for (int i = 0; i < kSumLanes; ++i) {
            auto of = [&](uint64_t x) __attribute__((always_inline)) {
                return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)x, i) |
                       ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), i) << 32);
            };
            sum = (sum - (uint32_t)__builtin_amdgcn_readlane((int)start, i)) * of(power) + of(chain);
        }
    }
    // Left in the header words the checksums belong to; the frame kernel reads
    // them there.
    if (lane == 0) {
        uint32_t *words = reinterpret_cast<uint32_t *>(static_cast<unsigned char *>(a.frames) + (int64_t)rec * a.frame_bytes);
        words[kKeySumWord + 2 * part] = (uint32_t)sum;
        words[kKeySumWord + 2 * part + 1] = (uint32_t)(sum >> 32);
    }
}

// ---- SHA-256 (FIPS 180-4) -------------------------------------------------

__device__ __constant__ uint32_t kSha256K[64] = {
    0x428a2f98u, 0x71374491u, 0xb5c0fbcfu, 0xe9b5dba5u, 0x3956c25bu, 0x59f111f1u, 0x923f82a4u, 0xab1c5ed5u,
    0xd807aa98u, 0x12835b01u, 0x243185beu, 0x550c7dc3u, 0x72be5d74u, 0x80deb1feu, 0x9bdc06a7u, 0xc19bf174u,
    0xe49b69c1u, 0xefbe4786u, 0x0fc19dc6u, 0x240ca1ccu, 0x2de92c6fu, 0x4a7484aau, 0x5cb0a9dcu, 0x76f988dau,
    0x983e5152u, 0xa831c66du, 0xb00327c8u, 0xbf597fc7u, 0xc6e00bf3u, 0xd5a79147u, 0x06ca6351u, 0x14292967u,
    0x27b70a85u, 0x2e1b2138u, 0x4d2c6dfcu, 0x53380d13u, 0x650a7354u, 0x766a0abbu, 0x81c2c92eu, 0x92722c85u,
    0xa2bfe8a1u, 0xa81a664bu, 0xc24b8b70u, 0xc76c51a3u, 0xd192e819u, 0xd6990624u, 0xf40e3585u, 0x106aa070u,
    0x19a4c116u, 0x1e376c08u, 0x2748774cu, 0x34b0bcb5u, 0x391c0cb3u, 0x4ed8aa4au, 0x5b9cca4fu, 0x682e6ff3u,
    0x748f82eeu, 0x78a5636fu, 0x84c87814u, 0x8cc70208u, 0x90befffau, 0xa4506cebu, 0xbef9a3f7u, 0xc67178f2u};

__device__ __forceinline__ uint32_t rotr(uint32_t x, int n) { return (x >> n) | (x << (32 - n)); }
// Three-input bit functions in one instruction each (v_bitop3_b32; the truth
// table is the function of 0xf0, 0xcc and 0xaa).
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}
__device__ __forceinline__ uint32_t choose(uint32_t a, uint32_t b, uint32_t c) {  // a ? b : c
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0xca);
}
__device__ __forceinline__ uint32_t majority(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0xe8);
}

// Sixteen message words (big-endian values) extended in place to the schedule
// of rounds r .. r + 15, r a multiple of 16 above zero.
__device__ __forceinline__ void sha256_extend(uint32_t w[16]) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const uint32_t w15 = w[(i + 1) & 15], w2 = w[(i + 14) & 15];
        const uint32_t s0 = xor3(rotr(w15, 7), rotr(w15, 18), w15 >> 3);
        const uint32_t s1 = xor3(rotr(w2, 17), rotr(w2, 19), w2 >> 10);
        w[i] += s0 + w[(i + 9) & 15] + s1;
    }
}

__device__ __forceinline__ uint32_t lo32(uint64_t x) { return (uint32_t)x; }
__device__ __forceinline__ uint32_t hi32(uint64_t x) { return (uint32_t)(x >> 32); }

// Three wavefronts per 64 records, lane = record, in step over the 64-byte
// blocks of header | tables | K | V | padding:
//   * the schedule wavefront loads block i + 2, extends it to its 64 round
//     words and leaves them, constants added, in LDS (and the sixteen message
//     words as they lie in the record);
//   * the rounds wavefront runs the 64 rounds of block i;
//   * the checksum wavefront runs the record's FNV-1a over block i.
// A lane's instructions issue every four clocks whatever its neighbours do, so
// the chain is as long as its instruction count: the rounds alone are 14
// instructions each, and everything else of SHA-256 (8 to 10 more, the loads
// and byte swaps) runs on another SIMD.  2,016 records of 64 KiB payloads:
// 4.41 ms with the schedule, the message ring and the payload checksums on
// the rounds' wavefront, 2.11 ms here (1,030 blocks of 64 rounds).
constexpr int kFrameThreads = 64;  // records per workgroup
constexpr int kFrameRoles = 3;
enum { kRounds = 0, kSchedule = 1, kChecksum = 2 };

__global__ __launch_bounds__(kFrameRoles * kFrameThreads) void frame_kernel(FramesCodecLaunch a) {
    // [block % 4][four words][lane]
    __shared__ u32x4_t rounds_lds[4][16][kFrameThreads];
    __shared__ u32x4_t message_lds[4][4][kFrameThreads];
    __shared__ uint64_t sums[kFrameRoles][kFrameThreads];
    const int lane = threadIdx.x & (kFrameThreads - 1);
    const int role = __builtin_amdgcn_readfirstlane(threadIdx.x / kFrameThreads);
    const int rec = blockIdx.x * kFrameThreads + lane;
    const bool live = rec < a.count;
    RecordDesc r = {};
    if (live) r = a.records[rec];
    const bool valid = live && record_ok(a, r);
    uint32_t *frame_words = reinterpret_cast<uint32_t *>(static_cast<unsigned char *>(a.frames) +
                                                         (int64_t)(live ? rec : 0) * a.frame_bytes);
    const int frame_words_n = (int)(a.frame_bytes / 4);
    const int tokens = valid ? (int)r.tokens : 0;
    const int row_bytes = a.head_dim * 2, row_chunks = row_bytes / 16;
    const int64_t payload_len = (int64_t)a.kv_heads * tokens * row_bytes;
    RecordDesc rv = r;
    if (!valid) rv = RecordDesc{0, 0, 0, 1, 0, 0};
    const PayloadAt kat = payload_at(a, a.k_pool, rv, valid ? rec : 0, row_bytes);
    const PayloadAt vat = payload_at(a, a.v_pool, rv, valid ? rec : 0, row_bytes);

    // Hash-table checksums over the little-endian u64 tables (written by
    // token_hashes_kernel into this frame): K's on one wavefront, V's on
    // another.
    const uint32_t *tables = frame_words + kHeaderWords;
    if (role != kChecksum) {
        uint64_t sum = kFnvOffset;
        const uint2 *t = reinterpret_cast<const uint2 *>(tables) + role * tokens;
        constexpr int kAhead = 8;
        for (int i0 = 0; i0 < tokens; i0 += kAhead) {
            uint2 h[kAhead];
#pragma unroll
            for (int i = 0; i < kAhead; ++i) h[i] = t[min(i0 + i, tokens - 1)];
#pragma unroll
            for (int i = 0; i < kAhead; ++i)
                if (i0 + i < tokens) sum = fnv_word(fnv_word(sum, h[i].x), h[i].y);
        }
        sums[role][lane] = sum;
    }
    __syncthreads();
    const uint64_t record_len =
        (uint64_t)kRecordHeaderBytes + 16ull * tokens + 2ull * (uint64_t)payload_len + kRecordFooterBytes;
    // The header (cold_store.rs:291-309); the payload checksums already lie in
    // it (payload_sums_kernel).
    if (role == kRounds && valid) {
        const uint64_t key_hashes_sum = sums[0][lane], value_hashes_sum = sums[1][lane];
        frame_words[0] = 0x564b5354u;  // "TSKV"
        frame_words[1] = 0x34304750u;  // "PG04"
        frame_words[2] = kRecordVersion;
        frame_words[3] = kRecordHeaderBytes;
        frame_words[4] = lo32(r.page_id);
        frame_words[5] = hi32(r.page_id);
        frame_words[6] = r.layer;
        frame_words[7] = 0u;
        frame_words[8] = lo32(r.token_start);
        frame_words[9] = hi32(r.token_start);
        frame_words[10] = r.tokens;
        frame_words[11] = (uint32_t)a.kv_heads;
        frame_words[12] = (uint32_t)a.head_dim;
        frame_words[13] = a.tile;
        frame_words[14] = lo32((uint64_t)payload_len);
        frame_words[15] = hi32((uint64_t)payload_len);
        frame_words[16] = lo32((uint64_t)payload_len);
        frame_words[17] = hi32((uint64_t)payload_len);
        frame_words[22] = lo32(key_hashes_sum);
        frame_words[23] = hi32(key_hashes_sum);
        frame_words[24] = lo32(value_hashes_sum);
        frame_words[25] = hi32(value_hashes_sum);
        for (int i = kHeaderWords + 4 * tokens; i < frame_words_n - kFooterWords; ++i) frame_words[i] = 0u;
    }
    __syncthreads();  // the header is read back as message words below

    // The message: head words (header and tables, as they lie in the frame),
    // payload words (K then V, whole 16-byte chunks), the 0x80 byte, zeros and
    // the bit length.  The payload starts at word 2 of a group of four.
    const int head_words = kHeaderWords + 4 * tokens;
    const int part_chunks = (int)(payload_len / 16);
    const int payload_words = 8 * part_chunks;
    const int message_words = head_words + payload_words;
    const int blocks = valid ? (message_words + 3 + 15) / 16 : 0;
    int most = blocks;
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) most = max(most, __shfl_xor(most, m, 64));
    most = __builtin_amdgcn_readfirstlane(most);

    // Where chunk i of K then V lies.  A payload whose heads follow each other
    // without a gap (a whole page, or staging) is one run.
    const bool run = kat.head_stride == (int64_t)tokens * row_bytes;
    auto chunk_at = [&](int i) __attribute__((always_inline)) {
        const bool v = i >= part_chunks;
        const int c = v ? i - part_chunks : i;
        const unsigned char *base = v ? vat.base : kat.base;
        if (run) return base + (int64_t)c * 16;
        const int row = c / row_chunks, head = row / tokens;
        return base + head * kat.head_stride + (int64_t)(row - head * tokens) * row_bytes + (c - row * row_chunks) * 16;
    };

    if (role == kSchedule) {
        // Block b is inside the payload for most of a record: its words are
        // the last two of chunk c, chunks c + 1 .. c + 3 and the first two of
        // chunk c + 4.
        auto inside = [&](int b) __attribute__((always_inline)) {
            const int o = b * 16 - head_words;
            return o >= 2 && o + 16 <= payload_words;
        };
        constexpr int kAhead = 2;  // blocks in flight
        u32x4_t ahead[kAhead][5];
        auto fetch = [&](u32x4_t (&c)[5], int b) __attribute__((always_inline)) {
            if (!inside(b)) return;
            const int c0 = (b * 16 - head_words - 2) / 4;
#pragma unroll
            for (int k = 0; k < 5; ++k) c[k] = *reinterpret_cast<const u32x4_t *>(chunk_at(c0 + k));
        };
        auto produce = [&](const u32x4_t (&c)[5], int b) __attribute__((always_inline)) {
            uint32_t w[16];
            if (inside(b)) {
                w[0] = c[0][2];
                w[1] = c[0][3];
#pragma unroll
                for (int k = 0; k < 12; ++k) w[2 + k] = c[1 + k / 4][k % 4];
                w[14] = c[4][0];
                w[15] = c[4][1];
            } else {
                const uint64_t bits = (record_len - kRecordFooterBytes) * 8;
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const int g = b * 16 + j, o = g - head_words;
                    uint32_t x = 0;
                    if (b < blocks) {
                        if (g < head_words) x = frame_words[g];
                        else if (o < payload_words) x = reinterpret_cast<const uint32_t *>(chunk_at(o / 4))[o % 4];
                        else if (g == message_words) x = 0x80u;
                        else if (g == blocks * 16 - 2) x = __builtin_bswap32(hi32(bits));
                        else if (g == blocks * 16 - 1) x = __builtin_bswap32(lo32(bits));
                    }
                    w[j] = x;
                }
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
                message_lds[b & 3][k][lane] = u32x4_t{w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]};
#pragma unroll
            for (int j = 0; j < 16; ++j) w[j] = __builtin_bswap32(w[j]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (q) sha256_extend(w);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    u32x4_t x;
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[e] = w[4 * k + e] + kSha256K[16 * q + 4 * k + e];
                    rounds_lds[b & 3][4 * q + k][lane] = x;
                }
            }
        };
#pragma unroll
        for (int k = 0; k < kAhead; ++k) fetch(ahead[k], k);
        produce(ahead[0], 0);
        fetch(ahead[0], kAhead);
        for (int b = 0; b < most; b += kAhead) {
#pragma unroll
            for (int k = 0; k < kAhead; ++k) {
                if (b + k >= most) break;
                const int next = (k + 1) % kAhead;
                produce(ahead[next], b + k + 1);
                fetch(ahead[next], b + k + 1 + kAhead);
                __syncthreads();
            }
        }
    } else if (role == kRounds) {
        uint32_t h[8] = {0x6a09e667u, 0xbb67ae85u, 0x3c6ef372u, 0xa54ff53au,
                         0x510e527fu, 0x9b05688cu, 0x1f83d9abu, 0x5be0cd19u};
        // Barrier b: blocks up to b + 1 are in LDS, and the place of block
        // b - 2 is free.  The first words of block b + 1 are read ahead of
        // the last rounds of block b.
        constexpr int kFirst = 4;
        u32x4_t first[kFirst] = {};
        for (int b = 0; b < most; ++b) {
            __syncthreads();
            if (b >= blocks) continue;
            if (b == 0) {
#pragma unroll
                for (int k = 0; k < kFirst; ++k) first[k] = rounds_lds[0][k][lane];
            }
            uint32_t s[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) s[i] = h[i];
#pragma unroll
            for (int i = 0; i < 64; i += 4) {
                const u32x4_t kw = i / 4 < kFirst ? first[i / 4 % kFirst] : rounds_lds[b & 3][i / 4][lane];
                if (i == 4 * kFirst) {
#pragma unroll
                    for (int k = 0; k < kFirst; ++k) first[k] = rounds_lds[(b + 1) & 3][k][lane];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    // s[(0 - i - e) & 7] is the round's a, and so on: the
                    // state turns instead of moving
                    const int n = (i + e) & 7;
                    const uint32_t A = s[(8 - n) & 7], B = s[(9 - n) & 7], C = s[(10 - n) & 7];
                    const uint32_t E = s[(12 - n) & 7], F = s[(13 - n) & 7], G = s[(14 - n) & 7];
                    const uint32_t t1 = s[(15 - n) & 7] + kw[e] + xor3(rotr(E, 6), rotr(E, 11), rotr(E, 25)) +
                                        choose(E, F, G);
                    s[(11 - n) & 7] += t1;
                    s[(15 - n) & 7] = t1 + xor3(rotr(A, 2), rotr(A, 13), rotr(A, 22)) + majority(A, B, C);
                }
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) h[i] += s[i];
        }
        __syncthreads();  // the checksum wavefront is done
        if (!live) return;
        if (!valid) {
            for (int i = 0; i < frame_words_n; ++i) frame_words[i] = 0u;
            return;
        }
        const uint64_t record_sum = sums[kChecksum][lane];
        uint32_t *footer = frame_words + frame_words_n - kFooterWords;
        footer[0] = 0x564b5354u;  // "TSKV"
        footer[1] = 0x54494d43u;  // "CMIT"
        footer[2] = lo32(record_sum);
        footer[3] = hi32(record_sum);
        footer[4] = lo32(record_len);
        footer[5] = hi32(record_len);
#pragma unroll
        for (int i = 0; i < 8; ++i) footer[6 + i] = __builtin_bswap32(h[i]);
        return;
    } else {
        uint64_t record_sum = kFnvOffset;
        for (int b = 0; b < most; ++b) {
            __syncthreads();
            const int n = message_words - b * 16;  // message words left
            if (!valid || n <= 0) continue;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const u32x4_t c = message_lds[b & 3][k][lane];
                if (n >= 16) {
                    record_sum = fnv_chunk(record_sum, c);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (4 * k + e < n) record_sum = fnv_word(record_sum, c[e]);
                }
            }
        }
        sums[kChecksum][lane] = record_sum;
    }
    __syncthreads();
}

// Payload moves between pool pages and contiguous staging: staging slot i
// (one pool page's bytes) holds record i's head-major payload compacted to
// its `tokens` rows per head.  One lane moves one 16-byte piece of K and of V;
// consecutive lanes take consecutive pieces of a pool page, so the pool side
// is coalesced and the staging side is coalesced within each row run.
template <bool TO_STAGING>
__global__ __launch_bounds__(256) void record_payloads_kernel(PayloadMoveLaunch a) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int cpr = a.head_dim * 2 / 16;  // 16-byte pieces per row
    const int64_t per_page = (int64_t)a.kv_heads * a.page_tokens * cpr;
    if (gid >= (int64_t)a.count * per_page) return;
    const int rec = (int)(gid / per_page);
    const int64_t c = gid - (int64_t)rec * per_page;
    const RecordDesc r = a.records[rec];
    if (!record_valid(r, a.page_tokens, a.pool_pages)) return;
    const int col = (int)(c % cpr);
    const int64_t hr = c / cpr;  // head * page_tokens + row of the pool page
    const int page_row = (int)(hr % a.page_tokens);
    const int head = (int)(hr / a.page_tokens);
    const int row = page_row - (int)r.first_row;  // row of the record
    if (row < 0 || row >= (int)r.tokens) return;
    const int64_t page_bytes = per_page * 16;
    const int64_t pool_off = (int64_t)r.pool_page * page_bytes + c * 16;
    const int64_t stage_off = (int64_t)rec * page_bytes + (((int64_t)head * r.tokens + row) * cpr + col) * 16;
    unsigned char *kp = static_cast<unsigned char *>(a.k_pool), *vp = static_cast<unsigned char *>(a.v_pool);
    unsigned char *ks = static_cast<unsigned char *>(a.k_stage), *vs = static_cast<unsigned char *>(a.v_stage);
    if constexpr (TO_STAGING) {
        *reinterpret_cast<u32x4_t *>(ks + stage_off) = *reinterpret_cast<const u32x4_t *>(kp + pool_off);
        *reinterpret_cast<u32x4_t *>(vs + stage_off) = *reinterpret_cast<const u32x4_t *>(vp + pool_off);
    } else {
        *reinterpret_cast<u32x4_t *>(kp + pool_off) = *reinterpret_cast<const u32x4_t *>(ks + stage_off);
        *reinterpret_cast<u32x4_t *>(vp + pool_off) = *reinterpret_cast<const u32x4_t *>(vs + stage_off);
    }
}

}  // namespace

int64_t record_frame_bytes(int page_tokens) {
    return (int64_t)kRecordHeaderBytes + 16ll * page_tokens + kRecordFooterBytes;
}

hipError_t launch_record_frames(const FramesCodecLaunch &a, hipStream_t stream) {
    if (a.count == 0) return hipSuccess;
    const int64_t lanes = (int64_t)a.count * 2 * a.page_tokens;
    hipLaunchKernelGGL(token_hashes_kernel, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, stream, a);
    if (hipError_t e = hipGetLastError()) return e;
    const int64_t sum_lanes = (int64_t)a.count * 2 * kSumLanes;
    hipLaunchKernelGGL(payload_sums_kernel, dim3((unsigned)((sum_lanes + 255) / 256)), dim3(256), 0, stream, a);
    if (hipError_t e = hipGetLastError()) return e;
    hipLaunchKernelGGL(frame_kernel, dim3((unsigned)((a.count + kFrameThreads - 1) / kFrameThreads)),
                       dim3(kFrameRoles * kFrameThreads), 0, stream, a);
    return hipGetLastError();
}

hipError_t launch_record_payloads(const PayloadMoveLaunch &a, bool to_staging, hipStream_t stream) {
    if (a.count == 0) return hipSuccess;
    const int64_t lanes = (int64_t)a.count * a.kv_heads * a.page_tokens * (a.head_dim * 2 / 16);
    const dim3 grid((unsigned)((lanes + 255) / 256));
    if (to_staging)
        hipLaunchKernelGGL(record_payloads_kernel<true>, grid, dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL(record_payloads_kernel<false>, grid, dim3(256), 0, stream, a);
    return hipGetLastError();
}

}  // namespace mslim
