// Attention of portions of prompts over the paged cache (prefill), bfloat16, on the MFMA units
// with 32 x 32 tiles.
//
// A wave owns 32 columns: R consecutive query rows of a request for each of GH = 32 / R query
// heads that share one key/value head (GH = the group size when that is a power of two up to 32,
// else 1), so one pass over the keys serves the whole group.  A block is four waves with four
// neighbouring row tiles of one request.  It walks the keys its rows see, 32 at a time, from the
// cache pages (keys written by this same step included): a block's loads write key and value tiles to shared memory
// directly, a ring of four tiles ahead, one barrier per tile; every wave reads its MFMA
// operands from shared memory, whose pieces are exchanged so that those reads do not collide.
//   S^T[key, col] = K[key, :] . Q[col, :]         v_mfma_f32_32x32x16_bf16, D / 16 of them;
//       lane (g, r), g = lane / 32, r = lane % 32, takes K[key r'][ks * 16 + g * 8 .. + 8], r' being r with its bits 2
//       and 3 exchanged, and ends up with 16 scores: keys 16 h + 8 g + j (h < 2, j < 8) of column r
//   online softmax per column in 32-bit, in the base-2 domain (scores are scaled by
//       scale * log2 e once); the accumulator is rescaled only when a score exceeds the column's
//       reference by more than 8
//   O^T[d, col] += V^T[d, key] . P^T[key, col]    v_mfma_f32_32x32x16_bf16, 2 * D / 32 of them;
//       the 8 probabilities of a half tile that a lane holds are its B operand as they lie, and
//       because value tiles are stored transposed ([D][P]) the A operand is the same 8 keys of
//       one row of V^T, one 16-byte read
// What bounds it: the vector units' 560 cycles and the matrix units' 512 of a wave's tile, which overlap only between the two waves of
// a SIMD.  (With tiles through registers, a barrier behind every tile's arrival and the scores of a tile right before its weights:
// 8192 tokens of 32 heads of 128 on 8, 637 us, now 588; 512 rows each behind 4096 keys, four requests, 204, now 171; 2048 tokens of
// 16 heads 49, now 44.7; 512 rows behind 7680 keys, with the merge of their segments, 62, now 56; 3000 tokens of 16 heads of 64 on 4 53, now 50.)
// The causal and window limits are applied per column, so the order of the sums for a row
// depends on its position and the window only.
//
// With NG = 2 a block has two such groups of four waves on the same four row tiles: group 0 takes
// the even key tiles and group 1 the odd ones, each through shared buffers of its own, and at the
// end group 0 merges the two partial results (maxima, sums, accumulators) through shared memory.
// That halves the length of the longest block, which is what the time of a causal prompt hangs on
// when there are no more blocks than compute units.  The longest blocks are started first.
//
// Key segments: with fewer blocks than compute units and many keys (a portion of a prompt far into
// its context) the keys are cut at absolute multiples of a segment length, and the blocks of the
// grid's second dimension walk one segment each.  A block whose rows' keys lie in one segment writes
// its result as before (the blocks of the other segments leave at once); else the blocks of the
// segments that hold keys of its rows leave their maxima, sums and accumulators, as the lanes hold
// them, in a workspace, and attention_prefill_merge_kernel, with the same lanes, weighs and adds them
// in the order of the segments.  The segment length comes from the host, or, where the host does not
// know the positions (a recorded step), from the position of the row that sees the most keys.
#include "common.h"

#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(16))) float floatx16;
typedef __attribute__((ext_vector_type(4))) unsigned int uint4_t;

// Lane i and lane i ^ 32 exchange a value without a trip through shared memory.
__device__ __forceinline__ float max_of_both_halves(float v) {
    float a, b;
    pair_across_halves(v, a, b);
    return fmaxf(a, b);
}
__device__ __forceinline__ float sum_of_both_halves(float v) {
    float a, b;
    pair_across_halves(v, a, b);
    return a + b;
}

#define QE_PREFILL_UNCUT_KEYS 1024
#define QE_PREFILL_MIN_SEGMENT 512

// Tiles of keys and values in a group's shared memory: 64 KB for heads of 128, for two groups a compute unit (eight tiles of heads of 64
// are no quicker).
#define RING 4

// The keys of a segment when ``keys`` keys are cut into ks segments: a multiple of 64, at least
// QE_PREFILL_MIN_SEGMENT; 0 (no cut) up to QE_PREFILL_UNCUT_KEYS keys.  One formula for the host's plan
// and for the kernels of a recorded step, which cut by a position they read on the device.
__host__ __device__ __forceinline__ int prefill_segment_length(int keys, int ks) {
    if (keys <= QE_PREFILL_UNCUT_KEYS || ks <= 1) return 0;
    const int seg = ((keys + ks - 1) / ks + 63) / 64 * 64;
    return seg < QE_PREFILL_MIN_SEGMENT ? QE_PREFILL_MIN_SEGMENT : seg;
}

// The keys of a segment when the host does not know the positions (a recorded step): seg_param < 0
// asks for -seg_param segments of the keys that row keys_row sees, each a multiple of 64 and at least
// QE_PREFILL_MIN_SEGMENT keys; up to QE_PREFILL_UNCUT_KEYS keys nothing is cut (0).  The same value
// in every block of the two kernels.
__device__ __forceinline__ int segment_keys(int seg_param, const int* __restrict__ positions, int keys_row) {
    if (seg_param >= 0) return seg_param;
    return prefill_segment_length(positions[keys_row] + 1, -seg_param);
}

// A lane's share of its column's result: the accumulators' element 4 b + j of block db is feature
// 32 db + 8 b + 4 g + j.
template <int D>
__device__ __forceinline__ void store_columns(bf16_t* __restrict__ out, const floatx16 (&acc)[D / 32], float inv,
                                              int row, int head, int g, const AttnTail& tail) {
    if (tail.plain) {
        bf16_t* orow = out + (long)row * tail.out_stride + (long)head * D + 4 * g;
#pragma unroll
        for (int db = 0; db < D / 32; ++db)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                bf16x4 o;
#pragma unroll
                for (int j = 0; j < 4; ++j) o[j] = (__bf16)(acc[db][4 * b + j] * inv);
                *(bf16x4*)(orow + db * 32 + 8 * b) = o;
            }
        return;
    }
    // (the pieces of four whose gates and places are whole pieces too go as such)
    const bool four = tail.dv % 4 == 0 && tail.out_stride % 4 == 0 && (((unsigned long)out) & 7) == 0 &&
                      (!tail.gate || (!tail.gate_f32 && tail.gate_stride % 4 == 0 && (((unsigned long)tail.gate) & 7) == 0));
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int d = db * 32 + 8 * b + 4 * g;
            if (four) {
                if (d >= tail.dv) continue;
                float v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = acc[db][4 * b + j] * inv;
                if (tail.gate) {
                    float z[4];
                    Vec4<bf16_t>::load((const bf16_t*)tail.gate + (long)row * tail.gate_stride + (long)head * tail.dv + d, z);
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] *= __builtin_amdgcn_rcpf(1.f + __expf(-z[j]));
                }
                Vec4<bf16_t>::store(out + (long)row * tail.out_stride + (long)head * tail.dv + d, v);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) tail.store(out, row, head, d + j, acc[db][4 * b + j] * inv);
            }
        }
}

// Two waves per SIMD (at most 256 registers a lane), as two blocks of one group or one block of
// two: while one wave waits for its next tile or at its barrier, the other computes.
// CAP: the scaled scores pass cap * tanh(. / cap): cap_in is the scores' scale times 2 log2(e) / cap, cap_out the cap
// in the base-2 domain, and scale_log2 is 1.
// DIRECT: the cache begins at a whole 16-byte piece, which loads that write to shared memory themselves want.  Tiles of a cache that lies
// elsewhere come through registers, asked for a round before they are stored to their place; the same bits (8192 tokens of 32 heads of 128 on 8
// 546 us and 609, 2048 of 16 heads 45 and 58, 512 rows behind 7680 keys 50 and 61).
// SINGLES: the first groups are single new tokens (its own form: the comparison with a number of the group's own instead of 8 cost prompts 0.6 %).
template <int D, int NG, bool CAP, bool DIRECT, bool SINGLES>
__global__ __launch_bounds__(256 * NG, NG == 1 ? 2 : 1) void attention_prefill_kernel(
    const bf16_t* __restrict__ q, bf16_t* __restrict__ out, const bf16_t* __restrict__ cache,
    const int* __restrict__ tiles, const int* __restrict__ positions, const int* __restrict__ tok_seq,
    const int* __restrict__ block_table, int max_blocks,
    int Hq, int Hkv, int P, int log2P, float scale_log2, int window, int R, int seg_param, int keys_row,
    float* __restrict__ part, int keep_first, int sink, float cap_in, float cap_out, int singles, AttnTail tail) {
    constexpr int KROW = D * 2, KBYTES = 32 * KROW, BUF = 2 * KBYTES;    // bytes of a key row, of a tile's keys, of a tile
    constexpr int LP = D / 64;                       // loads of a wave for a tile's keys, and for its values
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_all[];      // NG rings of RING tiles

    // (group and wave are the same for all lanes of a wave: kept in scalar registers, so that what
    // follows from them — tile keys, pages, addresses — is scalar arithmetic)
    const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x / 256);   // which half of the key tiles (NG = 2)
    const int tid = threadIdx.x % 256, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned char* smem = smem_all + grp * RING * BUF;
    const int g = lane >> 5, r = lane & 31;
    const int G = Hq / Hkv;
    const int GH = 32 / R;                                 // heads per wave
    // The grid is (head waves, segments, tile groups): blocks start in the order of the first
    // dimension first, so all heads and segments of the last rows (the longest walks) start before
    // anything of earlier rows, and a compute unit that is done takes the longest of what is left.
    const int bhead = blockIdx.x, bseg = blockIdx.y, bgroup = blockIdx.z;
    const int kvh = bhead / (G / GH);
    const int head = kvh * G + (bhead % (G / GH)) * GH + r / R;   // this lane's column: head and row

    // the block's four tiles belong to one request, in ascending rows; tiles of 0 rows pad the group
    const int* bt4 = tiles + 8 * (gridDim.z - 1 - bgroup);   // later rows see more keys: they start first
    if (bt4[1] <= 0) return;                               // a group without rows (a list filled up to a fixed length)
    const int row_first = bt4[0];
    const float slack = SINGLES && (int)(gridDim.z - 1 - bgroup) < singles ? 0.f : 8.f;
    int last = 0;
#pragma unroll
    for (int j = 1; j < 4; ++j) if (bt4[2 * j + 1] > 0) last = j;
    const int p_block = positions[row_first];
    int kmin = first_seen_key(p_block, window);
    int kmax = positions[bt4[2 * last]] + bt4[2 * last + 1];
    // the request's kept first keys that lie behind the block's window: [0, kfb) (never together with segments)
    const int kfb = keep_first < kmin ? keep_first : kmin;
    // key segments: this block walks the keys of segment bseg only
    bool partial = false;
    const int seg_keys = segment_keys(seg_param, positions, keys_row);
    if (seg_keys <= 0 && bseg > 0) return;                 // (asked for segments, but the keys are too few to cut)
    if (seg_keys > 0) {
        const int z = bseg, z_lo = kmin / seg_keys, z_hi = (kmax - 1) / seg_keys;
        if (z < z_lo || z > z_hi) return;                  // (the whole block: no barrier has been met yet)
        partial = z_hi > z_lo;
        if (partial) {
            kmin = max(kmin, z * seg_keys);
            kmax = min(kmax, (z + 1) * seg_keys);
        }
    }
    const int* bt = block_table + (long)tok_seq[row_first] * max_blocks;
    const long page_stride = 2L * Hkv * P * D;

    // this wave's tile
    const int row0 = bt4[2 * wave], cnt = bt4[2 * wave + 1];
    const bool wave_on = cnt > 0;
    const int rr = r % R;
    const bool col_ok = wave_on && rr < cnt;
    const int row = wave_on ? row0 + (rr < cnt ? rr : cnt - 1) : row_first;   // columns beyond the tile repeat its last row
    const int p = positions[row];
    const int hi = p + 1;
    const int lo = first_seen_key(p, window);
    const int p_first = positions[wave_on ? row0 : row_first];
    const int k_start = first_seen_key(p_first, window);
    const int k_stop = wave_on ? p_first + cnt : 0;       // positions of a tile's rows are consecutive
    // keys every column of the wave sees without a limit: [all_lo, all_hi)
    const int p_last = p_first + cnt - 1;
    const int all_hi = p_first + 1;
    const int all_lo = first_seen_key(p_last, window);

    float m = -INFINITY, l = 0.f;
    floatx16 acc[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[db][e] = 0.f;

    // ---- staging: global -> shared -------------------------------------------------------------
    // A 32-key tile has two halves of 16 keys with pages and offsets of their own; half of the waves bring one, half the
    // other.  A half that no
    // row of the block sees (beyond the request's keys, or wholly behind the window, where the page
    // may have been given back) is asked for with a descriptor of no bytes and arrives as zeros; what else lies outside
    // [kmin, kmax) is masked in the scores and zeroed in the value fragments (it may be unwritten memory, and anything times a
    // weight of 0 must still be 0).
    // The loads are buffer loads that write to shared memory directly, 64 pieces of 16 bytes side by side an instruction: the
    // page's address and the offset of the 16 keys in it are scalar, and a lane adds bytes that are constant over the
    // loop.  A ring of RING tiles, each tile's loads issued RING - 1 rounds or more ahead; the next tile's page
    // id is asked for a round before it is used.  Pieces are exchanged so that the fragment reads fall into distinct
    // banks: piece p of key row r lies at place p ^ (r % 16) (D = 64: p ^ (r / 2 % 8)), of value row d at p ^ (d / 8 % 2).
    // (So is a tile that does not exist: the number of loads in flight is always known.)  The loads and the waits for them are written as instructions: the compiler would wait for every
    // load in flight before it reads shared memory.
    int kconst[LP], vconst[LP];                            // bytes from the page's start, without the keys' offset
    const int half = wave >> 1;                            // of the tile, that this wave brings
#pragma unroll
    for (int i = 0; i < LP; ++i) {
        const int krow = (wave & 1) * 8 + (D == 128 ? i * 4 + (lane >> 4) : lane >> 3);
        const int piece = D == 128 ? (lane & 15) ^ krow : (lane & 7) ^ (((half * 16 + krow) >> 1) & 7);
        kconst[i] = ((kvh * P + krow) * D) * 2 + piece * 16;
        const int d = (wave & 1) * (D / 2) + i * 32 + (lane >> 1);
        vconst[i] = (((Hkv + kvh) * P) * D + d * P) * 2 + ((lane & 1) ^ ((d >> 3) & 1)) * 16;
    }
    const int pmask = P - 1;
    const int page_bytes = (int)page_stride * 2;
    const unsigned lds_k = (unsigned)(unsigned long)(__attribute__((address_space(3))) unsigned char*)smem + wave * (LP * 1024);
    const unsigned lds_v = lds_k + KBYTES;                 // (as many bytes of a tile's values before a wave's as of its keys)
    // (a tile's place, and the page of this wave's half of it; no more than the last key's page is ever asked for)
#define PAGE_OF(kk_) bt[min((kk_) + 16 * half, kmax - 1) >> log2P]
#define TILE_HALF(kk_)                                                                              \
        const int key_ = (kk_) + 16 * half, off_ = key_ & pmask;                                    \
        const bool there_ = (key_ < kmax) & ((key_ + 16 > kmin) | (key_ < kfb));
#define LOAD_TILE(kk_, page_, at_)                                                                  \
    {                                                                                               \
        TILE_HALF(kk_)                                                                              \
        const unsigned long base_ = (unsigned long)(cache + (long)(page_) * page_stride);           \
        const uint4_t rsrc_ = {(unsigned)base_, (unsigned)(base_ >> 32) & 0xffffu, there_ ? (unsigned)page_bytes : 0u, 0x00020000u}; \
        _Pragma("unroll") for (int i_ = 0; i_ < LP; ++i_) {                                         \
            if constexpr (CAP && D == 64) {   /* (these forms keep more scalars than there are registers) */ \
                QE_LOAD_TO_SHARED(lds_k + (at_) + i_ * 1024, kconst[i_], rsrc_, off_ * (D * 2), "4", ""); \
                QE_LOAD_TO_SHARED(lds_v + (at_) + i_ * 1024, vconst[i_], rsrc_, off_ * 2, "4", "");  \
            } else {                                                                                \
                QE_LOAD_TO_SHARED(lds_k + (at_) + i_ * 1024, kconst[i_], rsrc_, off_ * (D * 2), "0", ""); \
                QE_LOAD_TO_SHARED(lds_v + (at_) + i_ * 1024, vconst[i_], rsrc_, off_ * 2, "0", "");  \
            }                                                                                       \
        }                                                                                           \
    }
    // (the two steps of it through registers)
    [[maybe_unused]] uint4_t kst[LP], vst[LP];
#define FETCH_TILE(kk_, page_)                                                                      \
    {                                                                                               \
        TILE_HALF(kk_)                                                                              \
        const __amdgpu_buffer_rsrc_t rsrc_ = __builtin_amdgcn_make_buffer_rsrc(                     \
            (void*)(cache + (long)(page_) * page_stride), 0, there_ ? page_bytes : 0, 0x00020000);  \
        _Pragma("unroll") for (int i_ = 0; i_ < LP; ++i_) {                                         \
            kst[i_] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_, kconst[i_], off_ * (D * 2), 0);  \
            vst[i_] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_, vconst[i_], off_ * 2, 0);        \
        }                                                                                           \
    }
#define PUT_TILE(at_)                                                                               \
    _Pragma("unroll") for (int i_ = 0; i_ < LP; ++i_) {                                             \
        unsigned char* const to_ = smem + (at_) + wave * (LP * 1024) + i_ * 1024 + lane * 16;       \
        *(uint4_t*)to_ = kst[i_];                                                                   \
        *(uint4_t*)(to_ + KBYTES) = vst[i_];                                                        \
    }
    // waits until at most younger_ loads of the wave are in flight and its reads of shared memory are done, then for the other
    // waves; nothing is moved across
#define MEET(younger_)                                                                              \
    {                                                                                               \
        __builtin_amdgcn_sched_barrier(0);                                                          \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(younger_) : "memory");   \
        __builtin_amdgcn_sched_barrier(0);                                                          \
    }

    // The group's i-th tile holds the keys from kk0 + 32 (NG i + grp) on and uses place i % RING.
    // All groups make the same number of rounds (the barriers are the
    // block's); a round whose tile lies beyond the keys brings and computes nothing.
    // The walk's tiles: those of the kept first keys that lie wholly before the window's first tile, then
    // the tiles from the window's first on.
    const int kk0 = (kmin / 32) * 32;
    const int n_first = (kfb + 31) / 32 < kk0 / 32 ? (kfb + 31) / 32 : kk0 / 32;
    const int rounds = (n_first + (kmax - kk0 + 31) / 32 + NG - 1) / NG;
    const int gap = kk0 - 32 * n_first;
#define TILE_KEY(i_) (32 * (NG * (i_) + grp) + (NG * (i_) + grp < n_first ? 0 : gap))
    // some row of the wave sees some key of the tile, and it is a tile of this block's keys
    const int see_from = k_start - 32, see_to = wave_on ? min(k_stop, kmax) : 0;
#define SEEN(kk_) ((kk_) < see_to && ((kk_) > see_from || (kk_) < keep_first))
    bf16x8 qreg[D / 16];
    int kk_r = TILE_KEY(RING), page;                       // the tile that is asked for next, and its page
    {
        int pages[RING];
#pragma unroll
        for (int t = 0; t < RING; ++t) pages[t] = PAGE_OF(TILE_KEY(t));
        page = PAGE_OF(kk_r);
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks)
            qreg[ks] = *(const bf16x8*)(q + ((long)row * Hq + head) * D + ks * 16 + g * 8);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (DIRECT) {
            LOAD_TILE(TILE_KEY(0), pages[0], 0)
            LOAD_TILE(TILE_KEY(1), pages[1], BUF)
        }
        // Wait for q here, with an instruction the compiler sees: else it waits for these loads where q
        // is first used, inside the loop, where its count of loads in flight knows nothing of the loop's own,
        // and every round would end up waiting for the loads it has just issued.
        __builtin_amdgcn_s_waitcnt(0x0f70);                // vmcnt(0)
        if constexpr (DIRECT) {
            if (rounds > 2) {                              // (else nobody reads them)
#pragma unroll
                for (int t = 2; t < RING; ++t) LOAD_TILE(TILE_KEY(t), pages[t], t * BUF)
            }
        } else {
#pragma unroll
            for (int t = 0; t < RING - 1; ++t) {
                FETCH_TILE(TILE_KEY(t), pages[t])
                PUT_TILE(t * BUF)
            }
            FETCH_TILE(TILE_KEY(RING - 1), pages[RING - 1])
        }
    }
    // The rows of the MFMA's first operand are the tile's keys in an order in which the eight weights of a half tile that a
    // lane ends up with belong to eight neighbouring keys, 16 h + 8 g + 0 .. 7: row r is key r with its bits 2 and 3
    // exchanged.  A value fragment is then one piece of a row of V^T.
    const int kr = (r & 19) | ((r & 4) << 1) | ((r & 8) >> 1);
    const unsigned char* const k_frag = smem + kr * KROW;
    const int kx = D == 128 ? (kr & 15) : ((kr >> 1) & 7);
    const unsigned char* const v_frag = smem + KBYTES + r * 32 + ((g ^ ((r >> 3) & 1)) * 16);
    bf16x8 kf[D / 16];
    bf16x8 vf[D / 32][2];
    floatx16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.f;
#define READ_KEYS(at_)                                                                              \
    _Pragma("unroll") for (int ks = 0; ks < D / 16; ++ks) kf[ks] = *(const bf16x8*)(k_frag + (at_) + (((ks * 2 + g) ^ kx) * 16));
    // A round: the weights of tile i from its scores, on the vector units, while the fragments of its values and of
    // the next tile's keys come from shared memory; then the products of the weights and the values; and behind the barrier the scores of
    // tile i + 1, under which the loads of tile i + RING and their addresses pass.  So nothing waits for shared memory, one
    // barrier a round is enough, and two blocks on a unit fill each other's phases.  (Products and scores in turn before the barrier, the
    // loads alone behind it: 2048 tokens of 16 heads 43.2 us, 40.0; 512 rows behind 7680 keys 51.1, 48.9.)  Tiles the wave sees nothing of are
    // multiplied like the others, as zeros: with branches around the MFMAs the accumulators are copied.
    constexpr int LT = 2 * LP;                             // loads of a wave for a tile
    int at = 0, kk = TILE_KEY(0);
    bool seen = SEEN(kk);
    MEET((RING - 2) * LT)
    READ_KEYS(0)
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks], qreg[ks], s, 0, 0, 0);
    // The last round (LAST) reads nothing ahead: a walk of one tile or a few would pay for scores that nobody wants and for loads that are only
    // waited for (8 rows of 16 heads 7.5 us with the same round to the end, 6.8; 300 behind a window of 64 11.5, 10.9).
    const auto round = [&](int i, auto last) {
        constexpr bool LAST = decltype(last)::value;
        const int next = at + BUF == RING * BUF ? 0 : at + BUF;
        const int kk_1 = TILE_KEY(i + 1);
        const bool seen_1 = SEEN(kk_1);
        bf16x8 pb[2];
        if constexpr (!LAST) { READ_KEYS(next) }
        if (!seen) {                                       // (a tile that the wave sees nothing of adds nothing; without a branch around the MFMAs)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                pb[h] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                for (int db = 0; db < D / 32; ++db) vf[db][h] = pb[h];
            }
        } else {
#pragma unroll
            for (int db = 0; db < D / 32; ++db)
#pragma unroll
                for (int h = 0; h < 2; ++h) vf[db][h] = *(const bf16x8*)(v_frag + at + (h * D + db * 32) * 32);
            __builtin_amdgcn_sched_barrier(0);
            if (CAP) {
#pragma unroll
                for (int e = 0; e < 16; ++e) s[e] = soft_capped(s[e] * cap_in, cap_out);
            }
            // (the scores stay unscaled: the scale is positive, so it is applied to the maximum, and
            // to each score by the multiply-add that also subtracts the maximum)
            float tmax = -INFINITY;
            if ((kk >= all_lo || kk + 32 <= keep_first) && kk + 32 <= all_hi) {   // every column sees every key of the tile
#pragma unroll
                for (int e = 0; e < 16; ++e) tmax = fmaxf(tmax, s[e]);
            } else {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int key = kk + 16 * (e >> 3) + 8 * g + (e & 7);
                    s[e] = ((key >= lo || key < keep_first) && key < hi) ? s[e] : -INFINITY;
                    tmax = fmaxf(tmax, s[e]);
                }
            }
            tmax = max_of_both_halves(tmax) * scale_log2;
            // m is the reference the weights are taken against, not the exact maximum: a column moves
            // it only when a score exceeds it by more than 8 (a weight above 2^8), which after the
            // first tiles is rare, so that the accumulators are seldom rescaled.  The decision is the
            // column's own: its sums do not depend on the other columns of the wave.  (A single new token's is the exact maximum,
            // as in the decode kernel: its largest weight is then 1 and not rounded, without which it errs by a tenth to a third more.)
            const bool moves = tmax > m + slack;               // (never for a tile without a visible key)
            if (__any(moves)) {
                const float alpha = moves ? __builtin_amdgcn_exp2f(m - tmax) : 1.f;   // 0 from a column's first keys
                m = moves ? tmax : m;
                l *= alpha;
#pragma unroll
                for (int db = 0; db < D / 32; ++db) acc[db] *= alpha;
            }
            const float ref = (m == -INFINITY) ? 0.f : m;      // a column that has seen no key yet: all weights 0
            float psum = 0.f;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float pe = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], scale_log2, -ref));   // 0 for keys that are not seen
                psum += pe;
                pb[e >> 3][e & 7] = (__bf16)pe;
            }
            l += psum;
            if (kk < kmin || kk + 32 > kmax) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    unsigned keep[4];
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const int key = kk + 16 * h + 8 * g + e;
                        const unsigned on = (key >= kmin || key < kfb) && key < kmax ? 0xffffu : 0u;
                        keep[e / 2] = e % 2 ? keep[e / 2] | on << 16 : on;
                    }
#pragma unroll
                    for (int db = 0; db < D / 32; ++db) {
                        uint4_t pv = __builtin_bit_cast(uint4_t, vf[db][h]);
#pragma unroll
                        for (int e = 0; e < 4; ++e) pv[e] &= keep[e];
                        vf[db][h] = __builtin_bit_cast(bf16x8, pv);
                    }
                }
            }
        }
        if constexpr (!DIRECT && !LAST) {                  // (to the place of the tile before this one)
            PUT_TILE(at == 0 ? (RING - 1) * BUF : at - BUF)
            FETCH_TILE(kk_r, page)
        }
#pragma unroll
        for (int u = 0; u < D / 16; ++u)
            acc[u % (D / 32)] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[u % (D / 32)][u / (D / 32)], pb[u / (D / 32)],
                                                                        acc[u % (D / 32)], 0, 0, 0);
        if constexpr (!LAST) {
            MEET((RING - 3) * LT)
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] = 0.f;
            if constexpr (DIRECT) LOAD_TILE(kk_r, page, at)    // the place was read for the last time before the last barrier
#pragma unroll
            for (int ks = 0; ks < D / 16; ++ks) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[ks], qreg[ks], s, 0, 0, 0);
            kk_r = TILE_KEY(i + RING + 1);
            page = PAGE_OF(kk_r);
            at = next;
            kk = kk_1;
            seen = seen_1;
        }
    };
    for (int i = 0; i + 1 < rounds; ++i) round(i, std::false_type());
    round(rounds - 1, std::true_type());
    MEET(0)                                                // (what was asked for beyond the end arrives too, before the memory is used again)
#undef LOAD_TILE
#undef FETCH_TILE
#undef PUT_TILE
#undef TILE_HALF
#undef PAGE_OF
#undef MEET
#undef TILE_KEY
#undef SEEN
#undef READ_KEYS
    l = sum_of_both_halves(l);
    if (NG == 2) {
        // group 1 hands its maxima, sums and accumulators to group 0, 16 values of every lane at a
        // time, through the staging memory (free after the loop's last barrier): [wave][value][lane]
        float* xch = (float*)smem_all + wave * 18 * 64 + lane;
        float a_own = 1.f, a_other = 0.f;
        if (grp == 1) { xch[0] = m; xch[64] = l; }
        __syncthreads();
        if (grp == 0) {
            const float m1 = xch[0], l1 = xch[64];
            const float mt = fmaxf(m, m1);
            const float ref = (mt == -INFINITY) ? 0.f : mt;
            a_own = __builtin_amdgcn_exp2f(m - ref);       // 0 for a side that has seen no key
            a_other = __builtin_amdgcn_exp2f(m1 - ref);
            l = l * a_own + l1 * a_other;
            m = mt;
        }
#pragma unroll
        for (int db = 0; db < D / 32; ++db) {
            if (grp == 1) {
#pragma unroll
                for (int e = 0; e < 16; ++e) xch[(2 + e) * 64] = acc[db][e];
            }
            __syncthreads();
            if (grp == 0) {
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[db][e] = acc[db][e] * a_own + xch[(2 + e) * 64] * a_other;
            }
            __syncthreads();
        }
        if (grp == 1) return;
    }
    if (partial) {
        // as the lanes hold them: [segment][block][wave][value][lane], value = m, l, then the accumulators
        constexpr int NV = 2 + (D / 32) * 16;
        float* dst = part + ((((long)bseg * gridDim.x + bhead) * gridDim.z + bgroup) * 4 + wave) * NV * 64 + lane;
        dst[0] = m;
        dst[64] = l;
        if (m != -INFINITY) {                              // (a column that saw no key of the segment: nothing else is read of it)
#pragma unroll
            for (int db = 0; db < D / 32; ++db)
#pragma unroll
                for (int e = 0; e < 16; ++e) dst[(2 + db * 16 + e) * 64] = acc[db][e];
        }
        return;
    }
    // (sink: one more entry that carries no value; m is the scaled reference of the weights)
    if (sink) l += __builtin_amdgcn_exp2f(fminf(tail.sink_of(head) * 1.4426950408889634f - m, 126.f));
    if (col_ok) store_columns<D>(out, acc, 1.f / l, row, head, g, tail);
}

// The segments' partial results of the blocks that left some: the same first two grid dimensions
// and the same lanes as the kernel above, the third dimension being the block of 32 features;
// lane by lane, in the order of the segments.
template <int D>
__global__ __launch_bounds__(256) void attention_prefill_merge_kernel(
    const float* __restrict__ part, bf16_t* __restrict__ out, const int* __restrict__ tiles,
    const int* __restrict__ positions, int Hq, int Hkv, int window, int R, int seg_param, int keys_row, AttnTail tail) {
    constexpr int NV = 2 + (D / 32) * 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 5, r = lane & 31;
    const int G = Hq / Hkv, GH = 32 / R;
    const int bhead = blockIdx.x, db = blockIdx.y, bgroup = blockIdx.z;     // (head waves, feature blocks, tile groups)
    const int kvh = bhead / (G / GH);
    const int head = kvh * G + (bhead % (G / GH)) * GH + r / R;
    const int* bt4 = tiles + 8 * (gridDim.z - 1 - bgroup);
    if (bt4[1] <= 0) return;
    const int row_first = bt4[0];
    int last = 0;
#pragma unroll
    for (int j = 1; j < 4; ++j) if (bt4[2 * j + 1] > 0) last = j;
    const int p_block = positions[row_first];
    const int kmin = first_seen_key(p_block, window);
    const int kmax = positions[bt4[2 * last]] + bt4[2 * last + 1];
    const int seg_keys = segment_keys(seg_param, positions, keys_row);
    if (seg_keys <= 0) return;                             // nothing was cut
    const int z_lo = kmin / seg_keys, z_hi = (kmax - 1) / seg_keys;
    if (z_hi <= z_lo) return;                              // the block wrote its result itself
    const int row0 = bt4[2 * wave], cnt = bt4[2 * wave + 1];
    const int rr = r % R;
    if (cnt <= 0 || rr >= cnt) return;
    const int row = row0 + rr;
    const long zstride = (long)gridDim.x * gridDim.z * 4 * NV * 64;
    const float* src = part + (((long)bhead * gridDim.z + bgroup) * 4 + wave) * NV * 64 + lane;
    // Four segments are asked for at once, their accumulators without waiting for the maxima (those of a segment of which the column saw
    // no key were never written and are not used; a segment beyond the last is the last again).  One after the other, with a trip
    // to memory for each of its loops' rounds, four segments of 512 rows of 16 heads took 8.0 us,
    // now 6.7.
    constexpr int AT = 4;
    float ms[AT], ls[AT], as[AT][16];
    const auto ask = [&](int z0) {
#pragma unroll
        for (int k = 0; k < AT; ++k) {
            const float* at = src + min(z0 + k, z_hi) * zstride;
            ms[k] = at[0];
            ls[k] = at[64];
#pragma unroll
            for (int e = 0; e < 16; ++e) as[k][e] = at[(2 + db * 16 + e) * 64];
        }
    };
    ask(z_lo);
    float M = -INFINITY;
#pragma unroll
    for (int k = 0; k < AT; ++k) M = fmaxf(M, ms[k]);
    for (int z = z_lo + AT; z <= z_hi; ++z) M = fmaxf(M, src[z * zstride]);
    float l = 0.f;
    floatx16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.f;
    for (int z = z_lo; z <= z_hi; z += AT) {
        if (z > z_lo) ask(z);
#pragma unroll
        for (int k = 0; k < AT; ++k) {
            if (z + k > z_hi || ms[k] == -INFINITY) continue;
            const float wgt = __builtin_amdgcn_exp2f(ms[k] - M);
            l += wgt * ls[k];
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[e] += wgt * as[k][e];
        }
    }
    const float inv = 1.f / l;
    bf16_t* orow = out + (long)row * tail.out_stride + (long)head * D + 4 * g + db * 32;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        bf16x4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = (__bf16)(acc[4 * b + j] * inv);
        if (tail.plain) *(bf16x4*)(orow + 8 * b) = o;
        else
#pragma unroll
            for (int j = 0; j < 4; ++j) tail.store(out, row, head, db * 32 + 8 * b + 4 * g + j, acc[4 * b + j] * inv);
    }
}

// The tile list of qe_attention_prefill from the step's portions, made on the device (a recorded step
// does not know its portions' lengths on the host): portions [n_portions][2] = (first row, rows), each
// cut into tiles of at most `rows_per_tile` rows in groups of four, a group filled up with tiles of no
// rows; the list is filled up to max_groups groups with groups of no rows.  The step's first `singles` rows, each of a
// request of its own, are a group each before those.  One thread per group.
__global__ void prefill_tiles_kernel(const int* __restrict__ portions, int n_portions, int rows_per_tile,
                                     int* __restrict__ tiles, int max_groups, int singles) {
    int grp = blockIdx.x * blockDim.x + threadIdx.x;
    if (grp >= singles + max_groups) return;
    if (grp < singles) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            tiles[8 * grp + 2 * j] = grp;
            tiles[8 * grp + 2 * j + 1] = j == 0;
        }
        return;
    }
    grp -= singles;
    tiles += 8 * singles;
    int first = 0, start = 0, rows = 0, in_portion = -1;   // which portion the group lies in, and the group's place in it
    for (int i = 0; i < n_portions; ++i) {
        const int n = portions[2 * i + 1];
        const int groups = n > 0 ? (n + 4 * rows_per_tile - 1) / (4 * rows_per_tile) : 0;
        if (in_portion < 0 && grp < first + groups) {
            in_portion = grp - first;
            start = portions[2 * i];
            rows = n;
        }
        first += groups;
    }
    int* out = tiles + 8 * grp;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = in_portion < 0 ? rows : (4 * in_portion + j) * rows_per_tile;    // rows before this tile in its portion
        const int cnt = in_portion < 0 || r >= rows ? 0 : min(rows_per_tile, rows - r);
        out[2 * j] = cnt > 0 ? start + r : start;
        out[2 * j + 1] = cnt;
    }
}

int qe_attention_prefill_tiles(const int* portions, int n_portions, int rows_per_tile, int* tiles, int max_groups,
                               int singles, hipStream_t stream) {
    QE_REQUIRE(portions && tiles && n_portions >= 1 && n_portions <= 64 && rows_per_tile >= 1 && max_groups >= 1 && singles >= 0,
               "prefill tiles: %d portions, tiles of %d rows, %d groups, %d single rows", n_portions, rows_per_tile, max_groups, singles);
    prefill_tiles_kernel<<<qe_cdiv(singles + max_groups, 64), 64, 0, stream>>>(portions, n_portions, rows_per_tile, tiles, max_groups, singles);
    QE_LAUNCH_CHECK();
    return 0;
}

// Rows per tile for a model's head counts: 32 / (heads that one wave serves).
int qe_attention_prefill_tile_rows(int Hq, int Hkv) {
    const int G = Hq / Hkv;
    const bool pow2 = G > 0 && (G & (G - 1)) == 0 && G <= 32;
    return 32 / (pow2 ? G : 1);
}

// How the keys of a call are best cut into segments: 0 (not at all) or the keys a segment (a multiple
// of 64).  blocks: blocks of the grid without segments; max_keys: the most keys a row of the call
// sees.  Every segment costs a trip of the partial results through memory, and more blocks than
// compute units gained nothing where it was measured (a whole prompt of 1536 or 2048 tokens took
// longer in two segments than in one), so there are only as many segments as fill the chip, of at
// least 512 keys; up to QE_PREFILL_UNCUT_KEYS keys a walk is too short to be worth one.
int qe_attention_prefill_uncut_keys() { return QE_PREFILL_UNCUT_KEYS; }

int qe_attention_prefill_segments(long blocks) {
    const int units = qe_compute_units();
    if (blocks <= 0 || blocks > units / 2) return 1;
    const long ks = units / blocks;                        // as many blocks as there are compute units, not more
    return ks > 8 ? 8 : (int)ks;
}

int qe_attention_prefill_segment_keys(long blocks, int max_keys) {
    const int ks = qe_attention_prefill_segments(blocks);
    const int seg = prefill_segment_length(max_keys, ks);
    return seg >= max_keys ? 0 : seg;
}

// Wave groups a block: two where the blocks do not fill the compute units anyway, and up to twice as many blocks as units where the
// longest walk decides: one prompt from its start, or several beside one that is as long as they together.  (rows: 32 a tile, those
// that fill a tile up among them.  One group and two, 32 heads of 128 on 8: 2048 rows from the start 64 and 58 us, 16 prompts of 128 rows
// 18 and 25, four of 512 31 and 36, 512 rows each behind 4096 keys 185 and 189; 16 heads on 8, 4096 rows 134 and 109, eight prompts of
// 256 beside one of 2000 63 and 52, the same behind 4096 keys 195 and 215; 64 heads, 1000 rows 37 and 39.)
int qe_attention_prefill_choose_groups(long blocks, long rows, int window, int max_keys) {
    const int units = qe_compute_units();
    if (blocks <= units) return 2;
    return blocks <= 2L * units && window == 0 && max_keys >= 1536 && 5L * max_keys >= 2 * rows && 4L * max_keys <= 5 * rows ? 2 : 1;
}

size_t qe_attention_prefill_workspace(int num_tiles, int Hq, int Hkv, int D, int segments) {
    const int R = qe_attention_prefill_tile_rows(Hq, Hkv);
    const long blocks = (long)(num_tiles / 4) * Hkv * ((Hq / Hkv) / (32 / R));
    return (size_t)segments * blocks * 4 * (2 + (D / 32) * 16) * 64 * sizeof(float);
}

// tiles: num_tiles pairs (first row of q, number of rows <= qe_attention_prefill_tile_rows), in
// groups of four that belong to one request, in ascending rows, with consecutive positions
// through the group; a group is filled up with pairs of 0 rows.  num_tiles is a multiple of 4.
// seg_keys: 0; or the keys of a segment (a multiple of 64) with max_keys, the most keys a row sees; or,
// for a caller that does not know the positions, minus the number of segments (at most 8) into which
// the keys of row keys_row, which sees the most, are to be cut.  The workspace has
// qe_attention_prefill_workspace(..., segments) bytes.  singles: the first so many groups are single new tokens.
int qe_attention_prefill(const void* q, void* out, const void* cache, const int* tiles, int num_tiles,
                         const int* positions, const int* tok_seq, const int* block_table, int max_blocks,
                         int Hq, int Hkv, int D, int P, float scale, int window, int groups,
                         int seg_keys, int max_keys, int keys_row, void* workspace, size_t workspace_bytes,
                         hipStream_t stream, int keep_first, int sink, float softcap, int singles, const AttnTail& tail) {
    QE_REQUIRE(seg_keys == 0 || (keep_first == 0 && !sink),
               "prefill attention: kept first keys and a sink go with uncut walks only");
    QE_REQUIRE(singles >= 0 && (singles == 0 || softcap == 0.f), "prefill attention: %d single tokens, which go without a soft cap", singles);
    QE_REQUIRE((D == 64 || D == 128) && P >= 16 && (P & (P - 1)) == 0 && Hq % Hkv == 0,
               "prefill attention: sizes not taken");
    int log2P = 0;
    while ((1 << log2P) < P) ++log2P;
    QE_REQUIRE(num_tiles % 4 == 0, "prefill attention: tiles come in groups of four");
    QE_REQUIRE(4L * Hkv * P * D < (1L << 31), "prefill attention: a page of %ld bytes is too large", 4L * Hkv * P * D);
    if (num_tiles == 0) return 0;
    const int R = qe_attention_prefill_tile_rows(Hq, Hkv);
    const int waves_per_kv = (Hq / Hkv) / (32 / R);
    int segments = 1;
    if (seg_keys > 0) {
        QE_REQUIRE(seg_keys % 64 == 0 && max_keys > 0, "prefill attention: segments of %d keys (a multiple of 64), %d keys", seg_keys, max_keys);
        segments = qe_cdiv(max_keys, seg_keys);
        QE_REQUIRE(segments <= 64, "prefill attention: %d segments", segments);
        if (segments <= 1) { seg_keys = 0; segments = 1; }
    } else if (seg_keys < 0) {
        segments = -seg_keys;
        QE_REQUIRE(segments <= 8 && keys_row >= 0, "prefill attention: %d segments of the keys of row %d", segments, keys_row);
        if (segments == 1) seg_keys = 0;
    }
    if (segments > 1)
        QE_REQUIRE(workspace && workspace_bytes >= qe_attention_prefill_workspace(num_tiles, Hq, Hkv, D, segments),
                   "prefill attention: workspace of %zu bytes is too small", workspace_bytes);
    QE_REQUIRE(num_tiles / 4 <= 65535, "prefill attention: %d tiles are too many for one launch", num_tiles);
    dim3 grid(Hkv * waves_per_kv, segments, num_tiles / 4);
    dim3 mgrid(Hkv * waves_per_kv, D / 32, num_tiles / 4);
    const float scale_log2 = softcap > 0.f ? 1.f : scale * 1.4426950408889634f;
    const float cap_in = softcap > 0.f ? scale * 2.f * 1.4426950408889634f / softcap : 0.f, cap_out = softcap * 1.4426950408889634f;
    if (groups == 0) groups = qe_attention_prefill_choose_groups((long)grid.x * grid.z, (long)num_tiles * R, window, max_keys);
    QE_REQUIRE(groups == 1 || groups == 2, "prefill attention: %d groups a block", groups);
    // (a cache may begin at any element of a larger buffer)
    const bool direct = ((unsigned long)cache & 15) == 0;
#define QE_PREFILL_FORM(D_, NG_, CAP_, DIRECT_, SINGLES_)                                                     \
    {                                                                                               \
        constexpr int shmem_ = NG_ * RING * 2 * 32 * D_ * 2;                                       \
        QE_RAISE_SHARED((attention_prefill_kernel<D_, NG_, CAP_, DIRECT_, SINGLES_>), shmem_);      \
        attention_prefill_kernel<D_, NG_, CAP_, DIRECT_, SINGLES_><<<grid, 256 * NG_, shmem_, stream>>>(      \
        (const bf16_t*)q, (bf16_t*)out, (const bf16_t*)cache, tiles, positions, tok_seq, block_table, \
        max_blocks, Hq, Hkv, P, log2P, scale_log2, window, R, seg_keys, keys_row, (float*)workspace, keep_first, sink, \
        cap_in, cap_out, singles, tail);                                                            \
    }
#define QE_PREFILL_CAP(D_, NG_, CAP_, S_) { if (direct) QE_PREFILL_FORM(D_, NG_, CAP_, true, S_) else QE_PREFILL_FORM(D_, NG_, CAP_, false, S_) }
#define QE_PREFILL(D_, NG_) do { if (softcap > 0.f) QE_PREFILL_CAP(D_, NG_, true, false) else if (singles) QE_PREFILL_CAP(D_, NG_, false, true) else QE_PREFILL_CAP(D_, NG_, false, false) } while (0)
    if (D == 128) { if (groups == 2) QE_PREFILL(128, 2); else QE_PREFILL(128, 1); }
    else          { if (groups == 2) QE_PREFILL(64, 2); else QE_PREFILL(64, 1); }
#undef QE_PREFILL
#undef QE_PREFILL_CAP
#undef QE_PREFILL_FORM
    if (seg_keys != 0) {
        if (D == 128)
            attention_prefill_merge_kernel<128><<<mgrid, 256, 0, stream>>>((const float*)workspace, (bf16_t*)out, tiles,
                                                                           positions, Hq, Hkv, window, R, seg_keys, keys_row, tail);
        else
            attention_prefill_merge_kernel<64><<<mgrid, 256, 0, stream>>>((const float*)workspace, (bf16_t*)out, tiles,
                                                                          positions, Hq, Hkv, window, R, seg_keys, keys_row, tail);
    }
    QE_LAUNCH_CHECK();
    return 0;
}
