// The layers of a step of single new tokens in one launch (pre-norm blocks: norm, q|k|v, attention over the paged cache, output
// product, norm, gate|up, down; bfloat16, heads of 128).
//
// What bounds such a step is not its bytes but the chain of its kernels: six a layer, each of which waits for the last block of the one
// before, starts its blocks, asks for its weights and has them 1.5 us later, for some 5 us in the mean (16 heads of 128, width 1024).
// Here a block a compute unit stays for all layers.  The blocks hand their few numbers on through memory (1.65 us from one product to
// the next with nothing else on the way, about what a dependent kernel costs before its first load), and the weights and keys of what comes next
// travel meanwhile:
//
//   * Eight of a block's waves (the feeding ones) ask for what the step reads once, in the order in which it will be used and
//     whatever layer it belongs to, straight to rings in shared memory, and multiply it.
//   * Four (the waiting ones) read what the other blocks publish, norm it, leave it in shared memory as the products' operand, and
//     publish the products' results.
//
// A step of 28 layers (16 heads of 128 on 8, width 1024), logits and all, with six kernels a layer and so, in us: one request at 64 keys
// 919, 600; at 2000 922, 643; at 8192 1129, 784; four at 128 1070, 757; eight at 1024 1324, 1128; at 4000 1746, 1586; at 12288 3310, 2967.  Of six
// layers of width 4096 with 12288 in the middle, at 512 keys, one request 873, 715, two 878, 744.  What is left above the bytes is the waiting: with
// the same kilobyte asked for again and again in the place of all weights and keys, a layer (of the first model) takes 14.5 us instead of 16.3 with one
// request at 64 keys, 14.9 instead of 17.2 at 2040, and eight at 4000 take 35.5 instead of 50.7.  A look for numbers stands behind the
// kilobytes that its compute unit has asked for before.
//
// A number that is not there yet is told by its bits: every place of the exchange holds ~0 (a NaN that no result has: a result of these
// bits is published as another NaN) until its one writer fills it, and every reader asks until nothing is ~0.  So nothing beyond the
// numbers themselves is waited for: no counter that all blocks add to, no second trip for a flag.  A place is written once a launch (an
// earlier launch on the stream has filled the exchange with ~0), but for the parts of the attention, of which each has one
// reader, which puts ~0 back; they lie in two sets, layer by layer in turn: a set is written again only after all of the layer between is
// published, and a reader of it has published there behind its ~0.
//
// No block waits for one that is not running: which blocks take part is settled at the start by a roll call, and the
// work is dealt out among those.  Every wait has an end: at its limit a wave takes NaN for what has not come, which makes the rows NaN, and says so
// in a word of the host's memory (`late`), which whoever takes the results looks at.
//
// The sums of a product have one order, whatever the number of rows and blocks: K goes to the eight waves in chunks of 128 dealt out in turn, whose
// sums are added in the order of the waves.  A token's keys are cut in segments that follow its own position (segment_keys).
#include "attention_tile.h"
#include <type_traits>

namespace {

constexpr int FEED = 8, WAIT = 4, THREADS = (FEED + WAIT) * 64;
constexpr int D = 128;
constexpr int MAX_LAYERS = 40;         // of one launch: what 4 KB of arguments hold
constexpr int MAX_ROWS = 8;
constexpr int MAX_GROUP = 8;
constexpr int MAX_SEGMENTS = 32;       // a token's keys are cut in
constexpr unsigned NONE = ~0u;
constexpr unsigned A_NAN = 0x7fc07fc0u;                    // as a float and as two bfloat16
constexpr unsigned CLOSED = 0x80000000u;
constexpr unsigned GAP = 1000000u;                         // of the 100 MHz clock: 10 ms
constexpr unsigned long CALL = 5000ul;                     // 50 us
constexpr unsigned long KILOBYTE = 5ul;                    // 50 ns: what a block takes for one by itself (10 to 29 GB/s a block with 1 to 32 blocks)

typedef unsigned u4 __attribute__((ext_vector_type(4)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));

struct ChainLayer {
    const bf16_t *w_qkv, *w_o, *w_gu, *w_down;
    const float *norm1, *norm2, *q_norm, *k_norm;
    bf16_t* cache;
    float eps1, eps2;
};

struct ChainArgs {
    ChainLayer layer[MAX_LAYERS];
    float* h;
    const int *positions, *tok_seq, *table, *slots, *shared_keys;
    const float* rope;
    unsigned* work;
    float scale, qk_eps;
    int layers, M, H, Hq, Hkv, I, logP, max_blocks, segments, max_position;
    int* late;                         // host memory, or null: 1 once a wait has been given up
    unsigned limit;                    // of a wait, in ticks of the 100 MHz clock
    long layer_bytes;                  // of a layer's matrices
    int absent;                        // blocks that the roll call counts beside those that come
};

// How long something has been waited for.  The clock also runs while the device has set the whole queue aside for another process, so a gap
// between two looks counts as GAP at most: what is waited for stood still as well.
struct Waited {
    unsigned ticks = 0;
    unsigned long last = 0;
    __device__ __forceinline__ unsigned look() {
        const unsigned long t = __builtin_amdgcn_s_memrealtime();
        if (last) ticks += (unsigned)min(t - last, (unsigned long)GAP);
        last = t;
        return ticks;
    }
};

// The exchange, in words from its start: the roll call's, the attention's parts (two sets), then a layer's numbers, layer after layer.
// A part is a quarter of a head's features of one segment with the segment's maximum and sum: PART words.
constexpr int PART = 36;

struct Exchange {
    unsigned parts, set, layers, per_layer, qkv, att, act, x1, x2, total;
    __host__ __device__ Exchange(int M, int H, int Hq, int Hkv, int I, int segments, int n_layers) {
        parts = 64;
        set = (unsigned)M * Hq * segments * 4 * PART;
        layers = parts + 2 * set;
        qkv = 0;
        att = qkv + (unsigned)M * (Hq + 2 * Hkv) * (D / 2);
        act = att + (unsigned)M * Hq * (D / 2);
        x1 = act + (unsigned)M * (I / 2);
        x2 = x1 + (unsigned)M * H;
        per_layer = x2 + (unsigned)M * H;
        total = layers + per_layer * n_layers;
    }
};

// A token's keys are cut in segments by its own position alone, so that its sums, and its bits, are the same alone and in company: of 128 keys, a
// tile for each feeding wave, up to 20 of them; from 2560 keys on of 256, up to 32; then of as many 128s as make 32 at most.  More and
// smaller segments suit one row, which has the chip to itself, fewer and larger ones eight, whose units are several a block (us a step of 28 layers,
// width 1024 with 8 key/value heads, segments of 128 and of 256: at 2100 keys one row 648, 694, two 782, 770, four 978, 1005, eight 1327, 1332; at 2600
// one 663, 701, two 793, 783, four 1000, 1015, eight 1417, 1353; at 3900 one 683, 708, eight 1659, 1572.  us a layer, at 16000: 512 and 1024 keys, one
// row 31.1, 39, eight 117, 116).
__host__ __device__ constexpr int segment_keys(int p) { return 128 * (p < 2560 ? 1 : p < 8192 ? 2 : p / 4096 + 1); }

// A unit of the attention: the cached keys [lo, hi) of one segment for one row and key/value head; own: the token's own key belongs to it.
struct Unit { int m, kvh, seg, lo, hi, tiles, own; };

__device__ __forceinline__ u4 rsrc_of(const void* p, unsigned bytes) {
    const unsigned long b = (unsigned long)p;
    return u4{(unsigned)b, (unsigned)(b >> 32) & 0xffffu, bytes, 0x00020000u};
}

__device__ __forceinline__ unsigned published(unsigned bits) { return bits == NONE ? A_NAN : bits; }
__device__ __forceinline__ unsigned published(float v) { return published(__float_as_uint(v)); }
__device__ __forceinline__ unsigned pair_bits(float a, float b) {
    return (unsigned)float_to_bf16(a).bits | (unsigned)float_to_bf16(b).bits << 16;
}

// the same number in all lanes, told to the compiler
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <typename T>
__device__ __forceinline__ const T* uniform(const T* p) {
    const unsigned long v = (unsigned long)p;
    return (const T*)((unsigned long)(unsigned)uniform((int)(v >> 32)) << 32 | (unsigned)uniform((int)v));
}

__device__ __forceinline__ Unit uniform(const Unit& r) {
    return Unit{uniform(r.m), uniform(r.kvh), uniform(r.seg), uniform(r.lo), uniform(r.hi), uniform(r.tiles), uniform(r.own)};
}

// What every wave knows of the step's rows.
struct Rows {
    int pos[MAX_ROWS], slot[MAX_ROWS], table[MAX_ROWS], shared[MAX_ROWS];
    int first[MAX_ROWS + 1];           // the row's first unit of the attention
    int keys[MAX_ROWS], segments[MAX_ROWS];                // a segment's keys; how many segments
};

__device__ __forceinline__ void unit_ends(Unit& r, const Rows& rows) {
    const int pos = uniform(rows.pos[r.m]), keys = uniform(rows.keys[r.m]);
    r.lo = r.seg * keys;
    r.hi = min(r.lo + keys, pos);
    r.tiles = (max(0, r.hi - r.lo) + 15) >> 4;
    r.own = pos < r.lo + keys;
}
// the u-th: row by row, in a row head by head, in a head segment by segment
__device__ __forceinline__ Unit unit_at(const Rows& rows, int M, int u) {
    Unit r;
    r.m = 0;
    while (r.m + 1 < M && u >= rows.first[r.m + 1]) ++r.m;
    const int at = u - rows.first[r.m];
    r.kvh = at / rows.segments[r.m];
    r.seg = at - r.kvh * rows.segments[r.m];
    unit_ends(r, rows);
    return r;
}
// the one behind it, of which there has to be one
__device__ __forceinline__ void unit_next(Unit& r, const Rows& rows, int Hkv) {
    if (++r.seg == uniform(rows.segments[r.m])) {
        r.seg = 0;
        if (++r.kvh == Hkv) {
            r.kvh = 0;
            ++r.m;
        }
    }
    unit_ends(r, rows);
}

#define BLOCK_BARRIER()                                    \
    do {                                                   \
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); \
        __builtin_amdgcn_s_barrier();                      \
        asm volatile("" ::: "memory");                     \
    } while (0)

// The block's share of the work: from the first to before the last of a product's fours of outputs, of the attention's units.
struct Share { int qkv0, qkv1, out0, out1, act0, act1, unit0, unit1; };
// A wave's tile of keys: the page (with the sign bit for keys that other requests read too) and the place in it.
struct Tile { int page, place; };
constexpr int TILES = 32;              // that shared memory holds of a wave's

// What a feeding wave asks for, kilobyte by kilobyte: in a layer the chunks of K of its fours of rows of q|k|v, its tiles (four kilobytes
// of keys, four of values), its fours of output, gate|up and down rows, then the next layer's.  Where they lie is worked out for up to 64 of them at
// once, a lane each, so that asking takes a dozen instructions: for a whole layer if it has no more, and then once for all layers but for
// the operands' addresses; else for a stage or a part of it.
// PAIRS: of gate|up, the fours of outputs of one round: first their gates, then their ups.
template <int RING, int PAIRS>
struct Feed {
    int row, piece, keys, values;                          // a lane's place in four rows of a matrix (the row, the byte in it), in a tile of keys, of values
    int wave, logP;
    unsigned to;                                           // the ring's place in shared memory
    int tiles;                                             // the wave's in a layer
    int total;                                             // a layer's kilobytes
    int layer = 0, stage = 0, first = 0, next = 0, window = 0, slot = 0;    // the window's stage, its first kilobyte in that, the one that is asked for next, how many
    unsigned lo, hi;                                       // a lane's: where its kilobyte lies
    int kind;                                              // 0: of a matrix, with the bytes of a row; 1: of keys, with the pieces' exchange; 2: of values.  4: not streamed
    unsigned rel_lo, rel_hi;                               // of a whole layer: where in the operand, and which
    int which;

    __device__ __forceinline__ static int chunks_of(int K, int wave) { return K / 128 > wave ? (K / 128 - wave + FEED - 1) / FEED : 0; }
    __device__ __forceinline__ static Tile tile_at(const int* table, int max_blocks, int row, int key, int kvh, bool shared, int logP) {
        return Tile{table[(long)row * max_blocks + (key >> logP)] | (shared ? (int)0x80000000 : 0), kvh << (logP + 8) | (key & ((1 << logP) - 1))};
    }
    __device__ __forceinline__ static Tile tile_of(const int* table, int max_blocks, const Rows& rows, const Unit& un, int t, int logP) {
        return tile_at(table, max_blocks, rows.table[un.m], un.lo + t * 16, un.kvh, un.lo < rows.shared[un.m], logP);
    }
    // how many kilobytes stage s has
    template <typename Args>
    __device__ __forceinline__ int count_of(int s, const Args& a, const Share& share) const {
        if (s == 1) return tiles * 8;
        const int at = s == 0 ? 0 : s == 3 ? 4 : 2, n = uniform((&share.qkv0)[at + 1]) - uniform((&share.qkv0)[at]);
        return (s == 3 ? 2 * n : n) * chunks_of(s == 2 ? a.Hq * D : s == 4 ? a.I : a.H, wave);
    }
    // a lane's: where the x-th kilobyte of stage s (the same in all lanes) lies in its operand
    template <typename Args>
    __device__ __forceinline__ unsigned long place(int s, int x, int& of_kind, const Args& a, const Share& share, const Rows& rows, const Tile* held) const {
        if (s == 1) {
            const int t = x >> 3, part = x & 7;
            Tile mine = held[min(max(t, 0), TILES - 1)];
            if (tiles > TILES) {                           // (more than shared memory holds: its unit is found again)
                int before = 0, key = 0, row = 0, kvh = 0, shared = 0;
                const int units = uniform(share.unit1) - uniform(share.unit0);
                Unit un = unit_at(rows, a.M, uniform(share.unit0));
                for (int i = 0; i < units; ++i) {
                    if (i > 0) unit_next(un, rows, a.Hkv);
                    const int count = un.tiles > wave ? (un.tiles - wave + FEED - 1) / FEED : 0;
                    const bool here = t >= before && t < before + count;
                    key = here ? un.lo + (wave + (t - before) * FEED) * 16 : key;
                    row = here ? uniform(rows.table[un.m]) : row;
                    kvh = here ? un.kvh : kvh;
                    shared = here ? un.lo < uniform(rows.shared[un.m]) : shared;
                    before += count;
                }
                mine = tile_at(a.table, a.max_blocks, row, key, kvh, shared, logP);
            }
            const int inside = mine.place & ((1 << logP) - 1), head = mine.place - inside;
            of_kind = (part < 4 ? (part << 6) << 3 | 1 : 2) | (mine.page < 0 ? 4 : 0);
            return (unsigned long)(mine.page & 0x7fffffff) * (unsigned)(4 * a.Hkv * D << logP) +
                   (unsigned)(head + (part < 4 ? inside * (D * 2) + part * 1024 : (a.Hkv << (logP + 8)) + inside * 2 + (((part - 4) * 64) << logP)));
        }
        const int K = s == 2 ? a.Hq * D : s == 4 ? a.I : a.H, K2 = K * 2, chunks = max(1, chunks_of(K, wave));
        int four = x, c = 0;
        if (chunks > 1) {                                  // (numbers far below 2^20: the quotient is exact)
            four = (int)(((float)x + 0.5f) * __builtin_amdgcn_rcpf((float)chunks));
            c = x - four * chunks;
        }
        int at = 4 * (uniform(s == 0 ? share.qkv0 : share.out0) + four);
        if (s == 3) {
            const int round = four / (2 * PAIRS), in = four & (2 * PAIRS - 1), pair0 = uniform(share.act0) + round * PAIRS;
            const int pairs = min(PAIRS, uniform(share.act1) - pair0), up = in >= pairs, pair = pair0 + in - (up ? pairs : 0);
            at = (pair >> 3) * 64 + (pair & 7) * 4 + up * 32;
        }
        of_kind = K2 << 3;
        return (unsigned)at * (unsigned)K2 + (unsigned)(wave * 256 + c * (FEED * 256));
    }
    // the next window: from the end of this one on
    template <typename Args>
    __device__ __forceinline__ void open(const Args& a, const ChainLayer* layers, const Share& share, const Rows& rows, const Tile* held, int lane) {
        next = 0;
        if (total > 64) {
            first += window;
            for (int n; layer < a.layers; first = 0, stage == 4 ? (stage = 0, ++layer) : ++stage)
                if ((n = count_of(stage, a, share) - first) > 0) {
                    window = min(n, 64);
                    const unsigned long at = place(stage, first + min(lane, window - 1), kind, a, share, rows, held) +
                                             (unsigned long)(&layers[layer].w_qkv)[stage == 1 ? 8 : stage == 0 ? 0 : stage - 1];
                    lo = (unsigned)at;
                    hi = (unsigned)(at >> 32);
                    return;
                }
        } else {
            if (window > 0) ++layer;
            window = total;
            if (layer < a.layers && total > 0) {
                const unsigned long at = ((unsigned long)rel_hi << 32 | rel_lo) + (unsigned long)(&layers[layer].w_qkv)[which];
                lo = (unsigned)at;
                hi = (unsigned)(at >> 32);
                return;
            }
        }
        // nothing is left: the same kilobyte again and again, as the waits count loads
        window = 0x7fffffff;
        lo = (unsigned)(unsigned long)a.h;
        hi = (unsigned)((unsigned long)a.h >> 32);
        kind = 3;
    }
    template <typename Args>
    __device__ __forceinline__ void begin(const Args& a, const ChainLayer* layers, const Share& share, const Rows& rows, const Tile* held, int lane) {
        rel_lo = rel_hi = 0;
        which = kind = 0;
        total = 0;
        for (int s = 0; s < 5; ++s) {
            const int n = count_of(s, a, share);
            int k;
            const unsigned long at = place(s, min(max(lane - total, 0), max(n - 1, 0)), k, a, share, rows, held);
            if (lane >= total && lane < total + n) {
                rel_lo = (unsigned)at;
                rel_hi = (unsigned)(at >> 32);
                kind = k;
                which = s == 1 ? 8 : s == 0 ? 0 : s - 1;
            }
            total += n;
        }
        open(a, layers, share, rows, held, lane);
    }
    // so many kilobytes more
    template <typename Args>
    __device__ __forceinline__ void ask(int count, const Args& a, const ChainLayer* layers, const Share& share, const Rows& rows, const Tile* held, int lane) {
#pragma clang loop unroll(disable)
        for (int k = 0; k < count; ++k) {
            const int of = next & 63, what = __builtin_amdgcn_readlane(kind, of);
            const u4 rsrc = {(unsigned)__builtin_amdgcn_readlane(lo, of), (unsigned)__builtin_amdgcn_readlane(hi, of) & 0xffffu, 0x7fffffffu, 0x00020000u};
            int off = values;
            if ((what & 3) == 0) off = row * (what >> 3) + piece;
            else if ((what & 3) == 1) off = keys ^ (what >> 3);
            else if ((what & 3) == 3) off = 0;
            const unsigned here = uniform(to + slot * 1024);
            if (!(what & 4)) QE_LOAD_TO_SHARED(here, off, rsrc, 0, "4", " nt");
            else QE_LOAD_TO_SHARED(here, off, rsrc, 0, "4", "");
            slot = slot + 1 == RING ? 0 : slot + 1;
            if (++next >= window) open(a, layers, share, rows, held, lane);
        }
    }
};

// MV: at most so many rows; RING: kilobytes of a feeding wave's ring; NP: a row of the stream is at most NP * 1024 numbers
template <int MV, int RING, int NP>
__global__ __launch_bounds__(THREADS) void decode_chain_kernel(const ChainArgs) {
    // (read where they lie: the compiler copies an array of arguments that is indexed by a variable to scratch memory)
    const auto& a = *(const __attribute__((address_space(4))) ChainArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    constexpr int MT = MV > 4 ? 2 : 1, MR = MV, QR = 8;                // rows of a tile of results; quads of outputs between two barriers
    extern __shared__ __align__(16) unsigned char shared[];
    __shared__ Rows rows;
    __shared__ Share share;
    __shared__ Unit s_unit;
    __shared__ Tile tiles[FEED * TILES];
    __shared__ ChainLayer layers[MAX_LAYERS];              // (the arguments may lie in the host's memory)
    __shared__ __align__(16) float squares[MAX_ROWS][WAIT];
    __shared__ int s_worker, s_workers, s_units[2];
    __shared__ int s_late;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, n = lane & 15;
    const int M = a.M, H = a.H, Hq = a.Hq, Hkv = a.Hkv, I = a.I, G = Hq / Hkv, P = 1 << a.logP;
    const int CQ = (Hq + 2 * Hkv) * D;
    unsigned char* const ring = shared;
    float* const part = (float*)(shared + FEED * RING * 1024);                 // [2][FEED][QR][MR][4]
    unsigned char* const xbuf = (unsigned char*)(part + 2 * FEED * QR * MR * 4);
    // (where the products have their operand, the attention has its own: [2][FEED][G][128], [2][FEED][G][2], [3][G][64], [3][64] twice)
    float* const macc = (float*)xbuf;
    float* const mml = macc + 2 * FEED * G * D;
    unsigned* const qbuf = (unsigned*)(mml + 2 * FEED * G * 2);
    unsigned* const kbuf = qbuf + 3 * G * 64;
    unsigned* const vbuf = kbuf + 3 * 64;

    for (unsigned i = threadIdx.x; i < a.layers * (sizeof(ChainLayer) / 4); i += THREADS) ((unsigned*)layers)[i] = ((const __attribute__((address_space(4))) unsigned*)a.layer)[i];

    // ---- roll call: the blocks that run by the time it ends share the work, the others leave ----
    if (threadIdx.x == 0) {
        s_late = 0;
        const unsigned id = __hip_atomic_fetch_add(a.work, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int worker = (int)id, workers = 0;
        if (id & CLOSED) {
            worker = -1;
        } else if (id == 0) {                              // the first comer waits for the others ...
            // ... for as long as the step would take longer with those that are there than with all, as which blocks take part is settled for
            // the whole step.  (Begun after 200 us whoever was there, a step beside a product that leaves 120 of 256 units free for 0.73 ms took
            // until 4.0 ms, 28 layers of width 1024 and one request, and 5.5, 12 layers and eight requests of 2000 keys; so until 1.25 and 1.2.  Between
            // products of 7 ms each: 2.3 ms a step, the longest 2.8, 3.0 and 4.8 before; the kernels one after the other wait until the
            // products are done.)
            long bytes = a.layer_bytes;
            for (int m = 0; m < M; ++m) bytes += (long)min(a.positions[m], a.max_position) * (4 * Hkv * D);
            const unsigned long alone = (unsigned long)a.layers * (bytes >> 10) * KILOBYTE, t0 = __builtin_amdgcn_s_memrealtime();
            const unsigned grid = gridDim.x;
            for (;;) {
                const unsigned come = min(__hip_atomic_load(a.work, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), grid);
                const unsigned long wait = min(max(CALL, alone / come - alone / grid), (unsigned long)a.limit / 4);
                if (come == grid || __builtin_amdgcn_s_memrealtime() - t0 >= wait) break;
            }
            workers = (int)__hip_atomic_fetch_or(a.work, CLOSED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + a.absent;
            __hip_atomic_store(a.work + 16, (unsigned)workers, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {                                           // (the first comer runs and says so soon)
            Waited waited;
            do workers = (int)__hip_atomic_load(a.work + 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            while (workers == 0 && waited.look() < a.limit);
            if (workers == 0) {
                worker = -1;
                if (a.late) __hip_atomic_store(a.late, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
        s_worker = worker;
        s_workers = workers;
        // The units are dealt out in their order and by what they cost: the tiles a wave has of them, and one more for a unit's joining.
        int first = 0;
        long weight = 0;
        for (int m = 0; m < M; ++m) {
            const int p = min(a.positions[m], a.max_position), row = a.tok_seq[m];
            rows.pos[m] = p;
            rows.slot[m] = a.slots ? a.slots[m] : -1;
            rows.table[m] = row;
            rows.shared[m] = a.shared_keys ? a.shared_keys[row] : 0;
            rows.keys[m] = segment_keys(p);
            rows.segments[m] = p / rows.keys[m] + 1;
            rows.first[m] = first;
            first += rows.segments[m] * Hkv;
            weight += (long)(rows.segments[m] * Hkv) * (rows.keys[m] / 128 + 1);
        }
        rows.first[M] = first;
        const auto share_begins = [&](int w) {
            long left = weight * w;                        // (in parts of 1 / workers)
            for (int m = 0; m < M; ++m) {
                const long one = (long)(rows.keys[m] / 128 + 1) * workers, count = rows.first[m + 1] - rows.first[m];
                if (left <= one * count) return rows.first[m] + (int)((left + one - 1) / one);
                left -= one * count;
            }
            return first;
        };
        s_units[0] = worker < 0 ? 0 : share_begins(worker);
        s_units[1] = worker < 0 ? 0 : share_begins(worker + 1);
    }
    __syncthreads();
    const int worker = uniform(s_worker), workers = uniform(s_workers);
    if (worker < 0) return;
    const auto part_of = [&](int items, int w) __attribute__((always_inline)) { return uniform((int)((long)items * w / workers)); };
    const int qkv0 = part_of(CQ / 4, worker), qkv1 = part_of(CQ / 4, worker + 1);
    const int out0 = part_of(H / 4, worker), out1 = part_of(H / 4, worker + 1);
    const int act0 = part_of(I / 4, worker), act1 = part_of(I / 4, worker + 1);
    const int unit0 = uniform(s_units[0]), unit1 = uniform(s_units[1]);
    if (threadIdx.x == 0) share = Share{qkv0, qkv1, out0, out1, act0, act1, unit0, unit1};
    if (threadIdx.x == 64) s_unit = unit0 < unit1 ? unit_at(rows, M, unit0) : Unit{};
    __syncthreads();

    if (wave < FEED) {
        // ================================ the feeding waves ================================
        const unsigned char* const my_slots = ring + wave * RING * 1024;
        const int o = n >> 2, qq = n & 3;
        Tile* const held = tiles + wave * TILES;
        Feed<RING, QR / 2> feed;
        feed.wave = wave; feed.logP = a.logP;
        feed.row = o; feed.piece = g * 64 + qq * 16;
        feed.keys = (lane >> 4) * 256 + (((lane & 15) ^ (lane >> 4)) << 4); feed.values = (lane >> 1) * P * 2 + (lane & 1) * 16;
        feed.to = (unsigned)(unsigned long)(__attribute__((address_space(3))) unsigned char*)shared + wave * RING * 1024;
        int count = 0;
        Unit of = uniform(s_unit);
        for (int u = unit0; u < unit1; ++u) {
            if (u > unit0) unit_next(of, rows, Hkv);
            const Unit& un = of;
            for (int t = wave; t < un.tiles; t += FEED, ++count)
                if (count < TILES && lane == 0) held[count] = Feed<RING, QR / 2>::tile_of(a.table, a.max_blocks, rows, un, t, a.logP);
        }
        feed.tiles = count;
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        feed.begin(a, layers, share, rows, held, lane);
        feed.ask(RING, a, layers, share, rows, held, lane);

        // What a product has used up is asked for again behind its barrier, or, with few numbers on the way between the blocks, when the next
        // operand is there: a compute unit's loads come back in their order, and a look for the next numbers would wait for
        // the kilobytes before it (width 1024, a layer: one request at 2048 keys 21.0 us and 19.9 so, at 8192 25.6 and 25.0; eight rows
        // at 4060 53.4 and 56.1, width 4096 79 and 84).
        constexpr bool LATE = MV <= 2 && NP == 1;
        int debt = 0;
        int cur = 0;                                       // the ring's oldest kilobyte
        const auto slot_at = [&](int i) __attribute__((always_inline)) { const int s = cur + i; return s >= RING ? s - RING : s; };
        for (int turn = 0; turn < 5 * a.layers; ++turn) {
            const int stage = turn % 5;
            if (stage == 1) {
                if (unit0 < unit1) BLOCK_BARRIER();
                if (LATE) { feed.ask(debt, a, layers, share, rows, held, lane); debt = 0; }
                Unit un = uniform(s_unit);
                int turns = 0;
                for (int u = unit0; u < unit1; ++u) {
                    const int i = u - unit0;
                    if (i > 0) {
                        unit_next(un, rows, Hkv);
                        turns += un.seg == 0;              // (another head's)
                    }
                    if (wave < un.tiles) {
                        AttnState<D> st;
                        st.init();
                        bf16x8 qreg[D / 32];
                        const unsigned* qrow = qbuf + (turns % 3 * G + min(n, G - 1)) * 64;
#pragma unroll
                        for (int c = 0; c < D / 32; ++c) qreg[c] = *(const bf16x8*)(qrow + c * 16 + g * 4);
                        for (int t = wave; t < un.tiles; t += FEED) {
                            asm volatile("s_waitcnt vmcnt(%0)" : : "n"(RING - 8) : "memory");
                            KVTile<D> tile;
                            const unsigned char* krow = my_slots + slot_at(n >> 2) * 1024 + (n & 3) * 256;
#pragma unroll
                            for (int c = 0; c < D / 32; ++c) tile.k[c] = *(const bf16x8*)(krow + (((c * 4 + g) ^ n) << 4));
#pragma unroll
                            for (int db = 0; db < D / 16; ++db)
                                tile.v[db] = *(const short4_t*)(my_slots + slot_at(4 + (db >> 1)) * 1024 + ((db & 1) * 16 + n) * 32 + g * 8);
                            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                            cur = slot_at(8);
                            if (t + FEED < un.tiles) {     // (the last tile's place is asked for behind the barriers)
                                feed.ask(8, a, layers, share, rows, held, lane);
                            }
                            attn_tile_step<D>(st, tile, qreg, a.scale, un.lo + t * 16, g, un.lo, un.hi, un.lo, un.hi);
                        }
                        float s = st.l;
                        s += __shfl_xor(s, 16, 64);
                        s += __shfl_xor(s, 32, 64);
                        if (n < G) {
                            float* acc = macc + (((i & 1) * FEED + wave) * G + n) * D;
#pragma unroll
                            for (int db = 0; db < D / 16; ++db) *(floatx4*)(acc + db * 16 + g * 4) = st.acc[db];
                            if (g == 0) {
                                float* ml = mml + (((i & 1) * FEED + wave) * G + n) * 2;
                                ml[0] = st.m;
                                ml[1] = s;
                            }
                        }
                    }
                    BLOCK_BARRIER();
                    if (u + 1 == unit1) BLOCK_BARRIER();   // (the one behind the last unit's joining)
                    if (wave < un.tiles) feed.ask(8, a, layers, share, rows, held, lane);
                }
                if (unit0 == unit1) BLOCK_BARRIER();
                continue;
            }
            // a product against `quads` fours of outputs: the wave's chunks of K, to `part`
            const int quads = stage == 0 ? qkv1 - qkv0 : stage == 3 ? 2 * (act1 - act0) : out1 - out0;
            if (quads == 0) continue;
            const int K = stage == 2 ? Hq * D : stage == 4 ? I : H;
            const int chunks = K / 128 > wave ? (K / 128 - wave + FEED - 1) / FEED : 0;
            const unsigned char* xrow[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) xrow[t] = xbuf + min(t * 4 + o, M - 1) * (K * 2 + 64) + wave * 256 + g * 64 + qq * 16;
            if (stage == 0 || stage == 3) BLOCK_BARRIER();
            BLOCK_BARRIER();
            for (int r = 0; r * QR < quads; ++r) {
                float* const mine = part + (r & 1) * (FEED * QR * MR * 4) + wave * (QR * MR * 4);
                const int total = min(QR, quads - r * QR) * chunks;
                int c = 0, q = 0, owed = 0;
                if (LATE) { feed.ask(debt, a, layers, share, rows, held, lane); debt = 0; }
                float acc[MT];
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[t] = 0.f;
                for (int e = 0; e < total; e += 4) {
                    // (what has been used up is asked for again four kilobytes later, the round's last behind its barrier, and so all if it has few)
                    if (owed == 0) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(RING - 4) : "memory");
                    else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(RING - 8) : "memory");
                    bf16x8 wv[4], xv[4][MT];
                    int cc = c;
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        wv[u] = *(const bf16x8*)(my_slots + slot_at(u) * 1024 + lane * 16);
#pragma unroll
                        for (int t = 0; t < MT; ++t) xv[u][t] = *(const bf16x8*)(xrow[t] + cc * (FEED * 256));
                        cc = cc + 1 == chunks ? 0 : cc + 1;
                    }
                    const int here = min(4, total - e);
                    float v[4][MT];
#pragma unroll
                    for (int u = 0; u < 4; ++u)
#pragma unroll
                        for (int t = 0; t < MT; ++t) {
                            // rows (output o, quarter q of K), columns (row m, quarter q'): what counts has q = q', one a lane
                            const floatx4 r = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[u], xv[u][t], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                            const float lo = qq & 1 ? r[1] : r[0], hi = qq & 1 ? r[3] : r[2];
                            v[u][t] = qq & 2 ? hi : lo;
                        }
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (u < here) {
#pragma unroll
                            for (int t = 0; t < MT; ++t) acc[t] += v[u][t];
                            if (++c == chunks) {
#pragma unroll
                                for (int t = 0; t < MT; ++t) {
                                    float y = acc[t];
                                    y += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, y), 0xb1, 0xf, 0xf, false));
                                    y += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, y), 0x4e, 0xf, 0xf, false));
                                    if (qq == 0 && t * 4 + o < MR) mine[(q * MR + t * 4 + o) * 4 + g] = y;
                                    acc[t] = 0.f;
                                }
                                c = 0;
                                ++q;
                            }
                        }
                    }
                    cur = slot_at(here);
                    if (total > 8 && e > 0) { feed.ask(4, a, layers, share, rows, held, lane); owed -= 4; }
                    owed += here;
                }
                if (chunks == 0) {                         // (a narrow matrix: nothing of it is this wave's)
                    for (int k = lane; k < QR * MR * 4; k += 64) mine[k] = 0.f;
                }
                BLOCK_BARRIER();
                if (LATE) debt += owed; else feed.ask(owed, a, layers, share, rows, held, lane);
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (no load may come to shared memory that is another block's by then)
        return;
    }

    // ================================ the waiting waves ================================
    const Exchange ex(M, H, Hq, Hkv, I, a.segments, a.layers);
    __builtin_amdgcn_s_setprio(3);                         // (what they wait for holds all blocks up, what the others ask for does not)
    const int hw = wave - FEED, ht = threadIdx.x - FEED * 64;
    const auto ex_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)a.work, 0, ex.total * 4u, 0x00020000);
    const auto h_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)a.h, 0, (unsigned)M * H * 4u, 0x00020000);
    // (16: past this compute die's L2, which the others' writes do not reach)
    const auto get4 = [&](unsigned word) __attribute__((always_inline)) { return __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(ex_rsrc, word * 4, 0, 16)); };
    // Through the L2, where a compute die's blocks find what one of them has fetched.  It may hold a place as it was before it was written: then it
    // still says ~0, as every place is written once, and get4 has to be asked.  (Not for the attention's parts.)
    const auto near4 = [&](unsigned word) __attribute__((always_inline)) { return __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(ex_rsrc, word * 4, 0, 0)); };
    const auto get2 = [&](unsigned word) __attribute__((always_inline)) { return __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(ex_rsrc, word * 4, 0, 16)); };
    const auto get1 = [&](unsigned word) __attribute__((always_inline)) { return (unsigned)__builtin_amdgcn_raw_buffer_load_b32(ex_rsrc, word * 4, 0, 16); };
    const auto put1 = [&](unsigned word, unsigned v) __attribute__((always_inline)) { __builtin_amdgcn_raw_buffer_store_b32(v, ex_rsrc, word * 4, 0, 16); };
    const auto put2 = [&](unsigned word, unsigned v, unsigned w) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_buffer_store_b64(u2{v, w}, ex_rsrc, word * 4, 0, 16);
    };
    const auto there = [&](const u4& v) __attribute__((always_inline)) {
        return ((v.x != NONE) & (v.y != NONE) & (v.z != NONE) & (v.w != NONE)) != 0;
    };
    // Asks (get(): false while something is missing) until all lanes have all, or until the limit of a wait: then false, and the host is told.
    // (No load of a get() stands under a condition: the compiler would wait for it before the next.)
    const auto await = [&](auto get) __attribute__((always_inline)) {
        Waited waited;
        for (unsigned i = 1;; ++i) {
            if (__all(get())) return true;
            if (i % 64 == 0 && (waited.look() > a.limit || __hip_atomic_load(&s_late, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP))) break;
            asm volatile("" ::: "memory");
        }
        __hip_atomic_store(&s_late, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);   // (nobody in this block waits again)
        if (a.late && lane == 0) __hip_atomic_store(a.late, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return false;
    };
    const auto or_nan = [&](u4& v) __attribute__((always_inline)) {
        v.x = published(v.x); v.y = published(v.y); v.z = published(v.z); v.w = published(v.w);
    };

    // The stream's rows from word `from` of the exchange (first: from h), normed, to xbuf: a quarter of each row a wave.
    const auto gather_normed = [&](bool first, unsigned from, const float* gain, float eps) __attribute__((always_inline)) {
        const int stride = H * 2 + 64;
        const auto column = [&](int p) __attribute__((always_inline)) { return min((p * WAIT + hw) * 256 + lane * 4, H - 4); };
        const auto within = [&](int p) __attribute__((always_inline)) { return (p * WAIT + hw) * 256 + lane * 4 < H; };
        u4 v[MV][NP], w[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) w[p] = *(const u4*)(gain + column(p));
        if (first) {
#pragma unroll
            for (int m = 0; m < MV; ++m)
#pragma unroll
                for (int p = 0; p < NP; ++p) v[m][p] = *(const u4*)(a.h + min(m, M - 1) * H + column(p));
        } else {
            const auto get_by = [&](auto load) __attribute__((always_inline)) {
                bool ok = true;
#pragma unroll
                for (int m = 0; m < MV; ++m)
#pragma unroll
                    for (int p = 0; p < NP; ++p) v[m][p] = load(from + min(m, M - 1) * H + column(p));
#pragma unroll
                for (int m = 0; m < MV; ++m)
#pragma unroll
                    for (int p = 0; p < NP; ++p) ok = ok & there(v[m][p]);
                return ok;
            };
            // (many rows: asked for again and again is one of them, until it is there; all of them would be some megabytes each time)
            bool all = false;
            if constexpr (MV > 2) {
                u4 u[NP];
                await([&]() __attribute__((always_inline)) {
                    bool ok = true;
#pragma unroll
                    for (int p = 0; p < NP; ++p) u[p] = get4(from + (M - 1) * H + column(p));
#pragma unroll
                    for (int p = 0; p < NP; ++p) ok = ok & there(u[p]);
                    return ok;
                });
                all = __all(get_by(near4));
            }
            if (!all && !await([&]() __attribute__((always_inline)) { return get_by(get4); })) {
#pragma unroll
                for (int m = 0; m < MV; ++m)
#pragma unroll
                    for (int p = 0; p < NP; ++p) or_nan(v[m][p]);
            }
        }
        float sq[MV];
#pragma unroll
        for (int m = 0; m < MV; ++m) {
            float ss = 0.f;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                float s4 = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) s4 += __uint_as_float(v[m][p][e]) * __uint_as_float(v[m][p][e]);
                ss += within(p) ? s4 : 0.f;
            }
            sq[m] = ss;
        }
        // The rows' sums over the wave: two rows' halves, then two pairs' quarters change places, so that half of the sums is left each time.
        if constexpr (MV >= 4) {
            float a4[MV / 4];
#pragma unroll
            for (int m = 0; m < MV / 4; ++m) {
                float two[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(sq[4 * m + k]), __float_as_uint(sq[4 * m + 2 + k]), false, false);
                    const unsigned r0 = r[0], r1 = r[1];
                    two[k] = __uint_as_float(r0) + __uint_as_float(r1);
                }
                const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(two[0]), __float_as_uint(two[1]), false, false);
                const unsigned r0 = r[0], r1 = r[1];
                a4[m] = row16_sum(__uint_as_float(r0) + __uint_as_float(r1));
            }
            // (lanes of row g of 16: the row m of the four that the swaps left there)
#pragma unroll
            for (int m = 0; m < MV / 4; ++m)
                if (n == 0) squares[4 * m + g][hw] = a4[m];
        } else {
#pragma unroll
            for (int m = 0; m < MV; ++m) {
                const float ss = wave_sum(sq[m]);
                if (lane == 0) squares[m][hw] = ss;
            }
        }
        BLOCK_BARRIER();
#pragma unroll
        for (int m = 0; m < MV; ++m) {
            const float4 ss = *(const float4*)squares[m];
            const float rstd = rsqrtf((ss.x + ss.y + ss.z + ss.w) / (float)H + eps);
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                float y[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) y[e] = __uint_as_float(v[m][p][e]) * rstd * __uint_as_float(w[p][e]);
                if (m < M && within(p)) Vec4<bf16_t>::store((bf16_t*)(xbuf + m * stride) + (p * WAIT + hw) * 256 + lane * 4, y);
            }
        }
    };
    // Rows of K bfloat16 from word `from` of the exchange, as they are: B pieces of 16 bytes a thread at once.
    const auto gather_some = [&](auto count, unsigned from, int K, int i0) __attribute__((always_inline)) {
        constexpr int B = decltype(count)::value;
        const int stride = K * 2 + 64, per = K / 8, all = M * per;
        u4 v[B];
        const auto get_by = [&](auto load) __attribute__((always_inline)) {
            bool ok = true;
#pragma unroll
            for (int b = 0; b < B; ++b) v[b] = load(from + min(i0 + b * WAIT * 64 + ht, all - 1) * 4);
#pragma unroll
            for (int b = 0; b < B; ++b) ok = ok & there(v[b]);
            return ok;
        };
        bool found = false;
        if constexpr (B > 2) {                             // (one of many first, as above)
            u4 u;
            await([&]() __attribute__((always_inline)) {
                u = get4(from + min(i0 + (B - 1) * WAIT * 64 + ht, all - 1) * 4);
                return there(u);
            });
            found = __all(get_by(near4));
        }
        if (!found && !await([&]() __attribute__((always_inline)) { return get_by(get4); })) {
#pragma unroll
            for (int b = 0; b < B; ++b) or_nan(v[b]);
        }
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const int i = min(i0 + b * WAIT * 64 + ht, all - 1);       // (the last piece several times: the same bytes)
            int m = 0;
#pragma unroll
            for (int k = 1; k < MR; ++k) m += i >= k * per;
            *(u4*)(xbuf + m * stride + (i - m * per) * 16) = v[b];
        }
    };
    const auto gather_rows = [&](unsigned from, int K) __attribute__((always_inline)) {
        const int all = M * (K / 8);
        for (int i0 = 0; i0 < all;) {
            const int need = (all - i0 + WAIT * 64 - 1) / (WAIT * 64);
            constexpr int FEW = MV > 4 ? 8 : 2, MANY = MV > 4 ? 12 : 6;
            if (need > FEW) { gather_some(std::integral_constant<int, MANY>{}, from, K, i0); i0 += MANY * WAIT * 64; }
            else { gather_some(std::integral_constant<int, FEW>{}, from, K, i0); i0 += FEW * WAIT * 64; }
        }
    };
    // q's heads of a unit (and the token's own key and value), normed and rotated, to shared memory; key and value to the cache
    const auto prepare = [&](const Unit& un, int i, bool with_q, unsigned qkv, const float* q_norm, const float* k_norm, bf16_t* cache) __attribute__((always_inline)) {
        const int tasks = un.own ? G + 2 : G, task0 = with_q ? hw : G + hw;
        const int p = uniform(rows.pos[un.m]), slot = uniform(rows.slot[un.m]);
        constexpr int MOST = (MAX_GROUP + 2 + WAIT - 1) / WAIT;
        unsigned v[MOST];
        float2 cs = {1.f, 1.f}, sn = {0.f, 0.f};
        if (a.rope) {
            cs = *(const float2*)(a.rope + (long)p * D + (lane & 31) * 2);
            sn = *(const float2*)(a.rope + (long)p * D + D / 2 + (lane & 31) * 2);
        }
        const auto task = [&](int t) __attribute__((always_inline)) { return min(task0 + t * WAIT, tasks - 1); };
        float2 w[MOST];
#pragma unroll
        for (int t = 0; t < MOST; ++t) w[t] = float2{1.f, 1.f};
        if (q_norm && k_norm) {
#pragma unroll
            for (int t = 0; t < MOST; ++t) w[t] = *(const float2*)((task(t) < G ? q_norm : k_norm) + lane * 2);
        }
        const auto get = [&]() __attribute__((always_inline)) {
            bool ok = true;
#pragma unroll
            for (int t = 0; t < MOST; ++t) {
                const int j = task(t), head = j < G ? un.kvh * G + j : j == G ? Hq + un.kvh : Hq + Hkv + un.kvh;
                v[t] = get1(qkv + un.m * (CQ / 2) + head * 64 + lane);
            }
#pragma unroll
            for (int t = 0; t < MOST; ++t) ok = ok & (v[t] != NONE);
            return ok;
        };
        if (!await(get)) {
#pragma unroll
            for (int t = 0; t < MOST; ++t) v[t] = published(v[t]);
        }
        // (the parts that this wave put back to ~0 in the layer before have arrived when anything of this layer is published)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        bf16_t* page = cache + (long)(slot >> a.logP) * (2L * Hkv * P * D);
        const int in = slot & (P - 1);
#pragma unroll
        for (int t = 0; t < MOST; ++t) {
            const int j = task0 + t * WAIT;
            if (j >= tasks) break;
            if (j == G + 1) {                              // the value
                vbuf[i % 3 * 64 + lane] = v[t];
                if (slot >= 0) {
                    bf16_t* vt = page + (long)((Hkv + un.kvh) * P) * D + in;
                    vt[(long)(2 * lane) * P].bits = (uint16_t)(v[t] & 0xffffu);
                    vt[(long)(2 * lane + 1) * P].bits = (uint16_t)(v[t] >> 16);
                }
                continue;
            }
            float x = bf16_bits_to_float(v[t] & 0xffffu), y = bf16_bits_to_float(v[t] >> 16);
            if (q_norm && k_norm) {
                const float rstd = rsqrtf(wave_sum(x * x + y * y) / (float)D + a.qk_eps);
                x = x * rstd * w[t].x;
                y = y * rstd * w[t].y;
            }
            // (the other of a rotated pair, 64 features on, is 32 lanes on)
            const float ox = __shfl_xor(x, 32, 64), oy = __shfl_xor(y, 32, 64);
            x = lane < 32 ? cs.x * x - sn.x * ox : sn.x * ox + cs.x * x;
            y = lane < 32 ? cs.y * y - sn.y * oy : sn.y * oy + cs.y * y;
            const unsigned b = pair_bits(x, y);
            if (j < G) {
                qbuf[(i % 3 * G + j) * 64 + lane] = b;
            } else {
                kbuf[i % 3 * 64 + lane] = b;
                if (slot >= 0) *(unsigned*)(page + ((long)(un.kvh * P) + in) * D + lane * 2) = b;
            }
        }
    };
    // A unit's result from its waves' and the token's own key, to the exchange: a thread a feature.  The own key's score and value are
    // looked up while the feeding waves have the unit.
    constexpr int TURNS = MAX_GROUP * D / (WAIT * 64);
    float own_score[TURNS], own_value = 0.f;
    const auto look_up_own = [&](const Unit& un, int i) __attribute__((always_inline)) {
        if (!un.own) return;
        const unsigned k = kbuf[i % 3 * 64 + lane], v = vbuf[i % 3 * 64 + ((ht & 127) >> 1)];
        own_value = bf16_bits_to_float(ht & 1 ? v >> 16 : v & 0xffffu);
#pragma unroll
        for (int t = 0; t < TURNS; ++t) {
            const int j = uniform((ht + t * WAIT * 64) >> 7);
            if (j < G) {
                const unsigned q = qbuf[(i % 3 * G + j) * 64 + lane];
                own_score[t] = wave_sum(bf16_bits_to_float(q & 0xffffu) * bf16_bits_to_float(k & 0xffffu) +
                                        bf16_bits_to_float(q >> 16) * bf16_bits_to_float(k >> 16)) * a.scale;
            }
        }
    };
    const auto join_waves = [&](const Unit& un, int i, unsigned parts) __attribute__((always_inline)) {
        const int waves = min(un.tiles, FEED), d = ht & 127;
#pragma unroll
        for (int t = 0; t < TURNS; ++t) {
            const int j = uniform((ht + t * WAIT * 64) >> 7);          // (a wave has features of one head)
            if (j >= G) break;
            const float* ml = mml + ((i & 1) * FEED * G + j) * 2;
            const float* acc = macc + ((i & 1) * FEED * G + j) * D + d;
            float2 mw[FEED];
            float o[FEED];
#pragma unroll
            for (int w = 0; w < FEED; ++w) mw[w] = *(const float2*)(ml + w * G * 2);
#pragma unroll
            for (int w = 0; w < FEED; ++w) o[w] = acc[w * G * D];
            const float own = un.own ? own_score[t] : -INFINITY;
            float top = own;
#pragma unroll
            for (int w = 0; w < FEED; ++w) {
                mw[w].x = w < waves ? mw[w].x : -INFINITY;
                top = fmaxf(top, mw[w].x);
            }
            const float ref = attn_reference(top);
            const float f = __expf(own - ref);
            float x = un.own ? f * own_value : 0.f, sum = f;
#pragma unroll
            for (int w = 0; w < FEED; ++w) {
                const float e = __expf(mw[w].x - ref);
                x = w < waves ? x + e * o[w] : x;
                sum = w < waves ? sum + e * mw[w].y : sum;
            }
            const unsigned to = parts + (((un.m * Hq + un.kvh * G + j) * a.segments + un.seg) * 4 + (d >> 5)) * PART;
            put1(to + (d & 31), published(x));
            if ((d & 31) == 0) put2(to + 32, published(top), published(sum));
        }
    };
    // A quarter of a head of a row a wave: the segments' parts, every eighth of them eight lanes', added up.
    const int joins = M * Hq * 4, join0 = part_of(joins, worker), join1 = part_of(joins, worker + 1);
    const auto join_some = [&](auto count, int t, int segments, unsigned parts, unsigned att) __attribute__((always_inline)) {
        constexpr int S = decltype(count)::value;
        const int head = t >> 2, piece = lane & 7, group = lane >> 3;
        const auto place = [&](int s) __attribute__((always_inline)) {
            return parts + ((head * a.segments + min(group + s * 8, segments - 1)) * 4 + (t & 3)) * PART;
        };
        u4 v[S];
        u2 ml[S];
        const auto get = [&]() __attribute__((always_inline)) {
            bool ok = true;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                v[s] = get4(place(s) + piece * 4);
                ml[s] = get2(place(s) + 32);
            }
#pragma unroll
            for (int s = 0; s < S; ++s) ok = ok & there(v[s]) & (ml[s].x != NONE) & (ml[s].y != NONE);
            return ok;
        };
        if (!await(get)) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                or_nan(v[s]);
                ml[s].x = published(ml[s].x);
            }
        }
        float top = -INFINITY, sum = 0.f, r[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < S; ++s) top = fmaxf(top, __uint_as_float(ml[s].x));
        top = wave_max(top);
        const float ref = attn_reference(top);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const bool mine = group + s * 8 < segments;
            const float f = __expf(__uint_as_float(ml[s].x) - ref);
            sum = mine ? sum + f * __uint_as_float(ml[s].y) : sum;
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = mine ? r[e] + f * __uint_as_float(v[s][e]) : r[e];
        }
        const auto over_groups = [&](float x) __attribute__((always_inline)) {
            float y, z;
            x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x128, 0xf, 0xf, false));
            pair_across_rows(x, y, z);
            x = y + z;
            pair_across_halves(x, y, z);
            return y + z;
        };
        sum = over_groups(sum);
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = over_groups(r[e]) / sum;
        if (lane < 8) put2(att + head * 64 + (t & 3) * 16 + piece * 2, published(pair_bits(r[0], r[1])), published(pair_bits(r[2], r[3])));
        // back to ~0 for the layer after the next
#pragma unroll
        for (int s = 0; s < S; ++s) {
            if (group + s * 8 < segments) {
                __builtin_amdgcn_raw_buffer_store_b128(u4{NONE, NONE, NONE, NONE}, ex_rsrc, (place(s) + piece * 4) * 4, 0, 16);
                if (piece == 0) put2(place(s) + 32, NONE, NONE);
            }
        }
    };
    const auto join_segments = [&](unsigned parts, unsigned att) __attribute__((always_inline)) {
        for (int t = join0 + hw; t < join1; t += WAIT) {
            const int m = uniform((t >> 2) / Hq), segments = uniform(rows.segments[m]);
            if (segments <= 8) join_some(std::integral_constant<int, 1>{}, t, segments, parts, att);
            else join_some(std::integral_constant<int, MAX_SEGMENTS / 8>{}, t, segments, parts, att);
        }
    };

    // a thread has an output of a row of a round's; two neighbours' as one word of bfloat16, in the even lane
    const int q1 = (ht >> 2) / M, m1 = (ht >> 2) - q1 * M;
    const auto pair_of = [&](float v) __attribute__((always_inline)) {
        return pair_bits(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xb1, 0xf, 0xf, false)));
    };
    for (int turn = 0; turn < 5 * a.layers; ++turn) {
        const int l = turn / 5, stage = turn - l * 5;
        const ChainLayer& L = layers[l];
        const unsigned base = ex.layers + ex.per_layer * l;
        const unsigned before = base - ex.per_layer + ex.x2;           // the stream as the layer before left it
        if (stage == 1) {
            const unsigned parts = ex.parts + (l & 1) * ex.set;
            if (unit0 < unit1) {
                // (a unit is prepared while the feeding waves have the one before)
                Unit un = uniform(s_unit);
                int turns = 0;
                prepare(un, 0, true, base + ex.qkv, L.q_norm, L.k_norm, L.cache);
                BLOCK_BARRIER();
                for (int u = unit0; u < unit1; ++u) {
                    const int i = u - unit0;
                    const Unit now = un;
                    look_up_own(now, turns);
                    if (u + 1 < unit1) {
                        unit_next(un, rows, Hkv);
                        const bool another = un.seg == 0;
                        turns += another;
                        if (another || un.own) prepare(un, turns, another, base + ex.qkv, L.q_norm, L.k_norm, L.cache);
                    }
                    BLOCK_BARRIER();
                    join_waves(now, i, parts);
                }
            } else {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // (as in prepare)
            }
            BLOCK_BARRIER();                               // (what the units left in shared memory gives way to the operand)
            join_segments(parts, base + ex.att);
            continue;
        }
        const int first_quad = stage == 0 ? qkv0 : stage == 3 ? act0 : out0;
        const int quads = stage == 0 ? qkv1 - qkv0 : stage == 3 ? 2 * (act1 - act0) : out1 - out0;
        if (quads == 0) continue;
        const int K = stage == 2 ? Hq * D : stage == 4 ? I : H;
        const bool from_h = l == 0 && stage <= 2, to_h = l + 1 == a.layers && stage == 4;
        const unsigned old = stage == 2 ? before : base + ex.x1;       // the stream before the branch that stage 2 or 4 adds
        if (stage == 0 || stage == 3) gather_normed(from_h, stage == 0 ? before : base + ex.x1, stage == 0 ? L.norm1 : L.norm2, stage == 0 ? L.eps1 : L.eps2);
        else gather_rows(base + (stage == 2 ? ex.att : ex.act), K);
        const bool adds = stage == 2 || stage == 4;
        const auto place = [&](int r) __attribute__((always_inline)) { return m1 * H + (out0 + r * QR + q1) * 4 + (ht & 3); };
        float was = 0.f;
        const auto ask_was = [&](int r) __attribute__((always_inline)) {
            if (adds && q1 < min(QR, quads - r * QR)) {
                if (from_h) was = a.h[place(r)];
                else was = __uint_as_float(get1(old + place(r)));
            }
        };
        ask_was(0);
        BLOCK_BARRIER();                                   // (the operand is there)
        for (int r = 0; r * QR < quads; ++r) {
            BLOCK_BARRIER();
            const float* round = part + (r & 1) * (FEED * QR * MR * 4);
            const int count = min(QR, quads - r * QR);
            const auto summed = [&](int q, int m, int e) __attribute__((always_inline)) {
                const float* p = round + (q * MR + m) * 4 + e;
                float v = 0.f, t[FEED];
#pragma unroll
                for (int w = 0; w < FEED; ++w) t[w] = p[w * (QR * MR * 4)];
#pragma unroll
                for (int w = 0; w < FEED; ++w) v += t[w];
                return v;
            };
            if (adds) {
                if (q1 < count) {
                    const float y = was + summed(q1, m1, ht & 3);
                    if (to_h) a.h[place(r)] = y;
                    else put1(base + (stage == 2 ? ex.x1 : ex.x2) + place(r), published(y));
                }
                if ((r + 1) * QR < quads) ask_was(r + 1);
            } else if (stage == 0) {
                if (q1 < count) {
                    const unsigned pair = pair_of(summed(q1, m1, ht & 3));
                    if (!(ht & 1)) put1(base + ex.qkv + m1 * (CQ / 2) + (first_quad + r * QR + q1) * 2 + ((ht & 3) >> 1), published(pair));
                }
            } else if (2 * q1 < count) {                   // (the round's gates, then its ups)
                const float gate = summed(q1, m1, ht & 3), up = summed(count / 2 + q1, m1, ht & 3);
                const unsigned pair = pair_of(gate / (1.f + __expf(-gate)) * up);
                if (!(ht & 1)) put1(base + ex.act + m1 * (I / 2) + (first_quad + r * (QR / 2) + q1) * 2 + ((ht & 3) >> 1), published(pair));
            }
        }
    }
}

// ~0 to the exchange, 0 to the roll call's words (a launch of its own in front: see above)
__global__ __launch_bounds__(256) void decode_chain_clear_kernel(u4* work, unsigned pieces) {
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < pieces; i += gridDim.x * 256) {
        const unsigned v = i < 16 ? 0u : NONE;
        work[i] = u4{v, v, v, v};
    }
}

int chain_segments(int max_position) {
    const int small = max_position / 128 + 1, large = max_position / 256 + 1;      // (segment_keys() for all positions up to it)
    return max(min(small, 20), min(large, MAX_SEGMENTS));
}

// Shared memory for rings of `ring` kilobytes.
size_t chain_shared(int ring, int M, int H, int Hq, int Hkv, int I) {
    const int G = Hq / Hkv, rows = M > 4 ? 8 : M > 2 ? 4 : M;
    long K = H > I ? H : I;
    if ((long)Hq * D > K) K = (long)Hq * D;
    const size_t x = (size_t)M * (K * 2 + 64);
    const size_t at = (size_t)4 * (2 * FEED * G * (D + 2) + 3 * (G + 2) * 64);
    return (size_t)FEED * ring * 1024 + 4ul * 2 * FEED * 8 * rows * 4 + (x > at ? x : at);
}
constexpr size_t SHARED_LIMIT = 160 * 1024 - 512 - sizeof(ChainLayer) * MAX_LAYERS - sizeof(Tile) * FEED * TILES;         // (the kernel's few words besides)

int chain_ring(int M, int H, int Hq, int Hkv, int I) {
    const int most = M > 4 ? 10 : 12;
    if (chain_shared(most, M, H, Hq, Hkv, I) <= SHARED_LIMIT) return most;
    return chain_shared(8, M, H, Hq, Hkv, I) <= SHARED_LIMIT ? 8 : 0;
}

}  // namespace

// What the chain takes: rows of single new tokens, up to 8; heads of 128, up to 8 queries to a key; widths in multiples of 128; pages
// of 16, 32, 64 ... tokens; an operand that fits shared memory beside the rings.
extern "C" int qe_decode_chain_supported(int M, int H, int Hq, int Hkv, int head_dim, int I, int P) {
    if (M < 1 || M > MAX_ROWS || head_dim != D || Hkv < 1 || Hq < 1 || Hq % Hkv || Hq / Hkv > MAX_GROUP) return 0;
    if (H < 128 || H % 128 || H > (M > 4 ? 2048 : 5120) || I < 128 || I % 128 || P < 16 || (P & (P - 1))) return 0;
    if ((double)(Hq + 2 * Hkv) * D * H * 2 > 4e9 || 4.0 * I * H > 4e9 || 2.0 * Hq * D * H > 4e9 || 4.0 * Hkv * P * D > 2e9) return 0;
    return chain_ring(M, H, Hq, Hkv, I) > 0;
}

// Whether the chain is the quicker way (us a layer, the kernels one after the other and the chain, 200 keys a row, and at 8000):
//   * Up to some 600 MB of matrices a layer.  Larger ones stream for so long that the kernels' starts count for little, and each product's own kernel
//     streams them as fast or faster (width 5120 with 25600 in the middle, 975 MB, one request: 300 and 312; 13824, 550 MB, two: 134, 111).
//   * Of widths beyond 3072, two rows at most: with more the rows' way to all blocks and back costs what the starts do (width 4096, three: 142, 143).
//   * Rings of twelve (ten) kilobytes, or a narrow layer.  Where an operand of many rows, a wide middle or seven or eight queries to a key leave
//     room for rings of eight, a compute unit has a third less on the way: up to width 2304 that costs less than the starts (2048 with 6144, six rows:
//     56, 46 and 88, 83; 2304 with 9216, three: 66, 61 and 82, 79), with one or two rows up to 3072 (with 12288 and seven queries to a key, two:
//     84, 80 and 89, 86), and up to 4096 where the width comes out even, four chunks of K a wave and four fours of outputs a unit (4096 with
//     16384, two: 133, 116 and 144, 129).  Not beyond: three rows of 2560 with 9728 76, 74 and 92, 94, of 3072 with 12288 84, 84 and 101, 103 (at
//     32000 keys 155, 143 and 164, 152; but which way a row goes, and so its bits, is not to follow how far the rows beside it are); 3584 with
//     18944 and seven queries to a key, one 122, 122 and 122, 128, two 121, 128 and 126, 135; 4224 with 12288 and eight, two 108, 113; 5120
//     with 14592, two 136, 144.
//   * One request with one key/value head up to some 48 keys a number of the width: its keys are cut in 32 segments, which leave most of the chip
//     idle (width 1024, 45000 keys 47, 46, 64000 53, 56, 120000 76, 85; width 2048, 60000 71, 66, 120000 95, 98).  Two key/value heads: 120000
//     keys 89, 87.
// max_position: no row stands beyond it.
extern "C" int qe_decode_chain_preferred(int M, int H, int Hq, int Hkv, int head_dim, int I, int P, int max_position) {
    if (!qe_decode_chain_supported(M, H, Hq, Hkv, head_dim, I, P)) return 0;
    if (2.0 * H * ((Hq * 2.0 + 2.0 * Hkv) * head_dim + 3.0 * I) > 600e6 || (M > 2 && H > 3072)) return 0;
    if (chain_ring(M, H, Hq, Hkv, I) == 8 && H > (M > 2 ? 2304 : H % 1024 ? 3072 : 4096)) return 0;
    return M * Hkv > 1 || max_position / 48 < H;
}

extern "C" int qe_decode_chain_layers() { return MAX_LAYERS; }

extern "C" long qe_decode_chain_workspace_bytes(int M, int H, int Hq, int Hkv, int I, int layers, int max_position) {
    const Exchange ex(M, H, Hq, Hkv, I, chain_segments(max_position), layers);
    return ((long)ex.total * 4 + 15) / 16 * 16;
}

// h: float32 [M, H], the stream in front of the first layer, and behind the last one afterwards.  layers: for each nine pointers: q|k|v, output, gate|up
// (rows of gate and up in alternating blocks of 32) and down matrices, the weights of the two norms and of q's and k's (null: none), the cache.  eps: two a layer.
// rope: rows [cos | sin] of 128 numbers a position, or null.  units: blocks (0: one a compute unit).  late: a word of pinned host memory that
// becomes 1 if a block has waited for others for limit_us in vain (the rows are then NaN), or null.  absent: so many blocks more are given work than
// come, so that what they should do is waited for in vain.  Every row is the one new token of its request, at positions[m] <= max_position.
extern "C" int qe_decode_chain(void* h, const void* const* layers, const float* eps, int n_layers, const int* positions, const int* tok_seq,
                               const int* block_table, int max_blocks, const int* shared_keys, const int* slots, const float* rope, float qk_eps,
                               float scale, int M, int H, int Hq, int Hkv, int I, int P, int max_position, int units, int* late, int limit_us,
                               int absent, void* workspace, long workspace_bytes, hipStream_t stream) {
    QE_REQUIRE(qe_decode_chain_supported(M, H, Hq, Hkv, D, I, P), "decode chain: sizes not taken");
    QE_REQUIRE(n_layers >= 1 && n_layers <= MAX_LAYERS, "decode chain: %d layers in a launch", n_layers);
    QE_REQUIRE(max_position >= 0, "decode chain: position %d", max_position);
    QE_REQUIRE(limit_us > 0 && limit_us <= 10000000 && absent >= 0 && absent <= 1024, "decode chain: a limit of %d us, %d blocks absent", limit_us, absent);
    for (int l = 0; l < n_layers; ++l) QE_REQUIRE(!layers[9 * l + 6] == !layers[9 * l + 7], "decode chain: a norm of q or of k alone");
    QE_REQUIRE(workspace_bytes >= qe_decode_chain_workspace_bytes(M, H, Hq, Hkv, I, n_layers, max_position),
               "decode chain: workspace of %ld bytes is too small", workspace_bytes);
    // (three or four rows beyond width 3072 go two by two: a form that held them all spilled 37 registers, and the rule above never picks them)
    if (M > 2 && H > 3072) {
        for (int m = 0; m < M; m += 2) {
            const int rc = qe_decode_chain((float*)h + (long)m * H, layers, eps, n_layers, positions + m, tok_seq + m, block_table, max_blocks, shared_keys,
                                           slots ? slots + m : nullptr, rope, qk_eps, scale, min(2, M - m), H, Hq, Hkv, I, P, max_position, units, late,
                                           limit_us, absent, workspace, workspace_bytes, stream);
            if (rc) return rc;
        }
        return 0;
    }
    ChainArgs a{};
    for (int l = 0; l < n_layers; ++l) {
        const void* const* p = layers + 9 * l;
        for (int i = 0; i < 9; ++i) QE_REQUIRE(((uintptr_t)p[i] & 15) == 0 && (p[i] || i == 6 || i == 7), "decode chain: operand %d of layer %d", i, l);
        a.layer[l] = ChainLayer{(const bf16_t*)p[0], (const bf16_t*)p[1], (const bf16_t*)p[2], (const bf16_t*)p[3], (const float*)p[4],
                                (const float*)p[5], (const float*)p[6], (const float*)p[7], (bf16_t*)p[8], eps[2 * l], eps[2 * l + 1]};
    }
    QE_REQUIRE((((uintptr_t)h | (uintptr_t)rope | (uintptr_t)workspace) & 15) == 0, "decode chain: operands at odd addresses");
    a.h = (float*)h;
    a.positions = positions; a.tok_seq = tok_seq; a.table = block_table; a.slots = slots; a.shared_keys = shared_keys;
    a.rope = rope;
    a.work = (unsigned*)workspace;
    a.scale = scale; a.qk_eps = qk_eps;
    a.layers = n_layers; a.M = M; a.H = H; a.Hq = Hq; a.Hkv = Hkv; a.I = I;
    a.logP = __builtin_ctz(P);
    a.late = late; a.limit = (unsigned)limit_us * 100u; a.absent = absent;
    a.layer_bytes = 2l * H * ((2l * Hq + 2l * Hkv) * D + 3l * I);
    a.max_blocks = max_blocks; a.segments = chain_segments(max_position); a.max_position = max_position;
    const Exchange ex(M, H, Hq, Hkv, I, a.segments, n_layers);
    const int ring = chain_ring(M, H, Hq, Hkv, I);
    const size_t bytes = chain_shared(ring, M, H, Hq, Hkv, I);
    const int blocks = units > 0 && units < qe_compute_units() ? units : qe_compute_units();
    decode_chain_clear_kernel<<<4 * blocks, 256, 0, stream>>>((u4*)workspace, (ex.total + 3) / 4);
    QE_LAUNCH_CHECK();
#define QE_CHAIN3(MV_, RING_, NP_)                                                            \
    do {                                                                                      \
        QE_RAISE_SHARED((decode_chain_kernel<MV_, RING_, NP_>), SHARED_LIMIT);                \
        decode_chain_kernel<MV_, RING_, NP_><<<blocks, THREADS, bytes, stream>>>(a);          \
    } while (0)
#define QE_CHAIN2(MV_, NP_)                                                                   \
    do {                                                                                      \
        if (ring > 8) QE_CHAIN3(MV_, (MV_ > 4 ? 10 : 12), NP_);                               \
        else QE_CHAIN3(MV_, 8, NP_);                                                          \
    } while (0)
#define QE_CHAIN(MV_)                                                                         \
    do {                                                                                      \
        if (H <= 1024) QE_CHAIN2(MV_, 1);                                                     \
        else if (H <= 2048) QE_CHAIN2(MV_, 2);                                                \
        else QE_CHAIN2(MV_, 3);                                                               \
    } while (0)
    if (M == 1 && H > 3072) QE_CHAIN2(1, 5);
    else if (M == 2 && H > 3072) QE_CHAIN2(2, 5);
    else if (M == 1) QE_CHAIN(1);
    else if (M == 2) QE_CHAIN(2);
    else if (M <= 4) QE_CHAIN(4);
    else if (H <= 1024) QE_CHAIN2(8, 1);
    else QE_CHAIN2(8, 2);
#undef QE_CHAIN
#undef QE_CHAIN2
#undef QE_CHAIN3
    QE_LAUNCH_CHECK();
    return 0;
}
