// Matrix product for many rows of activations (prefill): out[M, N] = x[M, K] . W[N, K]^T (+ bias),
// bfloat16 in, 32-bit accumulation with v_mfma_f32_32x32x16_bf16, output bfloat16 or float32.
//
// A block of NW waves (NW / 2 down, 2 across) computes a BM x BN tile of the output; each wave its
// part as MFMA tiles of 32 x 32.  K is walked in stages of 64 through shared memory.  Both operands are
// K-contiguous in memory, so they are staged alike, by loads that write to shared memory directly.
//
// What the time of such a block goes to: a compute unit takes 64 bytes a cycle from its L1 and 128 from its shared
// memory, a wave issues in order, and a load needs up to two microseconds to arrive.  So whatever is not an MFMA stands between
// MFMAs, fragments are read a good part of a stage before they are wanted, and a stage's loads are issued one and a half to
// two stages ahead.  (With the loads in registers first, stored to shared memory a stage later, and all fragments of a k
// step read in a row behind each stage's barrier: 8192 x 8192 x 8192 took 829 us, now 769; 8192 rows against gate and up of 24576 x 4096
// 1316, now 1220; 512 rows against 6144 x 1024 12.2, now 10.7; 512 against q, k and v of 4096 x 1024 11.8, now 9.9.  Stages of 32 of K,
// half lines of 64 bytes a row, are 5 to 25 % slower than the whole lines of 64.)
//
// 128 x 128 by four waves (two blocks a compute unit), 64 x 128 where there would be too few blocks otherwise, 256 x 128
// (eight waves) and 256 x 256 (four waves, a wave's part 128 x 128, which reads half the bytes per MFMA
// from the L1 and from shared memory) where there are many: see qe_gemm_mfma_shape.
//
// Rows of x beyond M and rows of W beyond N are read as zero and never stored; K must be a
// multiple of 8 (16-byte loads), a tail shorter than 64 is filled with zeros.
// The blocks of one XCD (every eighth block) take a compact part of the tiles, see the kernel.
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float floatx16;
typedef __attribute__((ext_vector_type(4))) unsigned int uint4_t;
union Piece16 {   // 16 bytes, addressable by element
    uint4_t q;
    unsigned short e[8];
};

// SILU (1; 2: with biases, which lie as W's rows do): W holds gate and up rows interleaved in blocks of 32 (gate 0..31, up 0..31, gate 32..63,
// ...), N counts all of them, and the result is silu(gate) * up, N / 2 wide: the two MFMA tiles a
// lane holds side by side are the gate and the up of the same outputs.
// What the q|k|v product of an attention layer does with its result instead of storing it (QKV):
// per-head RMSNorm of q and k (weights or null), half-split rotation from the table's row of the
// token's position (or null), then q to q_out [M, Hq, 128], k and v into the cache at the token's
// slot (negative: nowhere), exactly as the kernels of qk_rope_store.hip do on a stored product, in
// the same arithmetic: the product is rounded to bfloat16 first.  Heads are 128 wide, so that a
// tile's 128 columns are one head.
struct QkvTail {
    const int* positions;
    const int* slots;
    const float* q_w;
    const float* k_w;
    const float* table;
    bf16_t* q_out;
    bf16_t* cache;
    float eps;
    int Hq, Hkv, P;
    int lp;   // log2 P: the page size is a power of two, and a division by a number known only at run time costs dozens of instructions an item
    // Rows grouped by expert (a mixture of experts): the block's row tile is entry blockIdx of ``tiles``
    // (expert, first row, rows <= BM), of which the device knows how many there are (n_tiles); W holds
    // one [N, K] matrix per expert.  A block beyond the tiles leaves at once, so the grid follows the
    // shapes alone.  null: one matrix, M rows.
    const int* tiles;
    const int* n_tiles;
    // With SILU: act_limit > 0 makes the activation min(g, limit) sigmoid(act_slope g) (clamp(u, -limit, limit) + 1)
    // instead of silu(g) u.
    float act_limit, act_slope;
    // Without SILU: the result is relu(.)^2 instead of the product itself.
    int relu_sq;
    // The first column of the product that this launch computes (a multiple of 256).
    int n_first;
    // With SILU over grouped rows: sorted row i is row_w[perm[i]] times its row of x (null: that row itself); the
    // factor meets gate and up in 32-bit.
    const float* row_w;
    const int* perm;
};

// Bytes of shared memory: the ring, or the tile of results with the rows' positions, slots and lists where that takes more.
constexpr int gemm_mfma_shared_bytes(int BM, int BN, int RING, bool QKV) {
    const int ring = RING * (BM + BN) * 128, tile = BM * (BN * 2 + 16) + 2 * BM * 4 + (BM + BM / 8 + 8) * 4;
    return QKV && tile > ring ? tile : ring;
}

// DIRECT: x and w begin at a whole 16-byte piece, which loads that write to shared memory themselves want.  Operands that lie elsewhere come
// through registers, asked for a stage before they are stored; every shape is then a ring (both operands at an odd element: 8192 rows against gate
// and up of 24576 x 4096 2051 us, 1238 aligned; 512 against 6144 x 1024 22, 11; copied by elements they took 12976 and 69).
template <typename TO, int BM, int BN, int RING, int NW, int MINB, int SILU, bool QKV = false, bool DIRECT = true>
__global__ __launch_bounds__(64 * NW, MINB) void gemm_mfma_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const float* __restrict__ bias,
    TO* __restrict__ out, int M, int N, int K, int tiles_m, int tiles_n, int k_per_split, int xcd_m, int xcd_n,
    int rotate, QkvTail tail) {
    constexpr bool PAIR = SILU > 0;
    constexpr int WM = BM / (NW / 2), WN = BN / 2;   // a wave's part: NW / 2 waves down, 2 across
    constexpr int MI = WM / 32, NJ = WN / 32;
    constexpr int LDA = BM / (8 * NW), LD = (BM + BN) / (8 * NW);   // a wave's loads of a stage: LDA of x, then of W
    static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && LD >= 2 && (RING - 2) * LD + (LD + 1) / 2 < 64 && RING >= 2,
                  "the rows of a stage must be whole loads of every wave, the loads in flight no more than can be counted");
    constexpr bool BIG = DIRECT && BM == 256 && BN == 256 && NW == 4, TWO = DIRECT && BM == 128 && BN == 128 && RING == 2;
    constexpr int STAGE = (BM + BN) * 128;   // bytes of a stage: the x rows, then the W rows
    [[maybe_unused]] constexpr int SMEM = gemm_mfma_shared_bytes(BM, BN, RING, QKV);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // Consecutive blocks go to the eight XCDs in turn, and each XCD has an L2 of its own: the blocks
    // of one XCD take a compact part of the tiles, xcd_m parts down by xcd_n across (the host picks
    // the cut that makes the XCDs read the fewest rows of x and W altogether; 0: no cut into equal parts), so
    // that they share what they read through that L2.  (A single row of tiles shares nothing of W and goes as the blocks
    // come.)
    int tile_m, tile_n;
    const int rows_m = tail.tiles ? tail.n_tiles[0] : tiles_m;       // (grouped rows: the grid has blocks for the most tiles there can be)
    if (rows_m > 1) {
        int local, part_m = 0, part_n = 0, per_m = rows_m, per_n = tiles_n;
        const int xcd = blockIdx.x % 8;
        local = blockIdx.x / 8;
        if (xcd_m > 0) {
            per_m /= xcd_m;
            per_n /= xcd_n;
            part_m = (xcd / xcd_n) * per_m;
            part_n = (xcd % xcd_n) * per_n;
        } else {
            // no cut into equal parts: each XCD takes an eighth of the walk below through all tiles (dealt out block by
            // block, every XCD read nearly all of W: 1600 rows against 5120 x 25600 in three cuts, 7 by 20 tiles of
            // 256 x 256: 455 us, then 435; 8192 rows of 32 experts of 2048 x 2048: 137 us, then 122)
            const int all = rows_m * tiles_n, each = all / 8, over = all % 8;
            if (local >= each + (xcd < over)) return;
            local += xcd * each + min(xcd, over);
        }
        // Inside the part the tiles go in bands of 8 tile rows (the last band has what is left), across the band
        // column by column: the 32 or 64 blocks that an XCD runs at a time are then a patch of 8 by 4 or 8
        // tiles, which reads 12 or 16 tiles' worth of rows where a column of 32 reads 33 (what
        // the XCDs fetch through the fabric is what bounds a large product).  With bands of a divisor of the tile rows
        // instead, five tile rows went one after the other, each through all of W: 272 rows
        // against 51200 x 5120 in tiles of 64 rows 470 us, then 266; 528 rows in tiles of 128 rows 476, then 337.
        const int band = local / (8 * per_n), within = local - band * 8 * per_n;
        const int rows = min(8, per_m - band * 8);
        tile_m = part_m + band * 8 + within % rows;
        tile_n = part_n + within / rows;
    } else {
        tile_m = 0;
        tile_n = blockIdx.x;
        if (tile_n >= rows_m * tiles_n) return;
    }
    if (tail.tiles) {
        const int expert = tail.tiles[3 * tile_m], first = tail.tiles[3 * tile_m + 1];
        if (PAIR && tail.row_w) tail.perm += first;        // (from here on by the tile's own rows)
        M = tail.tiles[3 * tile_m + 2];
        x += (long)first * K;
        w += (long)expert * N * K;
        out += (long)first * (PAIR ? N / 2 : N);
        tile_m = 0;
    }
    const int m0 = tile_m * BM, n0 = tail.n_first + tile_n * BN;
    const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
    // (QKV: thread i fetches the position and the slot of the tile's row i now, for the end)
    int my_pos = 0, my_slot = -1;
    if constexpr (QKV) {
        static_assert(!QKV || BM <= 64 * NW, "a thread for every row of the tile");
        if (tid < BM && m0 + tid < M) {
            if (tail.table) my_pos = tail.positions[m0 + tid];
            if (tail.slots) my_slot = tail.slots[m0 + tid];
        }
    }

    // blockIdx.y cuts K: this block sums the k values [k0, k0 + klen) and writes the partial product
    // number blockIdx.y (out is then [splits][M][N]); without a cut k_per_split = K
    const int k0 = blockIdx.y * k_per_split;
    const int klen = K - k0 < k_per_split ? K - k0 : k_per_split;
    const int nk = (klen + 63) / 64;
    // rotate: the block walks its k steps from another start than its neighbours (and wraps round).  Few rows
    // of x against a large matrix: the blocks stream their rows of W in step, and with a row stride that is a
    // power of two all their loads of a moment have the same address bits below the stride, which land on the
    // same few memory channels (the logits' matrix of 151936 x 4096 against 64 rows: 4.4 TB/s, and 5.1 with a
    // row of 4160; where the stride is no such power, walking in step is the quicker: the blocks then share
    // their rows of x through the caches).  The order of a tile's sum is then a function of its place, not of
    // the batch.
    const int rot = rotate ? (tile_n * 5 + (int)blockIdx.y * 3) % nk : 0;
#define QE_KK(kt_) ((kt_) < nk ? ((kt_) + rot < nk ? (kt_) + rot : (kt_) + rot - nk) : (kt_))
    // A stage is 64 values of K of all the tile's rows, 128 bytes a row (a line of the caches) without padding.  The loads
    // go to shared memory directly (no registers, no stores of the waves' own): one instruction
    // brings 8 rows, 16 bytes a lane, side by side.  The eight pieces of a row are exchanged by the row's number
    // (piece p of row r lies at place p ^ (r / 2 % 8)), so that the fragment reads of 16 rows fall into distinct banks;
    // the exchange is made by the addresses that the lanes ask for.
    //
    // The loads are buffer loads: one descriptor for the tile's rows of x and one for its rows of W,
    // each ending with the last row that exists, so that a row beyond the matrix is "out of range"
    // and arrives as zeros by itself.  The thread's byte offset never changes and the stage's k offset
    // is a scalar.  A thread whose piece lies beyond K (in a last stage shorter than 64) picks an
    // offset that is out of range.
    //
    // The loads and the waits for them are written as instructions: the compiler would wait for every load in flight
    // before it reads shared memory.
    const int wave_s = __builtin_amdgcn_readfirstlane(wave);
    const int pc = (lane & 7) ^ ((wave & 1) * 4 + (lane >> 4));            // the lane's piece of its row (of the 8 of an instruction)
    const int a_rows = M - m0 < BM ? M - m0 : BM, b_rows = N - n0 < BN ? N - n0 : BN;
    const unsigned long a_addr = (unsigned long)(x + (long)m0 * K + k0), b_addr = (unsigned long)(w + (long)n0 * K + k0);
    uint4_t rsrc_a, rsrc_b;   // base, base high 16 bits (stride 0), bytes, format: 32-bit raw buffer
    rsrc_a[0] = (unsigned)a_addr; rsrc_a[1] = (unsigned)(a_addr >> 32) & 0xffffu;
    rsrc_a[2] = (unsigned)(((a_rows - 1) * K + klen) * 2); rsrc_a[3] = 0x00020000u;   // up to the last row's last k of this cut
    rsrc_b[0] = (unsigned)b_addr; rsrc_b[1] = (unsigned)(b_addr >> 32) & 0xffffu;
    rsrc_b[2] = (unsigned)(((b_rows - 1) * K + klen) * 2); rsrc_b[3] = 0x00020000u;
#pragma unroll
    for (int c = 0; c < 4; ++c) {   // the same in every lane: into scalar registers
        rsrc_a[c] = __builtin_amdgcn_readfirstlane(rsrc_a[c]);
        rsrc_b[c] = __builtin_amdgcn_readfirstlane(rsrc_b[c]);
    }
    const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) unsigned char*)smem + wave_s * 1024;
#define LOAD_LDS(to_, vo_, rsrc_, soff_) QE_LOAD_TO_SHARED(to_, vo_, rsrc_, soff_, "0", "");
    // waits until at most younger_ loads of the wave are in flight and its reads of shared memory are done, then for
    // the other waves
#define MEET(younger_)                                                                   \
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(younger_) : "memory");

    floatx16 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    // A lane's fragment: row lane % 32, of its 16-wide k step ks the 8 values from 8 (lane / 32) on; that of k step 0, the
    // others: ^ 32 ks
    const int fr = lane & 31;
    const int f0 = fr * 128 + (((lane >> 5) ^ ((fr >> 1) & 7)) * 16);
    if constexpr (BIG) {
        // 256 x 256 by four waves, one wave a SIMD, its accumulators in the 256 AGPRs.  The halves of a wave's rows of x and of W
        // are four regions of a stage, each read once into registers and kept there: a stage is four quarters (a half of x with a
        // half of W, 16 MFMAs), in an order in which one quarter's last operands are no operands of the next, so that
        // each quarter reads the region that is first wanted in the next one or the one after it.  Behind the barrier at its end that
        // region's memory takes the same rows two stages later: seven quarters, over two microseconds, for a load to
        // arrive, and 24 loads of a wave always in flight.  The order alternates: even stages x0 w0, x0 w1, x1 w1, x1 w0,
        // odd ones x0 w1, x0 w0, x1 w0, x1 w1.
        int voff[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                voff[h][i] = ((i / 2) * 128 + h * 64 + (i % 2) * 32 + wave * 8 + (lane >> 3)) * K * 2 + pc * 16;
        bf16x8 fa[2][2][4], fb[2][2][4];
        const unsigned char* const fa0 = smem + (wave >> 1) * 8192;
        const unsigned char* const fb0 = smem + (wave & 1) * 8192;
        // region rg_: 0, 1: the halves of x; 2, 3: of W; its place for a stage of parity st_
#define REGION_AT(rg_, st_) ((((st_) & 1) * 4 + (rg_)) * 16384)
#define LOAD_REGION(rg_, st_, par_, i_)                                                  \
        {                                                                                \
            const int kk = QE_KK(st_);                                                   \
            const int vo = kk * 64 + pc * 8 < klen ? voff[(rg_) & 1][i_] : 0x7fffffff;   \
            const int soff = kk * 128;                                                   \
            const unsigned to = lds0 + REGION_AT(rg_, par_) + (i_) * 4096;               \
            if ((rg_) < 2) LOAD_LDS(to, vo, rsrc_a, soff) else LOAD_LDS(to, vo, rsrc_b, soff) \
        }
#define READ_REGION(rg_, par_, p_)                                                       \
        {                                                                                \
            if ((rg_) < 2) fa[(rg_) & 1][(p_) & 1][(p_) >> 1] = *(const bf16x8*)(fa0 + REGION_AT(rg_, par_) + ((p_) & 1) * 4096 + (f0 ^ (((p_) >> 1) * 32))); \
            else fb[(rg_) & 1][(p_) & 1][(p_) >> 1] = *(const bf16x8*)(fb0 + REGION_AT(rg_, par_) + ((p_) & 1) * 4096 + (f0 ^ (((p_) >> 1) * 32))); \
        }
        // half ha_ of x with half hb_ of W; meanwhile region rrg_ of a stage of parity rpar_ is read and region lrg_ of stage lst_ (parity
        // lpar_) asked for
#define QUAD(ha_, hb_, rrg_, rpar_, lrg_, lst_, lpar_)                                   \
        _Pragma("unroll") for (int sl = 0; sl < 16; ++sl) {                              \
            if (sl < 8) READ_REGION(rrg_, rpar_, sl)                                     \
            acc[(ha_) * 2 + (sl / 2) % 2][(hb_) * 2 + sl % 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16( \
                fb[hb_][sl % 2][sl / 4], fa[ha_][(sl / 2) % 2][sl / 4], acc[(ha_) * 2 + (sl / 2) % 2][(hb_) * 2 + sl % 2], 0, 0, 0); \
            if (sl % 4 == 1) LOAD_REGION(lrg_, lst_, lpar_, sl / 4)                      \
            __builtin_amdgcn_sched_barrier(0);                                           \
        }                                                                                \
        MEET(24)
#define EVEN(st_)                                                                        \
        QUAD(0, 0, 3, 0, 2, (st_) + 2, 0)                                                \
        QUAD(0, 1, 1, 0, 3, (st_) + 2, 0)                                                \
        QUAD(1, 1, 0, 1, 1, (st_) + 2, 0)                                                \
        QUAD(1, 0, 3, 1, 0, (st_) + 3, 1)
#define ODD(st_)                                                                         \
        QUAD(0, 1, 2, 1, 3, (st_) + 2, 1)                                                \
        QUAD(0, 0, 1, 1, 2, (st_) + 2, 1)                                                \
        QUAD(1, 0, 0, 0, 1, (st_) + 2, 1)                                                \
        QUAD(1, 1, 2, 0, 0, (st_) + 3, 0)
        constexpr int first[8] = {0, 2, 3, 1, 0 + 4, 3 + 4, 2 + 4, 1 + 4};      // in the order in which they are read (4: of the second stage)
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) LOAD_REGION(first[r] & 3, first[r] >> 2, first[r] >> 2, i)
        MEET(24)
#pragma unroll
        for (int p = 0; p < 8; ++p) READ_REGION(0, 0, p)
#pragma unroll
        for (int p = 0; p < 8; ++p) READ_REGION(2, 0, p)
        MEET(24)
#pragma unroll
        for (int i = 0; i < 4; ++i) LOAD_REGION(0, 2, 0, i)
        MEET(24)
        int st = 0;
        for (; st + 1 < nk; st += 2) {
            EVEN(st)
            ODD(st + 1)
        }
        if (st < nk) { EVEN(st) }
#undef EVEN
#undef ODD
#undef QUAD
#undef READ_REGION
#undef LOAD_REGION
#undef REGION_AT
    } else if constexpr (TWO) {
        // 128 x 128 by four waves in the same way, with room for two blocks a compute unit (64 KB each): half stages (a half of x with
        // all of W, 8 MFMAs), the next stage's W in registers of its own, and three half stages for a load to arrive.  (As a
        // ring of whole stages as below, which leaves one stage: 512 rows against 4096 x 4096 54 us, now 37; 2048 against
        // 6144 x 2048 57, now 51.)
        int voff[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 2; ++i) voff[h][i] = (i * 64 + h * 32 + wave * 8 + (lane >> 3)) * K * 2 + pc * 16;
        bf16x8 fa[2][4], fb[2][2][4];
        const unsigned char* const fa0 = smem + (wave >> 1) * 4096;
        const unsigned char* const fb0 = smem + (wave & 1) * 4096;
#define REGION_AT(rg_, st_) ((((st_) & 1) * 4 + (rg_)) * 8192)
#define LOAD_REGION(rg_, st_, par_, i_)                                                  \
        {                                                                                \
            const int kk = QE_KK(st_);                                                   \
            const int vo = kk * 64 + pc * 8 < klen ? voff[(rg_) & 1][i_] : 0x7fffffff;   \
            const int soff = kk * 128;                                                   \
            const unsigned to = lds0 + REGION_AT(rg_, par_) + (i_) * 4096;               \
            if ((rg_) < 2) LOAD_LDS(to, vo, rsrc_a, soff) else LOAD_LDS(to, vo, rsrc_b, soff) \
        }
#define READ_A(h_, par_, ks_) fa[h_][ks_] = *(const bf16x8*)(fa0 + REGION_AT(h_, par_) + (f0 ^ ((ks_) * 32)));
#define READ_B(h_, par_, ks_) fb[par_][h_][ks_] = *(const bf16x8*)(fb0 + REGION_AT(2 + (h_), par_) + (f0 ^ ((ks_) * 32)));
#define HALF_STAGE(ha_, par_, st_)                                                       \
        _Pragma("unroll") for (int sl = 0; sl < 8; ++sl) {                               \
            if (sl % 2 == 0) { READ_A((ha_) ^ 1, (ha_) ? (par_) ^ 1 : (par_), sl / 2) }  \
            else { READ_B(ha_, (par_) ^ 1, sl / 2) }                                     \
            acc[ha_][sl % 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[par_][sl % 2][sl / 2], fa[ha_][sl / 2], acc[ha_][sl % 2], 0, 0, 0); \
            if (sl == 1) LOAD_REGION(ha_, (st_) + 2, par_, 0)                            \
            if (sl == 3) LOAD_REGION(ha_, (st_) + 2, par_, 1)                            \
            if (sl == 5) LOAD_REGION(3 - (ha_), (st_) + 2 + (ha_), (par_) ^ (ha_), 0)    \
            if (sl == 7) LOAD_REGION(3 - (ha_), (st_) + 2 + (ha_), (par_) ^ (ha_), 1)    \
            __builtin_amdgcn_sched_barrier(0);                                           \
        }                                                                                \
        MEET(8)
        constexpr int first[8] = {0, 2, 3, 1, 2 + 4, 0 + 4, 3 + 4, 1 + 4};
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
            for (int i = 0; i < 2; ++i) LOAD_REGION(first[r] & 3, first[r] >> 2, first[r] >> 2, i)
        MEET(10)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            READ_A(0, 0, ks)
            READ_B(0, 0, ks)
            READ_B(1, 0, ks)
        }
        MEET(10)
        LOAD_REGION(2, 2, 0, 0)
        LOAD_REGION(2, 2, 0, 1)
        MEET(8)
        int st = 0;
        for (; st + 1 < nk; st += 2) {
            HALF_STAGE(0, 0, st)
            HALF_STAGE(1, 0, st)
            HALF_STAGE(0, 1, st + 1)
            HALF_STAGE(1, 1, st + 1)
        }
        if (st < nk) {
            HALF_STAGE(0, 0, st)
            HALF_STAGE(1, 0, st)
        }
#undef HALF_STAGE
#undef READ_A
#undef READ_B
#undef LOAD_REGION
#undef REGION_AT
    } else {
    // The other shapes: a ring of RING stages, three where two blocks of 64 x 128 share a unit and for 256 x 128.
    int voff[LD];                                          // of the wave's instructions of a stage: LDA for x, then for W
#pragma unroll
    for (int i = 0; i < LD; ++i)
        voff[i] = (((i < LDA ? i : i - LDA) * NW + wave) * 8 + (lane >> 3)) * K * 2 + pc * 16;
    // the wave's i_-th load of stage st_, into the ring's place that begins at byte at_; through registers: the piece that was asked for a
    // stage ago goes there, and the next stage's is asked for
    [[maybe_unused]] uint4_t held[LD];
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t piece_a = __builtin_amdgcn_make_buffer_rsrc((void*)a_addr, 0, rsrc_a[2], 0x00020000);
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t piece_b = __builtin_amdgcn_make_buffer_rsrc((void*)b_addr, 0, rsrc_b[2], 0x00020000);
#define PLACE(at_, i_) ((at_) + ((i_) < LDA ? (i_) * NW * 1024 : BM * 128 + ((i_) - LDA) * NW * 1024))
#define HOLD_PIECE(st_, i_)                                                              \
    {                                                                                    \
        const int kk = QE_KK(st_);                                                       \
        const int vo = kk * 64 + pc * 8 < klen ? voff[i_] : 0x7fffffff;                  \
        held[i_] = __builtin_amdgcn_raw_buffer_load_b128((i_) < LDA ? piece_a : piece_b, vo, kk * 128, 0); \
    }
#define PUT_PIECE(at_, i_) *(uint4_t*)(smem + PLACE(at_, i_) + wave * 1024 + lane * 16) = held[i_];
#define LOAD_PIECE(st_, at_, i_)                                                         \
    {                                                                                    \
        if constexpr (!DIRECT) {                                                         \
            PUT_PIECE(at_, i_)                                                           \
            HOLD_PIECE((st_) + 1, i_)                                                    \
        } else {                                                                         \
            const int kk = QE_KK(st_);                                                   \
            const int vo = kk * 64 + pc * 8 < klen ? voff[i_] : 0x7fffffff;              \
            if ((i_) < LDA) LOAD_LDS(lds0 + PLACE(at_, i_), vo, rsrc_a, kk * 128) else LOAD_LDS(lds0 + PLACE(at_, i_), vo, rsrc_b, kk * 128) \
        }                                                                                \
    }
    const unsigned char *a_frag[4], *b_frag[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        a_frag[ks] = smem + wm * 128 + (f0 ^ (32 * ks));
        b_frag[ks] = smem + (BM + wn) * 128 + (f0 ^ (32 * ks));
    }
    bf16x8 fa[2][MI], fb[2][NJ];
    constexpr int R = MI + NJ;                             // fragments of a k step: of W and of x in turn
#define READ_FRAG(ks_, at_, p_)                                                          \
    {                                                                                    \
        const bool of_a = (p_) < 2 * MI && (p_) < 2 * NJ ? (p_) % 2 : MI > NJ;           \
        const int i_ = (p_) < 2 * MI && (p_) < 2 * NJ ? (p_) / 2 : (p_) - (MI > NJ ? NJ : MI); \
        if (of_a) fa[(ks_) & 1][i_ < MI ? i_ : 0] = *(const bf16x8*)(a_frag[ks_] + (at_) + i_ * 4096); \
        else fb[(ks_) & 1][i_ < NJ ? i_ : 0] = *(const bf16x8*)(b_frag[ks_] + (at_) + i_ * 4096); \
    }
    // The MFMAs of k step ks_ of a stage, and between them (a wave issues in order) what is wanted next: the fragments of
    // the k step behind it, from place rd_, and the wave's loads [l0_, l1_) of stage st_ to place ld_.
    constexpr int PER = MI * NJ, RSLOTS = PER >= 2 * R ? R : (PER + 1) / 2;
#define K_STEP(ks_, rd_, st_, ld_, l0_, l1_)                                             \
    _Pragma("unroll") for (int sl = 0; sl < PER; ++sl) {                                 \
        _Pragma("unroll") for (int p = 0; p < R; ++p)                                    \
            if (p * RSLOTS / R == sl) READ_FRAG(((ks_) + 1) & 3, rd_, p)                 \
        acc[sl / NJ][sl % NJ] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[(ks_) & 1][sl % NJ], fa[(ks_) & 1][sl / NJ], acc[sl / NJ][sl % NJ], 0, 0, 0); \
        _Pragma("unroll") for (int p = (l0_); p < (l1_); ++p)                            \
            if ((p - (l0_)) * PER / ((l1_) > (l0_) ? (l1_) - (l0_) : 1) == sl) LOAD_PIECE(st_, ld_, p)       \
        __builtin_amdgcn_sched_barrier(0);                                               \
    }
    // A place of the ring is read for the last time in the third k step of its stage (by then the last k step's fragments are
    // in registers); behind the barrier there it takes the stage RING later: half of that stage's loads go with
    // the last k step, half with the first of the next stage.
    constexpr int HALF = (LD + 1) / 2;
    if constexpr (!DIRECT) {
#pragma unroll
        for (int i = 0; i < LD; ++i) HOLD_PIECE(0, i)
    }
#pragma unroll
    for (int st = 0; st < RING; ++st)
#pragma unroll
        for (int i = 0; i < LD; ++i)
            if (st + 1 < RING || i < HALF) LOAD_PIECE(st, st * STAGE, i)
    MEET((RING - 2) * LD + HALF)
#pragma unroll
    for (int p = 0; p < R; ++p) READ_FRAG(0, 0, p)
    int at = 0, before = (RING - 1) * STAGE;               // this stage's place, and that of the stage before
    for (int st = 0; st < nk; ++st) {
        const int next = at + STAGE == RING * STAGE ? 0 : at + STAGE;
        K_STEP(0, at, st + RING - 1, before, HALF, LD)
        K_STEP(1, at, 0, 0, 0, 0)
        K_STEP(2, at, 0, 0, 0, 0)
        MEET((RING - 2) * LD)
        K_STEP(3, next, st + RING, at, 0, HALF)
        before = at;
        at = next;
    }
#undef K_STEP
#undef LOAD_PIECE
#undef HOLD_PIECE
#undef PUT_PIECE
#undef PLACE
#undef READ_FRAG
    }
    MEET(0)                                                // (what was asked for beyond the end arrives too, before the memory is used again)
#undef QE_KK
#undef LOAD_LDS
#undef MEET

    // The MFMA is given the W rows as its first operand and the x rows as its second, so its
    // result is the tile transposed: a lane holds, for the token row m = lane % 32, the outputs
    // n = 8 b + 4 (lane / 32) + r (e = 4 b + r), four consecutive n at a time.  Stored from there,
    // one instruction would touch 32 rows with 16 bytes each.  So each wave turns its part round
    // in shared memory, a strip of 32 rows at a time (the staging buffers are free: every wave has
    // passed the loop's last barrier): it writes the strip as rows and reads it back 16 bytes a
    // lane, so that a store instruction covers whole rows of the strip.
    if constexpr (QKV) {
        // The whole tile goes to shared memory as bfloat16 rows (the staging buffers are free), then
        // 16 lanes take a row of a head each, as in qk_rope_store_vec_kernel: lane j has the features
        // 4 j .. 4 j + 3 and 64 + 4 j .. 64 + 4 j + 3, the two halves that rotate together.
        constexpr int TROW = BN * 2 + 16;                  // bytes of a row of the tile
        static_assert(BM * TROW <= SMEM && BN % 128 == 0, "the tile must fit the staging buffers, in whole heads");
        // positions and slots of the tile's rows, once, into shared memory behind the tile
        int* pos_sh = (int*)(smem + BM * TROW);
        int* slot_sh = pos_sh + BM;
        static_assert(BM * TROW + 2 * BM * 4 <= SMEM, "the rows' positions and slots must fit too");
        if (tid < BM) { pos_sh[tid] = my_pos; slot_sh[tid] = my_slot; }
        __syncthreads();
        const int D = 128, half = 64;
        const int j16 = tid % 16;
        const long page_stride = 2L * tail.Hkv * tail.P * D;
        constexpr int GROUPS = 64 * NW / 16, ITEMS = BM * (BN / 128);
        constexpr int NIT = (ITEMS + GROUPS - 1) / GROUPS;         // items a group of 16 lanes takes, one after the other
        constexpr int CHUNK = NIT < 8 ? NIT : 8;
        // The only loads from memory in the items' loop are the table's rows, and an item is short
        // beside a trip to memory: the rows of eight items are asked for at once, the first eight
        // before the tile is written to shared memory.
        float c[CHUNK][4], sn[CHUNK][4];
#define LOAD_TABLE_ROWS(it0_)                                                            \
        _Pragma("unroll") for (int k = 0; k < CHUNK; ++k) {                              \
            const int idx = tid / 16 + ((it0_) + k) * GROUPS;                            \
            _Pragma("unroll") for (int e = 0; e < 4; ++e) { c[k][e] = 1.f; sn[k][e] = 0.f; } \
            if (tail.table && idx < ITEMS && n0 / 128 + idx / BM < tail.Hq + tail.Hkv) {  \
                const float* cs = tail.table + (long)pos_sh[idx % BM] * D;               \
                Vec4<float>::load(cs + 4 * j16, c[k]);                                   \
                Vec4<float>::load(cs + half + 4 * j16, sn[k]);                           \
            }                                                                            \
        }
        LOAD_TABLE_ROWS(0)
        float wq_a[4], wq_b[4], wk_a[4], wk_b[4];
        if (tail.q_w) {
            Vec4<float>::load(tail.q_w + 4 * j16, wq_a);
            Vec4<float>::load(tail.q_w + half + 4 * j16, wq_b);
            Vec4<float>::load(tail.k_w + 4 * j16, wk_a);
            Vec4<float>::load(tail.k_w + half + 4 * j16, wk_b);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int bq = 0; bq < 4; ++bq) {
                    const int nl = wn + j * 32 + 8 * bq + 4 * (lane >> 5);
                    float v[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = acc[i][j][4 * bq + r];
                    if (bias) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) v[r] += bias[n0 + nl + r < N ? n0 + nl + r : N - 1];
                    }
                    Vec4<bf16_t>::store((bf16_t*)(smem + (wm + i * 32 + (lane & 31)) * TROW) + nl, v);
                }
        __syncthreads();
        for (int it0 = 0; it0 < NIT; it0 += CHUNK) {
            if (it0 > 0) { LOAD_TABLE_ROWS(it0) }
#pragma unroll
            for (int k = 0; k < CHUNK; ++k) {
                const int idx = tid / 16 + (it0 + k) * GROUPS;
                if (idx >= ITEMS) continue;
                const int hd = idx / BM, row = idx % BM;
                const int m = m0 + row, head = n0 / 128 + hd;
                if (m < M && head < tail.Hq + tail.Hkv) {                   // (values: below, by tiles)
                    const bool is_q = head < tail.Hq;
                    const bf16_t* src = (const bf16_t*)(smem + row * TROW) + hd * 128;
                    float a[4], b[4];
                    Vec4<bf16_t>::load(src + 4 * j16, a);
                    Vec4<bf16_t>::load(src + half + 4 * j16, b);
                    if (tail.q_w) {
                        float ss = 0.f;
#pragma unroll
                        for (int e = 0; e < 4; ++e) ss += a[e] * a[e] + b[e] * b[e];
                        ss = row16_sum(ss);                                  // (the item's 16 lanes are a row)
                        const float rstd = rsqrtf(ss / (float)D + tail.eps);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            a[e] = a[e] * rstd * (is_q ? wq_a[e] : wk_a[e]);
                            b[e] = b[e] * rstd * (is_q ? wq_b[e] : wk_b[e]);
                        }
                    }
                    if (tail.table) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) rotate_pair(c[k][e], sn[k][e], a[e], b[e]);
                    }
                    bf16_t* dst = nullptr;
                    if (is_q) {
                        dst = tail.q_out + ((long)m * tail.Hq + head) * D;
                    } else {
                        const int sl = slot_sh[row];
                        if (sl >= 0) dst = tail.cache + (long)(sl >> tail.lp) * page_stride + ((long)(head - tail.Hq) * tail.P + (sl & (tail.P - 1))) * D;
                    }
                    if (dst) {
                        Vec4<bf16_t>::store(dst + 4 * j16, a);
                        Vec4<bf16_t>::store(dst + half + 4 * j16, b);
                    }
                }
            }
        }
#undef LOAD_TABLE_ROWS
        // values: where eight tokens' slots lie side by side from a multiple of eight on, eight tokens of a feature are one
        // 16-byte store into the transposed value tile [D][P], whichever row of the tile the first of them is (a prompt's portion
        // begins behind any number of other rows); the other rows' values are stored one by one.  Which rows begin such a
        // piece and which stand alone is found once, by a thread a row, and listed in the order of the rows.  (With
        // pieces only where sixteen rows from a multiple of sixteen fill a page, 2048 rows of 4096 x 1024 behind ten others took
        // 53 us, now 26, and 528 of 6144 x 4096 60, now 50.)
        int* pieces = slot_sh + BM;
        int* singles = pieces + BM / 8;
        int* counts = singles + BM;                       // of the pieces, then of the single rows, found by each wave
        static_assert(BM * TROW + 2 * BM * 4 + (BM + BM / 8 + 8) * 4 <= SMEM && BM <= 256, "the lists must fit too");
        const bool has_values = tail.slots && n0 / 128 + BN / 128 > tail.Hq + tail.Hkv;   // the same for the whole block
        int n_pieces = 0, n_singles = 0;
        if (has_values) {
            const auto begins = [&](int r) {
                const int s0 = slot_sh[r];
                bool run = s0 >= 0 && (s0 & 7) == 0 && r + 8 <= BM;
#pragma unroll
                for (int i = 1; i < 8; ++i) run = run && slot_sh[min(r + i, BM - 1)] == s0 + i;
                return run;
            };
            bool piece = false, single = false;
            if (tid < BM) {
                const int sl = slot_sh[tid], first = tid - (sl & 7);
                piece = begins(tid);
                single = sl >= 0 && !(first >= 0 && slot_sh[max(first, 0)] == (sl & ~7) && begins(max(first, 0)));
            }
            const unsigned long long mp = __ballot(piece), msg = __ballot(single), below = (1ull << lane) - 1;
            if (tid < BM && lane == 0) {
                counts[wave] = __popcll(mp);
                counts[4 + wave] = __popcll(msg);
            }
            __syncthreads();
            int bp = 0, bs = 0;
#pragma unroll
            for (int v = 0; v < BM / 64; ++v) {
                if (v == wave) { bp = n_pieces; bs = n_singles; }
                n_pieces += counts[v];
                n_singles += counts[4 + v];
            }
            if (piece) pieces[bp + __popcll(mp & below)] = tid;
            if (single) singles[bs + __popcll(msg & below)] = tid;
            __syncthreads();
        }
        for (int hd = 0; hd < BN / 128; ++hd) {
            const int kh = n0 / 128 + hd - tail.Hq - tail.Hkv;
            if (!has_values || kh < 0 || kh >= tail.Hkv) continue;      // the same for the whole block
            bf16_t* const plane = tail.cache + ((long)(tail.Hkv + kh) * tail.P) * D;
            // a thread: the features d and d + 1 of one of two neighbouring pieces (two features at a time: half the reads
            // from shared memory)
            for (int idx = tid; idx < (n_pieces + 1) / 2 * D; idx += 64 * NW) {
                const int k = idx / D * 2 + idx % 2, d = idx % D / 2 * 2;
                if (k >= n_pieces) continue;
                const int r0 = pieces[k], s0 = slot_sh[r0];
                Piece16 lo, hi;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const unsigned two = *(const unsigned*)(smem + (r0 + e) * TROW + (hd * 128 + d) * 2);
                    lo.e[e] = (unsigned short)(two & 0xffffu);
                    hi.e[e] = (unsigned short)(two >> 16);
                }
                bf16_t* vt = plane + (long)(s0 >> tail.lp) * page_stride + (s0 & (tail.P - 1));
                *(uint4_t*)(vt + (long)d * tail.P) = lo.q;
                *(uint4_t*)(vt + (long)(d + 1) * tail.P) = hi.q;
            }
            for (int idx = tid; idx < n_singles * (D / 2); idx += 64 * NW) {
                const int r0 = singles[idx / (D / 2)], d = idx % (D / 2) * 2, s0 = slot_sh[r0];
                bf16_t* vt = plane + (long)(s0 >> tail.lp) * page_stride + (s0 & (tail.P - 1));
                const bf16_t* from = (const bf16_t*)(smem + r0 * TROW + (hd * 128 + d) * 2);
                vt[(long)d * tail.P] = from[0];
                vt[(long)(d + 1) * tail.P] = from[1];
            }
        }
        return;
    }
    const int NO = PAIR ? N / 2 : N;                       // width of the output
    constexpr int WNO = PAIR ? WN / 2 : WN;                // output columns of a wave's strip
    constexpr int ESZ = (int)sizeof(TO);
    constexpr int CH = 16 / ESZ;                           // outputs in 16 bytes
    constexpr int CPR = WNO / CH;                          // 16-byte chunks in a row of the strip
    constexpr int SROW = WNO * ESZ + 16;                   // bytes of a staged row
    static_assert(NW * 32 * SROW <= SMEM, "the strips of the waves must fit the staging buffers");
    unsigned char* strip = smem + wave * 32 * SROW;
    const int no0 = PAIR ? (n0 + wn) / 2 : n0 + wn;        // first output column of the wave's strip
    const bool vec_ok = (NO % CH) == 0 && (((unsigned long)out) & 15) == 0;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        __builtin_amdgcn_sched_barrier(0);   // one strip after the other: nothing of the next is computed early
        float row_w = 1.f;
        if (PAIR && tail.row_w) {
            const int m = wm + i * 32 + (lane & 31);       // (a grouped tile starts at row 0 of its rows)
            row_w = tail.row_w[tail.perm[m < M ? m : M - 1]];
        }
#pragma unroll
        for (int j = 0; j < NJ; j += (PAIR ? 2 : 1))
#pragma unroll
            for (int bq = 0; bq < 4; ++bq) {
                const int nl = (PAIR ? j * 16 : j * 32) + 8 * bq + 4 * (lane >> 5);   // column within the strip
                float v[4], bg[4], bu[4];
                if (SILU == 2) {                           // (columns beyond the output are never stored: any bias does)
                    const int ng = min(n0 + wn + j * 32 + 8 * bq + 4 * (lane >> 5), N - 36);
                    Vec4<float>::load(bias + ng, bg);
                    Vec4<float>::load(bias + ng + 32, bu);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (PAIR) {
                        float gt = acc[i][j][4 * bq + r], up = acc[i][j + (PAIR ? 1 : 0)][4 * bq + r];
                        float slope = 1.f;
                        if (SILU == 2) { gt += bg[r]; up += bu[r]; }
                        if (tail.row_w) { gt *= row_w; up *= row_w; }
                        if (tail.act_limit > 0.f) {
                            gt = fminf(gt, tail.act_limit);
                            up = fminf(fmaxf(up, -tail.act_limit), tail.act_limit) + 1.f;
                            slope = tail.act_slope;
                        }
                        v[r] = gt * __builtin_amdgcn_rcpf(1.f + __expf(-slope * gt)) * up;   // rcp: within 1 ulp
                    } else {
                        v[r] = acc[i][j][4 * bq + r];
                        if (tail.relu_sq) { const float z = fmaxf(v[r], 0.f); v[r] = z * z; }
                        if (SILU < 0) v[r] = gelu_of(v[r]);
                    }
                }
                if (!PAIR && bias && blockIdx.y == 0) {                       // (a column beyond the output is never stored: any bias does)
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] += bias[no0 + nl + r < NO ? no0 + nl + r : NO - 1];
                }
                Vec4<TO>::store((TO*)(strip + (lane & 31) * SROW) + nl, v);
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // the wave's writes before its reads
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int c = lane; c < 32 * CPR; c += 64) {
            const int row = c / CPR, col = (c % CPR) * CH;
            const int m = m0 + wm + i * 32 + row, n = no0 + col;
            if (m >= M || n >= NO) continue;
            const uint4_t piece = *(const uint4_t*)(strip + row * SROW + col * ESZ);
            TO* o = out + ((long)blockIdx.y * M + m) * NO + n;
            if (vec_ok) {
                *(uint4_t*)o = piece;                      // n + CH <= NO: both are multiples of CH
            } else {
                const TO* pv = (const TO*)&piece;
#pragma unroll
                for (int e = 0; e < CH; ++e) if (n + e < NO) o[e] = pv[e];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // the reads before the next strip's writes
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

bool qe_gemm_mfma_ok(int M, int N, int K, int dt_a, int dt_w) {
    return dt_a == QE_BF16 && dt_w == QE_BF16 && M > 16 && K % 8 == 0 && K >= 64;
}

// The columns tail.n_first .. tail.n_first + n_cols - 1 of the product (rounded up to whole tiles).
template <typename TO, int BM, int BN, int RING, int NW, int MINB, int SILU, bool QKV = false, bool DIRECT = true>
static int launch_mfma(const void* x, const void* w, const float* bias, void* out, int M, int N, int K,
                       int n_cols, int splits, hipStream_t stream, const QkvTail& tail) {
    if constexpr (DIRECT) {
        if (((unsigned long)x | (unsigned long)w) & 15)
            return launch_mfma<TO, BM, BN, BM == 64 || BN < BM ? 3 : 2, NW, BM <= 128 ? 2 : 1, SILU, QKV, false>(x, w, bias, out, M, N, K, n_cols, splits,
                                                                                                      stream, tail);
    }
    const int tiles_m = qe_cdiv(M, BM), tiles_n = qe_cdiv(n_cols, BN);
    const long blocks = (long)tiles_m * tiles_n;
    QE_REQUIRE(blocks <= 2147483647L, "mfma gemm: too many tiles");
    const size_t shmem = gemm_mfma_shared_bytes(BM, BN, RING, QKV);
    QE_RAISE_SHARED((gemm_mfma_kernel<TO, BM, BN, RING, NW, MINB, SILU, QKV, DIRECT>), shmem);
    // a cut of K is a multiple of 64 long (the last may be shorter)
    const int k_per_split = splits > 1 ? qe_cdiv(qe_cdiv(K, splits), 64) * 64 : K;
    QE_REQUIRE(splits >= 1 && splits <= 65535 && (long)(splits - 1) * k_per_split < K,
               "mfma gemm: K=%d cannot be cut into %d parts", K, splits);
    // the eight XCDs as a by b parts of the tiles (a b = 8): every XCD reads M / a rows of x and
    // N / b rows of W, so all of them together b M + a N rows
    int xcd_m = 0, xcd_n = 0;
    long fewest = 0;
    for (int a = 1; a <= 8; a *= 2) {
        const int b = 8 / a;
        if (tiles_m % a || tiles_n % b) continue;
        const long rows = (long)b * M + (long)a * n_cols;
        if (xcd_m == 0 || rows < fewest) { xcd_m = a; xcd_n = b; fewest = rows; }
    }
    gemm_mfma_kernel<TO, BM, BN, RING, NW, MINB, SILU, QKV, DIRECT><<<dim3((unsigned)blocks, (unsigned)splits), 64 * NW, shmem, stream>>>(
        (const bf16_t*)x, (const bf16_t*)w, bias, (TO*)out, M, N, K, tiles_m, tiles_n, k_per_split, xcd_m, xcd_n,
        (!QKV && M <= 64 && (K * 2) % 8192 == 0) ? 1 : 0, tail);
    QE_LAUNCH_CHECK();
    return 0;
}

// Rows grouped by expert against one matrix per expert (see QkvTail): tiles of 128 x 128.
template <typename TO, int SILU, bool DIRECT = true>
static int launch_grouped(const void* x, const void* w, void* out, const int* tiles, const int* n_tiles,
                          int max_tiles, int N, int K, float limit, float slope, hipStream_t stream, int relu_sq = 0,
                          const float* row_w = nullptr, const int* perm = nullptr) {
    constexpr int BM = 128, BN = 128, RING = 2, NW = 4, MINB = 2;
    if constexpr (DIRECT) {
        if (((unsigned long)x | (unsigned long)w) & 15)
            return launch_grouped<TO, SILU, false>(x, w, out, tiles, n_tiles, max_tiles, N, K, limit, slope, stream, relu_sq, row_w, perm);
    }
    const int tiles_n = qe_cdiv(N, BN);
    const long blocks = (long)max_tiles * tiles_n;
    QE_REQUIRE(blocks > 0 && blocks <= 2147483647L, "mfma gemm (grouped): too many tiles");
    const size_t shmem = gemm_mfma_shared_bytes(BM, BN, RING, false);
    QE_RAISE_SHARED((gemm_mfma_kernel<TO, BM, BN, RING, NW, MINB, SILU, false, DIRECT>), shmem);
    QkvTail tail{};
    tail.tiles = tiles;
    tail.n_tiles = n_tiles;
    tail.act_limit = limit;
    tail.act_slope = slope;
    tail.relu_sq = relu_sq;
    tail.row_w = row_w;
    tail.perm = perm;
    gemm_mfma_kernel<TO, BM, BN, RING, NW, MINB, SILU, false, DIRECT><<<dim3((unsigned)blocks, 1), 64 * NW, shmem, stream>>>(
        (const bf16_t*)x, (const bf16_t*)w, nullptr, (TO*)out, 0, N, K, max_tiles, tiles_n, K, 0, 0, 0, tail);
    QE_LAUNCH_CHECK();
    return 0;
}

// x [rows, K] in the order of the tiles (an expert's rows side by side), w [E, N, K], out [rows, N] (silu: w's
// gate and up rows interleaved in blocks of 32, out [rows, N / 2], with the clamped activation when limit > 0; row i of
// x is then taken row_w[perm[i]] times, if row_w is given).
extern "C" int qe_gemm_mfma_grouped(const void* x, const void* w, void* out, const int* tiles, const int* n_tiles,
                                    int max_tiles, int N, int K, int silu, float limit, float slope, int dt_o,
                                    const float* row_w, const int* perm, hipStream_t stream) {
    QE_REQUIRE(K % 8 == 0 && K >= 64, "mfma gemm (grouped): K=%d", K);
    QE_REQUIRE(silu != 1 || N % 64 == 0, "mfma gemm (grouped): gate|up rows in blocks of 32");
    QE_REQUIRE(!row_w || (silu == 1 && perm), "mfma gemm (grouped): row factors go with gate|up rows and the rows' order");
    if (max_tiles == 0) return 0;
    if (silu == 2) {       // one matrix an expert, the result relu(.)^2
        QE_REQUIRE(dt_o == QE_BF16, "mfma gemm (grouped): the activation is stored in bfloat16");
        return launch_grouped<bf16_t, 0>(x, w, out, tiles, n_tiles, max_tiles, N, K, 0.f, 1.f, stream, 1);
    }
    if (silu) {
        QE_REQUIRE(dt_o == QE_BF16, "mfma gemm (grouped): the activation is stored in bfloat16");
        return launch_grouped<bf16_t, 1>(x, w, out, tiles, n_tiles, max_tiles, N, K, limit, slope, stream, 0, row_w, perm);
    }
    if (dt_o == QE_F32) return launch_grouped<float, 0>(x, w, out, tiles, n_tiles, max_tiles, N, K, 0.f, 1.f, stream);
    return launch_grouped<bf16_t, 0>(x, w, out, tiles, n_tiles, max_tiles, N, K, 0.f, 1.f, stream);
}
extern "C" int qe_gemm_mfma_grouped_tile_rows() { return 128; }

// The tile shape for a product in S cuts of K, and the microseconds it is taken to need (what the caller then does with
// partial products left out).
float qe_gemm_mfma_shape(int M, int N, int K, int splits, int* tile, bool largest = true) {
    // The busiest compute unit decides: its number of tiles (they are dealt out in turn) times what a tile costs, its
    // operations at the rate that the shape reaches in long products (256 x 256: 1.27 PFLOP/s over the chip, 256 x 128
    // 1.18, 128 x 128 1.07, 64 x 128 0.78) and 2.6 microseconds for the first trip to memory and the result's way out.
    // 128 x 128 and 64 x 128 reach their rates with two blocks on a compute unit: where the busiest unit gets an odd number of
    // them, the last runs alone and takes longer.  A chip with idle
    // units runs the others faster (two and a half times, were nearly all idle).  A shape is never taller than the rows need.
    // Against the best of all shapes (and, for a branch's last product, cuts) in products of 1024 to 51200 by 1024 to
    // 25600 with 80 to 3300 rows, 2900 measured one by one on rows that are in no L2 and weights that are in no cache, what this picks was
    // 0.3 % slower in the mean; in 639 others with 65 to 8192 rows, back to back and a branch's with its norm, 1.5 %, and a quarter at the most
    // (3300 to 4700 rows against a K of 1024, which mostly go in two launches: first_columns).
    const long cus = 256;
    struct Shape { int tile, bm, bn; float rate, alone_first, alone_later; };
    const Shape shapes[4] = {{64, 64, 128, 0.78f, 0.f, 0.15f}, {128, 128, 128, 1.07f, 0.05f, 0.41f},
                             {256, 256, 128, 1.18f, 0.f, 0.f}, {512, 256, 256, 1.27f, 0.f, 0.f}};
    const long cut = (long)qe_cdiv(qe_cdiv(K, splits), 64) * 64;
    float best = 0.f;
    *tile = 0;
    for (const Shape& sh : shapes) {
        if (sh.tile != 64 && M <= sh.bm / 2) continue;
        if (sh.tile == 512 && !largest) continue;
        const long blocks = (long)qe_cdiv(M, sh.bm) * qe_cdiv(N, sh.bn) * splits;
        const long turns = qe_cdiv(blocks, cus);
        const float alone = turns == 1 ? sh.alone_first : (turns % 2 ? sh.alone_later : 0.f);
        const float busy = (float)blocks / (float)(turns * cus);
        const float one = (float)(cut * sh.bm * sh.bn) * (2e-9f * (float)cus) / sh.rate;
        const float cost = ((float)turns + alone) * (one * (0.4f + 0.6f * busy) + 2.6f);
        if (*tile == 0 || cost < best) { *tile = sh.tile; best = cost; }
    }
    return best;
}

static int choose_tile(int M, int N, int K, int splits, bool largest = true) {
    int tile;
    qe_gemm_mfma_shape(M, N, K, splits, &tile, largest);
    return tile;
}

// Where the last turn of a product's tiles would leave most units idle, the columns that fill the turns before it go first, and the
// rest in a launch and a shape of its own: the number of the first columns, a multiple of 256, or 0; and what all that is taken to need.  Three
// microseconds for the second launch; less than 3 % is not worth it (4 to 8 us and 3 to 10 % were tried and leave more behind).  Of 639 products
// of 65 to 8192 rows 61 go in two, 57 of them faster than in one, a tenth in the mean: 4628 rows against 4096 x 1024 55.1 us, in two 47.3; 2048 against
// 10240 x 5120 225, 187; 1024 against 24576 x 4096 187, 174; 3300 against 5120 x 25600 in one part 1047, 806.  The four others are misjudged: 2600 rows
// against 6144 x 1024 37.5, 44.8, against 6144 x 4096 131, 139; 300 against 24576 x 4096 89, 100, against 51200 x 5120 224, 240.
static int first_columns(int M, int N, int K, bool largest = true, float* time = nullptr) {
    int tile;
    const float whole = qe_gemm_mfma_shape(M, N, K, 1, &tile, largest);
    float best = 0.97f * whole;
    int cut = 0;
    const int bms[4] = {64, 128, 256, 256}, bns[4] = {128, 128, 128, 256};
    for (int i = 0; i < 4; ++i) {
        const long tiles_m = qe_cdiv(M, bms[i]), turns = tiles_m * qe_cdiv(N, bns[i]) / 256;
        const long n1 = turns * 256 / tiles_m * bns[i] / 256 * 256;
        if (n1 <= 0 || n1 >= N) continue;
        const float t = qe_gemm_mfma_shape(M, (int)n1, K, 1, &tile, largest) + qe_gemm_mfma_shape(M, N - (int)n1, K, 1, &tile, largest) + 3.f;
        if (t < best) { best = t; cut = (int)n1; }
    }
    if (time) *time = cut ? best : whole;
    return cut;
}

// The microseconds that a product without a cut of K is taken to need, in one launch or in two.
float qe_gemm_mfma_uncut(int M, int N, int K) {
    float time;
    first_columns(M, N, K, true, &time);
    return time;
}

// The same for a caller that wants to know: the number of columns that a product of more than 64 rows gives a launch of their own, or 0
// (gelu: of one with that epilogue).
extern "C" int qe_gemm_first_columns(int M, int N, int K, int gelu) {
    return M > 64 && N > 0 && K >= 64 ? first_columns(M, N, K, !gelu) : 0;
}

template <typename TO, int SILU>
static int pick_mfma(const void* x, const void* w, const float* bias, void* out, int M, int N, int K,
                     int tile, int splits, hipStream_t stream, int n_first = 0, int n_cols = 0) {
    if (tile == 0 && splits == 1 && n_cols == 0 && M > 64) {
        const int n1 = first_columns(M, N, K, SILU >= 0);
        if (n1 > 0) {
            const int rc = pick_mfma<TO, SILU>(x, w, bias, out, M, N, K, choose_tile(M, n1, K, 1, SILU >= 0), 1, stream, 0, n1);
            return rc ? rc : pick_mfma<TO, SILU>(x, w, bias, out, M, N, K, choose_tile(M, N - n1, K, 1, SILU >= 0), 1, stream, n1, N - n1);
        }
    }
    if (n_cols == 0) n_cols = N;
    QkvTail tail{};
    tail.n_first = n_first;
    // Up to 64 rows against a gate|up matrix of at most one tile column a compute unit (its K cannot be
    // cut): a block streams its weights alone on its unit, and what it has in flight bounds it.  A ring of six stages
    // doubles that (24576 x 4096 against 64 rows, its weights in no cache: 38.8 us, 39.6 with three stages, 43.8 through registers with k steps of 128; as a
    // part of a step of 64 requests 44.7, and 45.9 through registers; with two blocks a unit, 51200 x 5120, a longer ring gains nothing).
    if (tile == 0 && SILU > 0 && M <= 64 && qe_cdiv(N, 128) <= 256) tile = 65;
    // (the gelu of 65536 values is 35 us in which nothing else runs on the unit: 256 x 256 is never its shape; 3000 rows against
    // 4096 x 1024: 65 us in it, 52 in 256 x 128, 47 in 128 x 128)
    if (tile == 0) tile = choose_tile(M, N, K, splits, SILU >= 0);
    if (tile == 65) return launch_mfma<TO, 64, 128, 6, 4, 1, SILU>(x, w, bias, out, M, N, K, n_cols, splits, stream, tail);
    if (tile == 512) return launch_mfma<TO, 256, 256, 2, 4, 1, SILU>(x, w, bias, out, M, N, K, n_cols, splits, stream, tail);
    if (tile == 256) return launch_mfma<TO, 256, 128, 3, 8, 1, SILU>(x, w, bias, out, M, N, K, n_cols, splits, stream, tail);
    if (tile == 128) return launch_mfma<TO, 128, 128, 2, 4, 2, SILU>(x, w, bias, out, M, N, K, n_cols, splits, stream, tail);
    return launch_mfma<TO, 64, 128, 3, 4, 2, SILU>(x, w, bias, out, M, N, K, n_cols, splits, stream, tail);
}

// tile: rows of the output tile (256, 128 or 64; 512 stands for 256 x 256, 65 for 64 x 128 with a ring of six stages), 0 to choose
// by the shape.  silu: w is [N, K] with
// gate and up rows interleaved in blocks of 32, out is [M, N / 2] = silu(gate) * up.
// splits > 1: out is float [splits, M, N], partial products along K (no silu then).
// gelu (without a bias, in bfloat16): out = gelu(product).
int qe_gemm_mfma(const void* x, const void* w, const float* bias, void* out, int M, int N, int K, int dt_o,
                 int tile, bool silu, int splits, hipStream_t stream, bool gelu) {
    QE_REQUIRE(splits >= 1 && (splits == 1 || (!silu && dt_o == QE_F32)), "mfma gemm: partial products are 32-bit and plain");
    QE_REQUIRE(K % 8 == 0 && K >= 64 && K < (1 << 22), "mfma gemm: K=%d is no multiple of 8 in [64, 2^22)", K);
    QE_REQUIRE(tile == 0 || tile == 512 || tile == 256 || tile == 128 || tile == 64 || tile == 65, "mfma gemm: tile of %d rows", tile);
    if (silu) {
        QE_REQUIRE(N % 64 == 0, "mfma gemm: silu-mul takes gate|up rows in blocks of 32");
        QE_REQUIRE((((unsigned long)bias) & 15) == 0, "mfma gemm: the biases of gate and up begin at a whole 16-byte piece");
        if (dt_o == QE_BF16)
            return bias ? pick_mfma<bf16_t, 2>(x, w, bias, out, M, N, K, tile, splits, stream)
                        : pick_mfma<bf16_t, 1>(x, w, bias, out, M, N, K, tile, splits, stream);
        return bias ? pick_mfma<float, 2>(x, w, bias, out, M, N, K, tile, splits, stream)
                    : pick_mfma<float, 1>(x, w, bias, out, M, N, K, tile, splits, stream);
    }
    if (gelu) {
        QE_REQUIRE(dt_o == QE_BF16 && !bias && splits == 1, "mfma gemm: gelu is stored in bfloat16, without a bias");
        return pick_mfma<bf16_t, -1>(x, w, bias, out, M, N, K, tile, splits, stream);
    }
    if (dt_o == QE_BF16) return pick_mfma<bf16_t, 0>(x, w, bias, out, M, N, K, tile, splits, stream);
    return pick_mfma<float, 0>(x, w, bias, out, M, N, K, tile, splits, stream);
}

// The q|k|v product of an attention layer with what follows it inside (see QkvTail): x [M, K] .
// w [(Hq + 2 Hkv) 128, K]^T (+ bias), then q to q_out [M, Hq, 128] and k, v into the cache
// [pages, 2, Hkv, P, 128] at slots[m] (negative or no slots: nowhere).  positions [M] index the
// table's rows [cos | sin] of 128 floats; q_w, k_w, table may be null.
int qe_gemm_qkv(const void* x, const void* w, const float* bias, int M, int K, int Hq, int Hkv, int P,
                const int* positions, const int* slots, const float* q_w, const float* k_w, float eps,
                const float* table, void* q_out, void* cache, int tile, hipStream_t stream) {
    const int N = (Hq + 2 * Hkv) * 128;
    QE_REQUIRE(K % 8 == 0 && K >= 64 && K < (1 << 22), "qkv gemm: K=%d is no multiple of 8 in [64, 2^22)", K);
    QE_REQUIRE(M > 16 && Hq > 0 && Hkv > 0 && P >= 16 && (P & (P - 1)) == 0, "qkv gemm: sizes not taken");
    QE_REQUIRE(tile == 0 || tile == 512 || tile == 256 || tile == 128 || tile == 64, "qkv gemm: tile of %d rows", tile);
    QE_REQUIRE(!table || positions, "qkv gemm: a rotation needs positions");
    int lp = 0;
    while ((1 << lp) < P) ++lp;
    QkvTail tail{positions, slots, q_w, k_w, table, (bf16_t*)q_out, (bf16_t*)cache, eps, Hq, Hkv, P, lp};
    const int n1 = tile == 0 ? first_columns(M, N, K) : 0;
    for (int part = 0; part < (n1 > 0 ? 2 : 1); ++part) {
        tail.n_first = part ? n1 : 0;
        const int n_cols = n1 == 0 ? N : (part ? N - n1 : n1), t = tile ? tile : choose_tile(M, n_cols, K, 1);
        int rc;
        if (t == 512) rc = launch_mfma<bf16_t, 256, 256, 2, 4, 1, 0, true>(x, w, bias, nullptr, M, N, K, n_cols, 1, stream, tail);
        else if (t == 256) rc = launch_mfma<bf16_t, 256, 128, 3, 8, 1, 0, true>(x, w, bias, nullptr, M, N, K, n_cols, 1, stream, tail);
        else if (t == 128) rc = launch_mfma<bf16_t, 128, 128, 2, 4, 2, 0, true>(x, w, bias, nullptr, M, N, K, n_cols, 1, stream, tail);
        else rc = launch_mfma<bf16_t, 64, 128, 3, 4, 2, 0, true>(x, w, bias, nullptr, M, N, K, n_cols, 1, stream, tail);
        if (rc) return rc;
    }
    return 0;
}
