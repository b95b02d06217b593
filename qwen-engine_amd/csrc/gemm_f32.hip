// out[M, N] = x[M, K] . W[N, K]^T (+ bias) with 32-bit operands on the matrix units: the product of
// the float32 mode.  v_mfma_f32_32x32x2_f32 and v_mfma_f32_16x16x4_f32 multiply 32-bit numbers and
// accumulate in 32-bit (no reduced-precision matrix mode), about ten times the rate of the vector
// units' multiply-adds.  Both are chains of fused multiply-adds in the order of k, bit for bit.
//
// Every output is summed in one order whatever M is and whichever kernel takes the rows, so a row's
// result does not depend on what else is in the batch.  K is cut into at most 16 chunks of chunk_len(K) (a
// multiple of 16, at least 64: with a chunk a step, 2000 rows of 3072 x 256 took 47 us, 40 now, 41 as one
// chain; the last one may be short).  Inside a chunk one chain runs over steps of 16,
// in a step over k = 0, 4, 8, 12, 1, 5, 9, 13, 2, ... (which is what lets a lane bring four neighbouring
// k by one load and use them in four instructions).  The chunks of a quarter are added in order, then
// the quarters in order.
//
// Four kernels share that order (those for the logits and for few rows and whole chunks stand by themselves):
//   few rows: a block owns 16 outputs (or 32) and has a wave per chunk (16 from K = 1024 on), so that the weights are asked for
//     by all its waves at once and the sums meet in shared memory.  Bound by the stream of the weights and
//     a kernel's fixed cost.  Two rows (as 64 x 64 tiles before): 4096 x 1024 7.1 us (42), 6144 x 1024 10.6 (42),
//     1024 x 3072 11.6 (117), weights of 151936 x 1024 that begin at no whole 16-byte piece 137 (215).  At most 64 registers a lane, so that two
//     blocks of 16 waves fit a compute unit (four steps at a time instead of two: 10.0, 17.7, 14.5 and 294 us).
//   more rows: tiles of 64 x 64, a wave a 32 x 32 quarter, K in steps of 16 through two buffers of shared
//     memory.  With fewer than TILES_FOR_FOUR tiles and a K that gives each something four groups of four
//     waves share a tile's K, one quarter each (a compute unit with one tile would else have a wave a SIMD and
//     wait for every step's loads: 235 rows of 3072 x 1024 took 38 us, now 28; with two tiles on some units one
//     group is the better one: 300 rows of 4096 x 512 33 us with four, 24 with one; a K of a chunk or two leaves
//     three groups idle: 744 rows of 2048 x 77 30 us, now 9).
// Loads stand under no condition: rows beyond the matrix read the last row again and are not stored, elements
// beyond a row its last ones and count as zeros.  (Behind a conditional load the compiler waits for all loads in flight: with
// such loads where K was no multiple of 16, 333 rows of 1024 x 1000 took 87.7 us.)
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef __attribute__((ext_vector_type(16))) float floatx16;

#define FT 64         // tile rows and columns
#define FK 16         // k step
#define FROW (FK + 4) // floats of a staged row: padded, so that the 32 rows a wave reads lie in different banks
#define CHUNKS 16
#define TILES_FOR_FOUR 257

__host__ __device__ __forceinline__ int chunk_len(int K) {
    const int even = (K + CHUNKS * FK - 1) / (CHUNKS * FK) * FK;
    return even < 4 * FK ? 4 * FK : even;
}

// How the rows of x and W lie: rows of whole steps, of whole fours (a four lies inside a row or behind its end), any of at least four
// numbers (the row's last four, moved up, stand for a four that passes its end), or shorter ones.
enum { ROWS_SHORT = 0, ROWS_ANY = 1, ROWS_FOURS = 2, ROWS_STEPS = 3 };

// Four consecutive elements of a row from k on, zeros behind its end (row may point behind the row's start: K is what is left of it
// from there on, perhaps less than nothing).  No load stands under a condition: one that would lie behind the end reads the row's last
// elements instead.  (A float is aligned to its own size and no more.)
typedef float floatx4_any __attribute__((ext_vector_type(4), aligned(4)));
template <int ROWS>
__device__ __forceinline__ floatx4 four_of_row(const float* __restrict__ row, int k, int K) {
    if (ROWS == ROWS_STEPS) return *(const floatx4_any*)(row + k);
    floatx4 v;
    if (ROWS == ROWS_FOURS) {
        v = *(const floatx4_any*)(row + min(k, K - 4));
        if (k >= K) v = floatx4{0.f, 0.f, 0.f, 0.f};
        return v;
    }
    if (ROWS == ROWS_ANY) {
        v = *(const floatx4_any*)(row + min(k, K - 4));
        const int past = k - (K - 4);
        if (past > 0) {
            const floatx4 u = v;
            v[0] = past == 1 ? u[1] : past == 2 ? u[2] : past == 3 ? u[3] : 0.f;
            v[1] = past == 1 ? u[2] : past == 2 ? u[3] : 0.f;
            v[2] = past == 1 ? u[3] : 0.f;
            v[3] = 0.f;
        }
        return v;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        v[e] = row[min(k + e, K - 1)];
        if (k + e >= K) v[e] = 0.f;
    }
    return v;
}

// The residual sum and the RMSNorm in front of a product of few rows: delta (or null): n_delta tensors [M, K] one after the other; the sums go to
// h_out [M, K].
struct RowsNorm {
    const float* weight;
    float eps;
    const float* delta;
    int n_delta;
    float* h_out;
};
constexpr int NORM_ROOM = 8192, NORM_PAD = 16;       // numbers of the normed rows; behind each (rows' reads in other banks)

// A row is normed by the number of threads that the norm's own kernel has for it (a thread a piece of four, at most 256), pieces and sums
// in its order, as many rows at once as the block has such groups.
__device__ __forceinline__ void norm_rows(const float* __restrict__ h, const RowsNorm& norm, float* normed, int M, int K, bool store) {
    __shared__ float red[CHUNKS];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int wide = min(4, (K + 255) / 256), threads = wide * 64, at_once = waves / wide, mine = wave / wide;
    const int tid = threadIdx.x - mine * threads;
    constexpr int NV = 4;                                   // (K <= 4096)
    for (int m0 = 0; m0 < M; m0 += at_once) {
        const int m = m0 + mine;
        const bool on = mine < at_once && m < M;
        const long row = (long)min(m, M - 1) * K;
        float v[NV][4], wv[NV][4];
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (i * threads * 4 < K) {
                const int c = (tid + i * threads) * 4, at = c < K ? c : 0;
                Vec4<float>::load(h + row + at, v[i]);
                Vec4<float>::load(norm.weight + at, wv[i]);
            }
        for (int s = 0; s < norm.n_delta; ++s) {
#pragma unroll
            for (int i = 0; i < NV; ++i)
                if (i * threads * 4 < K) {
                    const int c = (tid + i * threads) * 4, at = c < K ? c : 0;
                    float d[4];
                    Vec4<float>::load(norm.delta + (long)s * M * K + row + at, d);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[i][e] += d[e];
                }
        }
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if ((tid + i * threads) * 4 < K) ss = add_squares(ss, v[i], i == 0);
        ss = wave_sum(ss);
        if (m0) __syncthreads();                            // (the rows before have been read out)
        if ((threadIdx.x & 63) == 0) red[wave] = ss;
        __syncthreads();
        float sum = 0.f;
        for (int i = 0; i < wide; ++i) sum += red[min(mine * wide + i, waves - 1)];
        const float rstd = rsqrtf(sum / (float)K + norm.eps);
        if (on) {
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = (tid + i * threads) * 4;
                if (c < K) {
                    if (store && norm.delta) Vec4<float>::store(norm.h_out + row + c, v[i]);
                    float o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = v[i][e] * rstd * wv[i][e];
                    Vec4<float>::store(normed + m * (K + NORM_PAD) + c, o);
                }
            }
        }
    }
    __syncthreads();
}

// 16 MT rows a block (blockIdx.y: which).  Lane (g, r), g = lane / 16, r = lane % 16, brings W[n0 + r][k + 4 g .. + 4] and the same of x's row r.
// BATCH steps are asked for at once, the next batch before the current one is multiplied.
// SILU (NT = 2): w has the gate and up rows in alternating blocks of 32; a block has 16 outputs, their gate rows and their up rows, and stores
// silu(gate) * up.
// NORM (rows of at most NORM_ROOM numbers in all): x is the stream; what is to be added to it and the RMSNorm come first, with the sums and
// roundings of the norm's own kernel, while the first weights are on their way; the normed rows stay in shared memory.
// (Two rows against 4096 x 1024 8.6 us, with the norm before 7.4 + 3.4; 6144 x 1024 with norm and silu 12.5, as three kernels 11.0 + 3.4 + 2.5; and for the
// host two launches of some 12 us each less.)
template <int MT, int NT, int BATCH, int ROWS, bool SILU = false, bool NORM = false>
__global__ __launch_bounds__(64 * CHUNKS) void gemm_f32_rows_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                    const float* __restrict__ bias, float* __restrict__ out,
                                                                    int M, int N, int K, int chunk, RowsNorm norm) {
    __shared__ float sums[NORM ? 1 : CHUNKS * MT * NT * 256];
    extern __shared__ __attribute__((aligned(16))) float normed[];     // NORM: [M][K + NORM_PAD], then the chunks' sums in their place
    float* const part = NORM ? normed : sums;                          // [chunk][MT * NT][4][64]
    constexpr int TILE = 256, PART = MT * NT * TILE;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, r = lane & 15;
    const int n0 = blockIdx.x * (SILU ? 16 : 16 * NT), m0 = blockIdx.y * (16 * MT);
    const int k_lo = wave * chunk, k_hi = k_lo + chunk < K ? k_lo + chunk : K;   // (a block has a wave per chunk that holds some of K)
    const float* wrow[NT];
    const float* xrow[MT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int n = SILU ? (n0 & ~31) * 2 + 32 * j + (n0 & 31) + r : n0 + 16 * j + r;
        wrow[j] = w + (long)(SILU || n < N ? n : N - 1) * K + 4 * g;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = m0 + 16 * i + r;
        xrow[i] = x + (long)(m < M ? m : M - 1) * K + 4 * g;
    }
    floatx4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    floatx4 wv[2][BATCH][NT], xv[2][BATCH][MT];
    const int last = k_lo + (k_hi - k_lo - 1) / FK * FK;          // the chunk's last step (read again where a batch passes it)
    auto ask = [&](int buf, int k0) {
#pragma unroll
        for (int b = 0; b < BATCH; ++b) {
            const int k = k0 + b * FK < last ? k0 + b * FK : last;
#pragma unroll
            for (int j = 0; j < NT; ++j) wv[buf][b][j] = four_of_row<ROWS>(wrow[j], k, K - 4 * g);
#pragma unroll
            for (int i = 0; i < MT; ++i)
                if (!NORM) xv[buf][b][i] = four_of_row<ROWS>(xrow[i], k, K - 4 * g);
        }
    };
    auto multiply = [&](int buf, int k0) {
#pragma unroll
        for (int b = 0; b < BATCH; ++b) {
            if (k0 + b * FK > last) break;
            if (NORM) xv[buf][b][0] = *(const floatx4*)(normed + min(r, M - 1) * (K + NORM_PAD) + 4 * g + k0 + b * FK);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[buf][b][i][e], wv[buf][b][j][e], acc[i][j], 0, 0, 0);
        }
    };
    ask(0, k_lo);
    if constexpr (NORM) norm_rows(x, norm, normed, M, K, blockIdx.x == 0);
    for (int k0 = k_lo; k0 <= last; k0 += 2 * BATCH * FK) {
        ask(1, k0 + BATCH * FK);
        multiply(0, k0);
        ask(0, k0 + 2 * BATCH * FK);
        multiply(1, k0 + BATCH * FK);
    }
    if (NORM) __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[wave * PART + (i * NT + j) * TILE + e * 64 + lane] = acc[i][j][e];
    __syncthreads();
    const int waves = blockDim.x >> 6;
    const auto sum_of = [&](int tile, int e, int l) {
        const float* const of = part + tile * TILE + e * 64 + l;
        float total = 0.f;
        for (int q = 0; 4 * q < waves; ++q) {
            float quarter = of[4 * q * PART];
            for (int c = 4 * q + 1; c < 4 * q + 4 && c < waves; ++c) quarter += of[c * PART];
            total = q ? total + quarter : quarter;
        }
        return total;
    };
    if constexpr (SILU) {
        for (int at = threadIdx.x; at < 256; at += blockDim.x) {
            const int l = at & 63, e = at >> 6, m = m0 + 4 * (l >> 4) + e, n = n0 + (l & 15), row = (n & ~31) * 2 + (n & 31);
            float gate = sum_of(0, e, l), up = sum_of(1, e, l);
            if (bias) {
                gate += bias[row];
                up += bias[row + 32];
            }
            if (m < M) out[(long)m * N + n] = gate / (1.f + expf(-gate)) * up;
        }
        return;
    }
    for (int at = threadIdx.x; at < MT * NT * 256; at += blockDim.x) {
        const int l = at & 63, e = (at >> 6) & 3, tile = at >> 8;
        const float total = sum_of(tile, e, l);
        const int m = m0 + (tile / NT) * 16 + 4 * (l >> 4) + e, n = n0 + (tile % NT) * 16 + (l & 15);
        if (m < M && n < N) out[(long)m * N + n] = bias ? total + bias[n] : total;
    }
}

// The same for up to 16 rows against a matrix of very many rows (the logits'), K up to 1024 in whole lines of 32 numbers: blocks of 16
// outputs and four waves, a wave a quarter of K, its (up to) four chunks of 64 one after the other.  A chunk's 16 x 64 weights come as whole lines of 128
// bytes, 8 lanes a row, straight to shared memory, two chunks of a wave on their way; the row's pieces are exchanged there (piece p of row r at
// place p ^ (r / 2 % 8)) so that the reads in the operands' layout fall into distinct banks.  Five such blocks share a unit, and the
// end of one is hidden by the others (two rows against 151936 x 1024: 135 us with sixteen waves a block, now 100; one block's lines of all
// sixteen chunks at once, two blocks a unit, took 128; 32768 x 1024 32.0, now 25.0).
__global__ __launch_bounds__(256, 5) void gemm_f32_lines_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                const float* __restrict__ bias, float* __restrict__ out,
                                                                int M, int N, int K) {
    typedef __attribute__((ext_vector_type(4))) unsigned int uint4_t;
    constexpr int CHUNK = 4 * FK, QUARTER = 4 * CHUNK;
    __shared__ __attribute__((aligned(16))) float lines[4][2][1024];       // a wave's two chunks
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, r = lane & 15;
    const int n0 = blockIdx.x * 16, k_lo = wave * QUARTER, left = K - k_lo;        // (a block has a wave per quarter that holds some of K)
    const float* xrow = x + (long)min(r, M - 1) * K + 4 * g + k_lo;
    floatx4 xv[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) xv[s] = *(const floatx4_any*)(xrow + min(s * FK, left - FK));
    __builtin_amdgcn_sched_barrier(0);
    // (rows beyond the matrix are out of the descriptor's range and arrive as zeros, as does what lies beyond the last row's end; what lies
    // beyond another row's end is the next row's and is not multiplied)
    const unsigned long base = (unsigned long)(w + (long)n0 * K);
    const uint4_t rsrc = {(unsigned)base, (unsigned)(base >> 32) & 0xffffu, (unsigned)(min(16, N - n0) * K) * 4u, 0x00020000u};
    const unsigned to = (unsigned)(unsigned long)(__attribute__((address_space(3))) float*)lines + wave * 8192;
    int off[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) off[i] = ((8 * i + (lane >> 3)) * K + ((lane & 7) ^ (4 * i + (lane >> 4))) * 4) * 4;
    auto ask = [&](int c) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            QE_LOAD_TO_SHARED(to + (c & 1) * 4096 + i * 1024, off[i & 1], rsrc, (k_lo + c * CHUNK + (i >> 1) * 32) * 4, "0", " nt");
    };
    ask(0);
    ask(1);
    floatx4 quarter;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (c < 3) asm volatile("s_waitcnt vmcnt(4)" : : : "memory");      // (the wave's own lines: no barrier)
        else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        floatx4 wv[4], acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s) wv[s] = *(const floatx4*)(&lines[wave][c & 1][(s >> 1) * 512 + r * 32 + ((((s & 1) * 4 + g) ^ (r >> 1)) * 4)]);
        if (c < 2) {
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(wv[0]), "+v"(wv[1]), "+v"(wv[2]), "+v"(wv[3]) : : "memory");
            ask(c + 2);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (c * CHUNK + s * FK >= left) break;
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[c * 4 + s][e], wv[s][e], acc, 0, 0, 0);
        }
        if (c == 0) quarter = acc;
        else if (c * CHUNK < left) quarter += acc;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) lines[wave][0][e * 64 + lane] = quarter[e];
    __syncthreads();
    const int waves = blockDim.x >> 6;
    for (int at = threadIdx.x; at < 256; at += blockDim.x) {
        float total = lines[0][0][at];
        for (int q = 1; q < waves; ++q) total += lines[q][0][at];
        const int m = 4 * ((at & 63) >> 4) + (at >> 6), n = n0 + (at & 15);
        if (m < M && n < N) out[(long)m * N + n] = bias ? total + bias[n] : total;
    }
}

// The same for up to 16 rows where K is whole chunks of whole lines: a block has COLS rows of w (4, 8 or 16; the matrix instruction's other columns
// repeat them) and a wave a chunk of 16 STEPS numbers, which come in one trip, as whole lines, straight to shared memory (a row's piece p at
// place p ^ 4 (row % 4), so that the reads in the operands' layout fall into distinct banks); by pieces of half a line, two steps at a time, a chunk took a
// trip after the other.  Few columns a block where the matrix has few rows: 64 blocks of 16 would leave three units of four idle.  Bound by the
// trip and the launch.  (Two rows, by rows and so: 1024 x 1024 6.1 and 4.2 us, 1024 x 3072 11.7 and 7.0, 2048 x 1024 6.6 and 4.5, 4096 x 1024 7.1 and 6.1,
// 6144 x 1024 10.9 and 8.1, 12288 x 2048 23.6 and 23.1; sixteen: 1024 x 2048 12.4 and 6.8, 6144 x 1024 12.0 and 9.2.)
// (With the norm in front and silu behind, 384 blocks that norm the rows themselves took 13.7 us for 6144 x 1024 where 192 by rows take 12.5.)
template <int COLS, int STEPS>
__global__ __launch_bounds__(64 * CHUNKS) void gemm_f32_chunks_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                      const float* __restrict__ bias, float* __restrict__ out,
                                                                      int M, int N, int K) {
    typedef __attribute__((ext_vector_type(4))) unsigned int uint4_t;
    constexpr int C = STEPS * FK, PIECES = C / 4, LOADS = COLS * PIECES / 64;
    extern __shared__ __attribute__((aligned(16))) float chunks[];          // [wave][COLS][C], then a wave's sums [4][64] in its place
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, r = lane & 15;
    const int waves = blockDim.x >> 6, n0 = blockIdx.x * COLS, k_lo = wave * C;
    float* const mine = chunks + wave * (COLS * C);
    const float* xrow = x + (long)min(r, M - 1) * K + 4 * g + k_lo;
    floatx4 xv[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) xv[s] = *(const floatx4_any*)(xrow + s * FK);
    __builtin_amdgcn_sched_barrier(0);
    // (rows beyond the matrix are out of the descriptor's range and arrive as zeros)
    const unsigned long base = (unsigned long)(w + (long)n0 * K);
    const uint4_t rsrc = {(unsigned)base, (unsigned)(base >> 32) & 0xffffu, (unsigned)(min(COLS, N - n0) * K) * 4u, 0x00020000u};
    const unsigned to = (unsigned)(unsigned long)(__attribute__((address_space(3))) float*)chunks + wave * (COLS * C * 4);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int at = i * 64 + lane, col = at / PIECES, piece = (at % PIECES) ^ ((col & 3) * 4);
        QE_LOAD_TO_SHARED(to + i * 1024, (col * K + piece * 4) * 4, rsrc, k_lo * 4, "0", " nt");
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");                     // (the wave's own lines: no barrier)
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        const floatx4 wv = *(const floatx4*)(mine + (r % COLS) * C + ((s * 4 + g) ^ ((r & 3) * 4)) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[s][e], wv[e], acc, 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) mine[e * 64 + lane] = acc[e];
    __syncthreads();
    for (int at = threadIdx.x; at < 256; at += blockDim.x) {
        const int l = at & 63, m = 4 * (l >> 4) + (at >> 6), n = n0 + (l & 15);
        if ((l & 15) >= COLS || m >= M || n >= N) continue;
        float total = 0.f;
        for (int q = 0; 4 * q < waves; ++q) {
            float quarter = chunks[4 * q * (COLS * C) + at];
            for (int c = 4 * q + 1; c < 4 * q + 4 && c < waves; ++c) quarter += chunks[c * (COLS * C) + at];
            total = q ? total + quarter : quarter;
        }
        out[(long)m * N + n] = bias ? total + bias[n] : total;
    }
}

// Tiles of 64 x 64, GROUPS (1 or 4) groups of four waves.  For a step, lane (h, r), h = lane / 32, r = lane % 32, reads
// x[row r][4 h .. + 4] and [8 + 4 h .. + 4], and the same of W: with the instructions taking element j of the first and of
// the second piece in turn, the order is the one above.
template <int GROUPS, int ROWS>
__global__ __launch_bounds__(256 * GROUPS) void gemm_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                const float* __restrict__ bias, float* __restrict__ out,
                                                                int M, int N, int K, int chunk) {
    // (the groups' sums take the place of the staged steps at the end)
    constexpr int STAGE = 2 * FT * FROW, ALL = GROUPS * 2 * STAGE, SUMS = GROUPS > 1 ? GROUPS * 16 * 256 : 0;
    __shared__ __attribute__((aligned(16))) float lds[ALL > SUMS ? ALL : SUMS];
    const int group = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int h = lane >> 5, r = lane & 31;
    const int m0 = blockIdx.y * FT, n0 = blockIdx.x * FT;
    float* xs = lds + group * 2 * STAGE;              // [2 buffers][FT][FROW], then the same for w
    float* ws = xs + STAGE;
    // staging: thread tid brings four consecutive k of one row of each operand
    const int srow = tid >> 2, sk = (tid & 3) * 4;
    const float* xsrc = x + (long)(m0 + srow < M ? m0 + srow : M - 1) * K + sk;
    const float* wsrc = w + (long)(n0 + srow < N ? n0 + srow : N - 1) * K + sk;
    const int sat = srow * FROW + sk;

    const int quarters = GROUPS > 1 ? 1 : 4;          // quarters of K that this group walks
    const int k_begin = group * 4 * chunk;
    const int steps_chunk = chunk / FK, steps = quarters * 4 * steps_chunk;
    const int last = (K - 1) / FK * FK;               // K's last step
    // (steps behind the end of K are walked for the barriers' sake, their loads repeat the last step and nothing is multiplied)
    auto k_of = [&](int s) { const int k = k_begin + s * FK; return k < last ? k : last; };
    floatx16 acc, quarter, total;                     // (-0 is what leaves the first summand as it is)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        acc[e] = 0.f;
        quarter[e] = total[e] = -0.f;
    }
    floatx4 xv = four_of_row<ROWS>(xsrc, k_of(0), K - sk), wv = four_of_row<ROWS>(wsrc, k_of(0), K - sk);
    *(floatx4*)&xs[sat] = xv;
    *(floatx4*)&ws[sat] = wv;
    xv = four_of_row<ROWS>(xsrc, k_of(1), K - sk);
    wv = four_of_row<ROWS>(wsrc, k_of(1), K - sk);
    __syncthreads();
    int buf = 0, in_chunk = 0, chunk_no = 0;
    const int busy = k_begin >= K ? 0 : (K - k_begin + FK - 1) / FK < steps ? (K - k_begin + FK - 1) / FK : steps;
    const int walk = GROUPS > 1 ? (steps < (K + FK - 1) / FK ? steps : (K + FK - 1) / FK) : busy;   // (the first group's busy steps)
    for (int s = 0; s < walk; ++s) {
        const float* xa = &xs[(buf * FT + wm * 32 + r) * FROW + h * 4];
        const float* wa = &ws[(buf * FT + wn * 32 + r) * FROW + h * 4];
        const floatx4 a0 = *(const floatx4*)xa, a1 = *(const floatx4*)(xa + 8);
        const floatx4 b0 = *(const floatx4*)wa, b1 = *(const floatx4*)(wa + 8);
        // the next step, asked for a step ago, goes to the other buffer (its readers passed the last barrier); the step
        // after it is asked for
        *(floatx4*)&xs[(buf ^ 1) * FT * FROW + sat] = xv;
        *(floatx4*)&ws[(buf ^ 1) * FT * FROW + sat] = wv;
        xv = four_of_row<ROWS>(xsrc, k_of(s + 2), K - sk);
        wv = four_of_row<ROWS>(wsrc, k_of(s + 2), K - sk);
        if (s < busy) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[j], b0[j], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[j], b1[j], acc, 0, 0, 0);
            }
            if (++in_chunk == steps_chunk || s + 1 == busy) {     // the end of a chunk, perhaps of a quarter
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    quarter[e] += acc[e];
                    acc[e] = 0.f;
                }
                if ((chunk_no & 3) == 3 || s + 1 == busy) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        total[e] += quarter[e];
                        quarter[e] = -0.f;
                    }
                }
                in_chunk = 0;
                ++chunk_no;
            }
        }
        __syncthreads();
        buf ^= 1;
    }
    // lane (h, r) holds out[m0 + 32 wm + 8 b + 4 h + i][n0 + 32 wn + r] as element 4 b + i
    const int n = n0 + wn * 32 + r;
    const float bv = bias && n < N ? bias[n] : 0.f;
    auto put = [&](int e, float v) {
        const int m = m0 + wm * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
        if (m < M && n < N) out[(long)m * N + n] = bias ? v + bv : v;
    };
    if (GROUPS == 1) {
#pragma unroll
        for (int e = 0; e < 16; ++e) put(e, total[e]);
    } else {
        // the groups' quarters meet in shared memory; every group adds and stores four of a lane's 16 outputs
#pragma unroll
        for (int e = 0; e < 16; ++e) lds[(group * 16 + e) * 256 + tid] = total[e];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = group * 4 + i;
            float v = lds[e * 256 + tid];
#pragma unroll
            for (int q = 1; q < 4; ++q)
                if (q * 4 * chunk < K) v += lds[(q * 16 + e) * 256 + tid];
            put(e, v);
        }
    }
}

template <int MT, int NT, int BATCH>
static void launch_rows(const float* x, const float* w, const float* bias, float* out, int M, int N, int K, int rows,
                        hipStream_t stream) {
    const int chunk = chunk_len(K), waves = qe_cdiv(K, chunk);
    const dim3 grid(qe_cdiv(N, 16 * NT), qe_cdiv(M, 16 * MT));
#define QE_F32_ROWS(R_) gemm_f32_rows_kernel<MT, NT, BATCH, R_><<<grid, 64 * waves, 0, stream>>>(x, w, bias, out, M, N, K, chunk, RowsNorm{})
    if (rows == ROWS_STEPS) QE_F32_ROWS(ROWS_STEPS);
    else if (rows == ROWS_FOURS) QE_F32_ROWS(ROWS_FOURS);
    else if (rows == ROWS_ANY) QE_F32_ROWS(ROWS_ANY);
    else QE_F32_ROWS(ROWS_SHORT);
#undef QE_F32_ROWS
}

// gemm_f32_chunks_kernel takes up to 16 rows of these sizes.
static bool by_chunks(const float* w, int K) {
    const int chunk = chunk_len(K);
    return K % chunk == 0 && chunk % 64 == 0 && chunk <= 256 && (((unsigned long)w) & 15) == 0;
}

template <int COLS>
static int launch_chunks(const float* x, const float* w, const float* bias, float* out, int M, int N, int K, hipStream_t stream) {
    const int chunk = chunk_len(K), waves = K / chunk;
#define QE_F32_CHUNKS(S_)                                                                             \
    case S_: {                                                                                        \
        constexpr size_t most = CHUNKS * COLS * (S_) * FK * sizeof(float);                            \
        if constexpr (most <= 128 * 1024) {                                                           \
            QE_RAISE_SHARED((gemm_f32_chunks_kernel<COLS, S_>), most);                                 \
            gemm_f32_chunks_kernel<COLS, S_><<<qe_cdiv(N, COLS), 64 * waves, (size_t)K * COLS * sizeof(float), stream>>>(x, w, bias, out, M, N, K); \
            QE_LAUNCH_CHECK();                                                                        \
            return 0;                                                                                 \
        }                                                                                             \
        break;                                                                                        \
    }
    switch (chunk / FK) {
        QE_F32_CHUNKS(4) QE_F32_CHUNKS(8) QE_F32_CHUNKS(12) QE_F32_CHUNKS(16)
    }
#undef QE_F32_CHUNKS
    QE_REQUIRE(false, "gemm (32-bit): no kernel for chunks of %d numbers of %d rows a block", chunk, COLS);
}

// Whether up to 16 rows against a matrix [N, K] go by whole lines (see qe_gemm_f32).
static bool by_lines(int M, int N, int K) {
    return N >= 16384 && (K >= 608 || (K > 512 && (M > 2 || N >= 30000))) && K <= 4 * FK * CHUNKS && K % 32 == 0;
}

// The products of few rows with the steps beside them inside (N: the rows of w): silu(gate) * up over rows interleaved in blocks of 32, and
// the residual sum and the norm in front.  K in whole steps of 16.
extern int g_qe_matrix_f32;      // (switched off: the vector units' kernels do it all, one by one)
bool qe_gemm_f32_silu_ok(int M, int N, int K) { return g_qe_matrix_f32 && M <= 16 && N % 64 == 0 && K % FK == 0 && !by_lines(M, N, K); }
// Whether silu * up is best done in the product's launch (-1: it cannot be).  That form has 32 rows of w a block and asks for half as much at once: up to 128 blocks leave
// the units idle that four, eight or sixteen rows a block give work, beyond 256 their second turn is thin, but where the product by itself would have the same
// blocks.  (us, product and silu * up, then in one; two rows: 4096 x 512 6.5, 6.1, x 1536 10.9, 11.2, x 2048 10.9, 13.7, x 4096 18.8, 27.7; 2048 x 4096 12.3, 21.8;
// 4608 x 2048 15.4, 16.2, 6144 x 1024 9.7, 9.9, x 1536 17.5, 13.8, x 4096 28.6, 31.3 (behind the norm 35.3, 39.3), 8192 x 1024 11.3, 11.1, x 3072 25.2, 26.1; 9216 x 1024 12.1, 17.8; 24576 x 256 8.7,
// 8.2, x 512 12.5, 14.7, x 1536 43.7, 37.2, x 4096 77.7, 127; eight rows: 12288 x 2560 45.4, 43.4, 24576 x 2048 48.4, 57.7, x 4096 138, 127.  A launch less is some
// 12 us of the host's for a step that is not recorded.)
extern "C" int qe_gemm_f32_silu_inside(int M, int N, int K) {
    if (!qe_gemm_f32_silu_ok(M, N, K)) return -1;
    if (N <= 4096) return K <= 1536;
    if (N <= 8192) return M > 4 || K <= 3072;
    const bool chunks = K % chunk_len(K) == 0 && chunk_len(K) % 64 == 0 && chunk_len(K) <= 128;
    return K <= 256 || (!chunks && (M > 4 || K <= 1536));
}
bool qe_gemm_f32_norm_ok(int M, int N, int K) {
    return g_qe_matrix_f32 && M <= 16 && K % FK == 0 && K >= 256 && K <= 4096 && (long)M * K <= NORM_ROOM && !by_lines(M, N, K);
}

// N: outputs.  norm_w null: no norm.
int qe_gemm_f32_few(const float* x, const float* w, const float* bias, float* out, int M, int N, int K, bool silu, const float* norm_w,
                    float norm_eps, const float* delta, int n_delta, float* h_out, hipStream_t stream) {
    const int rows = silu ? 2 * N : N;
    QE_REQUIRE((silu || norm_w) && (!silu || qe_gemm_f32_silu_ok(M, rows, K)) && (!norm_w || qe_gemm_f32_norm_ok(M, rows, K)),
               "gemm (32-bit): %d rows against [%d, %d] are not taken with the steps beside them", M, rows, K);
    QE_REQUIRE(!delta || (n_delta >= 1 && h_out && h_out != x), "gemm (32-bit): the sums of %d tensors want a place of their own", n_delta);
    const int chunk = chunk_len(K), waves = qe_cdiv(K, chunk);
    const RowsNorm norm = {norm_w, norm_eps, delta, delta ? n_delta : 0, h_out};
    const long rows_room = (long)M * (K + NORM_PAD);
#define QE_F32_FEW(NT_, B_, S_, N_)                                                                                  \
    const size_t room = (N_) ? (rows_room > (NT_) * waves * 256L ? rows_room : (NT_) * waves * 256L) * sizeof(float) : 0; \
    gemm_f32_rows_kernel<1, NT_, B_, ROWS_STEPS, S_, N_><<<qe_cdiv(N, (S_) ? 16 : 16 * (NT_)), 64 * waves, room, stream>>>( \
        x, w, bias, out, M, N, K, chunk, norm)
    if (silu && norm_w) { QE_F32_FEW(2, 1, true, true); }
    else if (silu) { QE_F32_FEW(2, 1, true, false); }
    else if (M > 4 && N >= 6144) { QE_F32_FEW(2, 1, false, true); }
    else { QE_F32_FEW(1, 2, false, true); }
#undef QE_F32_FEW
    QE_LAUNCH_CHECK();
    return 0;
}

int qe_gemm_f32(const float* x, const float* w, const float* bias, float* out, int M, int N, int K,
                hipStream_t stream) {
    const int rows = K % FK == 0 ? ROWS_STEPS : (K % 4 == 0 ? ROWS_FOURS : (K > 4 ? ROWS_ANY : ROWS_SHORT));
    // More than 16 rows against a very wide matrix (logits): every block would read all rows again, and the tiles are
    // enough to fill the chip (33 rows, 151936 x 1024: 467 us by rows, 235 by tiles).  More than 32 rows with a single chunk of K
    // are one wave's work a block of rows (235 rows of 2048 x 64: 9.4 us by rows, 6.3 by tiles).  Up to 128 tiles leave half of the
    // compute units idle; blocks of 64 rows and 16 outputs do not (100 rows, 1024 x 3072: 73.5 us by tiles, 33.4 by rows).
    const long tiles = (long)qe_cdiv(N, FT) * qe_cdiv(M, FT);
    if (M <= 16 || ((K > 64 || M <= 32) && ((M <= 64 && N < 16384) || tiles <= 128))) {
        // 32 outputs a block halve the reads of x; they pay where the rows are some and the blocks enough (16 rows,
        // 6144 x 1024: 12.0 us against 14.3; 2 rows: 10.3 against 10.6; 16 rows, 4096 x 1024: 11.5 against 9.5)
        // Whole lines for the logits, with more than eight chunks of K and up to sixteen (chunks are longer than a wave's 64 beyond).  Up to two rows
        // and nine chunks, a matrix of fewer than 30000 rows goes by a wave a chunk (one row, by rows and by lines: 18000 x 544 12.7 us and
        // 14.5, 20001 x 576 13.5 and 15.6, 18000 x 608 13.9 and 14.8, 20001 x 608 15.5 and 15.7, 32768 x 544 20.6 and 19.1; eight rows: 20001 x 576 16.8 and
        // 15.9, 32768 x 608 26.6 and 21.0; with eight chunks or fewer a wave's walk is not worth a block: 20000 x 96 4.7 and 6.9)
        if (M <= 16 && by_lines(M, N, K) && (((unsigned long)w) & 15) == 0)
            gemm_f32_lines_kernel<<<qe_cdiv(N, 16), 64 * qe_cdiv(K, 16 * FK), 0, stream>>>(x, w, bias, out, M, N, K);
        // (two rows, us with 4, 8 and 16 columns a block: 1024 x 2048 5.5, 5.8, 6.5; 2048 x 1024 5.5, 4.5, 4.9; 4096 x 1024 9.6, 6.2, 6.1; 12288 x 1024
        // 24.9, 15.1, 12.1; 8192 x 3072, 8 columns, 29.5, and 25.2 by rows.  By rows and with 16 columns, beyond 12288 rows: 24576 x 512 14.7, 10.6, 151936 x 512
        // 71.0, 46.7, 16383 x 1024 18.5, 14.8, 24576 x 2048 41.6, 40.9, 151936 x 2048 238, 235, eight rows 326, 261; but one row 24576 x 2048 39.9, 40.6, 151936 x 2048
        // 225, 230: one block of 128 KB a unit, nothing beside it)
        else if (M <= 16 && N <= 1024 && by_chunks(w, K)) return launch_chunks<4>(x, w, bias, out, M, N, K, stream);
        else if (M <= 16 && N <= 2048 && by_chunks(w, K)) return launch_chunks<8>(x, w, bias, out, M, N, K, stream);
        else if (M <= 16 && by_chunks(w, K) && chunk_len(K) <= 128 && (M > 1 || chunk_len(K) == 64 || N <= 16384)) return launch_chunks<16>(x, w, bias, out, M, N, K, stream);
        else if (M > 4 && M <= 16 && N >= 6144) launch_rows<1, 2, 1>(x, w, bias, out, M, N, K, rows, stream);
        else if (M <= 16) launch_rows<1, 1, 2>(x, w, bias, out, M, N, K, rows, stream);
        else if (M <= 32) launch_rows<2, 1, 2>(x, w, bias, out, M, N, K, rows, stream);
        else launch_rows<4, 1, 1>(x, w, bias, out, M, N, K, rows, stream);
        QE_LAUNCH_CHECK();
        return 0;
    }
    QE_REQUIRE(qe_cdiv(M, FT) <= 65535, "gemm (32-bit): M=%d is too large for one launch", M);
    dim3 grid(qe_cdiv(N, FT), qe_cdiv(M, FT));
    const int chunk = chunk_len(K);
    const bool four = tiles < TILES_FOR_FOUR && K >= 512;
#define QE_F32_TILES(G_, R_) gemm_f32_kernel<G_, R_><<<grid, 256 * G_, 0, stream>>>(x, w, bias, out, M, N, K, chunk)
#define QE_F32_TILES2(R_) do { if (four) QE_F32_TILES(4, R_); else QE_F32_TILES(1, R_); } while (0)
    if (rows == ROWS_STEPS) QE_F32_TILES2(ROWS_STEPS);
    else if (rows == ROWS_FOURS) QE_F32_TILES2(ROWS_FOURS);
    else if (rows == ROWS_ANY) QE_F32_TILES2(ROWS_ANY);
    else QE_F32_TILES2(ROWS_SHORT);
#undef QE_F32_TILES2
#undef QE_F32_TILES
    QE_LAUNCH_CHECK();
    return 0;
}
