// Attention of single new tokens over the paged cache (decode), bfloat16, split over the keys
// ("flash decoding"), on the MFMA units.  All query heads of a key/value group are the columns
// of one wave (see attention_tile.h), so the cache is read from HBM once; this kernel is bound
// by that read.  Heads beyond the group size (lanes n >= G) compute on zeros and are not stored.
//
// W waves per (split of the keys, key/value head, token): one where the step has waves enough, four where it has few.  The
// splits are cut at absolute key positions (multiples of SPLIT), and four waves do the arithmetic of one in its order, so a
// token's result does not depend on what else is in the batch.  A second kernel merges the splits.
//
// What bounds a step of few tokens is a wave's chain: some 0.7 us of memory and some 0.4 of arithmetic for each of its tiles,
// eight of them in a split of 128 keys, whatever the other units do.  Of four waves each takes the scores and then the weights of
// every fourth tile, which meet in shared memory, and multiplies its quarter of the value rows by the weights of all tiles, in
// the order of the keys; everything a wave needs is asked for at its start.  (With the merge behind it, one token of 16 heads of
// 128 on 8 over 1000 keys: 8.6 us against 11.3 with one wave, over 40 keys 7.2 against 7.4; with the step before folded in
// 10.1 against 12.2, and 8.8 against 9.6.  With a softmax of its own for every wave, joined at the end, the sums had another
// order than one wave's and took 8.7 and 7.1, and 10.2 and 8.5.)
#include "attention_tile.h"
#include <type_traits>

// A split of so many tiles is the first wave's alone: what the waves would tell each other takes longer than a second tile (one token of
// 32 heads on 8 over 16 keys: 7.2 us with four waves at work, 6.2 so; where the host knows that there are no more, one wave is launched:
// 6.0).
#define ALONE 2

// What the waves of a block leave for each other about a split's tiles.
template <int TILES>
struct WaveShared {
    float tmax[16][TILES];
    short4_t weights[TILES][64];
    float sums[TILES][64];
};

// What wave ``wave`` of W asks for of the n tiles of a walk (1 <= n <= TILES): the key rows of the tiles wave, wave + W, ..., and of
// every tile its part of the value rows.  Beyond the last tile the last is asked for again: without a branch the waits are exact
// (for the same reason all loads are plain: so few splits, 16 MB at most, leave room in the caches).
// place(i, page, o): the i-th tile's page, and the place of its first key in it.
template <int D, int TILES, int W>
struct WaveTiles {
    static constexpr int NV = D / 16 / W;
    bf16x8 k[TILES / W][D / 32];
    short4_t v[TILES][NV];
    template <typename Place>
    __device__ __forceinline__ void ask(const bf16_t* cache, long page_stride, int kvh, int Hkv, int P, int n, int wave, int g, int lane_n,
                                        Place place) {
        int page, o;
#pragma unroll
        for (int j = 0; j < TILES / W; ++j) {
            place(min(j * W + wave, n - 1), page, o);
            const bf16_t* kbase = cache + page * page_stride + ((long)kvh * P + o) * D + (long)lane_n * D + g * 8;
#pragma unroll
            for (int c = 0; c < D / 32; ++c) k[j][c] = *(const bf16x8*)(kbase + c * 32);
        }
        __builtin_amdgcn_sched_barrier(0);                 // (the keys are wanted first)
#pragma unroll
        for (int i = 0; i < TILES; ++i) {
            place(min(i, n - 1), page, o);
            const bf16_t* vbase = cache + page * page_stride + ((long)(Hkv + kvh) * P) * D + o + (long)lane_n * P + g * 4;
#pragma unroll
            for (int b = 0; b < NV; ++b) v[i][b] = *(const short4_t*)(vbase + (long)(wave * NV + b) * 16 * P);
        }
    }
    floatx4 s[TILES / W];
    // The scores of the wave's tiles, and their maxima for the others; kk(i): the i-th tile's first key.  What stands for a tile behind
    // the last has no key that is seen: a maximum of minus infinity, a factor of 1 and weights of 0 below.
    template <bool CAP, int ALL, typename FirstKey>
    __device__ __forceinline__ void score(WaveShared<ALL>& sh, const bf16x8 (&qreg)[D / 32], float scale, int wave, int g, int lane_n, int lo, int hi,
                                          int kf, float cap, FirstKey kk) {
#pragma unroll
        for (int j = 0; j < TILES / W; ++j) {
            s[j] = attn_tile_scores<D, CAP>(k[j], qreg, scale, kk(j * W + wave), g, lo, hi, kf, cap);
            const float t = attn_tile_max(s[j]);
            if (g == 0) sh.tmax[lane_n][j * W + wave] = t;
        }
    }
    // Behind a barrier: the running maxima, the weights of the wave's tiles for the others, and, behind another, the walk with
    // all weights through the wave's value rows.  l: only the first wave's.
    template <int ALL, typename FirstKey>
    __device__ __forceinline__ void walk(WaveShared<ALL>& sh, int n, int wave, int g, int lane, int vlo, int vhi, int kf, FirstKey kk, float& m,
                                         float& l, floatx4 (&acc)[NV]) const {
        float tmax[TILES], ref[TILES], alpha[TILES];
#pragma unroll
        for (int i = 0; i < TILES; i += 4) Vec4<float>::load(&sh.tmax[lane & 15][i], *(float(*)[4])(tmax + i));
        m = -INFINITY;
#pragma unroll
        for (int i = 0; i < TILES; ++i) {
            const float mn = fmaxf(m, tmax[i]);
            ref[i] = attn_reference(mn);
            alpha[i] = __expf(m - ref[i]);
            m = mn;
        }
#pragma unroll
        for (int j = 0; j < TILES / W; ++j) {
            float mine = ref[j * W];
#pragma unroll
            for (int w = 1; w < W; ++w) mine = wave == w ? ref[j * W + w] : mine;
            float psum;
            sh.weights[j * W + wave][lane] = attn_tile_weights(s[j], mine, psum);
            sh.sums[j * W + wave][lane] = psum;
        }
        __syncthreads();
        l = 0.f;
#pragma unroll
        for (int b = 0; b < NV; ++b) acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i0 = 0; i0 < TILES; i0 += 4) {
            if (i0 >= n) break;
            short4_t pb[4];
            float psum[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) pb[u] = sh.weights[i0 + u][lane];
#pragma unroll
            for (int u = 0; u < 4; ++u) psum[u] = sh.sums[i0 + u][lane];
            // (value rows of tiles that lie wholly among the keys seen need no mask)
            const bool inside = i0 + 4 <= n && kk(i0) >= vlo && kk(i0 + 3) + 16 <= vhi && kk(i0 + 3) - kk(i0) == 48;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                l = l * alpha[i0 + u] + psum[u];
                short4_t vmask = {-1, -1, -1, -1};
                if (!inside) vmask = attn_value_mask(kk(i0 + u), g, vlo, vhi, kf);
#pragma unroll
                for (int b = 0; b < NV; ++b) {
                    acc[b] *= alpha[i0 + u];
                    acc[b] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v[i0 + u][b] & vmask, pb[u], acc[b], 0, 0, 0);
                }
            }
        }
    }
};

// SPLIT: keys per split (a multiple of 16, at most 64 tiles).  The next tile is loaded while the
// current one is computed, and the split's page ids are read before the loop.
// (Merging the splits in this same kernel, by the wave that finishes last, was tried: the
// device-wide fences it needs cost several times what the separate merge kernel costs.)
// CAP: a soft cap on the scores (scale then holds 2 log2(e) / cap, see attn_tile_step).
template <int D, int SPLIT, bool CAP, int W>
__global__ __launch_bounds__(64 * W) void attention_decode_split_kernel(
    const bf16_t* __restrict__ q, const bf16_t* cache,           // (not restrict: loads of a tile then stay where they are asked for)
    const int* __restrict__ dec_tokens, const int* __restrict__ positions, const int* __restrict__ tok_seq,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ shared_keys,
    float* __restrict__ part_acc, float* __restrict__ part_ml,
    int Hq, int Hkv, int P, float scale, int window, int keep_first, int num_splits, float cap) {
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    const int split = blockIdx.x, kvh = blockIdx.y, di = blockIdx.z;
    const int G = Hq / Hkv;
    const int t = dec_tokens ? dec_tokens[di] : di;       // (no list: every row, in order)
    const int p = positions[t];
    const int lo = first_seen_key(p, window);
    const int k_begin = max(split * SPLIT, lo);
    const int k_end = min((split + 1) * SPLIT, p + 1);
    // the request's kept first keys that lie behind the window, as far as they are this split's: [split * SPLIT, kf)
    const int kf = min(min(keep_first, lo), (split + 1) * SPLIT);
    const int first_tiles = kf > split * SPLIT ? (kf - split * SPLIT + 15) / 16 : 0;
    const int head = kvh * G + n;
    const bool head_ok = n < G;
    float* pacc = part_acc + (((long)di * Hq + head) * num_splits + split) * D;
    float* pml = part_ml + (((long)di * Hq + head) * num_splits + split) * 2;
    if (k_begin >= k_end && first_tiles == 0) {   // nothing of this split is seen by the token
        if (head_ok && g == 0 && wave == 0) { pml[0] = -INFINITY; pml[1] = 0.f; }
        return;
    }
    const int row = tok_seq[t];
    const int* bt = block_table + (long)row * max_blocks;
    // (keys that other requests read too are left in the caches, the others stream: see load_tile)
    const bool stream = !(shared_keys && split * SPLIT < shared_keys[row]);
    const long page_stride = 2L * Hkv * P * D;
    // the split's tiles that are walked: first_tiles from its start (kept first keys), then, from the window's
    // first tile on, tile0 .. tile1 - 1 (tiles between the two are not read: their pages may have gone back)
    const int tile1 = k_begin < k_end ? (k_end - split * SPLIT + 15) / 16 : first_tiles;
    const int tile0 = k_begin < k_end ? max((k_begin - split * SPLIT) / 16, first_tiles) : first_tiles;
    const int walk0 = first_tiles > 0 ? 0 : tile0;                    // first tile of the walk
    const int gap = first_tiles > 0 ? tile0 - first_tiles : 0;        // tiles left out behind the first ones
    // lane i holds the page of tile i (one vector load for the whole split); a tile's page is
    // then read from that lane
    int my_page = 0;
    if ((lane >= tile0 && lane < tile1) || lane < first_tiles) my_page = bt[(split * SPLIT + lane * 16) / P];
    const int my_place = (split * SPLIT + lane * 16) % P;             // (and the place of its first key in the page)

    bf16x8 qreg[D / 32];
    const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < D / 32; ++c)
        qreg[c] = head_ok ? *(const bf16x8*)(q + ((long)t * Hq + head) * D + c * 32 + g * 8) : zero8;

    // Two tile buffers used in turn: the loads of the next tile are issued before the current
    // one is computed, and nothing is copied from one buffer to the other.
    // (i_ counts the walk's tiles; TILE_OF: the tile of the split behind it)
#define TILE_OF(i_) ((i_) < first_tiles ? (i_) : (i_) + gap)
#define LOAD(buf_, i_) load_tile<D>(buf_, cache, __builtin_amdgcn_readlane(my_page, TILE_OF(i_)), page_stride, kvh, Hkv, P, \
                                    (split * SPLIT + TILE_OF(i_) * 16) % P, g, n, stream)
#define STEP(buf_, i_) attn_tile_step<D, CAP>(st, buf_, qreg, scale, split * SPLIT + TILE_OF(i_) * 16, g, k_begin, k_end, k_begin, k_end, kf, cap)
    const int walk1 = tile1 - gap;
    const bool alone = W > 1 && walk1 - walk0 <= ALONE;
    if (alone && wave > 0) return;
    if constexpr (W > 1) if (!alone) {
        constexpr int TILES = SPLIT / 16, NV = D / 16 / W;
        __shared__ WaveShared<TILES> shared;
        const int tiles = walk1 - walk0;
        const auto first_key = [&](int i) { return split * SPLIT + TILE_OF(walk0 + i) * 16; };
        const auto by_waves = [&](auto most) {             // (half of the loads where half of the tiles are all there are)
            WaveTiles<D, decltype(most)::value, W> wt;
            wt.ask(cache, page_stride, kvh, Hkv, P, tiles, wave, g, n, [&](int i, int& page, int& o) {
                page = __builtin_amdgcn_readlane(my_page, TILE_OF(walk0 + i));
                o = __builtin_amdgcn_readlane(my_place, TILE_OF(walk0 + i));
            });
            wt.template score<CAP>(shared, qreg, scale, wave, g, n, k_begin, k_end, kf, cap, first_key);
            __syncthreads();
            float m, l;
            floatx4 acc[NV];
            wt.walk(shared, tiles, wave, g, lane, k_begin, k_end, kf, first_key, m, l, acc);
            l += __shfl_xor(l, 16, 64);
            l += __shfl_xor(l, 32, 64);
            if (head_ok) {
#pragma unroll
                for (int b = 0; b < NV; ++b) *(floatx4*)(pacc + (wave * NV + b) * 16 + g * 4) = acc[b];
                if (g == 0 && wave == 0) { pml[0] = m; pml[1] = l; }
            }
        };
        if (tiles > TILES / 2) by_waves(std::integral_constant<int, TILES>{});
        else by_waves(std::integral_constant<int, TILES / 2>{});
        return;
    }
    AttnState<D> st;
    st.init();
    KVTile<D> ta, tb;
    int i = walk0;
    LOAD(ta, i);
    while (true) {
        if (i + 1 < walk1) LOAD(tb, i + 1);
        STEP(ta, i);
        if (++i >= walk1) break;
        if (i + 1 < walk1) LOAD(ta, i + 1);
        STEP(tb, i);
        if (++i >= walk1) break;
    }
#undef LOAD
#undef STEP
#undef TILE_OF
    float l = st.l;
    const float m = st.m;
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (head_ok) {
#pragma unroll
        for (int db = 0; db < D / 16; ++db)
            *(floatx4*)(pacc + db * 16 + g * 4) = st.acc[db];    // O^T rows d = db * 16 + g * 4 + j of column head n
        if (g == 0) { pml[0] = m; pml[1] = l; }
    }
}

// ---- the same with the step before it folded in ---------------------------------------------
// (Folding the output projection into the merge kernel, a block per head and 128 output features
// that merges the head's splits for all tokens and multiplies with its part of W_o, was tried for
// few tokens: it takes as long as the two kernels it replaces.)
//
// The q/k norm, the rotation and the cache write of the new token cost a kernel of their own
// that runs a few microseconds for a few kilobytes.  Here every wave norms and rotates the query
// heads it needs itself, straight from the q|k|v rows (the pairs d, d + D/2 of the rotation lie in
// the same lane in the MFMA operand layout), and the wave whose split holds the token's own
// position also norms and rotates the new key, takes it and the new value into its softmax from
// registers (the cached keys it reads stop before that position), and writes both to the cache.
// Roundings are where the separate kernels have them: q and k to bfloat16 after the rotation,
// the probability to bfloat16 before it meets the value.

// One head's features c * 32 + g * 8 + e in the MFMA operand layout: fetch() issues the loads (the
// head, the norm's weights, the position's row [cos | sin] of the table), finish() does the
// RMSNorm (w) and the rotation (cs), each optional, and rounds to bfloat16.  Apart, so that the
// loads of the first key tiles can be issued between the two.
template <int D>
struct NormRotate {
    static constexpr int H = D / 64;                       // chunk c and chunk c + H rotate together
    bf16x8 raw[D / 32];
    float wv[D / 32][8], co[H][8], sn[H][8];
    __device__ __forceinline__ void fetch(const bf16_t* __restrict__ src, bool active, const float* __restrict__ w,
                                          const float* __restrict__ cs, int g) {
#pragma unroll
        for (int c = 0; c < D / 32; ++c) {
            raw[c] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (active) raw[c] = *(const bf16x8*)(src + c * 32 + g * 8);
        }
        if (w) {
#pragma unroll
            for (int c = 0; c < D / 32; ++c) {
                Vec4<float>::load(w + c * 32 + g * 8, *(float(*)[4])wv[c]);
                Vec4<float>::load(w + c * 32 + g * 8 + 4, *(float(*)[4])(wv[c] + 4));
            }
        }
        if (cs) {
#pragma unroll
            for (int c = 0; c < H; ++c) {
                Vec4<float>::load(cs + c * 32 + g * 8, *(float(*)[4])co[c]);
                Vec4<float>::load(cs + c * 32 + g * 8 + 4, *(float(*)[4])(co[c] + 4));
                Vec4<float>::load(cs + D / 2 + c * 32 + g * 8, *(float(*)[4])sn[c]);
                Vec4<float>::load(cs + D / 2 + c * 32 + g * 8 + 4, *(float(*)[4])(sn[c] + 4));
            }
        }
    }
    __device__ __forceinline__ void finish(bf16x8 (&out)[D / 32], bool has_w, float eps, bool has_cs) {
        float x[D / 32][8];
#pragma unroll
        for (int c = 0; c < D / 32; ++c)
#pragma unroll
            for (int e = 0; e < 8; ++e) x[c][e] = (float)raw[c][e];
        if (has_w) {
            float ss = 0.f;
#pragma unroll
            for (int c = 0; c < D / 32; ++c)
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += x[c][e] * x[c][e];
            ss += __shfl_xor(ss, 16, 64);
            ss += __shfl_xor(ss, 32, 64);
            const float rstd = rsqrtf(ss / (float)D + eps);
#pragma unroll
            for (int c = 0; c < D / 32; ++c)
#pragma unroll
                for (int e = 0; e < 8; ++e) x[c][e] = x[c][e] * rstd * wv[c][e];
        }
        if (has_cs) {
#pragma unroll
            for (int c = 0; c < H; ++c)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x1 = x[c][e], x2 = x[c + H][e];
                    x[c][e] = co[c][e] * x1 - sn[c][e] * x2;
                    x[c + H][e] = sn[c][e] * x1 + co[c][e] * x2;
                }
        }
#pragma unroll
        for (int c = 0; c < D / 32; ++c)
#pragma unroll
            for (int e = 0; e < 8; ++e) out[c][e] = (__bf16)x[c][e];
    }
};

// The token's own key: its score from q and the key as normed and turned.
template <int D>
__device__ __forceinline__ float own_score(const bf16x8 (&qreg)[D / 32], const bf16x8 (&kreg)[D / 32]) {
    float dot = 0.f;
#pragma unroll
    for (int c = 0; c < D / 32; ++c)
#pragma unroll
        for (int e = 0; e < 8; ++e) dot += (float)qreg[c][e] * (float)kreg[c][e];
    dot += __shfl_xor(dot, 16, 64);
    dot += __shfl_xor(dot, 32, 64);
    return dot;
}
// It joins a running maximum and sum: its weight, rounded, and the factor for what was summed before it
// (the roundings are written out: one wave and four do the same).
__device__ __forceinline__ float own_weight(float dot, float scale, int g, float& m, float& l, float& alpha) {
    const float mn = fmaxf(m, dot * scale);
    alpha = __expf(m - mn);                                // 0 when no cached key was seen
    const float pn = __expf(__builtin_fmaf(dot, scale, -mn));
    l = __builtin_fmaf(l, alpha, g == 0 ? pn : 0.f);       // (a lane's share of the sum: once per column)
    m = mn;
    return (float)(__bf16)pn;
}
__device__ __forceinline__ void add_own(floatx4& acc, float alpha, float weight, const short4_t& vv) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = __builtin_fmaf(weight, bf16_bits_to_float((unsigned short)vv[j]), acc[j] * alpha);
}
// Key and value go to the cache.
template <int D>
__device__ __forceinline__ void store_own(bf16_t* cache, const bf16x8 (&kreg)[D / 32], const bf16_t* vsrc, int slot, long page_stride,
                                          int kvh, int Hkv, int P, int g, int n) {
    if (slot < 0) return;
    const long page = slot / P;
    const int off = slot % P;
    if (n == 0) {
#pragma unroll
        for (int c = 0; c < D / 32; ++c)
            *(bf16x8*)(cache + page * page_stride + ((long)kvh * P + off) * D + c * 32 + g * 8) = kreg[c];
    }
    if (n < D / 16) {                                      // the value tile is [D][P]: a column of single elements
        bf16_t* vt = cache + page * page_stride + ((long)(Hkv + kvh) * P) * D + off;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int d = n * 16 + g * 4 + j;
            vt[(long)d * P] = vsrc[d];
        }
    }
}

// AHEAD: how many tiles the loads of a whole split run ahead of the computation.  A wave with one
// tile in flight gets 8 KB per trip to memory (about 0.7 us); that is enough when the chip holds
// two waves or more per SIMD, whose loads together keep the memory busy, and far too little for one
// token's 256 waves.  With 3 the code of a whole split is straight-line (waits are then exact) and
// takes 64 registers more, which with many waves costs more than it brings.  The order of the
// arithmetic is the same either way.
// W: the waves that share a split, as above (AHEAD then means nothing).  Every wave prepares q for itself while its keys and values
// travel; one more wave prepares the token's own key, whose score it leaves for the others, and writes key and value to the cache.
template <int D, int SPLIT, int AHEAD, int W>
__global__ __launch_bounds__(64 * (W > 1 ? W + 1 : 1)) void attention_decode_fused_split_kernel(
    const bf16_t* __restrict__ qkv, bf16_t* cache,
    const int* __restrict__ dec_tokens, const int* __restrict__ positions, const int* __restrict__ tok_seq,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ shared_keys,
    const int* __restrict__ slots, const float* __restrict__ q_w, const float* __restrict__ k_w, float eps, const float* __restrict__ table,
    float* __restrict__ part_acc, float* __restrict__ part_ml,
    int Hq, int Hkv, int P, float scale, int window, int num_splits) {
    constexpr int TILES = SPLIT / 16;
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    const int split = blockIdx.x, kvh = blockIdx.y, di = blockIdx.z;
    const int G = Hq / Hkv;
    const int t = dec_tokens ? dec_tokens[di] : di;       // (no list: every row, in order)
    const int p = positions[t];
    const int lo = first_seen_key(p, window);
    const bool owns = split == p / SPLIT;                  // this block takes the token's own key and value
    const int k_begin = max(split * SPLIT, lo);
    const int k_end = min((split + 1) * SPLIT, p);         // cached keys: the token's own is not among them
    const int head = kvh * G + n;
    const bool head_ok = n < G;
    float* pacc = part_acc + (((long)di * Hq + head) * num_splits + split) * D;
    float* pml = part_ml + (((long)di * Hq + head) * num_splits + split) * 2;
    if (k_begin >= k_end && !owns) {   // nothing of this split is seen by the token
        if (head_ok && g == 0 && wave == 0) { pml[0] = -INFINITY; pml[1] = 0.f; }
        return;
    }
    const long width = (long)(Hq + 2 * Hkv) * D;
    const float* cs = table ? table + (long)p * D : nullptr;
    const long page_stride = 2L * Hkv * P * D;
    const bf16_t* vsrc = qkv + t * width + (long)(Hq + Hkv + kvh) * D;

    bf16x8 qreg[D / 32];
    bf16x8 kreg[D / 32];                                   // the token's own key, normed and turned
    const int tile0 = (k_begin - split * SPLIT) / 16;
    const int tile1 = k_begin < k_end ? (k_end - split * SPLIT + 15) / 16 : tile0;
    int my_page = 0;
    bool stream = false;
    if (k_begin < k_end) {
        const int row = tok_seq[t];
        const int* bt = block_table + (long)row * max_blocks;
        stream = !(shared_keys && split * SPLIT < shared_keys[row]);
        if (lane >= tile0 && lane < tile1) my_page = bt[(split * SPLIT + lane * 16) / P];
    }
    const bool alone = W > 1 && tile1 - tile0 <= ALONE;
    if (alone && wave > 0) return;
    if constexpr (W > 1) if (!alone) {
        constexpr int NV = D / 16 / W;
        __shared__ WaveShared<TILES> shared;
        __shared__ float own_dot[16];
        const int tiles = tile1 - tile0;
        if (wave == W) {                                   // the token's own key
            NormRotate<D> nq, nk;
            if (owns) {
                nk.fetch(qkv + t * width + (long)(Hq + kvh) * D, true, k_w, cs, g);
                nq.fetch(qkv + t * width + (long)head * D, head_ok, q_w, cs, g);
                nk.finish(kreg, k_w != nullptr, eps, cs != nullptr);
                nq.finish(qreg, q_w != nullptr, eps, cs != nullptr);
            }
            __syncthreads();
            if (owns) {
                const float dot = own_score<D>(qreg, kreg);
                if (g == 0) own_dot[n] = dot;
            }
            __syncthreads();
            if (owns) store_own<D>(cache, kreg, vsrc, slots ? slots[t] : -1, page_stride, kvh, Hkv, P, g, n);
            return;
        }
        const auto first_key = [&](int i) { return split * SPLIT + (tile0 + i) * 16; };
        const auto by_waves = [&](auto most) {
            constexpr int MOST = decltype(most)::value;    // tiles there can be; 0: none, the own key alone
            float m = -INFINITY, l = 0.f;
            floatx4 acc[NV];
#pragma unroll
            for (int b = 0; b < NV; ++b) acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
            short4_t vv[NV];
#pragma unroll
            for (int b = 0; b < NV; ++b) vv[b] = *(const short4_t*)(vsrc + (wave * NV + b) * 16 + g * 4);
            if constexpr (MOST > 0) {
                NormRotate<D> nq;
                nq.fetch(qkv + t * width + (long)head * D, head_ok, q_w, cs, g);
                const int my_place = (split * SPLIT + lane * 16) % P;
                WaveTiles<D, MOST, W> wt;
                wt.ask(cache, page_stride, kvh, Hkv, P, tiles, wave, g, n, [&](int i, int& page, int& o) {
                    page = __builtin_amdgcn_readlane(my_page, tile0 + i);
                    o = __builtin_amdgcn_readlane(my_place, tile0 + i);
                });
                __builtin_amdgcn_sched_barrier(0);         // (the tiles are asked for before anything waits for q)
                nq.finish(qreg, q_w != nullptr, eps, cs != nullptr);
                wt.template score<false>(shared, qreg, scale, wave, g, n, k_begin, k_end, 0, 0.f, first_key);
                __syncthreads();
                wt.walk(shared, tiles, wave, g, lane, k_begin, k_end, 0, first_key, m, l, acc);
            } else {
                __syncthreads();
                __syncthreads();
            }
            if (owns) {
                float alpha;
                const float weight = own_weight(own_dot[n], scale, g, m, l, alpha);
#pragma unroll
                for (int b = 0; b < NV; ++b) add_own(acc[b], alpha, weight, vv[b]);
            }
            l += __shfl_xor(l, 16, 64);
            l += __shfl_xor(l, 32, 64);
            if (head_ok) {
#pragma unroll
                for (int b = 0; b < NV; ++b) *(floatx4*)(pacc + (wave * NV + b) * 16 + g * 4) = acc[b];
                if (g == 0 && wave == 0) { pml[0] = m; pml[1] = l; }
            }
        };
        if (tiles > TILES / 2) by_waves(std::integral_constant<int, TILES>{});
        else if (tiles > 0) by_waves(std::integral_constant<int, TILES / 2>{});
        else by_waves(std::integral_constant<int, 0>{});
        return;
    }
    AttnState<D> st;
    st.init();
    if (k_begin < k_end) {
#define LOAD(buf_, i_) load_tile<D>(buf_, cache, __builtin_amdgcn_readlane(my_page, (i_)), page_stride, kvh, Hkv, P, \
                                    (split * SPLIT + (i_) * 16) % P, g, n, stream)
#define STEP(buf_, i_) attn_tile_step<D>(st, buf_, qreg, scale, split * SPLIT + (i_) * 16, g, k_begin, k_end, k_begin, k_end)
        NormRotate<D> nq;
        nq.fetch(qkv + t * width + (long)head * D, head_ok, q_w, cs, g);
        if (AHEAD > 1 && tile0 == 0 && tile1 == TILES) {
            KVTile<D> tl[AHEAD + 1];
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) LOAD(tl[j], j);   // the first tiles travel while q is prepared
            nq.finish(qreg, q_w != nullptr, eps, cs != nullptr);
#pragma unroll
            for (int j = 0; j < TILES; ++j) {
                if (j + AHEAD < TILES) LOAD(tl[(j + AHEAD) % (AHEAD + 1)], j + AHEAD);
                __builtin_amdgcn_sched_barrier(0);         // (the scheduler would move the loads down to their uses)
                STEP(tl[j % (AHEAD + 1)], j);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            KVTile<D> ta, tb;
            int i = tile0;
            LOAD(ta, i);                                   // the first tiles travel while q is prepared
            if (i + 1 < tile1) LOAD(tb, i + 1);
            nq.finish(qreg, q_w != nullptr, eps, cs != nullptr);
            while (true) {
                STEP(ta, i);
                if (++i >= tile1) break;
                if (i + 1 < tile1) LOAD(ta, i + 1);
                STEP(tb, i);
                if (++i >= tile1) break;
                if (i + 1 < tile1) LOAD(tb, i + 1);
            }
        }
#undef LOAD
#undef STEP
    } else {
        NormRotate<D> nq;
        nq.fetch(qkv + t * width + (long)head * D, head_ok, q_w, cs, g);
        nq.finish(qreg, q_w != nullptr, eps, cs != nullptr);
    }
    if (owns) {
        NormRotate<D> nk;
        nk.fetch(qkv + t * width + (long)(Hq + kvh) * D, true, k_w, cs, g);
        nk.finish(kreg, k_w != nullptr, eps, cs != nullptr);
        float alpha;
        const float weight = own_weight(own_score<D>(qreg, kreg), scale, g, st.m, st.l, alpha);
#pragma unroll
        for (int db = 0; db < D / 16; ++db) add_own(st.acc[db], alpha, weight, *(const short4_t*)(vsrc + db * 16 + g * 4));
        store_own<D>(cache, kreg, vsrc, slots ? slots[t] : -1, page_stride, kvh, Hkv, P, g, n);
    }
    float l = st.l;
    const float m = st.m;
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (head_ok) {
#pragma unroll
        for (int db = 0; db < D / 16; ++db)
            *(floatx4*)(pacc + db * 16 + g * 4) = st.acc[db];
        if (g == 0) { pml[0] = m; pml[1] = l; }
    }
}

// ---- a block a token and key/value head ---------------------------------------------------------
// With tokens enough to give every compute unit a block, a token's keys are one block's: W waves take its tiles in turn, each with a
// softmax of its own, and join them in shared memory, so that a walk's start (positions, table, pages, q: some 4 us before the first
// key is there) is paid once and not for every 128 keys, nothing partial goes through memory and no second kernel waits for the
// last block.  Where the tokens are too few for that, the keys go in segments (of whole tiles, cut at absolute positions), which the
// merge kernel below joins.
// FUSED: from the q|k|v rows, as the kernel above; the last wave takes the token's own key.
template <int D, int W, bool FUSED>
__global__ __launch_bounds__(64 * W, W == 4 ? (FUSED ? 2 : 3) : 1) void attention_decode_block_kernel(
    const bf16_t* __restrict__ q, bf16_t* cache, const int* __restrict__ dec_tokens, const int* __restrict__ positions,
    const int* __restrict__ tok_seq, const int* __restrict__ block_table, int max_blocks, const int* __restrict__ shared_keys,
    const int* __restrict__ slots, const float* __restrict__ q_w, const float* __restrict__ k_w, float eps, const float* __restrict__ table,
    bf16_t* __restrict__ out, float* __restrict__ part_acc, float* __restrict__ part_ml,
    int Hq, int Hkv, int P, float scale, int window, int segments, int seg_keys, AttnTail tail) {
    constexpr int ROW = D + 4;                             // floats of a wave's result for a head in shared memory
    extern __shared__ __attribute__((aligned(16))) float joined[];
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int seg = blockIdx.x, kvh = blockIdx.y, di = blockIdx.z;
    const int G = Hq / Hkv;
    const int t = dec_tokens ? dec_tokens[di] : di;       // (no list: every row, in order)
    const int p = positions[t], row = tok_seq[t];
    const int last = FUSED ? p : p + 1;                    // the cached keys end here
    const int lo = first_seen_key(p, window);
    const int k_begin = max(seg * seg_keys, lo);
    const int k_end = min((seg + 1) * seg_keys, last);
    const bool owns = FUSED && seg == p / seg_keys;        // this block takes the token's own key and value
    const int head = kvh * G + n;
    const bool head_ok = n < G;
    if (k_begin >= k_end && !owns) {                       // nothing of this segment is seen by the token (never if it is the only one)
        if (wave == 0 && head_ok && g == 0) {
            float* pml = part_ml + (((long)di * Hq + head) * segments + seg) * 2;
            pml[0] = -INFINITY;
            pml[1] = 0.f;
        }
        return;
    }
    const long page_stride = 2L * Hkv * P * D;
    const int* bt = block_table + (long)row * max_blocks;
    const int shared = shared_keys ? shared_keys[row] : 0;
    // the wave's i-th tile is the segment's (wave + W i)-th; lane l holds the page and the place of the l-th (a segment has at most 2048 keys)
    const int first = k_begin / 16 + wave, tiles = k_begin < k_end ? max(0, ((k_end + 15) / 16 - first + W - 1) / W) : 0;
    const int my_key = (first + lane * W) * 16, my_place = my_key % P;
    const int my_page = lane < tiles ? bt[my_key / P] : 0;
    bf16x8 qreg[D / 32];
    const long width = FUSED ? (long)(Hq + 2 * Hkv) * D : (long)Hq * D;
    const float* cs = FUSED && table ? table + (long)p * D : nullptr;
    [[maybe_unused]] NormRotate<D> nq;
    if constexpr (FUSED) {
        nq.fetch(q + t * width + (long)head * D, head_ok, q_w, cs, g);
    } else {
        const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < D / 32; ++c) qreg[c] = head_ok ? *(const bf16x8*)(q + t * width + (long)head * D + c * 32 + g * 8) : zero8;
    }
    AttnState<D> st;
    st.init();
    KVTile<D> ta, tb;
#define LOAD(buf_, i_) load_tile<D>(buf_, cache, __builtin_amdgcn_readlane(my_page, i_), page_stride, kvh, Hkv, P, \
                                    __builtin_amdgcn_readlane(my_place, i_), g, n, (first + (i_) * W) * 16 >= shared)
#define STEP(buf_, i_) attn_tile_step<D>(st, buf_, qreg, scale, (first + (i_) * W) * 16, g, k_begin, k_end, k_begin, k_end)
    if (tiles > 0) LOAD(ta, 0);
    if (tiles > 1) LOAD(tb, 1);
    if constexpr (FUSED) nq.finish(qreg, q_w != nullptr, eps, cs != nullptr);
    for (int i = 0; i < tiles;) {
        STEP(ta, i);
        if (i + 2 < tiles) LOAD(ta, i + 2);
        if (++i >= tiles) break;
        STEP(tb, i);
        if (i + 2 < tiles) LOAD(tb, i + 2);
        ++i;
    }
#undef LOAD
#undef STEP
    if constexpr (FUSED) {
        if (owns && wave == W - 1) {
            const bf16_t* vsrc = q + t * width + (long)(Hq + Hkv + kvh) * D;
            bf16x8 kreg[D / 32];
            NormRotate<D> nk;
            nk.fetch(q + t * width + (long)(Hq + kvh) * D, true, k_w, cs, g);
            short4_t vv[D / 16];
#pragma unroll
            for (int db = 0; db < D / 16; ++db) vv[db] = *(const short4_t*)(vsrc + db * 16 + g * 4);
            nk.finish(kreg, k_w != nullptr, eps, cs != nullptr);
            float alpha;
            const float weight = own_weight(own_score<D>(qreg, kreg), scale, g, st.m, st.l, alpha);
#pragma unroll
            for (int db = 0; db < D / 16; ++db) add_own(st.acc[db], alpha, weight, vv[db]);
            store_own<D>(cache, kreg, vsrc, slots ? slots[t] : -1, page_stride, kvh, Hkv, P, g, n);
        }
    }
    float l = st.l;
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    float* const ml = joined + W * G * ROW;
    if (head_ok) {
        float* acc = joined + (wave * G + n) * ROW;
#pragma unroll
        for (int db = 0; db < D / 16; ++db) *(floatx4*)(acc + db * 16 + g * 4) = st.acc[db];
        if (g == 0) {
            ml[(wave * G + n) * 2] = st.m;
            ml[(wave * G + n) * 2 + 1] = l;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < G * D; i += 64 * W) {
        const int j = i / D, d = i % D;
        float m[W], s[W], o[W], top = -INFINITY;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            m[w] = ml[(w * G + j) * 2];
            s[w] = ml[(w * G + j) * 2 + 1];
            o[w] = joined[(w * G + j) * ROW + d];
        }
#pragma unroll
        for (int w = 0; w < W; ++w) top = fmaxf(top, m[w]);
        float sum = 0.f, x = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float e = __expf(m[w] - top);            // (0 of a wave that had no tile)
            sum += e * s[w];
            x += e * o[w];
        }
        if (segments == 1) {
            tail.store(out, t, kvh * G + j, d, x * (1.f / sum));   // (as the merge of one segment has it)
        } else {
            const long at = ((long)di * Hq + kvh * G + j) * segments + seg;
            part_acc[at * D + d] = x;
            if (d == 0) {
                part_ml[at * 2] = top;
                part_ml[at * 2 + 1] = sum;
            }
        }
    }
}

// out[t, head, :] = sum_s e^{m_s - M} acc_s / sum_s e^{m_s - M} l_s,  M = max_s m_s.
// One block of 256 threads per (token, head): wave w sums the splits w, w + 4, ... in ascending
// order, the four sums are added in the order of the waves.
template <int D>
__global__ __launch_bounds__(256) void attention_decode_merge_kernel(
    const float* __restrict__ part_acc, const float* __restrict__ part_ml, const int* __restrict__ dec_tokens,
    bf16_t* __restrict__ out, int Hq, int num_splits, int sink, AttnTail tail) {
    constexpr int PER = (D + 63) / 64;
    __shared__ float red_o[4][D];
    __shared__ float red_l[4];
    __shared__ float red_m[4];
    const int di = blockIdx.x, head = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float* pml = part_ml + ((long)di * Hq + head) * num_splits * 2;
    const float* pacc = part_acc + ((long)di * Hq + head) * num_splits * D;
    // (the largest maximum is reduced only after the first eight splits' loads have been issued: its
    // own loads were issued before them, so waiting for those does not wait for these)
    const float sk = sink ? tail.sink_of(head) : 0.f;
    float M = -INFINITY;
    for (int s = lane; s < num_splits; s += 64) M = fmaxf(M, pml[2 * s]);
    bool reduced = false;
    float denom = 0.f;
    float o[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) o[i] = 0.f;
    // eight of the wave's splits at a time: their maxima, sums and accumulator rows are all asked
    // for before the first is used (one trip to memory for eight); added in ascending order
    for (int s0 = wave; s0 < num_splits; s0 += 32) {
        float ms[8], ls[8], a[8][PER];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int s = s0 + 4 * k;
            ms[k] = s < num_splits ? pml[2 * s] : -INFINITY;
            ls[k] = s < num_splits ? pml[2 * s + 1] : 0.f;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int s = s0 + 4 * k;
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int d = lane + i * 64;
                // (asked for without waiting for the maxima: an empty split's accumulator was never
                // written, and what is read of it is not used below; a split beyond the last reads the last)
                a[k][i] = d < D ? pacc[(long)(s < num_splits ? s : num_splits - 1) * D + d] : 0.f;
            }
        }
        // (sink: one more entry that carries no value)
        if (!reduced) { M = wave_max(M); if (sink) M = fmaxf(M, sk); reduced = true; }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (ms[k] == -INFINITY) continue;
            const float wgt = __expf(ms[k] - M);
            denom += wgt * ls[k];
#pragma unroll
            for (int i = 0; i < PER; ++i) o[i] += wgt * a[k][i];
        }
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int d = lane + i * 64;
        if (d < D) red_o[wave][d] = o[i];
    }
    if (lane == 0) red_l[wave] = denom;
    __syncthreads();
    if (wave == 0) {
        const float inv = 1.f / (red_l[0] + red_l[1] + red_l[2] + red_l[3] + (sink ? __expf(sk - M) : 0.f));
        const long row = dec_tokens ? dec_tokens[di] : di;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int d = lane + i * 64;
            if (d < D) tail.store(out, row, head, d, (red_o[0][d] + red_o[1][d] + red_o[2][d] + red_o[3][d]) * inv);
        }
    }
}

// also what the prefill kernel takes, but for the page size, which it wants to be a power of two
bool qe_attention_decode_ok(int Hq, int Hkv, int D, int P, int dt_a) {
    return dt_a == QE_BF16 && (D == 64 || D == 128) && P % 16 == 0 && Hq % Hkv == 0 && Hq / Hkv <= 16;
}

size_t qe_attention_decode_workspace(int n_dec, int Hq, int D, int num_splits) {
    return (size_t)n_dec * Hq * num_splits * (D + 2) * sizeof(float);
}

// The segments of a block's form: 0 (the splits are the better way), else how many, of seg_keys keys each.  (us, norm, rotation and cache write inside, 16 heads of 128
// on 8 if nothing else is said, rows of half to one and a half times the keys; splits of 128 and their merge, then blocks of four waves.)
// Up to eight tokens are the splits': four of 400 keys 13.0, 13.4, of 1000 14.3, 16.0, of 2000 16.2, 16.4.
// Up to 16 tokens, which every other kernel of their step takes in one order, the way is the model's and a token's segments follow its own position
// alone: its bits are the same beside any others.  With four key/value heads or fewer the blocks are too few: 9 tokens of one of 100 keys 10.4, 8.4, of 300 10.2, 11.4, of
// 640 10.6, 14.6, of 3000 13.5, 14.5; 12 of four of 200 10.8, 10.2, of 640 13.4, 14.8, of 1900 18.8, 21.2, of 6000 36.4, 36.2.  With more: 9 of 60 12.3, 6.7, of 300 13.5, 10.9, of 680 13.4, 15.3, of
// 1000 17.6, 20.4, of 3000 26.8, 25.7; 16 of 60 14.1, 6.8, of 300 15.7, 11.1, of 680 15.8, 16.0, of 1000 21.4, 21.5, of 3000 38.8, 37.5, of 6000 85.5, 82.0 (tokens at 512 to 1535 in segments of 384:
// 9 of 1000 19.2, but 16 of 680 18.6).
// More tokens: one segment up to 1024 positions, and up to 2048 for more than 128 blocks, but where the splits are few enough to run four waves each; else segments of 512.  The
// last position counts as recorded steps know it, as the end of a stretch of 1024 (the first two, of 512): a step has the same segments whether it is recorded or runs as it comes.
// (Splits, 512 keys and one segment: 20 tokens of one key/value head of 640 keys 10.6, 14.5, 16.8, 64 of 1000 16.1, 17.8, 23.6; 64 of two of 1000 22.9, 22.6, 24.5; 20 of eight of 1000 27.3, 28.5,
// 23.8, of 3000 47.9, 49.7, 55.3; 32 of 3000 86.7, 81.8, 84.3; 64 of 1000 64.0, 67.1, 46.7, of 1900 109.7, 103.9, 99.3; 48 of four of 3000 69.5, 61.2, 68.2.  Cut into as many as fill the units three
// times: 20 of 3000 63.4, 32 96.5.)
static int last_of_stretch(int position) { return position < 512 ? 511 : position | 1023; }
static int block_segments(int n_dec, int Hkv, int max_position, int window, int sink, float softcap, int& seg_keys) {
    if (n_dec <= 8 || window != 0 || sink || softcap > 0.f) return 0;
    if (n_dec <= 16) {
        seg_keys = 512;
        return Hkv <= 4 ? 0 : max_position / seg_keys + 1;
    }
    const long blocks = (long)Hkv * n_dec;
    const int last = last_of_stretch(max_position);
    if (last >= 512 && (last / 128 + 1) * blocks <= 544) return 0;
    seg_keys = last < 1024 || (last < 2048 && blocks > 128) ? last + 1 : 512;
    return max_position / seg_keys + 1;
}

template <int D, bool FUSED>
static void launch_block(const bf16_t* q, bf16_t* cache, const int* dec_tokens, int n_dec, const int* positions, const int* tok_seq,
                         const int* block_table, int max_blocks, const int* shared_keys, const int* slots, const float* q_w, const float* k_w,
                         float eps, const float* table, bf16_t* out, float* part, int Hq, int Hkv, int P, float scale, int window, int segments,
                         int seg_keys, hipStream_t stream, const AttnTail& tail) {
    constexpr int W = 4;                                   // (2048 keys a segment at the most: a wave's 32 tiles)
    float* part_ml = part + (size_t)n_dec * Hq * segments * D;
    attention_decode_block_kernel<D, W, FUSED><<<dim3(segments, Hkv, n_dec), 64 * W, (size_t)W * (Hq / Hkv) * (D + 6) * sizeof(float), stream>>>(
        q, cache, dec_tokens, positions, tok_seq, block_table, max_blocks, shared_keys, slots, q_w, k_w, eps, table, out, part, part_ml,
        Hq, Hkv, P, scale, window, segments, seg_keys, tail);
    if (segments > 1)
        attention_decode_merge_kernel<D><<<dim3(n_dec, Hq), 256, 0, stream>>>(part, part_ml, dec_tokens, out, Hq, segments, 0, tail);
}

// dec_tokens: the rows of q that are single new tokens of their requests (null: the rows
// 0 .. n_dec - 1, which saves every wave a dependent load).  max_position: the
// largest of their positions (fixes the number of splits).  workspace: at least
// qe_attention_decode_workspace(...) bytes.  shared_keys: null, or for every row of the block table
// the number of the request's first keys that other requests of the step may read as well (pages they
// hold together): a hint for the caches, results do not depend on it.  split_keys: 128 or 256; or 0, splits of 128 or, where that
// is quicker, a block a token and key/value head, whose sums have another order (the workspace is that of splits of 128).
int qe_attention_decode(const void* q, void* out, const void* cache, const int* dec_tokens, int n_dec,
                        const int* positions, const int* tok_seq, const int* block_table, int max_blocks,
                        const int* shared_keys, int Hq, int Hkv, int D, int P, float scale, int window, int keep_first,
                        int sink, float softcap, int max_position, int split_keys, void* workspace, size_t workspace_bytes,
                        hipStream_t stream, const AttnTail& tail) {
    QE_REQUIRE(qe_attention_decode_ok(Hq, Hkv, D, P, QE_BF16), "decode attention: sizes not taken");
    QE_REQUIRE(split_keys == 0 || split_keys == 128 || split_keys == 256, "decode attention: splits of 128 or 256 keys, not %d", split_keys);
    if (n_dec == 0) return 0;
    const bool blocks = split_keys == 0;
    if (blocks) split_keys = 128;
    const int num_splits = max_position / split_keys + 1;
    QE_REQUIRE(num_splits <= 65535 && n_dec <= 65535, "decode attention: too many splits or tokens");
    QE_REQUIRE(workspace_bytes >= qe_attention_decode_workspace(n_dec, Hq, D, num_splits),
               "decode attention: workspace of %zu bytes is too small", workspace_bytes);
    float* part_acc = (float*)workspace;
    float* part_ml = part_acc + (size_t)n_dec * Hq * num_splits * D;
    (void)qe_cdiv;
    dim3 grid(num_splits, Hkv, n_dec);
    dim3 mgrid(n_dec, Hq);
    int seg_keys = 0;
    if (const int segments = blocks ? block_segments(n_dec, Hkv, max_position, window, sink, softcap, seg_keys) : 0) {
#define QE_DECODE_BLOCK(D_)                                                                             \
        launch_block<D_, false>((const bf16_t*)q, (bf16_t*)cache, dec_tokens, n_dec, positions, tok_seq, block_table, max_blocks, shared_keys, \
                                nullptr, nullptr, nullptr, 0.f, nullptr, (bf16_t*)out, part_acc, Hq, Hkv, P, scale, window, segments, \
                                seg_keys, stream, tail)
        if (D == 128) QE_DECODE_BLOCK(128);
        else QE_DECODE_BLOCK(64);
#undef QE_DECODE_BLOCK
        QE_LAUNCH_CHECK();
        return 0;
    }
    // (512 splits of 8 tokens over 1000 keys: 14.0 us with one wave a split, 12.6 with four; from 576 on the two are within 3 %
    // of each other: 14.2 and 14.4, 1024 17.6 and 17.4)
    const bool four = (long)num_splits * Hkv * n_dec <= 512 && max_position >= 16 * ALONE;
    if (softcap > 0.f) scale = scale * 2.f * 1.4426950408889634f / softcap;
#define QE_DECODE_SPLIT2(D_, S_, CAP_, W_)                                                              \
        attention_decode_split_kernel<D_, S_, CAP_, W_><<<grid, 64 * W_, 0, stream>>>(                  \
            (const bf16_t*)q, (const bf16_t*)cache, dec_tokens, positions, tok_seq, block_table,        \
            max_blocks, shared_keys, part_acc, part_ml, Hq, Hkv, P, scale, window, keep_first, num_splits, softcap)
#define QE_DECODE_SPLIT(D_, S_, CAP_)                                                                   \
    do {                                                                                                \
        if (four) QE_DECODE_SPLIT2(D_, S_, CAP_, 4);                                                   \
        else QE_DECODE_SPLIT2(D_, S_, CAP_, 1);                                                         \
    } while (0)
#define QE_DECODE(D_, S_)                                                                               \
    do {                                                                                                \
        if (softcap > 0.f) QE_DECODE_SPLIT(D_, S_, true);                                               \
        else QE_DECODE_SPLIT(D_, S_, false);                                                            \
        attention_decode_merge_kernel<D_><<<mgrid, 256, 0, stream>>>(part_acc, part_ml, dec_tokens,     \
                                                                     (bf16_t*)out, Hq, num_splits, sink, tail); \
    } while (0)
    if (D == 128 && split_keys == 128) QE_DECODE(128, 128);
    else if (D == 128) QE_DECODE(128, 256);
    else if (split_keys == 128) QE_DECODE(64, 128);
    else QE_DECODE(64, 256);
#undef QE_DECODE
#undef QE_DECODE_SPLIT
#undef QE_DECODE_SPLIT2
    QE_LAUNCH_CHECK();
    return 0;
}

// The fused form: qkv [T, (Hq + 2 Hkv) D] as the projection left it; q_w, k_w (per-head norm weights)
// and table (rows [cos | sin] of D floats per position) may be null; slots: the cache slot of each
// row's own key and value (negative: not written).  Every row named in dec_tokens brings exactly
// its own new key; the cache holds the keys before it.
int qe_attention_decode_fused(const void* qkv, void* out, void* cache, const int* dec_tokens, int n_dec,
                              const int* positions, const int* tok_seq, const int* block_table, int max_blocks,
                              const int* shared_keys, const int* slots, const float* q_w, const float* k_w, float eps, const float* table,
                              int Hq, int Hkv, int D, int P, float scale, int window, int max_position,
                              int split_keys, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    QE_REQUIRE(qe_attention_decode_ok(Hq, Hkv, D, P, QE_BF16), "decode attention: sizes not taken");
    QE_REQUIRE(split_keys == 0 || split_keys == 128 || split_keys == 256, "decode attention: splits of 128 or 256 keys, not %d", split_keys);
    if (n_dec == 0) return 0;
    const bool blocks = split_keys == 0;
    if (blocks) split_keys = 128;
    const int num_splits = max_position / split_keys + 1;
    QE_REQUIRE(num_splits <= 65535 && n_dec <= 65535, "decode attention: too many splits or tokens");
    QE_REQUIRE(workspace_bytes >= qe_attention_decode_workspace(n_dec, Hq, D, num_splits),
               "decode attention: workspace of %zu bytes is too small", workspace_bytes);
    float* part_acc = (float*)workspace;
    float* part_ml = part_acc + (size_t)n_dec * Hq * num_splits * D;
    dim3 grid(num_splits, Hkv, n_dec);
    dim3 mgrid(n_dec, Hq);
    AttnTail tail{};
    tail.out_stride = (long)Hq * D;
    tail.dv = D;
    int seg_keys = 0;
    if (const int segments = blocks ? block_segments(n_dec, Hkv, max_position, window, 0, 0.f, seg_keys) : 0) {
#define QE_DECODE_BLOCK(D_)                                                                             \
        launch_block<D_, true>((const bf16_t*)qkv, (bf16_t*)cache, dec_tokens, n_dec, positions, tok_seq, block_table, max_blocks, shared_keys, \
                               slots, q_w, k_w, eps, table, (bf16_t*)out, part_acc, Hq, Hkv, P, scale, window, segments, seg_keys, stream, tail)
        if (D == 128) QE_DECODE_BLOCK(128);
        else QE_DECODE_BLOCK(64);
#undef QE_DECODE_BLOCK
        QE_LAUNCH_CHECK();
        return 0;
    }
    const long waves = (long)num_splits * Hkv * n_dec;
    const bool few = waves <= 1024;                            // at most a wave per SIMD: loads further ahead
    // (every wave prepares q: 256 splits of one request each take 11.4 us with four, 12.6 with one; 384 13.2 with one, 17.1 with four)
    const bool four = waves <= 256 && max_position > 16 * ALONE;
#define QE_DECODE_FUSED_ARGS(D_)                                                                        \
            (const bf16_t*)qkv, (bf16_t*)cache, dec_tokens, positions, tok_seq, block_table, max_blocks, \
            shared_keys, slots, q_w, k_w, eps, table, part_acc, part_ml, Hq, Hkv, P, scale, window, num_splits
#define QE_DECODE_FUSED(D_, S_)                                                                         \
    do {                                                                                                \
        if (four) attention_decode_fused_split_kernel<D_, S_, 1, 4><<<grid, 320, 0, stream>>>(QE_DECODE_FUSED_ARGS(D_)); \
        else if (few) attention_decode_fused_split_kernel<D_, S_, 3, 1><<<grid, 64, 0, stream>>>(QE_DECODE_FUSED_ARGS(D_)); \
        else attention_decode_fused_split_kernel<D_, S_, 1, 1><<<grid, 64, 0, stream>>>(QE_DECODE_FUSED_ARGS(D_)); \
        attention_decode_merge_kernel<D_><<<mgrid, 256, 0, stream>>>(part_acc, part_ml, dec_tokens,     \
                                                                     (bf16_t*)out, Hq, num_splits, 0, tail); \
    } while (0)
    if (D == 128 && split_keys == 128) QE_DECODE_FUSED(128, 128);
    else if (D == 128) QE_DECODE_FUSED(128, 256);
    else if (split_keys == 128) QE_DECODE_FUSED(64, 128);
    else QE_DECODE_FUSED(64, 256);
#undef QE_DECODE_FUSED
#undef QE_DECODE_FUSED_ARGS
    QE_LAUNCH_CHECK();
    return 0;
}
