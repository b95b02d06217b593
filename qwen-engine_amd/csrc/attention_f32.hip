// Attention in 32-bit on the matrix units: the kernel of the float32 mode for head sizes in
// steps of 16.  Every product and sum is an IEEE 32-bit operation (v_mfma_f32_16x16x4_f32 takes
// 32-bit operands and accumulates in 32-bit; no reduced-precision matrix mode).
//
// One block of four or eight waves per (token, key/value head, 16 query heads of its group): the heads are
// the 16 columns, so the keys and values of a key/value head are read once for all heads of the
// group.  The keys the token sees, lo .. p, are taken 16 at a time from absolute multiples of 16
// in eight walks: walk w takes the tiles w, w + 8, ..., the results of the walks w and w + 4 are put together,
// and the four of those in their order, through shared memory (a single new token over a long context would else
// be one wave's walk).  The order of the sums so depends on the position and the window only: not on whether
// four waves take two walks each, one after the other (many tokens), or eight one each (few).  For a tile
// of 16 keys:
//   S^T[key, col] = K[key, :] . Q[col, :]       D / 4 MFMAs of 16 x 16 x 4;
//       lane (g, r), g = lane / 16, r = lane % 16, holds K[key r][16 c + 4 g .. + 4] of feature block
//       c as one 16-byte load, and its element j goes into the j-th MFMA of the block (which
//       feature stands at which place of the sum does not matter as long as Q has it at the same)
//   online softmax per column over the lanes (g, n) that share column n, in 32-bit
//   O^T[d, col] += V^T[d, key] . P^T[key, col]   4 MFMAs per 16 rows of d: the j-th takes, at place
//       g of its sum, key 4 g + j: that is the probability a lane already holds as its element j,
//       and of V^T the lane needs row d = 16 db + r at keys 4 g .. 4 g + 3
// Any page size.  Keys outside lo .. p are never read
// (their memory may be unwritten): they enter as zeros with a score of minus infinity.
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float floatx4;

__device__ __forceinline__ float max_over_rows_of_lanes(float v) {
    float a, b;
    pair_across_rows(v, a, b);
    v = fmaxf(a, b);
    pair_across_halves(v, a, b);
    return fmaxf(a, b);
}

#define F32_WALKS 8
#define F32_SLOTS 4           // results in shared memory: one for the walks w and w + 4 together

// NW waves.  AHEAD: 1: a tile's values are asked for before its scores, the next tile's keys before this tile's softmax; 2 (pages of whole
// tiles): the next tile whole before this one's scores.  Few tokens are bound by their walks' trips to memory (2 tokens of 16 heads on 8
// over 744 keys: 55 us with four waves, each with 12 tiles one after the other and every load where it is used, 32 with eight and AHEAD 1; over 512 keys
// 27.8, with 2 22.7, over 2048 93 and 63; what is left is what a compute unit alone gets, some 35 GB/s); with many tokens other waves fill the time, and the
// registers that this takes cost more.
//
// ROWS (no window, at most eight heads a key/value head): the 16 columns are 16 / G tokens' heads, which see the keys of one
// request up to their own positions, so that many tokens read and multiply a tile once instead of each by itself; neighbours in the list that belong to
// different requests are walked by blocks of their own, block z the z-th request's, the last block what is left, one after the other.  A column's sums are those it has alone: a tile it sees nothing of leaves
// them as they are.  (Portions of 328 and 416 rows of 16 heads of 128 on 8: 200 us, a block a token, and 42; 2048 rows 1980, 300; 400 of 64
// heads 120, 78; 40 rows 11.7, 11.2.)
//
// FUSED (eight waves, AHEAD 2, at most 16 heads a key/value head): q is the q|k|v rows; the waves first norm and turn the token's heads and write its key
// and value to the cache, with the sums and roundings of the kernel that does this for few tokens, while the walks' first tiles are on their
// way.  The walk with the token's own key takes it, and its value, from shared memory: they may be written nowhere, and their page may not be
// there.  (2 tokens of 16 heads on 8 over 512 keys: the two kernels 22.6 and 3.9 us, in one 21.6, and a launch
// less for the host, some 12 us of a step that is not recorded; of 414 and 731 keys 27.3, 26.5 with the own key read back from the cache.)
struct OwnToken {
    const float* q_w;
    const float* k_w;
    float eps;
    const float* table;
    const int* slots;
};
template <int DB, int NW, int AHEAD, bool ROWS, bool FUSED = false>      // DB: head size / 16
__global__ __launch_bounds__(64 * NW, NW == F32_SLOTS && DB <= 8 ? (ROWS || AHEAD ? 2 : 3) : 1) void attention_f32_kernel(
    const float* __restrict__ q, float* __restrict__ out, const float* __restrict__ cache,
    const int* __restrict__ positions, const int* __restrict__ tok_seq,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ tokens, int T,
    int Hq, int Hkv, int P, float scale, int window, int keep_first, int sink, float softcap, AttnTail tail, OwnToken own) {
    static_assert(!FUSED || (NW == F32_WALKS && AHEAD == 2 && !ROWS), "");
    constexpr int D = DB * 16;
    // [F32_SLOTS][DB * 4 + 2][64]; FUSED: the token's query heads before that, [G][D], and behind it its key and its value
    extern __shared__ float merge_lds[];
    [[maybe_unused]] float* const own_kv = merge_lds + (long)F32_SLOTS * (DB * 4 + 2) * 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, n = lane & 15;
    const int G = Hq / Hkv, R = ROWS ? 16 / G : 1;         // (R: tokens a block)
    const int groups16 = ROWS ? 1 : (G + 15) / 16;
    // (ROWS: a compute die has the blocks of every eighth key/value head, whose keys its L2 holds; later tokens, which see more keys, start first)
    const int kvh = ROWS ? blockIdx.x : blockIdx.y / groups16, hg = ROWS ? 0 : blockIdx.y % groups16;
    const int mine = ROWS ? n / G : 0, first = ROWS ? (int)(gridDim.y - 1 - blockIdx.y) * R : blockIdx.x;      // the column's token of the block's
    const int at = min(first + min(mine, R - 1), T - 1);
    const long t = tokens ? tokens[at] : at;
    const int head = kvh * G + (ROWS ? n - mine * G : hg * 16 + n);
    const bool head_ok = ROWS ? mine < R && first + mine < T : hg * 16 + n < G;
    const int p = positions[t], seq = tok_seq[t];
    const long page_stride = 2L * Hkv * P * D;
    const bool vec_v = (P & 3) == 0;                      // four consecutive keys of a value row lie in one page, aligned

    floatx4 qv[DB];
#pragma unroll
    for (int c = 0; c < DB; ++c) {
        qv[c] = floatx4{0.f, 0.f, 0.f, 0.f};
        if (!FUSED && head_ok) qv[c] = *(const floatx4*)(q + (t * Hq + head) * D + c * 16 + g * 4);
    }
    // (one round, but for a block whose tokens belong to several requests, and for one with a value that is infinite or NaN: where a column does
    // not see it, it has met a weight of 0, so each token then has a round of its own)
    unsigned long todo = ROWS ? __ballot(head_ok) : 1ul;
    if (ROWS) {
        const auto of_first = [&]() { return __ballot(head_ok && seq == __builtin_amdgcn_readlane(seq, __builtin_ctzl(todo))); };
        for (int z = blockIdx.z; z > 0; --z) {
            todo &= ~of_first();
            if (!todo) return;                             // (the whole block: no barrier has been met yet)
        }
        if (blockIdx.z + 1 < gridDim.z) todo &= of_first();
    }
    bool one_by_one = false;
    do {
    const int next = ROWS ? __builtin_ctzl(todo) : 0;
    const int first_seq = ROWS ? __builtin_amdgcn_readlane(seq, next) : seq;
    // the column's token is of this round's request
    const bool on = head_ok && seq == first_seq && (!one_by_one || mine == __builtin_amdgcn_readlane(mine, next));
    if (ROWS) todo &= ~__ballot(on);
    bool odd = false;
    int top = p, first_p = p;                              // no column of the round sees a key beyond top, all see those up to first_p
    if (ROWS) {
        top = on ? p : -1;
        first_p = on ? p : 0x7fffffff;
#pragma unroll
        for (int k = 1; k < 16; k <<= 1) {
            top = max(top, __shfl_xor(top, k, 64));
            first_p = min(first_p, __shfl_xor(first_p, k, 64));
        }
        top = __builtin_amdgcn_readfirstlane(top);
        first_p = __builtin_amdgcn_readfirstlane(first_p);
    }
    const int lo = ROWS ? 0 : first_seen_key(p, window);
    const int* bt = block_table + (long)first_seq * max_blocks;
    // The tiles of the walks: those of the kept first keys 0 .. kf - 1 that lie wholly before the window's
    // first tile, then the tiles from the window's first on (which holds the rest of the kept keys, if
    // any); tile number i of this list is walk i % F32_WALKS's.
    const int kf = keep_first < lo ? keep_first : lo;
    const int tile_lo = lo / 16;
    const int n_first = (kf + 15) / 16 < tile_lo ? (kf + 15) / 16 : tile_lo;
    const int n_tiles = n_first + top / 16 - tile_lo + 1;
    const auto tile_key = [&](int ti) { return 16 * (ti < n_first ? ti : tile_lo + ti - n_first); };
    // Pages of whole tiles: lane i holds the page of the walk's i-th tile of 64 (one load for all of them, where each tile's lookups
    // were two trips to memory of their own); a tile's page is then the same for the wave, and so is its place in it.  Other page sizes:
    // every lane looks its own keys' pages up.
    const bool whole = P % 16 == 0;
    // (FUSED: the last tile may hold no key but the token's own; its page is then not looked up, and what is read is some page of the cache)
    const bool own_alone = FUSED && max(p / 16 * 16, lo) >= p;
    int my_page = 0;
    const auto page_of = [&](int ti, int walk) {               // asked for tile by tile, in order
        const int j = (ti - walk) / F32_WALKS;
        if (!whole) return 0;
        if ((j & 63) == 0) {
            const int tl = ti + lane * F32_WALKS;
            if (tl < n_tiles - own_alone) my_page = bt[tile_key(tl) / P];
        }
        return __builtin_amdgcn_readlane(my_page, j & 63);
    };
    const auto load_keys = [&](int kk, int page, floatx4 (&kr)[DB]) {      // S^T: this lane brings the key row kk + n
        const int key_r = kk + n;
        const bool row_ok = (key_r >= lo || key_r < kf) && key_r <= top;
        const float* krow = cache + (long)page * page_stride + ((long)kvh * P + kk % P + n) * D + g * 4;
        if (!whole && row_ok) krow = cache + (long)bt[key_r / P] * page_stride + ((long)kvh * P + key_r % P) * D + g * 4;
#pragma unroll
        for (int c = 0; c < DB; ++c) kr[c] = row_ok ? *(const floatx4*)(krow + c * 16) : floatx4{0.f, 0.f, 0.f, 0.f};
    };
    const auto value_places = [&](int kk, int page, const bool (&ok)[4], long (&voff)[4]) {
        if (whole) {
            voff[0] = (long)page * page_stride + ((long)(Hkv + kvh) * P) * D + kk % P + 4 * g;
#pragma unroll
            for (int i = 1; i < 4; ++i) voff[i] = voff[0] + i;
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int kc = ok[i] ? kk + 4 * g + i : top;   // (an address that is valid; the value is not used)
            voff[i] = (long)bt[kc / P] * page_stride + ((long)(Hkv + kvh) * P) * D + kc % P;
        }
    };
    const auto load_value = [&](int db, const bool (&ok)[4], const long (&voff)[4]) {
        floatx4 vf;
        const long drow = (long)(db * 16 + n) * P;
        if (vec_v && ok[0] && ok[3]) {
            vf = *(const floatx4*)(cache + voff[0] + drow);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) vf[i] = ok[i] ? cache[voff[i] + drow] : 0.f;
        }
        return vf;
    };
    // a result of a walk, or of two: the accumulators, the maximum and the whole sum of column n
    float* const slot = merge_lds + (long)(wave % F32_SLOTS) * (DB * 4 + 2) * 64 + lane;
    floatx4 acc[DB];
    float m, l;
    const auto leave = [&]() {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) slot[(db * 4 + i) * 64] = acc[db][i];
        slot[(DB * 4) * 64] = m;
        slot[(DB * 4 + 1) * 64] = l;
    };
    // the result in the slot (of the walk F32_SLOTS before this one, or after it) and this one together: the earlier walk first
    const auto join = [&](bool own_first) {
        const float mo = slot[(DB * 4) * 64], lo_ = slot[(DB * 4 + 1) * 64];
        const float mt = fmaxf(m, mo);
        const float a = m == -INFINITY ? 0.f : expf(m - mt), b = mo == -INFINITY ? 0.f : expf(mo - mt);
        l = own_first ? fmaf(lo_, b, l * a) : fmaf(l, a, lo_ * b);
        m = mt;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float o = slot[(db * 4 + i) * 64];
                acc[db][i] = own_first ? fmaf(o, b, acc[db][i] * a) : fmaf(acc[db][i], a, o * b);
            }
    };
    // the token's heads to shared memory, normed and turned, its key and value to the cache too; a wave a head
    [[maybe_unused]] const auto prepare = [&]() {
        const int slot = own.slots ? own.slots[t] : -1;
        float* const kv = const_cast<float*>(cache) + (slot < 0 ? 0 : (long)(slot / P) * page_stride);
        const float* const cs = own.table ? own.table + (long)p * D : nullptr;
        for (int j = wave; j < G + 2; j += NW) {
            const float* src = q + (t * (Hq + 2 * Hkv) + (j < G ? kvh * G + j : j == G ? Hq + kvh : Hq + Hkv + kvh)) * D;
            if (j > G) {                                   // the value tile is [D][P]
                for (int d = lane; d < D; d += 64) own_kv[D + d] = src[d];
                if (slot >= 0)
                    for (int d = lane; d < D; d += 64) kv[((long)(Hkv + kvh) * D + d) * P + slot % P] = own_kv[D + d];
                continue;
            }
            const float* w = j < G ? own.q_w : own.k_w;
            float* const row = j < G ? merge_lds + j * D : own_kv;
            float ss = 0.f;
            for (int d = lane; d < D; d += 64) {
                const float v = src[d];
                row[d] = v;
                ss = __builtin_fmaf(v, v, ss);
            }
            if (w) {
                ss = wave_sum(ss);
                const float rstd = rsqrtf(ss / (float)D + own.eps);
                for (int d = lane; d < D; d += 64) row[d] = row[d] * rstd * w[d];
            }
            __builtin_amdgcn_wave_barrier();               // (a wave's accesses to shared memory are done in their order)
            if (cs)
                for (int i = lane; i < D / 2; i += 64) {
                    float x1 = row[i], x2 = row[D / 2 + i];
                    rotate_pair(cs[i], cs[D / 2 + i], x1, x2);
                    row[i] = x1;
                    row[D / 2 + i] = x2;
                }
            __builtin_amdgcn_wave_barrier();
            if (j == G && slot >= 0)
                for (int d = lane; d < D; d += 64) kv[((long)kvh * P + slot % P) * D + d] = row[d];
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < DB; ++c)
            if (head_ok) qv[c] = *(const floatx4*)(merge_lds + n * D + c * 16 + g * 4);
        __syncthreads();                                   // (the walks' results take the query heads' place)
    };
    // (a walk without a tile changes nothing where it is joined: where a wave's second walk, or every walk from the fifth on, has none,
    // there is nothing to join)
    const bool second = wave + F32_SLOTS < n_tiles, joins = F32_SLOTS < n_tiles;
    for (int walk = wave; walk < F32_WALKS && (walk == wave || second); walk += NW) {
        m = -INFINITY;
        l = 0.f;                                           // this lane's share of the column's sum
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[db] = floatx4{0.f, 0.f, 0.f, 0.f};
        // From a tile's scores its weights (s holds those of keys kk + 4 g + i of column n), with the running maximum and sum; returns the factor for
        // what was summed before.  sees: the keys that the column sees.
        const auto weigh = [&](floatx4& s, const bool (&sees)[4]) {
            float tmax = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[i] *= scale;
                if (softcap > 0.f) s[i] = softcap * tanhf(s[i] / softcap);
                if (!sees[i]) s[i] = -INFINITY;
                tmax = fmaxf(tmax, s[i]);
            }
            tmax = max_over_rows_of_lanes(tmax);
            const float mn = fmaxf(m, tmax);               // finite, as every tile of the walk holds a key that is seen (ROWS: by some column)
            const float ref = ROWS && mn == -INFINITY ? 0.f : mn;
            const float alpha = expf(m - ref);             // 0 on the first tile
            float psum = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[i] = sees[i] ? expf(s[i] - ref) : 0.f;
                psum += s[i];
            }
            l = l * alpha + psum;
            m = mn;
            return alpha;
        };
        const auto score = [&](const floatx4 (&kr)[DB]) {
            floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < DB; ++c)
#pragma unroll
                for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[c][j], qv[c][j], s, 0, 0, 0);
            return s;
        };
        // O^T: the lane brings, of the value rows d = 16 db + n, the keys kk + 4 g .. + 3
        const auto add_values = [&](int db, const floatx4& vf, const floatx4& pr, float alpha) {
            acc[db] *= alpha;
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[j], pr[j], acc[db], 0, 0, 0);
        };
        // the keys of the lane's four that are there, and those of them that the column sees
        const auto look = [&](int kk, bool (&ok)[4], bool (&sees)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = kk + 4 * g + i;
                ok[i] = (key >= lo || key < kf) && key <= top;
                sees[i] = ROWS ? key <= p && on : ok[i];
            }
        };
        if constexpr (AHEAD == 2) {
            // (pages of whole tiles.  What of a tile is not there lies in its page all the same: it is read, and zeros take its place)
            floatx4 ka[DB], va[DB], kb[DB], vb[DB];
            const auto ask = [&](int ti, floatx4 (&kr)[DB], floatx4 (&vr)[DB]) {
                const int in = tile_key(ti) % P;
                const float* const page = cache + (long)page_of(ti, walk) * page_stride;
                const float* const krow = page + ((long)kvh * P + in + n) * D + g * 4;
                const float* const vrow = page + ((long)(Hkv + kvh) * D + n) * P + in + 4 * g;
#pragma unroll
                for (int c = 0; c < DB; ++c) kr[c] = *(const floatx4*)(krow + c * 16);
#pragma unroll
                for (int db = 0; db < DB; ++db) vr[db] = *(const floatx4*)(vrow + (long)db * 16 * P);
            };
            const auto step = [&](int ti, floatx4 (&kr)[DB], floatx4 (&vr)[DB]) {
                const int kk = tile_key(ti);
                bool ok[4], sees[4];
                look(kk, ok, sees);
                if (kk < lo || kk + 15 > top) {
                    const bool row_ok = (kk + n >= lo || kk + n < kf) && kk + n <= top;
#pragma unroll
                    for (int c = 0; c < DB; ++c)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            kr[c][i] = row_ok ? kr[c][i] : 0.f;
                            vr[c][i] = ok[i] ? vr[c][i] : 0.f;
                        }
                }
                if (FUSED && ti == n_tiles - 1) {          // (what was read in the own key's place, written by now or not, is not used)
                    const int in = p % 16;
                    int here = lane;                       // (so that nothing of this is kept in registers through the walk)
                    asm volatile("" : "+v"(here));
                    const int g = here >> 4, n = here & 15;
                    if (n == in) {
#pragma unroll
                        for (int c = 0; c < DB; ++c) kr[c] = *(const floatx4*)(own_kv + c * 16 + g * 4);
                    }
                    if (g == in / 4) {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (in % 4 == i) {
#pragma unroll
                                for (int c = 0; c < DB; ++c) vr[c][i] = own_kv[D + c * 16 + n];
                            }
                    }
                }
                floatx4 pr = score(kr);
                const float alpha = weigh(pr, sees);
#pragma unroll
                for (int db = 0; db < DB; ++db) add_values(db, vr[db], pr, alpha);
            };
            int ti = walk;
            if (ti < n_tiles) ask(ti, ka, va);
            if constexpr (FUSED) prepare();
            while (ti < n_tiles) {
                if (ti + F32_WALKS < n_tiles) ask(ti + F32_WALKS, kb, vb);
                step(ti, ka, va);
                ti += F32_WALKS;
                if (ti >= n_tiles) break;
                if (ti + F32_WALKS < n_tiles) ask(ti + F32_WALKS, ka, va);
                step(ti, kb, vb);
                ti += F32_WALKS;
            }
        } else {
            floatx4 kr[DB], vr[AHEAD ? DB : 1];
            int page = 0;
            if (AHEAD && walk < n_tiles) {
                page = page_of(walk, walk);
                load_keys(tile_key(walk), page, kr);
            }
            for (int ti = walk; ti < n_tiles; ti += F32_WALKS) {
                const int kk = tile_key(ti);
                bool ok[4], sees[4];
                look(kk, ok, sees);
                if (!AHEAD) {
                    page = page_of(ti, walk);
                    load_keys(kk, page, kr);
                }
                long voff[4];
                if (AHEAD) {
                    value_places(kk, page, ok, voff);
#pragma unroll
                    for (int db = 0; db < DB; ++db) vr[AHEAD ? db : 0] = load_value(db, ok, voff);
                    __builtin_amdgcn_sched_barrier(0);
                }
                floatx4 pr = score(kr);
                if (AHEAD && ti + F32_WALKS < n_tiles) {
                    page = page_of(ti + F32_WALKS, walk);
                    load_keys(tile_key(ti + F32_WALKS), page, kr);
                }
                const float alpha = weigh(pr, sees);
                if (!AHEAD) value_places(kk, page, ok, voff);
#pragma unroll
                for (int db = 0; db < DB; ++db) add_values(db, AHEAD ? vr[AHEAD ? db : 0] : load_value(db, ok, voff), pr, alpha);
            }
        }
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        if (ROWS) {
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int i = 0; i < 4; ++i) odd = odd || !(fabsf(acc[db][i]) < INFINITY);
        }
        if (NW == F32_SLOTS && walk < F32_SLOTS) leave();  // (read again by the same lane)
    }
    if (ROWS && __syncthreads_or(odd && on) && !one_by_one && first_p < top) {
        todo |= __ballot(on);
        one_by_one = true;
        continue;
    }
    // walks w and w + 4
    if (NW == F32_SLOTS) {
        if (second) {
            join(false);
            leave();
        }
    } else {
        if (joins) {
            if (wave >= F32_SLOTS) leave();
            __syncthreads();
        }
        if (wave < F32_SLOTS) {
            if (joins) join(true);
            leave();
        }
    }
    __syncthreads();
    if (wave == 0) {
    // the four results, merged by the first wave in their order (one without a tile has m = -inf and weighs nothing)
    const float sk = sink && head_ok ? tail.sink_of(head) : 0.f;
    float M = sink ? sk : -INFINITY;                      // (the sink: one more entry without a value)
#pragma unroll
    for (int w = 0; w < F32_SLOTS; ++w) M = fmaxf(M, merge_lds[((long)w * (DB * 4 + 2) + DB * 4) * 64 + lane]);
    float wgt[F32_SLOTS], lsum = sink ? expf(sk - M) : 0.f;
#pragma unroll
    for (int w = 0; w < F32_SLOTS; ++w) {
        const float mw = merge_lds[((long)w * (DB * 4 + 2) + DB * 4) * 64 + lane];
        wgt[w] = (mw == -INFINITY) ? 0.f : expf(mw - M);
        lsum += wgt[w] * merge_lds[((long)w * (DB * 4 + 2) + DB * 4 + 1) * 64 + lane];
    }
    if (ROWS ? on : head_ok) {
        const float inv = 1.f / lsum;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            floatx4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float a = 0.f;
#pragma unroll
                for (int w = 0; w < F32_SLOTS; ++w) a += wgt[w] * merge_lds[((long)w * (DB * 4 + 2) + db * 4 + i) * 64 + lane];
                o[i] = a * inv;
            }
            if (tail.plain) *(floatx4*)(out + t * tail.out_stride + (long)head * D + g * 4 + db * 16) = o;
            else
#pragma unroll
                for (int i = 0; i < 4; ++i) tail.store(out, t, head, db * 16 + g * 4 + i, o[i]);
        }
    }
    }
    if (ROWS && todo) __syncthreads();                     // (the results' places are written again)
    } while (ROWS && todo);
}

bool qe_attention_f32_ok(int Hq, int Hkv, int D, int P) {
    return D % 16 == 0 && D >= 16 && D <= 256 && Hq % Hkv == 0 && P >= 1;
}

// requests: to how many requests the tokens belong (0: not known).  Tokens each of a request of its own share nothing, and a few short portions
// little that a block a token, with a third more waves on a unit, does not make up for.  (us, 16 heads of 128 on 8, tokens several to a block with the blocks' requests one after
// the other, each by a block, and a token a block: 33 single tokens of 400 keys 271, 56.9, 56.2; 64 of 400 346, 78.6, 82.0, of 1000 762, 168, 184; 256 of 100 143,
// 104, 78.3, of 400 366, 258, 220.  16 portions of 4 from the start 15.9, 11.5, 9.8; 64 of 4 16.2, 14.7, 25.7; 64 of 2 behind 500 keys 202, 73.3, 129; 8 of 9 behind 1000
// 144, 74.7, 113; 50 and 30 rows 16.3, 11.5, 12.1; one of 40 10.5, 11.1, 10.9.)  Where there are more blocks than units the requests of a block
// take turns: others fill the time (32 portions of 20 behind 100 keys 46.7 and 41.9, 117 a token a block; 328 and 416 rows 39.6 and 43.3).
int qe_attention_f32(const float* q, float* out, const float* cache, const int* positions, const int* tok_seq,
                     const int* block_table, int max_blocks, const int* tokens, int T, int Hq, int Hkv, int D,
                     int P, float scale, int window, int keep_first, int sink, float softcap, int requests, hipStream_t stream, const AttnTail& tail) {
    QE_REQUIRE(qe_attention_f32_ok(Hq, Hkv, D, P), "attention (32-bit): sizes not taken");
    const int groups16 = (Hq / Hkv + 15) / 16;
    QE_REQUIRE((long)Hkv * groups16 <= 65535, "attention (32-bit): too many heads");
    dim3 grid(T, Hkv * groups16);
    // eight waves while the blocks leave compute units idle
    const bool few = (long)T * Hkv * groups16 <= 256;
    const int G = Hq / Hkv;
    const bool apart = requests > 0 && (requests >= T || (T < 8L * requests && (long)T * Hkv <= 512));
    const bool rows = !few && !apart && window == 0 && keep_first == 0 && G <= 8 && T / (16 / G) < 65535;
    if (rows) {
        grid = dim3(Hkv, qe_cdiv(T, 16 / G));
        if (requests != 1 && (long)grid.x * grid.y <= 256) grid.z = min(4, 16 / G);
    }
#define QE_ATTN_F32_FORM(DB_, NW_, AHEAD_, ROWS_)                                                     \
    do {                                                                                              \
        const size_t lds = (size_t)F32_SLOTS * (DB_ * 4 + 2) * 64 * sizeof(float);                    \
        if (lds > 48 * 1024) QE_RAISE_SHARED((attention_f32_kernel<DB_, NW_, AHEAD_, ROWS_>), lds);   \
        attention_f32_kernel<DB_, NW_, AHEAD_, ROWS_><<<grid, 64 * NW_, lds, stream>>>(q, out, cache, positions, tok_seq, \
                                                    block_table, max_blocks, tokens, T, Hq, Hkv, P, scale, window, keep_first, sink, softcap, tail, OwnToken{}); \
    } while (0)
#define QE_ATTN_F32_RUN(DB_, NW_, AHEAD_) QE_ATTN_F32_FORM(DB_, NW_, AHEAD_, false)
    // (beyond heads of 128 a tile ahead does not fit the registers)
    const bool whole = P % 16 == 0;
#define QE_ATTN_F32(DB_)                                                                              \
    case DB_:                                                                                         \
        if (few) { if (DB_ <= 8 && whole) QE_ATTN_F32_RUN(DB_, 8, (DB_ <= 8 ? 2 : 0)); else QE_ATTN_F32_RUN(DB_, 8, (DB_ <= 8)); } \
        else if (rows) QE_ATTN_F32_FORM(DB_, 4, (DB_ <= 8), true);                                    \
        else QE_ATTN_F32_RUN(DB_, 4, 0);                                                              \
        break;
    switch (D / 16) {
        QE_ATTN_F32(1) QE_ATTN_F32(2) QE_ATTN_F32(3) QE_ATTN_F32(4) QE_ATTN_F32(5) QE_ATTN_F32(6)
        QE_ATTN_F32(7) QE_ATTN_F32(8) QE_ATTN_F32(9) QE_ATTN_F32(10) QE_ATTN_F32(11) QE_ATTN_F32(12)
        QE_ATTN_F32(13) QE_ATTN_F32(14) QE_ATTN_F32(15) QE_ATTN_F32(16)
    }
#undef QE_ATTN_F32
#undef QE_ATTN_F32_RUN
#undef QE_ATTN_F32_FORM
    QE_LAUNCH_CHECK();
    return 0;
}

// The same for single new tokens from the q|k|v rows, with the norm, the rotation (over the whole head) and the cache write inside: for as many tokens
// as leave compute units idle and as have a wave for each head where these steps have a kernel of their own (whose order of sums this is).
extern int g_qe_matrix_f32;      // (switched off: the vector units' kernel and the one before it)
bool qe_attention_f32_fused_ok(int T, int Hq, int Hkv, int D, int P) {
    return g_qe_matrix_f32 && D % 16 == 0 && D >= 16 && D <= 128 && Hq % Hkv == 0 && Hq / Hkv <= 16 && P % 16 == 0 && (long)T * Hkv <= 256 &&
           (long)T * (Hq + 2 * Hkv) <= 2048;
}

int qe_attention_f32_fused(const float* qkv, float* out, float* cache, const int* positions, const int* tok_seq, const int* block_table,
                           int max_blocks, const int* slots, const float* q_w, const float* k_w, float eps, const float* table,
                           const int* tokens, int T, int rows, int Hq, int Hkv, int D, int P, float scale, int window, hipStream_t stream) {
    QE_REQUIRE(qe_attention_f32_fused_ok(rows, Hq, Hkv, D, P) && T <= rows, "attention (32-bit, fused): sizes not taken");
    if (T == 0) return 0;
    AttnTail tail{};
    tail.out_stride = (long)Hq * D;
    tail.dv = D;
    tail.plain = true;
    const OwnToken own = {q_w, k_w, eps, table, slots};
#define QE_ATTN_F32_FUSED(DB_)                                                                        \
    case DB_: {                                                                                       \
        constexpr size_t walks = (size_t)F32_SLOTS * (DB_ * 4 + 2) * 64, heads = 16 * 16 * DB_;   \
        static_assert(heads <= walks, "");                                                            \
        attention_f32_kernel<DB_, F32_WALKS, 2, false, true><<<dim3(T, Hkv), 64 * F32_WALKS, (walks + 2 * 16 * DB_) * sizeof(float), stream>>>( \
            qkv, out, cache, positions, tok_seq, block_table, max_blocks, tokens, T, Hq, Hkv, P, scale, window, 0, 0, 0.f, tail, own); \
        break;                                                                                        \
    }
    switch (D / 16) {
        QE_ATTN_F32_FUSED(1) QE_ATTN_F32_FUSED(2) QE_ATTN_F32_FUSED(3) QE_ATTN_F32_FUSED(4)
        QE_ATTN_F32_FUSED(5) QE_ATTN_F32_FUSED(6) QE_ATTN_F32_FUSED(7) QE_ATTN_F32_FUSED(8)
    }
#undef QE_ATTN_F32_FUSED
    QE_LAUNCH_CHECK();
    return 0;
}
