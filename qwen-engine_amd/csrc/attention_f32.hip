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

// NW waves.  AHEAD: a tile's values are asked for before its scores, the next tile's keys before this tile's softmax.  Few
// tokens are bound by their walks' trips to memory (2 tokens of 16 heads on 8 over 744 keys: 32 us, 55 with four waves, each
// with 12 tiles one after the other and every load where it is used); with many tokens other waves fill the time, and the
// registers that this takes cost more.
template <int DB, int NW, bool AHEAD>     // DB: head size / 16
__global__ __launch_bounds__(64 * NW, NW == F32_SLOTS && DB <= 8 ? 3 : 1) void attention_f32_kernel(
    const float* __restrict__ q, float* __restrict__ out, const float* __restrict__ cache,
    const int* __restrict__ positions, const int* __restrict__ tok_seq,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ tokens,
    int Hq, int Hkv, int P, float scale, int window, int keep_first, int sink, float softcap, AttnTail tail) {
    constexpr int D = DB * 16;
    extern __shared__ float merge_lds[];                  // [F32_SLOTS][DB * 4 + 2][64]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, n = lane & 15;
    const long t = tokens ? tokens[blockIdx.x] : blockIdx.x;
    const int G = Hq / Hkv;
    const int groups16 = (G + 15) / 16;
    const int kvh = blockIdx.y / groups16, hg = blockIdx.y % groups16;
    const int head = kvh * G + hg * 16 + n;
    const bool head_ok = hg * 16 + n < G;
    const int p = positions[t];
    const int lo = first_seen_key(p, window);
    const int* bt = block_table + (long)tok_seq[t] * max_blocks;
    const long page_stride = 2L * Hkv * P * D;
    const bool vec_v = (P & 3) == 0;                      // four consecutive keys of a value row lie in one page, aligned

    floatx4 qv[DB];
#pragma unroll
    for (int c = 0; c < DB; ++c) {
        qv[c] = floatx4{0.f, 0.f, 0.f, 0.f};
        if (head_ok) qv[c] = *(const floatx4*)(q + (t * Hq + head) * D + c * 16 + g * 4);
    }
    // The tiles of the walks: those of the kept first keys 0 .. kf - 1 that lie wholly before the window's
    // first tile, then the tiles from the window's first on (which holds the rest of the kept keys, if
    // any); tile number i of this list is walk i % F32_WALKS's.
    const int kf = keep_first < lo ? keep_first : lo;
    const int tile_lo = lo / 16;
    const int n_first = (kf + 15) / 16 < tile_lo ? (kf + 15) / 16 : tile_lo;
    const int n_tiles = n_first + p / 16 - tile_lo + 1;
    const auto tile_key = [&](int ti) { return 16 * (ti < n_first ? ti : tile_lo + ti - n_first); };
    // Pages of whole tiles: lane i holds the page of the walk's i-th tile of 64 (one load for all of them, where each tile's lookups
    // were two trips to memory of their own); a tile's page is then the same for the wave, and so is its place in it.  Other page sizes:
    // every lane looks its own keys' pages up.
    const bool whole = P % 16 == 0;
    int my_page = 0;
    const auto page_of = [&](int ti, int walk) {               // asked for tile by tile, in order
        const int j = (ti - walk) / F32_WALKS;
        if (!whole) return 0;
        if ((j & 63) == 0) {
            const int tl = ti + lane * F32_WALKS;
            if (tl < n_tiles) my_page = bt[tile_key(tl) / P];
        }
        return __builtin_amdgcn_readlane(my_page, j & 63);
    };
    const auto load_keys = [&](int kk, int page, floatx4 (&kr)[DB]) {      // S^T: this lane brings the key row kk + n
        const int key_r = kk + n;
        const bool row_ok = (key_r >= lo || key_r < kf) && key_r <= p;
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
            const int kc = ok[i] ? kk + 4 * g + i : p;     // (an address that is valid; the value is not used)
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
    // (a walk without a tile changes nothing where it is joined: where a wave's second walk, or every walk from the fifth on, has none,
    // there is nothing to join)
    const bool second = wave + F32_SLOTS < n_tiles, joins = F32_SLOTS < n_tiles;
    for (int walk = wave; walk < F32_WALKS && (walk == wave || second); walk += NW) {
        m = -INFINITY;
        l = 0.f;                                           // this lane's share of the column's sum
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[db] = floatx4{0.f, 0.f, 0.f, 0.f};
        floatx4 kr[DB], vr[AHEAD ? DB : 1];
        int page = 0;
        if (AHEAD && walk < n_tiles) {
            page = page_of(walk, walk);
            load_keys(tile_key(walk), page, kr);
        }
        for (int ti = walk; ti < n_tiles; ti += F32_WALKS) {
            const int kk = tile_key(ti);
            bool ok[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = kk + 4 * g + i;
                ok[i] = (key >= lo || key < kf) && key <= p;
            }
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
            floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < DB; ++c)
#pragma unroll
                for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[c][j], qv[c][j], s, 0, 0, 0);
            if (AHEAD && ti + F32_WALKS < n_tiles) {
                page = page_of(ti + F32_WALKS, walk);
                load_keys(tile_key(ti + F32_WALKS), page, kr);
            }
            // the lane now holds the scores of keys kk + 4 g + i of column n
            float tmax = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[i] *= scale;
                if (softcap > 0.f) s[i] = softcap * tanhf(s[i] / softcap);
                if (!ok[i]) s[i] = -INFINITY;
                tmax = fmaxf(tmax, s[i]);
            }
            tmax = max_over_rows_of_lanes(tmax);
            const float mn = fmaxf(m, tmax);               // finite: every tile of the walk holds a key that is seen
            const float alpha = expf(m - mn);              // 0 on the first tile
            floatx4 pr;
            float psum = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pr[i] = ok[i] ? expf(s[i] - mn) : 0.f;
                psum += pr[i];
            }
            l = l * alpha + psum;
            m = mn;
            // O^T: this lane brings, of the value rows d = 16 db + n, the keys kk + 4 g .. + 3
            if (!AHEAD) value_places(kk, page, ok, voff);
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const floatx4 vf = AHEAD ? vr[AHEAD ? db : 0] : load_value(db, ok, voff);
                acc[db] *= alpha;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[j], pr[j], acc[db], 0, 0, 0);
            }
        }
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        if (NW == F32_SLOTS && walk < F32_SLOTS) leave();  // (read again by the same lane)
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
    if (wave != 0) return;
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
    if (head_ok) {
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

bool qe_attention_f32_ok(int Hq, int Hkv, int D, int P) {
    return D % 16 == 0 && D >= 16 && D <= 256 && Hq % Hkv == 0 && P >= 1;
}

int qe_attention_f32(const float* q, float* out, const float* cache, const int* positions, const int* tok_seq,
                     const int* block_table, int max_blocks, const int* tokens, int T, int Hq, int Hkv, int D,
                     int P, float scale, int window, int keep_first, int sink, float softcap, hipStream_t stream, const AttnTail& tail) {
    QE_REQUIRE(qe_attention_f32_ok(Hq, Hkv, D, P), "attention (32-bit): sizes not taken");
    const int groups16 = (Hq / Hkv + 15) / 16;
    QE_REQUIRE((long)Hkv * groups16 <= 65535, "attention (32-bit): too many heads");
    dim3 grid(T, Hkv * groups16);
    // eight waves while the blocks leave compute units idle
    const bool few = (long)T * Hkv * groups16 <= 256;
#define QE_ATTN_F32_RUN(DB_, NW_, AHEAD_)                                                             \
    do {                                                                                              \
        const size_t lds = (size_t)F32_SLOTS * (DB_ * 4 + 2) * 64 * sizeof(float);                    \
        if (lds > 48 * 1024) QE_RAISE_SHARED((attention_f32_kernel<DB_, NW_, AHEAD_>), lds);          \
        attention_f32_kernel<DB_, NW_, AHEAD_><<<grid, 64 * NW_, lds, stream>>>(q, out, cache, positions, tok_seq, \
                                                    block_table, max_blocks, tokens, Hq, Hkv, P, scale, window, keep_first, sink, softcap, tail); \
    } while (0)
    // (beyond heads of 128 a tile ahead does not fit the registers)
#define QE_ATTN_F32(DB_)                                                                              \
    case DB_:                                                                                         \
        if (few) QE_ATTN_F32_RUN(DB_, 8, (DB_ <= 8)); else QE_ATTN_F32_RUN(DB_, 4, false);            \
        break;
    switch (D / 16) {
        QE_ATTN_F32(1) QE_ATTN_F32(2) QE_ATTN_F32(3) QE_ATTN_F32(4) QE_ATTN_F32(5) QE_ATTN_F32(6)
        QE_ATTN_F32(7) QE_ATTN_F32(8) QE_ATTN_F32(9) QE_ATTN_F32(10) QE_ATTN_F32(11) QE_ATTN_F32(12)
        QE_ATTN_F32(13) QE_ATTN_F32(14) QE_ATTN_F32(15) QE_ATTN_F32(16)
    }
#undef QE_ATTN_F32
#undef QE_ATTN_F32_RUN
    QE_LAUNCH_CHECK();
    return 0;
}
