// Latent attention of portions of prompts with the keys and values expanded (bfloat16, matrix units).
//
// See latent_attention.hip for what is cached: a row [R + Dr] a token, from which every head's keys and values are
// linear maps.  With the maps folded into the queries (what single new tokens do) a pair of a row and a key costs
// 2 R + Dr multiply-adds a head; with expanded keys and values it costs Dn + Dr + Dv, and every key once R (Dn + Dv).
// So rows that share their keys with some dozens of others are better off expanded: with R = 512, Dn = Dv = 128,
// Dr = 64 a prompt of 2048 has 3.4 times fewer operations, and the walk is that of an ordinary attention kernel with
// registers for two waves a SIMD.  2048 rows of 16 heads: 366 us folded and 90 for the products per head before and behind
// it; expanded 57 us (the walk: 21 GFLOP, 375 TFLOP/s; its longest block of 64 key tiles decides), some 100 with gather and
// both products.  Bound as attention_prefill.hip is: shared memory and exponentials beside the matrix instructions.
//
//   latent_gather_kernel   the rows' keys from the cache pages into [keys][R] and [keys][Dr], in the order of the
//                          positions, portion after portion, each from a multiple of 64 on; zeros behind a portion's
//                          last key, so that what the products make of them is zero and not unwritten memory
//   two products (gemm)    keys [keys][H Dn] = c . Uk^T, and the values transposed, [H Dv][keys] = Uv . c^T: the
//                          operand order of the second product of attention wants eight keys of one feature side by side
//   latent_prefill_kernel  a wave owns 32 rows of one head, a block four neighbouring tiles of 32 rows of one portion;
//                          the block walks the keys 32 at a time through shared memory, two buffers and two sets of
//                          staging registers, as attention_prefill.hip does (S^T = K Q^T, online softmax per column in
//                          the base-2 domain with a lazy reference, O^T += V^T P^T); NG = 2: two groups of four waves
//                          take the even and the odd tiles and merge at the end, where blocks are few.  A window's lower
//                          end and a sink as in latent_attention_mfma.hip; the output gate is applied as rows are stored.
//
// Positions are read on the device, so that a recorded step serves every place: the host fixes the rows, the portions'
// places in the key buffers and the buffers' lengths.
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float floatx16;
typedef __attribute__((ext_vector_type(4))) unsigned int uint4_t;

union Piece {
    uint4_t q;
    uint2 u[2];
};
union PackV {
    bf16x8 v;
    uint2 u[2];
};

// the first key that a portion's rows see (its first row sees the farthest back)
__device__ __forceinline__ int portion_first_key(const int* __restrict__ positions, int first_row, int window) {
    const int p = positions[first_row];
    return window > 0 && p - window + 1 > 0 ? p - window + 1 : 0;
}

// portions [n][3] = (first row, rows, place of its first key); owner [keys / 64]: the portion of every 64 keys.
// A thread brings 16 bytes.
__global__ __launch_bounds__(256) void latent_gather_kernel(const bf16_t* __restrict__ cache, const int* __restrict__ positions,
                                                            const int* __restrict__ tok_seq, const int* __restrict__ block_table,
                                                            int max_blocks, const int* __restrict__ portions,
                                                            const int* __restrict__ owner, bf16_t* __restrict__ ck,
                                                            bf16_t* __restrict__ kr, long keys, int R, int Dr, int P, int window) {
    const int per_row = (R + Dr) / 8;
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    const long j = idx / per_row;
    if (j >= keys) return;
    const int d = (int)(idx - j * per_row) * 8;
    const int* po = portions + 3 * owner[j >> 6];
    const int first = po[0], rows = po[1];
    const long key = portion_first_key(positions, first, window) + (j - po[2]);
    uint4_t v = {0u, 0u, 0u, 0u};
    if (key <= positions[first + rows - 1]) {
        const int* bt = block_table + (long)tok_seq[first] * max_blocks;
        v = *(const uint4_t*)(cache + ((long)bt[key / P] * P + key % P) * (R + Dr) + d);
    }
    if (d < R) *(uint4_t*)(ck + j * R + d) = v;
    else *(uint4_t*)(kr + j * Dr + (d - R)) = v;
}

#define LP_VROW 48   // bytes of a staged value row: 16 keys = 32 bytes of data + 16 of padding

template <int KS, int DV, int NG>     // KS = (Dn + Dr) / 16
__global__ __launch_bounds__(256 * NG, NG == 1 ? 2 : 1) void latent_prefill_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ kx, const bf16_t* __restrict__ kr,
    const bf16_t* __restrict__ vt, long keys, bf16_t* __restrict__ out, const int* __restrict__ tiles,
    const int* __restrict__ group_portion, const int* __restrict__ portions, const int* __restrict__ positions,
    int H, int Dn, float scale_log2, int window, const float* __restrict__ sink, const bf16_t* __restrict__ gate,
    long gs_t, int gs_h, int gs_n) {
    constexpr int DQ = KS * 16, KROW = DQ * 2 + 16;
    constexpr int KBYTES = 32 * KROW, VBYTES = 2 * DV * LP_VROW, BUF = KBYTES + VBYTES;
    constexpr int KN = 32 * (DQ / 8), KP = (KN + 255) / 256;     // 16-byte key pieces of a tile, and per thread
    constexpr int VP = DV * 4 / 256;                             // 16-byte value pieces per thread
    __shared__ __attribute__((aligned(16))) unsigned char smem_all[NG * 2 * BUF];
    const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x / 256);
    const int tid = threadIdx.x % 256, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned char* smem = smem_all + grp * 2 * BUF;
    const int g = lane >> 5, r = lane & 31;
    const int head = blockIdx.x;
    const int group = gridDim.y - 1 - blockIdx.y;                // later rows see more keys: they start first
    const int* bt4 = tiles + 8 * group;
    const int row_first = bt4[0];
    int last = 0;
#pragma unroll
    for (int j = 1; j < 4; ++j) if (bt4[2 * j + 1] > 0) last = j;
    const int* po = portions + 3 * group_portion[group];
    const int base = po[2] - portion_first_key(positions, po[0], window);   // place in the key buffers = position + base
    auto first_place = [&](int p) { return base + (window > 0 && p - window + 1 > 0 ? p - window + 1 : 0); };
    const int jmin = first_place(positions[row_first]);
    const int jmax = positions[bt4[2 * last]] + bt4[2 * last + 1] + base;

    const int row0 = bt4[2 * wave], cnt = bt4[2 * wave + 1];
    const bool wave_on = cnt > 0;
    const int row = wave_on ? row0 + (r < cnt ? r : cnt - 1) : row_first;
    const int p = positions[row];
    const int hi = p + 1 + base, lo = first_place(p);
    const int p_first = positions[wave_on ? row0 : row_first];
    const int j_start = first_place(p_first), j_stop = wave_on ? p_first + cnt + base : 0;
    const int all_hi = p_first + 1 + base, all_lo = first_place(p_first + cnt - 1);

    const int Dr = DQ - Dn;
    bf16x8 qreg[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
        qreg[ks] = *(const bf16x8*)(q + ((long)row * H + head) * DQ + ks * 16 + g * 8);
    __builtin_amdgcn_s_waitcnt(0x0f70);                          // vmcnt(0): the loop's loads are counted from here

    float m = -INFINITY, l = 0.f;
    floatx16 acc[DV / 32];
#pragma unroll
    for (int db = 0; db < DV / 32; ++db)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[db][e] = 0.f;

    // staging, as in attention_prefill.hip: a tile's loads are issued two tiles ahead and stored one tile ahead.  A key
    // row is put together from its own part and the part that all heads share.
    Piece kst[2][KP], vst[2][VP];
    const bf16_t* ksrc[KP];
    long kstep[KP];
    int kat[KP];
#pragma unroll
    for (int i = 0; i < KP; ++i) {
        const int id = tid + 256 * i < KN ? tid + 256 * i : tid;  // (a piece too many is a copy of the thread's first)
        const int krow = id / (DQ / 8), d = id % (DQ / 8) * 8;
        const bool mine = d < Dn;
        kstep[i] = mine ? (long)H * Dn : Dr;
        ksrc[i] = mine ? kx + ((long)krow * H + head) * Dn + d : kr + (long)krow * Dr + (d - Dn);
        kat[i] = krow * KROW + d * 2;
    }
    const bf16_t* vsrc[VP];
    int vat[VP];
#pragma unroll
    for (int i = 0; i < VP; ++i) {
        const int id = tid + 256 * i, d = id >> 2, part = id & 3;   // eight keys: half part / 2, piece part % 2 of it
        vsrc[i] = vt + ((long)head * DV + d) * keys + part * 8;
        vat[i] = KBYTES + ((part >> 1) * DV + d) * LP_VROW + (part & 1) * 8;
    }
#define STAGE_LOAD(set_, jj_)                                                                        \
    {                                                                                                \
        _Pragma("unroll") for (int i = 0; i < KP; ++i) kst[set_][i].q = *(const uint4_t*)(ksrc[i] + (jj_) * kstep[i]); \
        _Pragma("unroll") for (int i = 0; i < VP; ++i) vst[set_][i].q = *(const uint4_t*)(vsrc[i] + (jj_));           \
    }
#define STAGE_STORE(buf_, set_)                                                                      \
    {                                                                                                \
        unsigned char* b_ = smem + (buf_) * BUF;                                                     \
        _Pragma("unroll") for (int i = 0; i < KP; ++i) *(uint4_t*)(b_ + kat[i]) = kst[set_][i].q;    \
        _Pragma("unroll") for (int i = 0; i < VP; ++i) {                                             \
            *(uint2*)(b_ + vat[i]) = vst[set_][i].u[0];                                              \
            *(uint2*)(b_ + vat[i] + 16) = vst[set_][i].u[1];                                         \
        }                                                                                            \
    }
    const int jj0 = jmin & ~31;                                   // (the buffers' lengths are multiples of 64: whole tiles)
    const int rounds = ((jmax - jj0 + 31) / 32 + NG - 1) / NG;
#define TILE_AT(i_) (jj0 + 32 * (NG * (i_) + grp))
#define EXISTING(jj_) ((jj_) < jmax ? (jj_) : jj0)
    const int jj_first = TILE_AT(0), jj_second = TILE_AT(1);
    STAGE_LOAD(0, EXISTING(jj_first))
    STAGE_STORE(0, 0)
    STAGE_LOAD(1, EXISTING(jj_second))
    __syncthreads();
    for (int i2 = 0; i2 < rounds; i2 += 2) {
#pragma unroll
      for (int buf = 0; buf < 2; ++buf) {
        const int i = i2 + buf;
        if (i >= rounds) break;                                   // the same for all threads of the block
        const int jj = TILE_AT(i), jj_2 = TILE_AT(i + 2);
        STAGE_LOAD(buf, EXISTING(jj_2))
        __builtin_amdgcn_sched_barrier(0);
        if (wave_on && jj < j_stop && jj + 32 > j_start && jj < jmax) {
            const unsigned char* ks_ = smem + buf * BUF + r * KROW + g * 16;
            const unsigned char* vs_ = smem + buf * BUF + KBYTES + r * LP_VROW + g * 16;
            floatx16 s;
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(ks_ + ks * 32), qreg[ks], s, 0, 0, 0);
            PackV vf[DV / 32][2];
#pragma unroll
            for (int db = 0; db < DV / 32; ++db)
#pragma unroll
                for (int h = 0; h < 2; ++h) vf[db][h].v = *(const bf16x8*)(vs_ + (h * DV + db * 32) * LP_VROW);
            float tmax = -INFINITY;
            if (jj >= all_lo && jj + 32 <= all_hi) {              // every column sees every key of the tile
#pragma unroll
                for (int e = 0; e < 16; ++e) tmax = fmaxf(tmax, s[e]);
            } else {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int j = jj + 8 * (e >> 2) + 4 * g + (e & 3);
                    s[e] = (j >= lo && j < hi) ? s[e] : -INFINITY;
                    tmax = fmaxf(tmax, s[e]);
                }
            }
            {
                float a, b;
                pair_across_halves(tmax, a, b);
                tmax = fmaxf(a, b) * scale_log2;
            }
            const bool moves = tmax > m + 8.f;                    // (see attention_prefill.hip)
            if (__any(moves)) {
                const float alpha = moves ? __builtin_amdgcn_exp2f(m - tmax) : 1.f;
                m = moves ? tmax : m;
                l *= alpha;
#pragma unroll
                for (int db = 0; db < DV / 32; ++db) acc[db] *= alpha;
            }
            const float ref = (m == -INFINITY) ? 0.f : m;
            PackV pb[2];
            float psum = 0.f;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float pe = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], scale_log2, -ref));
                psum += pe;
                pb[e >> 3].v[e & 7] = (__bf16)pe;
            }
            l += psum;
#pragma unroll
            for (int db = 0; db < DV / 32; ++db)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[db][h].v, pb[h].v, acc[db], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        STAGE_STORE(buf ^ 1, buf ^ 1)                             // that buffer's readers finished before the last barrier
        __syncthreads();
      }
    }
#undef STAGE_LOAD
#undef STAGE_STORE
#undef TILE_AT
#undef EXISTING
    {
        float a, b;
        pair_across_halves(l, a, b);
        l = a + b;
    }
    if (NG == 2) {
        // group 1 hands over to group 0 through the staging memory, 16 values of every lane at a time: [wave][value][lane]
        float* xch = (float*)smem_all + wave * 18 * 64 + lane;
        float a_own = 1.f, a_other = 0.f;
        if (grp == 1) { xch[0] = m; xch[64] = l; }
        __syncthreads();
        if (grp == 0) {
            const float m1 = xch[0], l1 = xch[64];
            const float mt = fmaxf(m, m1);
            const float ref = (mt == -INFINITY) ? 0.f : mt;
            a_own = __builtin_amdgcn_exp2f(m - ref);
            a_other = __builtin_amdgcn_exp2f(m1 - ref);
            l = l * a_own + l1 * a_other;
            m = mt;
        }
#pragma unroll
        for (int db = 0; db < DV / 32; ++db) {
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
    if (!wave_on || r >= cnt) return;
    if (sink) l += __builtin_amdgcn_exp2f(fminf(sink[head] * 1.4426950408889634f - m, 126.f));
    const float inv = 1.f / l;
    bf16_t* o = out + ((long)row * H + head) * DV;
    const bf16_t* gt = gate ? gate + row * gs_t + (long)head * gs_h : nullptr;
#pragma unroll
    for (int db = 0; db < DV / 32; ++db)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int d = db * 32 + 8 * b + 4 * g;
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[j] = acc[db][4 * b + j] * inv;
                if (gt) v[j] /= 1.f + __expf(-bf16_to_float(gt[(long)(d + j) * gs_n]));
            }
            Vec4<bf16_t>::store(o + d, v);
        }
}

static int key_steps(int Dn, int Dr, int Dv) {
    const int dq = Dn + Dr;
    if (Dn <= 0 || Dn % 8 || Dr < 0 || Dr % 8) return 0;
    if (Dv == 64 && (dq == 64 || dq == 96 || dq == 128)) return dq / 16;
    if (Dv == 128 && (dq == 128 || dq == 192)) return dq / 16;
    return 0;
}

// 1 if the kernels take these sizes of a head and of a latent row
extern "C" int qe_latent_prefill_supported(int R, int Dn, int Dr, int Dv) {
    return (R > 0 && R % 8 == 0 && key_steps(Dn, Dr, Dv) != 0) ? 1 : 0;
}

// ck [keys, R] and kr [keys, Dr] (null where Dr is 0); keys is a multiple of 64
extern "C" int qe_latent_gather(const void* cache, const int* positions, const int* tok_seq, const int* block_table,
                                int max_blocks, const int* portions, const int* owner, void* ck, void* kr, long keys,
                                int R, int Dr, int P, int window, hipStream_t stream) {
    QE_REQUIRE(keys >= 0 && keys % 64 == 0 && R > 0 && R % 8 == 0 && Dr >= 0 && Dr % 8 == 0 && P > 0 && window >= 0 &&
               (Dr == 0 || kr), "latent_gather: bad sizes keys=%ld R=%d Dr=%d", keys, R, Dr);
    if (keys == 0) return 0;
    const long blocks = (keys * ((R + Dr) / 8) + 255) / 256;
    QE_REQUIRE(blocks < (1L << 31), "latent_gather: %ld keys are too many for one launch", keys);
    latent_gather_kernel<<<(unsigned)blocks, 256, 0, stream>>>((const bf16_t*)cache, positions, tok_seq, block_table, max_blocks,
                                                               portions, owner, (bf16_t*)ck, (bf16_t*)kr, keys, R, Dr, P, window);
    QE_LAUNCH_CHECK();
    return 0;
}

// q [T, H, Dn + Dr] (rotated), kx [keys, H Dn], kr [keys, Dr], vt [H Dv, keys] -> out [T, H Dv] at the rows that tiles
// names: n_groups groups of four tiles (first row, rows <= 32) of one portion, in ascending rows at consecutive positions, filled up
// with tiles of 0 rows; group_portion: their portions.  gate (or null): element (row, head, d) at row gs_t + head gs_h + d gs_n.
extern "C" int qe_latent_prefill(const void* q, const void* kx, const void* kr, const void* vt, long keys, void* out,
                                 const int* tiles, const int* group_portion, int n_groups, const int* portions,
                                 const int* positions, int H, int Dn, int Dr, int Dv, float scale, int window,
                                 const float* sink, const void* gate, long gs_t, int gs_h, int gs_n, hipStream_t stream) {
    const int ks = key_steps(Dn, Dr, Dv);
    QE_REQUIRE(ks && keys % 64 == 0 && keys < (1L << 30), "latent_prefill: sizes not taken");
    QE_REQUIRE(H > 0 && n_groups >= 0 && n_groups <= 65535 && window >= 0, "latent_prefill: bad sizes");
    if (n_groups == 0) return 0;
    const dim3 grid(H, n_groups);
    const float scale_log2 = scale * 1.4426950408889634f;
    const bool two = (long)H * n_groups <= qe_compute_units();    // (see attention_prefill.hip: no more blocks than compute units)
#define QE_LP_NG(KS_, DV_, NG_)                                                                                            \
    latent_prefill_kernel<KS_, DV_, NG_><<<grid, 256 * NG_, 0, stream>>>(                                                  \
        (const bf16_t*)q, (const bf16_t*)kx, (const bf16_t*)kr, (const bf16_t*)vt, keys, (bf16_t*)out, tiles, group_portion, \
        portions, positions, H, Dn, scale_log2, window, sink, (const bf16_t*)gate, gs_t, gs_h, gs_n)
#define QE_LP(KS_, DV_) do { if (two) QE_LP_NG(KS_, DV_, 2); else QE_LP_NG(KS_, DV_, 1); } while (0)
    if (Dv == 64) {
        if (ks == 4) QE_LP(4, 64);
        else if (ks == 6) QE_LP(6, 64);
        else QE_LP(8, 64);
    } else {
        if (ks == 8) QE_LP(8, 128);
        else QE_LP(12, 128);
    }
#undef QE_LP
#undef QE_LP_NG
    QE_LAUNCH_CHECK();
    return 0;
}
