// A short causal convolution over time on each channel of the 32-bit stream, added to its input:
//   out_t = x_t + sum_{k=0}^{taps-1} w[:, taps-1-k] * x_(t-k)        (zeros before a request's start)
// over a flat batch of portions of several requests.  What lies before a portion comes from the
// request's state: its last taps - 1 inputs, state[slot][j] being the input at position
// (tokens so far) - (taps - 1) + j, zeros where that is negative (the state of a new request is
// cleared by the step function).
//
// The rows of one request are consecutive and no request comes twice in a step, so a row finds its
// place inside its portion by looking back: row t - k belongs to the same request exactly if its
// table row (tok_seq) is the same.  No list of portions is needed, and a recorded step's rows that
// only fill it up (all on the tables' spare row) are taken as one portion.
#include "common.h"

template <typename TA>
__global__ void short_conv_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                  const float* __restrict__ state, const int* __restrict__ tok_seq,
                                  TA* __restrict__ out, int T, int H, int taps) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const long t = blockIdx.y;
    if (c >= H) return;
    const int n1 = taps - 1;
    const int s = tok_seq[t];
    int before = 0;                                   // rows of the same request right before this one, up to n1
    while (before < n1 && t - 1 - before >= 0 && tok_seq[t - 1 - before] == s) ++before;
    const float* wc = w + (long)c * taps;
    const float xt = x[t * H + c];
    float acc = xt;
    for (int k = n1; k >= 0; --k) {                   // oldest input first: the same order however the request was cut
        float v;
        if (k <= before) v = x[(t - k) * H + c];
        else v = state[((long)s * n1 + (n1 - k + before)) * H + c];
        acc = fmaf(wc[n1 - k], v, acc);
    }
    Elem<TA>::store(out + t * H + c, acc);
}

// After the convolution: the state takes the portion's last taps - 1 inputs.  A portion shorter than
// that moves the state's old entries up first; its first row's thread does all of it, so that no
// thread reads what another writes.
__global__ void short_conv_update_kernel(const float* __restrict__ x, float* __restrict__ state,
                                         const int* __restrict__ tok_seq, int T, int H, int taps) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const long t = blockIdx.y;
    if (c >= H) return;
    const int n1 = taps - 1;
    const int s = tok_seq[t];
    int before = 0, after = 0;
    while (before < n1 && t - 1 - before >= 0 && tok_seq[t - 1 - before] == s) ++before;
    while (after < n1 && t + 1 + after < T && tok_seq[t + 1 + after] == s) ++after;
    float* st = state + (long)s * n1 * H + c;
    if (before + after + 1 < n1) {                    // the whole portion is shorter than the state
        if (before != 0) return;
        const int q = after + 1;
        for (int j = 0; j + q < n1; ++j) st[(long)j * H] = st[(long)(j + q) * H];
        for (int m = 0; m < q; ++m) st[(long)(n1 - q + m) * H] = x[(t + m) * H + c];
    } else if (after < n1) {
        st[(long)(n1 - 1 - after) * H] = x[t * H + c];
    }
}

// The two kernels for channels in whole fours and up to eight taps: a thread has four channels of CV_ROWS neighbouring rows, which are
// asked for together with the taps - 1 rows before them, so that a row is read 1 + (taps - 1) / CV_ROWS times and not taps times, by
// two bytes a trip; the update's blocks look at CV_ROWS rows at once, of which mostly none is among the last of its portion (one request of
// 2048 rows of 2048, four taps: 8.0 us and 7.2 for the update; a thread a number took 23.4 and 17.7).
#define CV_ROWS 8

// the requests of the rows t0 - n1 .. t0 + CV_ROWS + n1 - 1 (-1: no such row)
__device__ __forceinline__ void rows_requests(int* seq, const int* __restrict__ tok_seq, int t0, int n1, int T) {
    for (int i = threadIdx.x; i < CV_ROWS + 2 * n1; i += blockDim.x) {
        const int t = t0 - n1 + i;
        seq[i] = t >= 0 && t < T ? tok_seq[t] : -1;
    }
    __syncthreads();
}

template <typename TA, int TAPS>
__global__ __launch_bounds__(256) void short_conv_rows_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                              const float* __restrict__ state, const int* __restrict__ tok_seq,
                                                              TA* __restrict__ out, int T, int H) {
    constexpr int N1 = TAPS - 1;
    __shared__ int seq[CV_ROWS + 2 * N1 + 1];
    const int c = (blockIdx.x * 256 + threadIdx.x) * 4, t0 = blockIdx.y * CV_ROWS;
    rows_requests(seq, tok_seq, t0, N1, T);
    if (c >= H) return;
    float v[CV_ROWS + N1][4], wc[4][TAPS];
#pragma unroll
    for (int i = 0; i < CV_ROWS + N1; ++i) {
        const int t = min(max(t0 - N1 + i, 0), T - 1);     // (a row beyond them is never used)
        Vec4<float>::load(x + (long)t * H + c, v[i]);
    }
#pragma unroll
    for (int k = 0; k < 4 * TAPS; ++k) wc[k / TAPS][k % TAPS] = w[(long)c * TAPS + k];
#pragma unroll
    for (int r = 0; r < CV_ROWS; ++r) {
        const int t = t0 + r;
        if (t >= T) break;
        const int s = seq[r + N1];
        int before = 0;                                   // rows of the same request right before this one, up to N1
#pragma unroll
        for (int k = 1; k <= N1; ++k) before += before == k - 1 && seq[r + N1 - k] == s;
        float acc[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = v[r + N1][e];
#pragma unroll
        for (int k = N1; k >= 0; --k) {                   // oldest input first
            float u[4];
            if (k <= before) {
#pragma unroll
                for (int e = 0; e < 4; ++e) u[e] = v[r + N1 - k][e];
            } else {
                Vec4<float>::load(state + ((long)s * N1 + (N1 - k + before)) * H + c, u);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = fmaf(wc[e][N1 - k], u[e], acc[e]);
        }
        Vec4<TA>::store(out + (long)t * H + c, acc);
    }
}

__global__ __launch_bounds__(256) void short_conv_rows_update_kernel(const float* __restrict__ x, float* __restrict__ state,
                                                                     const int* __restrict__ tok_seq, int T, int H, int taps) {
    __shared__ int seq[CV_ROWS + 2 * 7];
    const int n1 = taps - 1;
    const int c = (blockIdx.x * 256 + threadIdx.x) * 4, t0 = blockIdx.y * CV_ROWS;
    rows_requests(seq, tok_seq, t0, n1, T);
    if (c >= H) return;
    for (int r = 0; r < CV_ROWS; ++r) {
        const int t = t0 + r, s = seq[r + n1];
        if (t >= T) break;
        int before = 0, after = 0;
        while (before < n1 && seq[r + n1 - 1 - before] == s) ++before;
        while (after < n1 && seq[r + n1 + 1 + after] == s) ++after;
        float* st = state + (long)s * n1 * H + c;
        float u[4];
        if (before + after + 1 < n1) {                    // the whole portion is shorter than the state
            if (before != 0) continue;
            const int q = after + 1;
            for (int j = 0; j + q < n1; ++j) {
                Vec4<float>::load(st + (long)(j + q) * H, u);
                Vec4<float>::store(st + (long)j * H, u);
            }
            for (int m = 0; m < q; ++m) {
                Vec4<float>::load(x + (long)(t + m) * H + c, u);
                Vec4<float>::store(st + (long)(n1 - q + m) * H, u);
            }
        } else if (after < n1) {
            Vec4<float>::load(x + (long)t * H + c, u);
            Vec4<float>::store(st + (long)(n1 - 1 - after) * H, u);
        }
    }
}

// Every row the only row of its request (single new tokens): the convolution and the state's shift in one launch;
// a thread reads its channel's state, forms the output and writes the state back moved up by one.
template <typename TA>
__global__ void short_conv_single_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ state,
                                         const int* __restrict__ tok_seq, TA* __restrict__ out, int H, int taps) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const long t = blockIdx.y;
    if (c >= H) return;
    const int n1 = taps - 1;
    float* st = state + (long)tok_seq[t] * n1 * H + c;
    const float* wc = w + (long)c * taps;
    const float xt = x[t * H + c];
    float acc = xt;
    for (int j = 0; j < n1; ++j) {                    // oldest input first, as in short_conv_kernel
        const float v = st[(long)j * H];
        acc = fmaf(wc[j], v, acc);
        if (j > 0) st[(long)(j - 1) * H] = v;
    }
    acc = fmaf(wc[n1], xt, acc);
    st[(long)(n1 - 1) * H] = xt;
    Elem<TA>::store(out + t * H + c, acc);
}

// update 2: the caller knows that every row is the only row of its request
extern "C" int qe_short_conv(const float* x, const float* w, float* state, const int* tok_seq, void* out,
                             int dt_a, int T, int H, int taps, int update, hipStream_t stream) {
    QE_REQUIRE(T >= 0 && H > 0 && taps >= 1, "short_conv: bad sizes T=%d H=%d taps=%d", T, H, taps);
    QE_REQUIRE(taps == 1 || state, "short_conv: %d taps need a state", taps);
    QE_REQUIRE(T <= 65535, "short_conv: more than 65535 rows in a step");
    if (T == 0) return 0;
    const int threads = H >= 256 ? 256 : 64;
    dim3 grid(qe_cdiv(H, threads), T);                // (blockIdx.y is the row)
    if (update == 2 && taps > 1) {
        if (dt_a == QE_F32) short_conv_single_kernel<float><<<grid, threads, 0, stream>>>(x, w, state, tok_seq, (float*)out, H, taps);
        else if (dt_a == QE_BF16) short_conv_single_kernel<bf16_t><<<grid, threads, 0, stream>>>(x, w, state, tok_seq, (bf16_t*)out, H, taps);
        else QE_REQUIRE(false, "short_conv: unknown output type %d", dt_a);
        QE_LAUNCH_CHECK();
        return 0;
    }
    // (whole fours everywhere; the out rows of four numbers are 8 bytes in bfloat16).  Eight rows a thread are worth it where a thread a
    // number fills the chip more than once; the sums are the same.  (Both launches, a thread a number and eight rows a thread: 64 rows
    // of 2048 4.9 us and 9.9, 300 9.0 and 10.0, 400 10.6 and 10.2, 700 of 1024 9.7 and 9.9, 200 of 4096 10.6 and 10.1.)
    const bool fours = (long)T * H >= 3L << 18 && H % 4 == 0 && taps >= 2 && taps <= 8 && (((uintptr_t)x | (uintptr_t)state | (uintptr_t)out) & 15) == 0;
    if (fours) {
        dim3 rgrid(qe_cdiv(H, 1024), qe_cdiv(T, CV_ROWS));
        const int rthreads = H >= 1024 ? 256 : (qe_cdiv(H / 4, 64) * 64);
#define QE_CONV(TA_, TAPS_) short_conv_rows_kernel<TA_, TAPS_><<<rgrid, rthreads, 0, stream>>>(x, w, state, tok_seq, (TA_*)out, T, H)
#define QE_CONVS(TA_)                                                                                    \
        switch (taps) {                                                                                  \
            case 2: QE_CONV(TA_, 2); break;                                                              \
            case 3: QE_CONV(TA_, 3); break;                                                              \
            case 4: QE_CONV(TA_, 4); break;                                                              \
            case 5: QE_CONV(TA_, 5); break;                                                              \
            case 6: QE_CONV(TA_, 6); break;                                                              \
            case 7: QE_CONV(TA_, 7); break;                                                              \
            default: QE_CONV(TA_, 8);                                                                    \
        }
        if (dt_a == QE_F32) { QE_CONVS(float) }
        else if (dt_a == QE_BF16) { QE_CONVS(bf16_t) }
        else QE_REQUIRE(false, "short_conv: unknown output type %d", dt_a);
#undef QE_CONVS
#undef QE_CONV
        QE_LAUNCH_CHECK();
        if (update) {
            short_conv_rows_update_kernel<<<rgrid, rthreads, 0, stream>>>(x, state, tok_seq, T, H, taps);
            QE_LAUNCH_CHECK();
        }
        return 0;
    }
    if (dt_a == QE_F32)
        short_conv_kernel<float><<<grid, threads, 0, stream>>>(x, w, state, tok_seq, (float*)out, T, H, taps);
    else if (dt_a == QE_BF16)
        short_conv_kernel<bf16_t><<<grid, threads, 0, stream>>>(x, w, state, tok_seq, (bf16_t*)out, T, H, taps);
    else
        QE_REQUIRE(false, "short_conv: unknown output type %d", dt_a);
    QE_LAUNCH_CHECK();
    if (update && taps > 1) {
        short_conv_update_kernel<<<grid, threads, 0, stream>>>(x, state, tok_seq, T, H, taps);
        QE_LAUNCH_CHECK();
    }
    return 0;
}
