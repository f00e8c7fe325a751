// Token timestamps on the device: the alignment heads' cross-attention rows of every clip -> per-column z-scores ->
// median filter over time -> mean over heads -> dynamic time warping -> the time of each token's first frame.
// Follows src/align.rs:8-106 (transformers' _extract_token_timestamps) and computes exactly what the host routine
// mz_jump_times computes: the column statistics are accumulated in row order (in float with the fp16 roundings, as
// src/align.rs:18-23 does, or in double without them), every binary16 round trip is a round-to-nearest-even
// conversion, the DTW cost cells are (float)(-(double)s + (double)c), and contraction into fused multiply-adds is
// off, so both give identical bits.
//
// Three launches per batch of clips:
//   ts_stats_kernel  one thread per (clip, head, column) (ts_stats4_kernel: four adjacent columns per thread): mean
//                    and population standard deviation over the rows (ts_stats_lds_kernel: up to 256 rows, from LDS)
//   ts_cost_kernel   one workgroup per 32 x 64 tile of (row, column): median of the width-w reflect-padded window
//                    of z-scores, summed over heads; the cells are stored in anti-diagonal-major order
//                    [d = i + j][i], so that the DTW reads each diagonal with consecutive addresses
//   ts_dtw_wave_kernel  tables of at most 256 rows: one row per lane of one to four waves per clip, the previous two
//                    anti-diagonals in registers and the moves in LDS, where one lane walks the path back
//   ts_dtw_kernel    larger tables: one workgroup per clip; the DTW table is filled one anti-diagonal per step (every
//                    cell of a diagonal depends only on the two previous diagonals, kept in LDS), the move taken into
//                    each cell goes to a trace in the same diagonal-major order, and one lane walks the path back.
#include <math.h>

#include <algorithm>
#include <memory>
#include <mutex>
#include <new>

#include "../../include/mimizuku.h"
#include "mz_common.h"
#include "mz_internal.h"
#include "mz_kernels.h"

#pragma clang fp contract(off)

namespace {

__device__ __forceinline__ float rh(float x) { return (float)(f16)x; }

__device__ __forceinline__ void cswap(float& a, float& b) {
    const float lo = a < b ? a : b, hi = a < b ? b : a;
    a = lo;
    b = hi;
}

// the middle of 7 values (the order statistic is the same whatever network computes it)
__device__ __forceinline__ float median7(float* a) {
    cswap(a[0], a[6]), cswap(a[2], a[3]), cswap(a[4], a[5]);
    cswap(a[0], a[2]), cswap(a[1], a[4]), cswap(a[3], a[6]);
    cswap(a[0], a[1]), cswap(a[2], a[5]), cswap(a[3], a[4]);
    cswap(a[1], a[2]), cswap(a[4], a[6]);
    cswap(a[2], a[3]), cswap(a[4], a[5]);
    cswap(a[1], a[2]), cswap(a[3], a[4]), cswap(a[5], a[6]);
    return a[3];
}

__global__ void __launch_bounds__(256) ts_stats_kernel(const MzTs p) {
    const int c = blockIdx.z, a = blockIdx.y, j = blockIdx.x * 256 + threadIdx.x;
    const int R = p.rc[c].x, C = p.rc[c].y;
    if (j >= C || R <= 0) return;
    const float* w = p.w + c * p.clip_stride + (long)a * p.cols_full + j;
    const long rs = (long)p.heads * p.cols_full;
    float mu, sd;
    if (p.half) {
        float sum = 0.f;
        for (int i = 0; i < R; i++) sum += w[i * rs];
        const float mean = sum / (float)R;
        float sq = 0.f;
        for (int i = 0; i < R; i++) {
            const float dv = w[i * rs] - mean;
            sq += dv * dv;
        }
        mu = rh(mean);
        sd = rh(__builtin_sqrtf(sq / (float)R));
    } else {
        double sum = 0.0;
        for (int i = 0; i < R; i++) sum += (double)w[i * rs];
        const float mean = (float)(sum / R);
        double sq = 0.0;
        for (int i = 0; i < R; i++) {
            const double dv = (double)(w[i * rs] - mean);
            sq += dv * dv;
        }
        mu = mean;
        sd = __builtin_sqrtf((float)(sq / R));
    }
    const long o = ((long)c * p.heads + a) * p.cols_full + j;
    p.mean[o] = mu;
    p.sd[o] = sd;
}

// The same statistics for four adjacent columns per thread through 16-byte loads (each column's sums in row order,
// exactly as above): for rows whose column count and clip stride are multiples of 4 at a 16-byte aligned base
// (every engine batch: 1500 columns). Columns past C are summed (their reads stay inside the row) but not stored.
__global__ void __launch_bounds__(256) ts_stats4_kernel(const MzTs p) {
    const int c = blockIdx.z, a = blockIdx.y, j = (blockIdx.x * 256 + threadIdx.x) * 4;
    const int R = p.rc[c].x, C = p.rc[c].y;
    if (j >= C || R <= 0) return;
    const float4* w = (const float4*)(p.w + c * p.clip_stride + (long)a * p.cols_full + j);
    const long rs = (long)p.heads * p.cols_full / 4;
    float mu[4], sd[4];
    if (p.half) {
        float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
#pragma unroll 4
        for (int i = 0; i < R; i++) {
            const float4 v = w[i * rs];
            s0 += v.x;
            s1 += v.y;
            s2 += v.z;
            s3 += v.w;
        }
        const float m0 = s0 / (float)R, m1 = s1 / (float)R, m2 = s2 / (float)R, m3 = s3 / (float)R;
        float q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
#pragma unroll 4
        for (int i = 0; i < R; i++) {
            const float4 v = w[i * rs];
            const float d0 = v.x - m0, d1 = v.y - m1, d2 = v.z - m2, d3 = v.w - m3;
            q0 += d0 * d0;
            q1 += d1 * d1;
            q2 += d2 * d2;
            q3 += d3 * d3;
        }
        mu[0] = rh(m0), mu[1] = rh(m1), mu[2] = rh(m2), mu[3] = rh(m3);
        sd[0] = rh(__builtin_sqrtf(q0 / (float)R)), sd[1] = rh(__builtin_sqrtf(q1 / (float)R));
        sd[2] = rh(__builtin_sqrtf(q2 / (float)R)), sd[3] = rh(__builtin_sqrtf(q3 / (float)R));
    } else {
        double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll 4
        for (int i = 0; i < R; i++) {
            const float4 v = w[i * rs];
            s0 += (double)v.x;
            s1 += (double)v.y;
            s2 += (double)v.z;
            s3 += (double)v.w;
        }
        const float m0 = (float)(s0 / R), m1 = (float)(s1 / R), m2 = (float)(s2 / R), m3 = (float)(s3 / R);
        double q0 = 0.0, q1 = 0.0, q2 = 0.0, q3 = 0.0;
#pragma unroll 4
        for (int i = 0; i < R; i++) {
            const float4 v = w[i * rs];
            const double d0 = (double)(v.x - m0), d1 = (double)(v.y - m1), d2 = (double)(v.z - m2),
                         d3 = (double)(v.w - m3);
            q0 += d0 * d0;
            q1 += d1 * d1;
            q2 += d2 * d2;
            q3 += d3 * d3;
        }
        mu[0] = m0, mu[1] = m1, mu[2] = m2, mu[3] = m3;
        sd[0] = __builtin_sqrtf((float)(q0 / R)), sd[1] = __builtin_sqrtf((float)(q1 / R));
        sd[2] = __builtin_sqrtf((float)(q2 / R)), sd[3] = __builtin_sqrtf((float)(q3 / R));
    }
    const long o = ((long)c * p.heads + a) * p.cols_full + j;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (j + e < C) {
            p.mean[o + e] = mu[e];
            p.sd[o + e] = sd[e];
        }
}

// The same statistics for at most ST_R rows from LDS, one workgroup per (clip, head, 64 columns): the block's rows go
// straight into LDS once (whole 256-byte row segments, every load in flight together), and the first wave takes both
// passes from there, a column per lane, each column's sums in row order as above. Bound by reading the rows: the two
// passes over memory of ts_stats4_kernel read a large batch's rows twice, and these are more than stays in the
// memory-side cache (275 MB for 32 clips of up to 220 rows and 1500 columns, 6.88 million cells of 10 heads: 110 -> 86 us;
// 32 of 220 x 1500, 422 MB, 113; one clip of 41 rows x 6 heads 6.8 -> 3.5). Two workgroups per CU, so that one's sums run
// under the other's loads.
constexpr int ST_R = 256;

__global__ void __launch_bounds__(256) ts_stats_lds_kernel(const MzTs p) {
#if defined(__HIP_DEVICE_COMPILE__)
    __shared__ __attribute__((aligned(16))) float x[ST_R][64];
    const int c = blockIdx.z, a = blockIdx.y, j0 = blockIdx.x * 64, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int R = p.rc[c].x, C = p.rc[c].y;
    if (j0 >= C || R <= 0) return;
    const long rs = (long)p.heads * p.cols_full;
    // rows 4 g .. 4 g + 3 per load, 16 lanes (64 columns) each; rows past R and columns past the row read zeros
    const __amdgpu_buffer_rsrc_t rw = rsrc(p.w + c * p.clip_stride + (long)a * p.cols_full, (unsigned)(((long)(R - 1) * rs + p.cols_full) * 4));
    const int col = j0 + (lane & 15) * 4;
    for (int g = wave; 4 * g < R; g += 4) {
        const int i = 4 * g + (lane >> 4);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (__attribute__((address_space(3))) void*)&x[4 * g][0], 16,
                                                 i < R && col < p.cols_full ? (unsigned)(i * rs + col) * 4u : 0x80000000u, 0,
                                                 0, 0);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    const int j = j0 + lane;
    if (wave || j >= C) return;
    float mu, sd;
    if (p.half) {
        float sum = 0.f;
#pragma unroll 8
        for (int i = 0; i < R; i++) sum += x[i][lane];
        const float mean = sum / (float)R;
        float sq = 0.f;
#pragma unroll 8
        for (int i = 0; i < R; i++) {
            const float dv = x[i][lane] - mean;
            sq += dv * dv;
        }
        mu = rh(mean);
        sd = rh(__builtin_sqrtf(sq / (float)R));
    } else {
        double sum = 0.0;
#pragma unroll 8
        for (int i = 0; i < R; i++) sum += (double)x[i][lane];
        const float mean = (float)(sum / R);
        double sq = 0.0;
#pragma unroll 8
        for (int i = 0; i < R; i++) {
            const double dv = (double)(x[i][lane] - mean);
            sq += dv * dv;
        }
        mu = mean;
        sd = __builtin_sqrtf((float)(sq / R));
    }
    const long o = ((long)c * p.heads + a) * p.cols_full + j;
    p.mean[o] = mu;
    p.sd[o] = sd;
#endif
}

// One workgroup per tile of COST_RT rows x COST_CT columns of a clip. Per head, the tile's z-scores (with the window's
// reflect-padded halo) are computed once into LDS, the next head's weights already requested; each thread then takes the
// medians of eight adjacent cells, summed over heads in head order. The tile's cells leave diagonal by diagonal: the
// cells of one anti-diagonal within the tile are consecutive rows, so each diagonal's run is one contiguous store.
// W = 7: median of the two outer triples and the middle value. With both triples sorted, it is the middle one of the larger
// low, the middle of the three middles and the smaller high (the 3 x 3 rule for the median of nine, the third triple being
// -inf, the middle value, +inf), and a triple serves two windows: 8.5 min / med3 / max per cell where a sorting network
// took 48 compares and selects. W = 0: any odd width up to MZ_TS_MAX_WIDTH (insertion sort). 32 clips of up to 220 rows
// and 1500 columns, 6.88 million cells of 10 heads: 285 -> 109 us (32 of 220 x 1500: 145), one clip of 41 rows x 6 heads
// 40 -> 13.
constexpr int COST_RT = 32, COST_CT = 64, COST_HALO = MZ_TS_MAX_WIDTH - 1;

template <int W>
__global__ void __launch_bounds__(256) ts_cost_kernel(const MzTs p) {
    // row strides: 79 floats puts the eight cells of 8 x 8 threads in 64 banks, 66 a diagonal's 32 rows in 32
    __shared__ float zt[COST_RT][COST_CT + COST_HALO + 1];
    __shared__ float val[COST_RT][COST_CT + 2];
    __shared__ int nan_seen[2];
    const int c = blockIdx.z, i0 = blockIdx.y * COST_RT, j0 = blockIdx.x * COST_CT, tid = threadIdx.x;
    const int R = p.rc[c].x, C = p.rc[c].y;
    if (i0 >= R || j0 >= C) return;
    const int width = W ? W : p.width, pad = width >> 1, halo = 2 * pad;
    if (tid < 2) nan_seen[tid] = 0;
    lds_barrier();
    // the z phase: tile column cl = tid % 64 of rows tid / 64 + 4 k, then the halo columns 64 .. 64 + halo - 1, NH of them
    // per thread. Tile column cl stands for time j0 + cl - pad, reflected into 0 .. C - 1 as the window reads it
    // (columns of cells past C, whose values are never stored, are clamped into range instead).
    constexpr int NM = COST_RT / 4, NH = W ? 1 : (COST_RT * COST_HALO + 255) / 256;
    static_assert(COST_RT * 6 <= 256, "one halo element per thread at width 7");
    auto time_of = [&](int cl) {
        int t = j0 + cl - pad;
        if (t < 0) t = -t;
        if (t >= C) t = 2 * (C - 1) - t;
        return t < 0 ? 0 : t > C - 1 ? C - 1 : t;
    };
    const int zl = tid & 63, zi = tid >> 6, zt0 = time_of(zl);
    int hi[NH], hc[NH], ht[NH];
#pragma unroll
    for (int k = 0; k < NH; k++) {
        const int e = tid + 256 * k;
        hi[k] = halo ? e / max(halo, 1) : COST_RT;
        hc[k] = COST_CT + e - hi[k] * halo;
        ht[k] = time_of(hc[k]);
    }
    const float* wc = p.w + c * p.clip_stride;
    const float *mu = p.mean + (long)c * p.heads * p.cols_full, *sd = p.sd + (long)c * p.heads * p.cols_full;
    float xm[NM], xh[NH], mm, sm, mh[NH], sh[NH];
    auto fetch = [&](int a) {
        const long o = (long)a * p.cols_full;
        mm = mu[o + zt0];
        sm = sd[o + zt0];
#pragma unroll
        for (int k = 0; k < NM; k++) {
            const int i = i0 + zi + 4 * k;
            xm[k] = i < R ? wc[((long)i * p.heads + a) * p.cols_full + zt0] : 0.f;
        }
#pragma unroll
        for (int k = 0; k < NH; k++) {
            const int i = i0 + hi[k];
            const bool on = hi[k] < COST_RT && i < R;
            mh[k] = on ? mu[o + ht[k]] : 0.f;
            sh[k] = on ? sd[o + ht[k]] : 0.f;
            xh[k] = on ? wc[((long)i * p.heads + a) * p.cols_full + ht[k]] : 0.f;
        }
    };
    auto zscore = [&](float x, float m, float s) { return s > 0.f ? (p.half ? rh(rh(x - m) / s) : (x - m) / s) : 0.f; };
    // the median phase, eight cells per thread: at width 7 columns jl .. jl + 7 of row il, otherwise column jl of rows
    // il + 4 q (a wave's cells of one q lie in one row, and the rows past R are left out: 5 rows, width 15, 287 us for the
    // whole call; with eight columns per thread, so that one wave had all the rows there are, 855)
    const int il = W ? tid >> 3 : tid >> 6, jl = W ? (tid & 7) * 8 : tid & 63;
    auto row = [&](int q) { return W ? il : il + 4 * q; };
    auto col = [&](int q) { return W ? jl + q : jl; };
    float acc[8];
#pragma unroll
    for (int q = 0; q < 8; q++) acc[q] = 0.f;
    fetch(0);
    for (int a = 0; a < p.heads; a++) {
        bool nan = false;
#pragma unroll
        for (int k = 0; k < NM; k++) {
            const float z = i0 + zi + 4 * k < R ? zscore(xm[k], mm, sm) : 0.f;
            nan |= z != z;
            zt[zi + 4 * k][zl] = z;
        }
#pragma unroll
        for (int k = 0; k < NH; k++)
            if (hi[k] < COST_RT) {
                const float z = zscore(xh[k], mh[k], sh[k]);
                nan |= z != z;
                zt[hi[k]][hc[k]] = z;
            }
        if (__ballot(nan) && (tid & 63) == 0) nan_seen[a & 1] = 1;
        if (a + 1 < p.heads) fetch(a + 1);
        lds_barrier();  // (the weights of the next head stay in flight)
        const bool slow = nan_seen[a & 1] != 0;
        const float* zr = &zt[il][jl];
        if (C <= pad) {
#pragma unroll
            for (int q = 0; q < 8; q++) acc[q] += zt[row(q)][col(q) + pad];  // fewer columns than the half width: no filter
        } else if (W == 7 && !slow) {
            float z[14], lo[12], md[12], up[12];
#pragma unroll
            for (int q = 0; q < 14; q++) z[q] = zr[q];
#pragma unroll
            for (int q = 0; q < 12; q++) {
                lo[q] = fminf(fminf(z[q], z[q + 1]), z[q + 2]);
                md[q] = __builtin_amdgcn_fmed3f(z[q], z[q + 1], z[q + 2]);
                up[q] = fmaxf(fmaxf(z[q], z[q + 1]), z[q + 2]);
            }
#pragma unroll
            for (int q = 0; q < 8; q++)
                acc[q] += __builtin_amdgcn_fmed3f(fmaxf(lo[q], lo[q + 4]),
                                                  __builtin_amdgcn_fmed3f(md[q], z[q + 3], md[q + 4]),
                                                  fminf(up[q], up[q + 4]));
        } else if (W == 7) {
            // a NaN in the tile (half mode: a z-score that overflowed): min / med3 / max drop it, the network, with the
            // host routine's comparisons, moves it like any value
#pragma unroll
            for (int q = 0; q < 8; q++) {
                float win[7];
#pragma unroll
                for (int e = 0; e < 7; e++) win[e] = zr[q + e];
                acc[q] += median7(win);
            }
        } else {
#pragma unroll
            for (int q = 0; q < 8; q++) {
                if (i0 + row(q) >= R) continue;
                float win[MZ_TS_MAX_WIDTH];
                for (int e = 0; e < width; e++) {
                    const float v = zt[row(q)][col(q) + e];
                    int r = e - 1;
                    while (r >= 0 && win[r] > v) {
                        win[r + 1] = win[r];
                        r--;
                    }
                    win[r + 1] = v;
                }
                acc[q] += win[pad];
            }
        }
        lds_barrier();  // zt is rewritten for the next head
        if (tid == 0) nan_seen[a & 1] = 0;  // (read again, after another barrier, two heads on)
    }
#pragma unroll
    for (int q = 0; q < 8; q++) {
        float v = acc[q] / (float)p.heads;
        if (p.half) v = rh(v);
        val[row(q)][col(q)] = v;
    }
    __syncthreads();
    // DTW cell (i + 1, j + 1) lies on anti-diagonal i + j + 2: tile diagonal dl = il + jl holds rows il of one run
    float* dst = p.cost + c * p.diag_stride + (long)(i0 + j0 + 2) * p.ldd + (i0 + 1);
    const int dr = tid & 31;
    for (int dl = tid >> 5; dl < COST_RT + COST_CT - 1; dl += 8) {
        const int cl = dl - dr;
        if (cl >= 0 && cl < COST_CT && i0 + dr < R && j0 + cl < C) dst[(long)dl * p.ldd + dr] = val[dr][cl];
    }
}

// One workgroup per clip. Row i of the table (0..R) is handled by threads i, i + blockDim, ... The costs are staged
// in LDS DTW_STAGE diagonals at a time (diagonal-major, so a chunk is one contiguous run, copied with direct-to-LDS
// loads) while the previous chunk is being used; within a chunk a diagonal waits only for the LDS traffic of the
// one before (lds_barrier), so the trace stores and the next chunk's loads stay in flight.
constexpr int DTW_STAGE = 12;

__global__ void __launch_bounds__(1024) ts_dtw_kernel(const MzTs p) {
#if defined(__HIP_DEVICE_COMPILE__)  // the buffer-resource type exists only in the device pass
    extern __shared__ float lds[];
    const int c = blockIdx.x, R = p.rc[c].x, C = p.rc[c].y, nt = blockDim.x, tid = threadIdx.x;
    float* out = p.out + (long)c * p.out_stride;
    if (R <= 0) return;
    if (C <= 0) {
        for (int k = tid; k < R; k += nt) out[k] = 0.f;
        return;
    }
    const int ld = p.ldd;
    float* diag = lds;                       // 3 x (R + 1): diagonals d, d - 1, d - 2 in rotation
    int* first = (int*)(lds + 3 * ld);       // per row: the column of the path's first cell in that row
    float* chunk = lds + 4 * ld;             // 2 x DTW_STAGE diagonals of costs
    const float* cost = p.cost + c * p.diag_stride;
    signed char* tr = p.trace + c * p.diag_stride;
    // reads past the clip's cost table return zeros (the descriptor's range check)
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(cost), (short)0,
                                                                         (int)(p.diag_stride * 4), 0x00020000);
    // a chunk buffer holds a whole number of 64-float wave copies (the last one may read past the chunk)
    const int lane = tid & 63, wave = tid >> 6, per = (DTW_STAGE * ld + 63) & ~63;
    auto stage = [&](int d0, float* dst) {
        // wave w's lanes copy floats w * 64 + lane, + nt, ... of diagonals d0 .. d0 + DTW_STAGE - 1
        for (int k = wave * 64; k < per; k += nt)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rc, (__attribute__((address_space(3))) void*)(dst + k), 4,
                                                     (unsigned)((d0 * ld + k + lane) * 4), 0, 0, 0);
    };
    stage(0, chunk);
    for (int d0 = 0; d0 <= R + C; d0 += DTW_STAGE) {
        float* cb = chunk + ((d0 / DTW_STAGE) & 1) * per;
        __builtin_amdgcn_s_waitcnt(0);  // this chunk's copies (and the trace stores so far) are done
        __syncthreads();                // ... in every wave, and the other buffer's last chunk is no longer read
        if (d0 + DTW_STAGE <= R + C) stage(d0 + DTW_STAGE, chunk + (((d0 / DTW_STAGE) + 1) & 1) * per);
        const int dend = min(d0 + DTW_STAGE, R + C + 1);
        for (int d = d0; d < dend; d++) {
            float* cur = diag + (d % 3) * ld;
            const float* p1 = diag + ((d + 2) % 3) * ld;
            const float* p2 = diag + ((d + 1) % 3) * ld;
            const float* cd = cb + (d - d0) * ld;
            const int lo = max(0, d - C), hi = min(R, d);
            for (int i = lo + tid; i <= hi; i += nt) {
                const int j = d - i;
                float v;
                signed char t;
                if (i == 0) {
                    v = d == 0 ? 0.f : INFINITY;
                    t = 2;
                } else if (j == 0) {
                    v = INFINITY;
                    t = 1;
                } else {
                    const float c0 = p2[i - 1], c1 = p1[i - 1], c2 = p1[i];
                    float m;
                    if (c0 < c1 && c0 < c2) {
                        m = c0;
                        t = 0;
                    } else if (c1 < c0 && c1 < c2) {
                        m = c1;
                        t = 1;
                    } else {
                        m = c2;
                        t = 2;
                    }
                    v = (float)(-(double)cd[i] + (double)m);
                }
                cur[i] = v;
                tr[(long)d * ld + i] = t;
            }
            lds_barrier();
        }
    }
    __builtin_amdgcn_s_waitcnt(0);
    // the trace stores went to global memory from every lane: make them visible to the walking lane
    __threadfence_block();
    __syncthreads();
    if (tid == 0) {
        int i = R, j = C;
        bool row0 = false;
        while (i > 0 || j > 0) {
            first[i] = j - 1;
            row0 |= i == 0;
            const signed char t = tr[(long)(i + j) * ld + i];
            if (t == 0) {
                i--;
                j--;
            } else if (t == 1) {
                i--;
            } else {
                j--;
            }
        }
        // the token rows start at text index -1 when the path ran along row 0, else at 0; one start per row
        const int r0 = row0 ? 0 : 1;
        for (int n = 0; n < R; n++) out[n] = (float)((double)first[r0 + n] * 0.02);
    }
#endif
}

// Tables of at most 64 NW token rows: NW waves per clip, one table row per lane, a diagonal per step. A cell needs its
// left neighbour (this lane, one diagonal back) and the row above at the two diagonals before, which is the lane before
// one and two steps ago: one cross-lane move (DPP wave_shr) per step and no LDS round trip. Row 64 w (the last of the
// wave before) reaches wave w in chunks of 64 diagonals through LDS: wave w works one chunk behind wave w - 1, with one
// barrier per chunk, and takes the chunk's values out of a register that shifts by a lane per step. The moves (a bit per
// lane and kind) collect in two registers per 32 diagonals and go to LDS, where the path is walked back a run of equal
// moves at a time. The time is the serial chain of about 20 instructions per diagonal, the longest clip's: 32 clips of up
// to 220 rows and 1500 columns 466 -> 145 us (all of 220 x 1500: 149), one of 41 rows 415 -> 91 (four rows per lane in one
// wave and a walk of one cell at a time before).
// Same comparisons and results as ts_dtw_kernel, so the same bits.
constexpr int DTW_CH = 64;   // diagonals per chunk
constexpr int DTW_NCH = 28;  // chunks of a table: its diagonals 2 .. R + C are at most 1792 (256 rows x 1500 columns: 1755)

// lane l gets lane l - 1's v, lane 0 first; lane l gets lane l + 1's v, lane 63 last (DPP wave_shr:1, wave_shl:1)
__device__ __forceinline__ float lane_prev(float v, float first) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, first), __builtin_bit_cast(int, v),
                                                                 0x138, 0xF, 0xF, false));
}
__device__ __forceinline__ float lane_next(float v, float last) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, last), __builtin_bit_cast(int, v),
                                                                 0x130, 0xF, 0xF, false));
}

template <int NW>
__global__ void __launch_bounds__(64 * NW, 1) ts_dtw_wave_kernel(const MzTs p) {
#if defined(__HIP_DEVICE_COMPILE__)
    // moves of 32 diagonals of a row: diagonal 2 + 32 g + k at bit 31 - k of x (diagonal move) and y (up); none: left
    __shared__ uint2 moves[2 * DTW_NCH][64 * NW];
    __shared__ float edge[NW][4 * DTW_CH];  // the last row of each wave, by diagonal modulo 256
    __shared__ int first[64 * NW + 2];      // per row; [R + 1]: the first token row's offset
    const int c = blockIdx.x, R = p.rc[c].x, C = p.rc[c].y, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float* out = p.out + (long)c * p.out_stride;
    if (R <= 0) return;
    if (C <= 0) {
        for (int k = tid; k < R; k += 64 * NW) out[k] = 0.f;
        return;
    }
    const int row = tid + 1, nch = (R + C - 1 + DTW_CH - 1) / DTW_CH;
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(p.cost + c * p.diag_stride), (short)0, (int)(p.diag_stride * 4), 0x00020000);
    // the chunk's costs of this row, one register per diagonal: the diagonal (none past the table's last) in the
    // scalar offset; rows past R, and the cells left of the table (column <= 0: only in the wave's first chunk), read
    // zero through the range check
    float cost[2][DTW_CH];
    auto load = [&](int ch, float(&x)[DTW_CH]) {
        const int d0 = 2 + ch * DTW_CH;
        const bool edge_cells = ch <= wave;
#pragma unroll
        for (int k = 0; k < DTW_CH; k++) {
            const int d = min(d0 + k, R + C);
            const bool on = row <= R && !(edge_cells && d0 + k <= row);
            x[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rc, on ? (unsigned)row * 4u : 0x80000000u,
                                                                                  d * p.ldd * 4, 0));
        }
    };
    // Every cell of a diagonal is computed, in or out of the table: a cell outside (row past R, column past C) feeds only
    // cells outside, and cells left of column 1 stay +inf, as column 0 and row 0 are (but for the 0 at (0, 0), the
    // value up and left of the first cell).
    float left = INFINITY, up2 = tid == 0 ? 0.f : INFINITY;
    auto chunk = [&](int ch, const float(&x)[DTW_CH]) {
        const int d0 = 2 + ch * DTW_CH;
        float in = wave ? edge[wave ? wave - 1 : 0][(d0 - 1 + lane) & (4 * DTW_CH - 1)] : INFINITY, sent = 0.f;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            unsigned m0 = 0, m1 = 0;
#pragma unroll
            for (int k = 0; k < 32; k++) {
                const float up1 = lane_prev(left, in);
                in = lane_next(in, in);
                // the reference's comparisons as written (align.rs:77-83), so a NaN cost (a NaN or infinite z-score in
                // half mode) picks the same move as the host routine and ts_dtw_kernel: fminf would drop the NaN
                const bool t0 = (up2 < up1) & (up2 < left), t1 = (up1 < up2) & (up1 < left);
                const float m = t0 ? up2 : t1 ? up1 : left;
                // ts_dtw_kernel's fp64 -x + m rounded to fp32 equals the fp32 m - x: a sum rounded first to 53 bits
                // and then to 24 rounds as if once, since 53 >= 2 x 24 + 2 (Figueroa, 1995)
                left = m - x[32 * h + k];
                up2 = up1;
                m0 = 2 * m0 + (t0 ? 1u : 0u);
                m1 = 2 * m1 + (t1 ? 1u : 0u);
                sent = lane_next(sent, left);
            }
            moves[2 * ch + h][tid] = make_uint2(m0, m1);
        }
        edge[wave][(d0 + lane) & (4 * DTW_CH - 1)] = sent;
    };
    // wave w's chunk s - w at step s; its chunks before w hold no cell of the table
    const bool live = 64 * wave < R;
    if (live) load(wave, cost[0]);
    for (int s = 0; s < nch + NW - 1; s += 2) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const int ch = s + b - wave;
            if (live && ch >= wave && ch < nch) {
                // (the chunk parity of a wave is that of s - 2 wave: buffer b)
                if (ch + 1 < nch) load(ch + 1, cost[(b + 1) & 1]);
                chunk(ch, cost[b]);
            }
            lds_barrier();
        }
    }
    __syncthreads();
    if (tid == 0) {
        // back from (R, C): in row i the path runs left to the last cell at or before this one whose move is another
        // (column 0 if there is none), which is the row's first cell, then up or diagonally
        int i = R, j = C;
        while (i > 0 && j > 0) {
            int q = i + j - 2, d = -1;  // diagonal - 2
            uint2 w;
            do {
                w = moves[q >> 5][i - 1];
                const unsigned any = (w.x | w.y) >> (31 - (q & 31)) << (31 - (q & 31));
                d = any ? (q | 31) - (__ffs(any) - 1) : -1;
                q = (q & ~31) - 1;
            } while (d < 0 && q >= i - 1);
            j = d < 0 ? 0 : d + 2 - i;
            if (j < 1) j = 0;
            first[i] = j - 1;
            if (j > 0 && (w.x >> (31 - (d & 31)) & 1)) j--;
            i--;
        }
        for (; i > 0; i--) first[i] = -1;  // column 0: up
        first[0] = 0;
        // the token rows start at text index -1 when the path ran along row 0, else at 0
        first[R + 1] = j > 0 ? 0 : 1;
    }
    __syncthreads();
    const int r0 = first[R + 1];  // one start per row
#pragma unroll 1
    for (int n = tid; n < R; n += 64 * NW) out[n] = (float)((double)first[r0 + n] * 0.02);
#endif
}

}  // namespace

// 3 diagonals, the first-column table and 2 chunks of DTW_STAGE diagonals of costs, ld = rmax + 1 floats each
size_t mz_ts_lds_bytes(int rmax) { return ((size_t)(rmax + 1) * 4 + 2 * (((size_t)DTW_STAGE * (rmax + 1) + 63) & ~(size_t)63)) * 4; }

hipError_t mz_ts_launch(hipStream_t s, const MzTs& p, int n) {
    if (n <= 0) return hipSuccess;
    if (p.width < 1 || p.width % 2 == 0 || p.width > MZ_TS_MAX_WIDTH || p.heads <= 0 || p.rmax < 0 ||
        p.ldd < p.rmax + 1 || p.cols_full <= 0)
        return hipErrorInvalidValue;
    const bool vec = p.cols_full % 4 == 0 && p.clip_stride % 4 == 0 && ((uintptr_t)p.w & 15) == 0;
    // (a clip's rows within 31-bit byte offsets)
    if (vec && p.rmax <= ST_R && (long)p.rmax * p.heads * p.cols_full * 4 < (1L << 31)) {
        hipLaunchKernelGGL(ts_stats_lds_kernel, dim3((p.cols_full + 63) / 64, p.heads, n), dim3(256), 0, s, p);
    } else if (vec) {
        const dim3 gs((p.cols_full / 4 + 255) / 256, p.heads, n);
        hipLaunchKernelGGL(ts_stats4_kernel, gs, dim3(256), 0, s, p);
    } else {
        const dim3 gs((p.cols_full + 255) / 256, p.heads, n);
        hipLaunchKernelGGL(ts_stats_kernel, gs, dim3(256), 0, s, p);
    }
    if (p.rmax > 0) {
        const dim3 gc((p.cols_full + COST_CT - 1) / COST_CT, (p.rmax + COST_RT - 1) / COST_RT, n);
        if (p.width == 7)
            hipLaunchKernelGGL(ts_cost_kernel<7>, gc, dim3(256), 0, s, p);
        else
            hipLaunchKernelGGL(ts_cost_kernel<0>, gc, dim3(256), 0, s, p);
    }
    // the wave kernel: at most 256 rows, and the moves of every diagonal in LDS
    if (p.rmax <= 256 && p.rmax + p.cols_full - 1 <= DTW_NCH * DTW_CH && p.diag_stride * 4 < (1L << 31)) {
        if (p.rmax <= 64) hipLaunchKernelGGL(ts_dtw_wave_kernel<1>, dim3(n), dim3(64), 0, s, p);
        else if (p.rmax <= 128) hipLaunchKernelGGL(ts_dtw_wave_kernel<2>, dim3(n), dim3(128), 0, s, p);
        else hipLaunchKernelGGL(ts_dtw_wave_kernel<4>, dim3(n), dim3(256), 0, s, p);
        return hipGetLastError();
    }
    int nt = ((p.rmax + 1 + 63) / 64) * 64;
    nt = nt < 256 ? 256 : nt > 1024 ? 1024 : nt;
    if (mz_ts_lds_bytes(p.ldd - 1) > 64 * 1024 || p.diag_stride * 4 >= (1L << 31)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(ts_dtw_kernel, dim3(n), dim3(nt), mz_ts_lds_bytes(p.ldd - 1), s, p);
    return hipGetLastError();
}

// ------------------------------------------------------------------ the entry point that allocates nothing

// Scratch of mz_jump_times_device_noalloc: a file-scope device array, one copy per GPU the library runs on, held until
// the process ends. In host code `scratch` names a host-side stand-in, never a device address: its address on each
// device comes from hipGetSymbolAddress (mz_ts_scratch_setup, called by mz_init with that device current) and only
// that address is passed to kernels and copies.
static __device__ __align__(256) unsigned char scratch[MZ_TS_SCRATCH_BYTES];

namespace {
constexpr int MZ_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void* g_scratch[MZ_MAX_DEVICES] = {};
// held by a call of mz_jump_times_device_noalloc for its whole use of that device's array
std::mutex g_scratch_use[MZ_MAX_DEVICES];
size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }
}  // namespace

int mz_ts_scratch_setup(int device) {
    if (device < 0 || device >= MZ_MAX_DEVICES) return mz_fail(MZ_ERR_ARG, "device %d: at most %d devices", device, MZ_MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[device]) return MZ_OK;
    int cur = -1;
    if (int r = mz_hip(hipGetDevice(&cur), "hipGetDevice")) return r;
    if (cur != device) return mz_fail(MZ_ERR_STATE, "timestamp scratch set-up: device %d is not current (%d)", device, cur);
    void* ptr = nullptr;
    if (int r = mz_hip(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)")) return r;
    if (!ptr) return mz_fail(MZ_ERR_HIP, "hipGetSymbolAddress(scratch) gave a null address");
    g_scratch[device] = ptr;
    return MZ_OK;
}

extern "C" int mz_jump_times_device_noalloc(mz_ctx* c, uint64_t w, int64_t clip_stride, int n, const int32_t* rows,
                                            const int32_t* cols, int heads, int cols_full, int width, int half,
                                            float* out, int64_t out_stride) {
    if (!c || !w || !rows || !cols || !out || n < 0 || heads <= 0 || cols_full <= 0 || clip_stride < 0)
        return mz_fail(MZ_ERR_ARG, "mz_jump_times_device_noalloc: bad argument");
    if (width < 1 || width % 2 == 0 || width > MZ_TS_MAX_WIDTH)
        return mz_fail(MZ_ERR_ARG, "mz_jump_times_device_noalloc: width %d (odd, at most %d)", width, MZ_TS_MAX_WIDTH);
    for (int i = 0; i < n; i++)
        if (rows[i] < 0 || cols[i] < 0 || cols[i] > cols_full || rows[i] > 4095 || rows[i] > out_stride)
            return mz_fail(MZ_ERR_ARG, "mz_jump_times_device_noalloc: clip %d has %d rows, %d columns", i, rows[i],
                           cols[i]);
    if (n == 0) return MZ_OK;
    if (int r = mz_hip(hipSetDevice(c->device), "hipSetDevice")) return r;
    if (int r = mz_ts_scratch_setup(c->device)) return r;
    unsigned char* base;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        base = (unsigned char*)g_scratch[c->device];
    }
    // the array is this device's only copy: calls from other threads (or contexts) on the same GPU wait until this
    // one's results are on the host (every chunk below ends with a synchronisation of the stream)
    std::lock_guard<std::mutex> use(g_scratch_use[c->device]);
    // scratch of k clips whose longest has rmax rows: (rows, columns), column statistics, DTW cost and trace, times
    auto need = [&](int k, int rmax) {
        return up256((size_t)k * sizeof(int2)) + 2 * up256((size_t)k * heads * cols_full * 4) +
               up256((size_t)k * mz_ts_diag_stride(rmax, cols_full) * 5) + up256((size_t)k * rmax * 4);
    };
    // the clips go through the array in chunks of at most MZ_TS_NOALLOC_CHUNK that fit in it, one after the other
    int2 rc[MZ_TS_NOALLOC_CHUNK];
    // a chunk's times on the host: requested before anything is in flight, and without an exception past the C entry
    const int longest = *std::max_element(rows, rows + n);
    const std::unique_ptr<float[]> times(new (std::nothrow) float[(size_t)std::min(n, (int)MZ_TS_NOALLOC_CHUNK) * std::max(longest, 1)]);
    if (!times) return mz_fail(MZ_ERR_STATE, "mz_jump_times_device_noalloc: out of host memory");
    for (int c0 = 0; c0 < n;) {
        int k = 0, rmax = 0;
        while (c0 + k < n && k < MZ_TS_NOALLOC_CHUNK && need(k + 1, std::max(rmax, (int)rows[c0 + k])) <= MZ_TS_SCRATCH_BYTES) {
            rmax = std::max(rmax, (int)rows[c0 + k]);
            k++;
        }
        if (k == 0)
            return mz_fail(MZ_ERR_ARG,
                           "mz_jump_times_device_noalloc: clip %d (%d rows, %d heads x %d columns) needs %zu bytes of "
                           "scratch; the static scratch holds %u",
                           c0, rows[c0], heads, cols_full, need(1, rows[c0]), (unsigned)MZ_TS_SCRATCH_BYTES);
        for (int i = 0; i < k; i++) rc[i] = int2{rows[c0 + i], cols[c0 + i]};
        const long ds = mz_ts_diag_stride(rmax, cols_full);
        unsigned char* q = base;
        auto carve = [&](size_t bytes) {
            unsigned char* r = q;
            q += up256(bytes);
            return r;
        };
        MzTs p{};
        p.w = (const float*)(uintptr_t)w + (size_t)c0 * clip_stride;
        p.clip_stride = clip_stride;
        p.heads = heads;
        p.cols_full = cols_full;
        p.width = width;
        p.half = half;
        p.rmax = rmax;
        p.rc = (const int2*)carve((size_t)k * sizeof(int2));
        p.mean = (float*)carve((size_t)k * heads * cols_full * 4);
        p.sd = (float*)carve((size_t)k * heads * cols_full * 4);
        p.cost = (float*)carve((size_t)k * ds * 5);
        p.trace = (signed char*)(p.cost + (size_t)k * ds);
        p.diag_stride = ds;
        p.ldd = mz_ts_ldd(rmax);
        p.out = (float*)carve((size_t)k * rmax * 4);
        p.out_stride = rmax;
        int r = mz_hip(hipMemcpyAsync((void*)p.rc, rc, (size_t)k * sizeof(int2), hipMemcpyHostToDevice, c->stream),
                       "upload");
        if (!r) r = mz_hip(mz_ts_launch(c->stream, p, k), "timestamp kernels");
        // the chunk's times in one copy (one per clip took longer than the kernels of a large chunk)
        if (!r && rmax > 0)
            r = mz_hip(hipMemcpyAsync(times.get(), p.out, (size_t)k * rmax * 4, hipMemcpyDeviceToHost, c->stream), "download");
        // the next chunk reuses the array (and rc): wait for this one
        const int rs = mz_hip(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
        if (r || rs) return r ? r : rs;
        for (int i = 0; i < k; i++)
            std::copy(times.get() + (size_t)i * rmax, times.get() + (size_t)i * rmax + rows[c0 + i],
                      out + (size_t)(c0 + i) * out_stride);
        c0 += k;
    }
    return MZ_OK;
}
