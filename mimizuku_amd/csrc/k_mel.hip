// Whisper's log-mel features on the device (Mel::features, src/audio.rs:195-249; WhisperFeatureExtractor): the
// 30 s buffer zero padded, centred 400-point frames every 160 samples with reflect padding, the periodic-Hann-
// windowed DFT as power spectra, n_mels Slaney filters over 201 bins, log10 floored at 1e-10, clamped to (max - 8) per
// clip, then (x + 4) / 4. Frames past the audio are log10(1e-10) = -10 without computing them.
//
// The DFT is in double, as the reference's: samples widened, products and sums in double, the power rounded to float.
// A real frame's 400-point sums fold twice by the symmetries of cos and sin (j and 400 - j, then j and 200 - j, for even
// and odd bins apart), which leaves four products of [frames][101] by [101][101] and runs them on the fp64 matrix
// cores: a quarter of the direct sum's products. Fewer terms per sum, each product and add rounded in double, so the
// spectra are as close to the exact ones as the reference's are, though not summed in its order. The filter sums
// are float, in bin order; log10 is the device library's.
//
//   mel_basis_kernel  the folded basis in the matrix cores' operand order, and the window
//   mel_spec_kernel   one workgroup per (16 M frames, clip): the frames' samples in LDS, wave w the bins 32 w .. 32 w + 31,
//                     the power spectra to LDS, then the filters, the logarithm and the workgroup's maximum
//   mel_norm_kernel   the clip's maximum from the workgroups', then the clamp and scale in place
#include <math.h>

#include "mz_common.h"
#include "mz_kernels.h"

#pragma clang fp contract(off)

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int NT = 7;             // 16-bin tiles of the even (0, 2, .. 200) and of the odd bins (1, 3, .. 199)
constexpr int NS = 26;            // steps of 4 terms over j = 0 .. 100
constexpr int HOPP = 164;         // LDS floats per hop of 160 samples: 16 frames' reads of 4 samples fall in 64 banks
constexpr int PWP = 205;          // LDS floats per power spectrum: odd, one bank per frame
static_assert(4 * NT * NS * 64 + 256 == MZ_MEL_BASIS, "basis size");

__device__ __forceinline__ int live_frames(int n) {
    return min((n + MZ_MEL_NFFT / 2 + MZ_MEL_HOP - 1) / MZ_MEL_HOP, MZ_NFR_HOST);
}

// [part][tile][step][lane]: term j = 4 step + lane / 16 of bin n = 16 tile + lane % 16, zero past the last bin and term;
// parts: cos of the even bins 2 n, cos of the odd bins 2 n + 1, sin of the even, sin of the odd. Then the window
// w[0 .. 200] (the other half mirrors it). Angles are reduced to whole fractions of pi first.
__global__ void __launch_bounds__(256) mel_basis_kernel(double* __restrict__ basis) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= MZ_MEL_BASIS) return;
    if (i >= 4 * NT * NS * 64) {
        basis[i] = 0.5 - 0.5 * cospi((double)(i - 4 * NT * NS * 64) / 200.0);
        return;
    }
    const int lane = i & 63, s = (i >> 6) % NS, t = (i >> 6) / NS % NT, part = (i >> 6) / (NS * NT);
    const int j = 4 * s + (lane >> 4), n = 16 * t + (lane & 15);
    const bool odd = part & 1, sine = part >= 2;
    double v = 0.0;
    if (j <= 100 && n <= (odd ? 99 : 100)) {
        const double a = odd ? (double)(j * (2 * n + 1) % 400) / 200.0 : (double)(j * n % 200) / 100.0;
        v = sine ? sinpi(a) : cospi(a);
        if (j == 100 && odd != sine) v = 0.0;  // cos of the odd, sin of the even bins
    }
    basis[i] = v;
}

// Bound by the fp64 matrix cores: 104 products of 16 x 16 x 4 per wave and 16 frames (a wave holds one 16-bin tile of all
// four parts, so a bin's real and imaginary sums meet in one lane), 64 cycles each. The left operands are made from
// the samples by every wave for itself (12 fp64 instructions per 4 products), so LDS holds the samples only. M = 2
// halves the basis' reads per frame (373 KB per workgroup, from L2); M = 1 is for few frames. 32 clips of 18 to 30 s
// (76,536 frames): 257 us, 35% of the matrix cores' fp64 rate (91 us of products), for the transform, filters and
// logarithm that took 1386 + 381 us (one bin per thread, multiply and add apart; one workgroup per frame with 12 KB strided
// stores); 32 of 30 s (96,000 frames) 297 us, 38%; one of 7 s 154 + 30 -> 19.
template <int M>
__global__ void __launch_bounds__(64 * NT) mel_spec_kernel(const MzMel p) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int FB = 16 * M, HOPS = FB + 2;  // frame f spans hops f, f + 1 and half of f + 2
    __shared__ float xs[HOPS * HOPP];
    __shared__ double win[208];
    __shared__ float pw[FB][PWP];
    __shared__ int odd_frame[FB];  // frames with a power that is not finite
    __shared__ int meta[256];
    __shared__ float wts[MZ_MEL_WTS];
    __shared__ float red[NT];
    const int c = blockIdx.y, t0 = blockIdx.x * FB, n = p.ns[c], live = live_frames(n), tid = threadIdx.x;
    if (t0 >= live) return;
    const float* y = p.audio + (long)c * MZ_MEL_NSAMPLES;
    // sample i of the padded buffer: reflect at both ends of the 30 s window, zero past the audio
    for (int q = tid; q < HOPS * MZ_MEL_HOP; q += 64 * NT) {
        int i = t0 * MZ_MEL_HOP + q - MZ_MEL_NFFT / 2;
        if (i < 0) i = -i;
        else if (i >= MZ_MEL_NSAMPLES) i = 2 * (MZ_MEL_NSAMPLES - 1) - i;
        xs[q / MZ_MEL_HOP * HOPP + q % MZ_MEL_HOP] = i >= 0 && i < n ? y[i] : 0.f;
    }
    if (tid < 201) win[tid] = p.basis[4 * NT * NS * 64 + tid];
    if (tid < FB) odd_frame[tid] = 0;
    for (int m = tid; m < p.n_mels; m += 64 * NT) meta[m] = p.meta[m];
    for (int i = tid; i < MZ_MEL_WTS; i += 64 * NT) wts[i] = p.wts[i];
    __syncthreads();

    const int lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lq = lane >> 4;
    const double* bl = p.basis + (long)wave * NS * 64 + lane;
    constexpr int PART = NT * NS * 64;
    f64x4 acc[4][M];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
        for (int m = 0; m < M; m++) acc[q][m] = f64x4{0.0, 0.0, 0.0, 0.0};
    double b[4], bn[4];
#pragma unroll
    for (int q = 0; q < 4; q++) bn[q] = bl[q * PART];
    for (int s = 0; s < NS; s++) {
#pragma unroll
        for (int q = 0; q < 4; q++) b[q] = bn[q];
        if (s + 1 < NS) {
#pragma unroll
            for (int q = 0; q < 4; q++) bn[q] = bl[q * PART + (s + 1) * 64];
        }
        // samples j, 400 - j, 200 - j, 200 + j of the frame (j = 0: its own partner, weight 0; the terms past 100 meet a
        // zero basis)
        const int j = 4 * s + lq, j4 = j ? 400 - j : 0, j2 = 200 - j;
        const int o1 = j4 + (HOPP - 160) * (j4 / 160), o2 = j2 + (HOPP - 160) * (j2 / 160), o3 = 200 + j + (HOPP - 160);
        const double w = win[min(j, 200)], w2 = j == 100 ? 0.0 : win[j2];
#pragma unroll
        for (int m = 0; m < M; m++) {
            const float* x = &xs[(16 * m + l16) * HOPP];
            const double x0 = x[j], x1 = x[o1], x2 = x[o2], x3 = x[o3];
            const double u = w * (x0 + x1), v = w * (x0 - x1);
            const double u2 = w2 * (j ? x2 + x3 : x2), v2 = w2 * (x2 - x3);  // (sample 200 has no partner)
            acc[0][m] = __builtin_amdgcn_mfma_f64_16x16x4f64(u + u2, b[0], acc[0][m], 0, 0, 0);
            acc[1][m] = __builtin_amdgcn_mfma_f64_16x16x4f64(u - u2, b[1], acc[1][m], 0, 0, 0);
            acc[2][m] = __builtin_amdgcn_mfma_f64_16x16x4f64(v - v2, b[2], acc[2][m], 0, 0, 0);
            acc[3][m] = __builtin_amdgcn_mfma_f64_16x16x4f64(v + v2, b[3], acc[3][m], 0, 0, 0);
        }
    }
    // element r of lane l: frame 4 r + l / 16 of the 16, bin l % 16 of the tile
    const int bin = 16 * wave + l16;
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int f = 16 * m + 4 * r + lq;
            const float e = (float)(acc[0][m][r] * acc[0][m][r] + acc[2][m][r] * acc[2][m][r]);
            const float o = (float)(acc[1][m][r] * acc[1][m][r] + acc[3][m][r] * acc[3][m][r]);
            if (bin <= 100) pw[f][2 * bin] = e;
            if (bin <= 99) pw[f][2 * bin + 1] = o;
            if ((bin <= 100 && !(e < INFINITY)) || (bin <= 99 && !(o < INFINITY))) odd_frame[f] = 1;
        }
    __syncthreads();
    // a filter's bins (meta: first | count << 8 | first weight << 16), in bin order; the bins outside add zeros, but for a
    // power that is not finite, whose zero products are NaN
    const int f = tid % FB, t = t0 + f;
    float mx = -INFINITY;
    if (t < live) {
        const bool odd = odd_frame[f];
        for (int m = tid / FB; m < p.n_mels; m += 64 * NT / FB) {
            const int lo = meta[m] & 255, cnt = (meta[m] >> 8) & 255, off = meta[m] >> 16;
            float a = 0.f;
            if (!odd) {
                for (int k = 0; k < cnt; k++) a = a + wts[off + k] * pw[f][lo + k];
            } else {
                for (int k = 0; k < MZ_MEL_BINS; k++)
                    a = a + (k >= lo && k < lo + cnt ? wts[off + k - lo] : 0.f) * pw[f][k];
            }
            const float v = log10f(fmaxf(a, 1e-10f));
            mx = fmaxf(mx, v);
            p.mel[((long)c * p.n_mels + m) * MZ_NFR_HOST + t] = v;
        }
    }
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < NT; w++) mx = fmaxf(mx, red[w]);
        p.mx[(long)c * MZ_MEL_BLOCKS + blockIdx.x] = mx;
    }
#endif
}

// Bound by its one read and write of the mel (98 MB in all for 32 clips of 128 mels: 17 us; one workgroup per clip took 237).
// V frames per thread (4: 16-byte accesses, for a 16-byte aligned mel; a row is 3000 frames)
template <int V>
__global__ void __launch_bounds__(256) mel_norm_kernel(const MzMel p, int fb) {
    typedef float vec __attribute__((ext_vector_type(V)));
    __shared__ float red[4];
    const int c = blockIdx.y, tid = threadIdx.x, live = live_frames(p.ns[c]), nb = (live + fb - 1) / fb;
    const float v0 = tid < nb ? p.mx[(long)c * MZ_MEL_BLOCKS + tid] : -INFINITY;
    const long i = ((long)blockIdx.x * 256 + tid) * V, total = (long)p.n_mels * MZ_NFR_HOST;
    vec* dst = (vec*)(p.mel + c * total + i);
    vec x = {};
    if (i < total) x = *dst;
    const float wm = wave_max(v0);
    if ((tid & 63) == 0) red[tid >> 6] = wm;
    __syncthreads();
    float mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    if (live < MZ_NFR_HOST) mx = fmaxf(mx, -10.f);
    const float lo = mx - 8.0f;
    if (i >= total) return;
    const int t = (int)(i % MZ_NFR_HOST);
#pragma unroll
    for (int e = 0; e < V; e++) x[e] = (fmaxf(t + e < live ? x[e] : -10.f, lo) + 4.0f) / 4.0f;
    *dst = x;
}

}  // namespace

hipError_t mz_log_mel_launch(hipStream_t s, const MzMel& p, long frames) {
    if (p.n <= 0 || p.n > 65535 || p.n_mels <= 0 || p.n_mels > 256) return hipErrorInvalidValue;
    hipLaunchKernelGGL(mel_basis_kernel, dim3((MZ_MEL_BASIS + 255) / 256), dim3(256), 0, s, p.basis);
    // 16 frames per workgroup until they give every CU two: a workgroup of 16 is done in half the time
    const int fb = frames <= 16L * 2 * mz_cu_count() ? 16 : 32;
    const dim3 grid((MZ_NFR_HOST + fb - 1) / fb, p.n);
    if (fb == 16)
        hipLaunchKernelGGL(mel_spec_kernel<1>, grid, dim3(64 * NT), 0, s, p);
    else
        hipLaunchKernelGGL(mel_spec_kernel<2>, grid, dim3(64 * NT), 0, s, p);
    const long total = (long)p.n_mels * MZ_NFR_HOST;
    if (((uintptr_t)p.mel & 15) == 0)
        hipLaunchKernelGGL(mel_norm_kernel<4>, dim3((total / 4 + 255) / 256, p.n), dim3(256), 0, s, p, fb);
    else
        hipLaunchKernelGGL(mel_norm_kernel<1>, dim3((total + 255) / 256, p.n), dim3(256), 0, s, p, fb);
    return hipGetLastError();
}
