// NeMo log-mel frontend on the GPU (include/ud_mel.h).
//
// The reference computes the features on the CPU (Sources/DictatorCore/Audio/NemoMel.swift:85-107):
// two sgemms of the [T, 400] frame matrix against window-folded cos/sin tables [257, 400], the
// power |X|^2 (as sqrt then square), a third sgemm against the filterbank and log(x + 2^-24).
// Here a workgroup of 4 waves takes 4, 8 or 16 frames of one job; each wave transforms its own frames
// and the workgroup sums the mel bands together:
//
//   frame    the 400 preemphasized, windowed samples, centred in 512 (offset 56), packed as 256
//            complex values z[m] = x[2m] + i x[2m+1]; lane l loads m = l + 64 j, j < 4; the
//            next frame's loads are in flight behind a frame's transform
//   FFT      256 points, four radix-4 passes (decimation in frequency; Cooley and Tukey 1965) on four
//            values per lane, with three exchanges through the wave's own LDS: no barrier
//   split    X[k] of the real signal from Z[k] and Z[256 - k]: X = E - i W512^k O with
//            E, O = (Z[k] +- conj Z[256 - k]) / 2 (O over i)
//   power    |X|^2 into LDS (the reference takes the square root and squares it again)
//   mel      thread (m, frame quad) sums w[m][k] * power[k][t] over the bins from band m's first to its
//            last nonzero weight (the products outside are +0, so the sum is the same as over all 257
//            bins for any finite power), then log.  A band's weights are stored from its first bin on,
//            bin-major (fbw[j][m]), so the threads of a wave read neighbouring words
//
// 8 clips of 15-30 s (18,000 frames): 182 us a launch with the direct form (two 400-term sums per bin
// against a cos table in LDS: 1.6 TFLOP/s of FMAs, where the transform needs a thirtieth of them),
// 34.7 with flat sample loads and one range check per sample, 24.4 now; 24 clips of 19-37 s with their
// call 544 -> 68 (repeated calls: the samples come from the last-level cache; a first call on new samples,
// with the wait for it, 191 -> 54 where a repeated one takes 164 -> 30).  What is left is VALU issue: about
// 300 instructions a frame for the transform and the split, as many for the bands and the logarithm.
//
// Rounding: the reference multiplies x by float(cos) * window (its table entries) and sums 400 terms;
// here x * window goes through the transform's 9 levels, whose rounding error is smaller.  Every frame
// is computed the same way wherever it sits in the grid and however many frames its wave has (fixed
// operation order), so a frame recomputed by a later streaming chunk is bit-identical to its first
// computation.  The preemphasis is evaluated as the reference writes it, a[i] - 0.97 * a[i-1] with
// both roundings (contraction off); the transform and the power may use fused multiply-adds, alike in every
// instantiation.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/ud_mel.h"
#include "kernels.hpp"

int ud_set_error(int code, const char* msg);   // encoder.hip

namespace ud {

constexpr int MEL_WIN = 400;
constexpr int MEL_HOP = 160;
constexpr int MEL_NB = 257;        // rfft bins of n_fft 512
constexpr int MEL_OFF = 56;        // (512 - 400) / 2
constexpr int MEL_THREADS = 256;

__device__ __forceinline__ float preemph(float a, float prev) {
#pragma clang fp contract(off)
    return a - 0.97f * prev;
}

typedef float __attribute__((address_space(1))) gfloat;   // global memory, for a pointer read from memory

struct cpx {
    float x, y;
};
__device__ __forceinline__ cpx operator+(cpx a, cpx b) { return {a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ cpx operator-(cpx a, cpx b) { return {a.x - b.x, a.y - b.y}; }
// a (c - i s): a twiddle factor W = e^(-i angle) held as (cos, sin)
__device__ __forceinline__ cpx twiddle(cpx a, cpx w) { return {a.x * w.x + a.y * w.y, a.y * w.x - a.x * w.y}; }

// (cos, sin) of 2 pi j / 512 from the 512-entry cos table
__device__ __forceinline__ cpx unit512(const float* cos512, int j) {
    return {cos512[j & 511], cos512[(j + 384) & 511]};
}

// z[q] <- sum_j z[j] W4^(j q), then z[q] *= w[q - 1] for q > 0
__device__ __forceinline__ void radix4(cpx (&z)[4], const cpx (&w)[3]) {
    const cpx a = z[0] + z[2], b = z[0] - z[2], c = z[1] + z[3], d = z[1] - z[3];
    z[0] = a + c;
    z[1] = twiddle(cpx{b.x + d.y, b.y - d.x}, w[0]);
    z[2] = twiddle(a - c, w[1]);
    z[3] = twiddle(cpx{b.x - d.y, b.y + d.x}, w[2]);
}

// LDS slot of the transform's value i: the four bits above the low four permute those, so that every
// pass reads and writes at most two lanes per bank
__device__ __forceinline__ int fft_slot(int i) { return i ^ ((i >> 4) & 15); }

// Orders a wave's LDS writes before its LDS reads of them (the wave's LDS operations run in order; this
// keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int FPW>                                  // frames per wave
__global__ __launch_bounds__(MEL_THREADS) void mel_kernel(const MelJob* __restrict__ jobs, MelTables tb) {
    static_assert(FPW == 1 || FPW == 2 || FPW == 4, "frames per wave");
    constexpr int FR = 4 * FPW;                     // frames per workgroup
    constexpr int QPT = FPW == 4 ? 2 : 1;           // frame quads per thread in the band sums
    constexpr int MT = MEL_THREADS / (FPW / QPT);   // threads over the bands
    constexpr int PRE = 8;                          // band weights a thread loads ahead
    __shared__ float4 pw[FR / 4][MEL_NB];
    __shared__ cpx ex[4][256];
    const MelJob J = jobs[blockIdx.y];
    const int j0 = blockIdx.x * FR;
    if (j0 >= J.nf) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nfr = min(FR, J.nf - j0);
    const long long fbase = J.f0 + j0;

    // ---- the samples at 2m - 1, 2m, 2m + 1 of frame t's 512 (m = lane + 64 j).  Sample s of the frame
    //      is clip sample base + s, base = 160 f - 256; a buffer over the part of the frame that the
    //      clip (and the window's end) covers returns zeros for the rest.  (Buffer loads also count as
    //      vector memory alone: flat ones, which these pointers would otherwise give, make every wait
    //      for an LDS exchange wait for the next frame's samples too.)
    struct Samples {
        float v[4][3];
        int end;                                    // the clip covers s < end
        bool live;
    };
    auto load = [&](int t) __attribute__((always_inline)) {
        Samples r;
        const long long f = fbase + t, base = f * MEL_HOP - 256;
        r.live = t < nfr && f < J.zero_from;
        const int first = (int)min(max(J.first - base, 0ll), 1024ll);
        r.end = r.live ? (int)min(max(J.n_audio - base, 0ll), 1024ll) : 0;
        const int records = max(min(r.end, MEL_OFF + MEL_WIN) - first, 0);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(J.src + (base + first - J.first)), 0, records * 4, 0x00020000);
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int e = 0; e < 3; e++) {
                // negative before the clip: beyond the buffer as an unsigned offset, if all of it is in
                // the address register (the empty asm keeps an immediate from being split off, whose
                // sum the range check would not wrap)
                int off = (2 * (lane + 64 * j) - 1 + e - first) * 4;
                asm volatile("" : "+v"(off));
                r.v[j][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
            }
        return r;
    };
    Samples cur = load(wave * FPW);

    // ---- window weights; twiddle factors (of pass p, W_(4^(4 - p))^((lane's low index) q)); the
    //      thread's band and its first weights
    float wv[4][2];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = 2 * (lane + 64 * j) - MEL_OFF;
        const bool in = i >= 0 && i < MEL_WIN;      // (the window's length is even)
        wv[j][0] = in ? tb.win[i] : 0.0f;
        wv[j][1] = in ? tb.win[i + 1] : 0.0f;
    }
    cpx w1[3], w2[3], w3[3], ws[4];
#pragma unroll
    for (int q = 1; q < 4; q++) {
        w1[q - 1] = unit512(tb.cos512, 2 * lane * q);
        w2[q - 1] = unit512(tb.cos512, 8 * (lane & 15) * q);
        w3[q - 1] = unit512(tb.cos512, 32 * (lane & 3) * q);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) ws[j] = unit512(tb.cos512, lane + 64 * j);
    const int band = tid % MT;
    int2 kr = band < tb.n_mels ? tb.krange[band] : make_int2(0, 0);
    float pre[PRE];
#pragma unroll
    for (int j = 0; j < PRE; j++) pre[j] = kr.x + j < kr.y ? tb.fbw[j * tb.n_mels + band] : 0.0f;

    cpx* x = ex[wave];
#pragma unroll
    for (int u = 0; u < FPW; u++) {
        const int t = wave * FPW + u;
        float* pt = reinterpret_cast<float*>(pw[t / 4]) + t % 4;     // power of bin k at pt[4 k]
        const Samples c = cur;
        if (u + 1 < FPW) cur = load(t + 1);         // in flight behind this frame
        if (!c.live) {                              // wave-uniform: a frame of zeros, or none
#pragma unroll
            for (int j = 0; j < 4; j++) pt[4 * (lane + 64 * j)] = 0.0f;
            if (lane == 0) pt[4 * 256] = 0.0f;
            continue;
        }
        cpx z[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            // (the clip's first sample is its own preemphasis: the one before it loads as 0)
            z[j].x = preemph(c.v[j][1], c.v[j][0]) * wv[j][0];
            z[j].y = preemph(c.v[j][2], c.v[j][1]) * wv[j][1];
        }
        if (lane < MEL_OFF / 2) z[0] = cpx{0.0f, 0.0f};              // outside the window
        if (lane >= (MEL_OFF + MEL_WIN) / 2 - 192) z[3] = cpx{0.0f, 0.0f};
        if (c.end < MEL_OFF + MEL_WIN) {            // wave-uniform: samples past the clip are zero padding
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int s = 2 * (lane + 64 * j);
                if (s >= c.end) z[j].x = 0.0f;
                if (s + 1 >= c.end) z[j].y = 0.0f;
            }
        }
        // values of m = lane + 64 j -> digits q1 (stride 64 of the exchange), then q2, q3, q4
        radix4(z, w1);
#pragma unroll
        for (int q = 0; q < 4; q++) x[fft_slot(64 * q + lane)] = z[q];
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; j++) z[j] = x[fft_slot((lane & 48) * 4 + (lane & 15) + 16 * j)];
        wave_lds_fence();
        radix4(z, w2);
#pragma unroll
        for (int q = 0; q < 4; q++) x[fft_slot((lane & 48) * 4 + 16 * q + (lane & 15))] = z[q];
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; j++) z[j] = x[fft_slot((lane & 60) * 4 + (lane & 3) + 4 * j)];
        wave_lds_fence();
        radix4(z, w3);
#pragma unroll
        for (int q = 0; q < 4; q++) x[fft_slot((lane & 60) * 4 + 4 * q + (lane & 3))] = z[q];
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; j++) z[j] = x[fft_slot(4 * lane + j)];
        wave_lds_fence();
        {
            const cpx a = z[0] + z[2], b = z[0] - z[2], d = z[1] + z[3], e = z[1] - z[3];
            z[0] = a + d;
            z[1] = cpx{b.x + e.y, b.y - e.x};
            z[2] = a - d;
            z[3] = cpx{b.x - e.y, b.y + e.x};
        }
        // lane = 16 q1 + 4 q2 + q3 holds Z[q1 + 4 q2 + 16 q3 + 64 q4]
        const int k0 = (lane >> 4) + (lane & 12) + 16 * (lane & 3);
#pragma unroll
        for (int q = 0; q < 4; q++) x[fft_slot(k0 + 64 * q)] = z[q];
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int k = lane + 64 * j;
            const cpx a = x[fft_slot(k)], b = x[fft_slot((256 - k) & 255)];
            const cpx o = twiddle(cpx{0.5f * (a.x - b.x), 0.5f * (a.y + b.y)}, ws[j]);
            const float re = 0.5f * (a.x + b.x) + o.y, im = 0.5f * (a.y - b.y) - o.x;
            pt[4 * k] = re * re + im * im;
            if (k == 0) pt[4 * 256] = (a.x - a.y) * (a.x - a.y);
        }
        wave_lds_fence();                           // the next frame's exchanges reuse x
    }
    __syncthreads();

    const int quad = tid / MT * QPT;                // frames 4 quad .. 4 (quad + QPT) - 1
    gfloat* dst = (gfloat*)J.dst;
    for (int m = band; m < tb.n_mels; m += MT) {
        if (m != band) kr = tb.krange[m];
        const float* w = tb.fbw + m;
        float acc[QPT][4] = {};
        auto add = [&](float fw, int k) __attribute__((always_inline)) {
#pragma unroll
            for (int h = 0; h < QPT; h++) {
                const float4 p = pw[quad + h][k];
                acc[h][0] = fmaf(fw, p.x, acc[h][0]);
                acc[h][1] = fmaf(fw, p.y, acc[h][1]);
                acc[h][2] = fmaf(fw, p.z, acc[h][2]);
                acc[h][3] = fmaf(fw, p.w, acc[h][3]);
            }
        };
        int k = kr.x;
        if (m == band) {
#pragma unroll
            for (int j = 0; j < PRE; j++)
                if (kr.x + j < kr.y) add(pre[j], kr.x + j);
            k += PRE;
        }
#pragma unroll 4
        for (; k < kr.y; k++) add(w[(k - kr.x) * tb.n_mels], k);
#pragma unroll
        for (int i = 0; i < 4 * QPT; i++) {
            const int t = 4 * quad + i;
            if (t < nfr)
                dst[(long long)(j0 + t) * tb.n_mels + m] =
                    fbase + t < J.zero_from ? logf(acc[i / 4][i % 4] + 5.9604644775390625e-8f) : 0.0f;
        }
    }
}

int launch_mel(const MelTables& t, const MelJob* jobs_dev, int n_jobs, int max_nf, hipStream_t st) {
    if (n_jobs < 1 || max_nf < 1) return 0;
    if (t.n_mels < 1 || t.n_mels > 256 || n_jobs > 65535) return -2;
    // The frames of a wave share its twiddle factors, its thread's band and the launch, and their loads
    // run behind each other's transforms; with fewer than two workgroups per CU, fewer frames per wave
    // fill more of the chip.
    auto blocks = [&](int fr) { return (max_nf + fr - 1) / fr; };
    if (blocks(16) * n_jobs >= 512) mel_kernel<4><<<dim3(blocks(16), n_jobs), MEL_THREADS, 0, st>>>(jobs_dev, t);
    else if (blocks(8) * n_jobs >= 512) mel_kernel<2><<<dim3(blocks(8), n_jobs), MEL_THREADS, 0, st>>>(jobs_dev, t);
    else mel_kernel<1><<<dim3(blocks(4), n_jobs), MEL_THREADS, 0, st>>>(jobs_dev, t);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ud

using namespace ud;

static int mfail(int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    return ud_set_error(code, buf);
}

constexpr int MEL_RING = 4;   // job lists of ud_mel_features in flight before a call waits

struct ud_mel {
    int n_mels = 0;
    float *cos512 = nullptr, *win = nullptr, *fbw = nullptr;
    int2* krange = nullptr;
    // ring of job lists for ud_mel_features: slot i's pinned staging is rewritten only after the
    // kernel that read slot i's device copy has finished (its event)
    MelJob* djobs[MEL_RING] = {};
    MelJob* hjobs[MEL_RING] = {};
    hipEvent_t done[MEL_RING] = {};
    int cap_jobs = 0, next = 0;
};

namespace ud {
MelTables mel_tables_of(const ::ud_mel* m) { return MelTables{m->cos512, m->win, m->krange, m->fbw, m->n_mels}; }
}  // namespace ud

static void free_mel(ud_mel* m) {
    if (!m) return;
    (void)hipDeviceSynchronize();
    for (void* p : {(void*)m->cos512, (void*)m->win, (void*)m->fbw, (void*)m->krange}) if (p) (void)hipFree(p);
    for (int i = 0; i < MEL_RING; i++) {
        if (m->djobs[i]) (void)hipFree(m->djobs[i]);
        if (m->hjobs[i]) (void)hipHostFree(m->hjobs[i]);
        if (m->done[i]) (void)hipEventDestroy(m->done[i]);
    }
    delete m;
}

extern "C" UD_API int ud_mel_create(const float* fb_host, int32_t n_mels, const float* window_host, ud_mel** out) {
    if (!out || !fb_host || !window_host) return mfail(UD_ERR_INVALID, "ud_mel_create: null argument");
    *out = nullptr;
    if (n_mels < 1 || n_mels > 256) return mfail(UD_ERR_SHAPE, "ud_mel_create: n_mels %d outside 1..256", n_mels);
    // cos(2 pi j / 512) in double, rounded to float (the reference's float(cos(phase)),
    // NemoMel.swift:33-35), the window as given, each band's filterbank weights from its first
    // nonzero bin on, bin-major [widest band][n_mels]
    std::vector<float> cs(512);
    for (int j = 0; j < 512; j++) cs[j] = (float)cos(2.0 * 3.14159265358979323846 * (double)j / 512.0);
    std::vector<int2> kr(n_mels);
    int width = 1;
    for (int m = 0; m < n_mels; m++) {
        int lo = MEL_NB, hi = 0;
        for (int k = 0; k < MEL_NB; k++)
            if (fb_host[(size_t)m * MEL_NB + k] != 0.0f) { lo = std::min(lo, k); hi = k + 1; }
        kr[m] = make_int2(lo < hi ? lo : 0, hi);
        width = std::max(width, kr[m].y - kr[m].x);
    }
    std::vector<float> fbw((size_t)width * n_mels);
    for (int m = 0; m < n_mels; m++)
        for (int k = kr[m].x; k < kr[m].y; k++) fbw[(size_t)(k - kr[m].x) * n_mels + m] = fb_host[(size_t)m * MEL_NB + k];
    ud_mel* m = new ud_mel();
    m->n_mels = n_mels;
    bool ok = hipMalloc(&m->cos512, 512 * 4) == hipSuccess && hipMalloc(&m->win, MEL_WIN * 4) == hipSuccess &&
              hipMalloc(&m->fbw, fbw.size() * 4) == hipSuccess && hipMalloc(&m->krange, n_mels * sizeof(int2)) == hipSuccess;
    for (int i = 0; ok && i < MEL_RING; i++) ok = hipEventCreateWithFlags(&m->done[i], hipEventDisableTiming) == hipSuccess;
    ok = ok && hipMemcpy(m->cos512, cs.data(), 512 * 4, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(m->win, window_host, MEL_WIN * 4, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(m->fbw, fbw.data(), fbw.size() * 4, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(m->krange, kr.data(), n_mels * sizeof(int2), hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) {
        free_mel(m);
        return mfail(UD_ERR_NOMEM, "ud_mel_create: device allocation or upload failed");
    }
    *out = m;
    return UD_OK;
}

extern "C" UD_API void ud_mel_destroy(ud_mel* m) { free_mel(m); }

extern "C" UD_API int32_t ud_mel_bins(const ud_mel* m) { return m ? m->n_mels : 0; }

extern "C" UD_API int ud_mel_features(ud_mel* m, int32_t n, const float* audio_dev, int64_t audio_stride,
                                      const int64_t* n_samples_host, float* out_dev, int32_t out_rows,
                                      int32_t* frames_host, void* hip_stream) {
    if (!m || !audio_dev || !n_samples_host || !out_dev) return mfail(UD_ERR_INVALID, "ud_mel_features: null argument");
    if (n < 1 || n > 65535) return mfail(UD_ERR_SHAPE, "ud_mel_features: n = %d outside 1..65535", n);
    int max_nf = 0;
    for (int b = 0; b < n; b++) {
        const int64_t ns = n_samples_host[b];
        if (ns < 0 || ns > audio_stride)
            return mfail(UD_ERR_SHAPE, "ud_mel_features: clip %d has %lld samples (stride %lld)", b, (long long)ns,
                         (long long)audio_stride);
        const int64_t T = ns / MEL_HOP + 1;
        if (T > out_rows) return mfail(UD_ERR_SHAPE, "ud_mel_features: clip %d needs %lld rows > out_rows %d", b, (long long)T, out_rows);
        if (T > max_nf) max_nf = (int)T;
    }
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    if (n > m->cap_jobs) {
        for (int i = 0; i < MEL_RING; i++) {
            (void)hipEventSynchronize(m->done[i]);
            if (m->djobs[i]) (void)hipFree(m->djobs[i]);
            if (m->hjobs[i]) (void)hipHostFree(m->hjobs[i]);
            m->djobs[i] = nullptr;
            m->hjobs[i] = nullptr;
        }
        m->cap_jobs = 0;
        for (int i = 0; i < MEL_RING; i++)
            if (hipMalloc(&m->djobs[i], (size_t)n * sizeof(MelJob)) != hipSuccess ||
                hipHostMalloc((void**)&m->hjobs[i], (size_t)n * sizeof(MelJob)) != hipSuccess)
                return mfail(UD_ERR_NOMEM, "ud_mel_features: job list allocation failed");
        m->cap_jobs = n;
    }
    const int slot = m->next;
    m->next = (m->next + 1) % MEL_RING;
    if (hipEventSynchronize(m->done[slot]) != hipSuccess) return mfail(UD_ERR_HIP, "ud_mel_features: event wait failed");
    MelJob* hj = m->hjobs[slot];
    for (int b = 0; b < n; b++) {
        const int64_t ns = n_samples_host[b];
        MelJob& j = hj[b];
        j.src = audio_dev + (int64_t)b * audio_stride;
        j.dst = out_dev + (int64_t)b * out_rows * m->n_mels;
        j.first = 0;
        j.n_audio = ns;
        j.f0 = 0;
        j.nf = (int)(ns / MEL_HOP + 1);
        j.zero_from = ns / MEL_HOP;
        j.pad_ = 0;
        if (frames_host) frames_host[b] = j.nf;
    }
    if (hipMemcpyAsync(m->djobs[slot], hj, (size_t)n * sizeof(MelJob), hipMemcpyHostToDevice, st) != hipSuccess)
        return mfail(UD_ERR_HIP, "ud_mel_features: job upload failed");
    const int rc = launch_mel(mel_tables_of(m), m->djobs[slot], n, max_nf, st);
    if (rc != 0) return mfail(rc == -2 ? UD_ERR_SHAPE : UD_ERR_HIP, "ud_mel_features: launch failed");
    if (hipEventRecord(m->done[slot], st) != hipSuccess) return mfail(UD_ERR_HIP, "ud_mel_features: event record failed");
    return UD_OK;
}
