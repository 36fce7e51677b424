// Kokoro's harmonic-plus-noise source and its short-time spectrum for gfx950
// (kokoro/source.cpp:60-184, build_harmonic_source; the host runs it between
// the prosody and generator graphs). Three launches on one stream:
//
//   k_source_phase (one block): the phase increments frac(f0 * (h+1) / rate) of
//     the upsampled grid, resampled linearly to the f0 grid (PyTorch's
//     align_corners=false mapping, in double, the weight rounded to f32), into
//     LDS, a harmonic's frames in a row; each harmonic's running f32 sum in
//     frame order -- one lane per harmonic, the order the host code adds in, so
//     the sums are bit for bit its own; and the phase running * 2 pi * scale
//     (double, rounded), staged in the spectrum output's own memory until the
//     excitation launch has read it;
//   k_source_excite (a lane per upsampled sample): the phase resampled back,
//     sin(phase) * amp for voiced samples plus the noise at its gain, merged
//     with the weights in harmonic order from the bias, tanh;
//   k_source_stft (blocks of whole frames): torch.stft's centred framing --
//     reflect padding by n_fft/2, the periodic Hann window rounded to f32 --
//     each windowed sample formed once into LDS, then a lane per frame and bin
//     for the DFT in double with the host code's twiddles (the angle
//     -2 pi b k / n_fft as it computes it), the magnitude by hypot and the phase
//     by atan2, each rounded to f32.
// The f32 sine and tanh are the device's, within an ulp or two of the host
// library's; everything else is the host code's arithmetic in its order.
//
// Latency-bound: 5 seconds of speech are 400 serial sums, 120,000 samples and
// 24,001 frames. Measured on MI355X at Kokoro's 9 harmonics, x300, n_fft 20, hop
// 5: 1 second 16.2 -> 13.8 us, 5 seconds 28.4 -> 20.3, 20 seconds 76.6 -> 52.8, against
// four launches with the increments in one of their own, the sums read one value
// at a time and the twiddles of a 256-lane block made for 23 frames.

#include <cmath>

#include "shp_internal.hpp"

namespace shp {
namespace {

constexpr double kSrcPi       = 3.14159265358979323846;
constexpr int    kSrcMaxH     = 64;    // harmonics
constexpr int    kSrcMaxNfft  = 64;    // window (the twiddle table holds (n_fft/2 + 1) x n_fft entries)
constexpr int    kSrcChunk    = 8192;  // coarse values per LDS chunk

struct SourceArgs {
    const float * f0;
    const float * mw;     // merge weights
    const float * ri;     // initial phases
    const float * noise;  // [U][H]
    float *       exc;    // [U]
    float *       har;    // [frames][2*bins]; first L*H floats stage the phase
    int64_t       L;
    int64_t       U;
    int64_t       frames;
    float         bias;
    float         amp;
    float         noise_std;
    float         threshold;
    float         rate;
    int32_t       H;
    int32_t       scale;
    int32_t       nfft;
    int32_t       hop;
    int32_t       bins;
    int32_t       fpb;    // frames per spectrum block
    int32_t       pad;
    FastDiv       fH;
    FastDiv       fscale;
    FastDiv       fnfft;
    FastDiv       fbins;
};

// The increment of harmonic h at a sample of frequency f0 (the initial phase
// apart).
__device__ __forceinline__ float increment(float f0, int h, float rate) {
    const float v = f0 * static_cast<float>(h + 1) / rate;
    return v - floorf(v);
}

// LDS floats per harmonic of a phase chunk: whole kSrcAhead runs of frames and
// four of padding, kSrcChunk values in all at most.
__host__ __device__ __forceinline__ int source_stride(int H) {
    return kSrcChunk / H / 16 * 16 + 4;
}

// PyTorch's align_corners=false source position for output o, clamped at 0:
// its lower index, upper index and f32 weight.
__device__ __forceinline__ void linear_at(int64_t o, double ratio, int64_t in_len, int64_t & lo, int64_t & hi,
                                          float & w) {
    double position = (static_cast<double>(o) + 0.5) * ratio - 0.5;
    position        = position < 0.0 ? 0.0 : position;
    lo              = static_cast<int64_t>(position);
    hi              = lo + 1 < in_len ? lo + 1 : in_len - 1;
    w               = static_cast<float>(position - static_cast<double>(lo));
}

// The increments, their running sums (one lane per harmonic in frame order) and
// the phases, over LDS chunks of whole frames. A harmonic's frames lie in a row
// of LDS, so its lane reads and writes four at a time, 16 ahead of their adds.
constexpr int kSrcPhaseBlock = 1024;
constexpr int kSrcAhead      = 16;

__global__ __launch_bounds__(kSrcPhaseBlock) void k_source_phase(const SourceArgs a) {
    extern __shared__ f32x4 s_run4[];  // [H][stride]
    float *       s_run  = reinterpret_cast<float *>(s_run4);
    const int     tid    = static_cast<int>(threadIdx.x);
    const int     H      = a.H;
    const int     stride = source_stride(H);
    const int     chunk  = stride - 4;  // frames per chunk, a multiple of kSrcAhead
    float         run    = 0.0f;        // lane h < H: harmonic h's running sum
    for (int64_t j0 = 0; j0 < a.L; j0 += chunk) {
        const int nj = static_cast<int>(a.L - j0 < chunk ? a.L - j0 : chunk);
        const int up = (nj + kSrcAhead - 1) / kSrcAhead * kSrcAhead;  // zeros past the last frame: x + 0 is x
        // a lane per frame, whose position and f0 serve all its harmonics: the
        // one block's lanes are few, and the increments' arithmetic is not
        for (int j = tid; j < up; j += kSrcPhaseBlock) {
            int64_t lo = 0, hi = 0;
            float   w = 0.0f, flo = 0.0f, fhi = 0.0f;
            if (j < nj) {
                linear_at(j0 + j, static_cast<double>(a.U) / static_cast<double>(a.L), a.U, lo, hi, w);
                flo = a.f0[fastdiv(static_cast<uint32_t>(lo), a.fscale)];
                fhi = a.f0[fastdiv(static_cast<uint32_t>(hi), a.fscale)];
            }
            const bool apart = j < nj && (lo == 0 || __float_as_uint(flo) != __float_as_uint(fhi));
            for (int h = 0; h < H; ++h) {
                float r0 = increment(flo, h, a.rate), r1 = r0;
                if (apart) {
                    r1 = increment(fhi, h, a.rate);
                    r0 = lo == 0 ? r0 + a.ri[h] : r0;
                    r1 = hi == 0 ? r1 + a.ri[h] : r1;
                }
                s_run[h * stride + j] = j < nj ? r0 * (1.0f - w) + r1 * w : 0.0f;
            }
        }
        __syncthreads();
        if (tid < H) {
            f32x4 * row = reinterpret_cast<f32x4 *>(s_run + tid * stride);
            f32x4   next[kSrcAhead / 4];
#pragma unroll
            for (int q = 0; q < kSrcAhead / 4; ++q) {
                next[q] = row[q];
            }
            for (int j = 0; j < up; j += kSrcAhead) {
                f32x4 v[kSrcAhead / 4];
#pragma unroll
                for (int q = 0; q < kSrcAhead / 4; ++q) {
                    v[q]    = next[q];
                    next[q] = row[(j + kSrcAhead < up ? j + kSrcAhead : j) / 4 + q];
                }
#pragma unroll
                for (int q = 0; q < kSrcAhead / 4; ++q) {
                    v[q].x = run + v[q].x;
                    v[q].y = v[q].x + v[q].y;
                    v[q].z = v[q].y + v[q].z;
                    v[q].w = v[q].z + v[q].w;
                    run    = v[q].w;
                }
#pragma unroll
                for (int q = 0; q < kSrcAhead / 4; ++q) {
                    row[j / 4 + q] = v[q];
                }
            }
        }
        __syncthreads();
        for (int t = tid; t < nj * H; t += kSrcPhaseBlock) {
            const int j       = static_cast<int>(fastdiv(static_cast<uint32_t>(t), a.fH));
            const int h       = t - j * H;
            a.har[j0 * H + t] = static_cast<float>(static_cast<double>(s_run[h * stride + j]) * 2.0 * kSrcPi *
                                                   static_cast<double>(a.scale));
        }
        __syncthreads();
    }
}

// Harmonics whose loads go out before the first one's sine.
constexpr int kSrcBatch = 5;

__global__ __launch_bounds__(256) void k_source_excite(const SourceArgs a) {
    const int64_t u = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (u >= a.U) {
        return;
    }
    int64_t lo, hi;
    float   w;
    linear_at(u, static_cast<double>(a.L) / static_cast<double>(a.U), a.L, lo, hi, w);
    const float   f0u    = a.f0[fastdiv(static_cast<uint32_t>(u), a.fscale)];
    const float   uv     = f0u > a.threshold ? 1.0f : 0.0f;
    const float   gain   = uv * a.noise_std + (1.0f - uv) * a.amp / 3.0f;
    const float * plo    = a.har + lo * a.H;
    const float * phi    = a.har + hi * a.H;
    const float * nz     = a.noise + u * a.H;
    float         merged = a.bias;
    for (int h0 = 0; h0 < a.H; h0 += kSrcBatch) {
        float p0[kSrcBatch], p1[kSrcBatch], n[kSrcBatch], mw[kSrcBatch];
#pragma unroll
        for (int q = 0; q < kSrcBatch; ++q) {
            const int h = h0 + q < a.H ? h0 + q : a.H - 1;
            p0[q]       = plo[h];
            p1[q]       = phi[h];
            n[q]        = nz[h];
            mw[q]       = a.mw[h];
        }
#pragma unroll
        for (int q = 0; q < kSrcBatch; ++q) {
            if (h0 + q < a.H) {
                const float fine  = p0[q] * (1.0f - w) + p1[q] * w;
                const float sine  = sinf(fine) * a.amp;
                const float value = sine * uv + gain * n[q];
                merged            = merged + mw[q] * value;
            }
        }
    }
    a.exc[u] = tanhf(merged);
}

// Frames per spectrum block: an item (frame, bin) per lane. (256 lanes with two
// items each: the f64 hypot and atan2 chains then run one after the other.)
constexpr int kSrcStftBlock = 512;

__global__ __launch_bounds__(kSrcStftBlock) void k_source_stft(const SourceArgs a) {
    extern __shared__ double2 s_tw[];  // [nfft][bins] twiddles, then [fpb][nfft] windowed samples, then the window
    float *       s_seg = reinterpret_cast<float *>(s_tw + a.bins * a.nfft);
    float *       s_win = s_seg + a.fpb * a.nfft;
    const int     tid   = static_cast<int>(threadIdx.x);
    const int64_t f0    = static_cast<int64_t>(blockIdx.x) * a.fpb;
    const int     nf    = static_cast<int>(a.frames - f0 < a.fpb ? a.frames - f0 : a.fpb);
    const int     half  = a.nfft / 2;
    const int64_t last  = a.U - 1;
    for (int i = tid; i < nf * a.nfft; i += kSrcStftBlock) {
        const int f   = static_cast<int>(fastdiv(static_cast<uint32_t>(i), a.fnfft));
        int64_t   src = (f0 + f) * a.hop + (i - f * a.nfft) - half;
        while (src < 0 || src > last) {  // reflection without repeating the edge sample
            src = src < 0 ? -src : 2 * last - src;
        }
        s_seg[i] = a.exc[src];
    }
    for (int i = tid; i < (a.bins + 1) * a.nfft; i += kSrcStftBlock) {
        const int k = static_cast<int>(fastdiv(static_cast<uint32_t>(i), a.fbins));  // by bins, one past the twiddles' rows
        if (i < a.bins * a.nfft) {
            const int    b     = i - k * a.bins;
            const double angle = -2.0 * kSrcPi * static_cast<double>(b) * static_cast<double>(k) / static_cast<double>(a.nfft);
            double       sn, cs;
            sincos(angle, &sn, &cs);
            s_tw[i] = double2{ cs, sn };
        } else {
            const int j = i - a.bins * a.nfft;
            s_win[j] = static_cast<float>(0.5 * (1.0 - cos(2.0 * kSrcPi * static_cast<double>(j) / static_cast<double>(a.nfft))));
        }
    }
    __syncthreads();
    for (int i = tid; i < nf * a.bins; i += kSrcStftBlock) {
        const int     f   = static_cast<int>(fastdiv(static_cast<uint32_t>(i), a.fbins));
        const int     b   = i - f * a.bins;
        const float * x   = s_seg + f * a.nfft;
        double        re = 0.0, im = 0.0;
#pragma unroll 4
        for (int k = 0; k < a.nfft; ++k) {
            const float   seg = x[k] * s_win[k];
            const double2 t   = s_tw[k * a.bins + b];
            re += static_cast<double>(seg) * t.x;
            im += static_cast<double>(seg) * t.y;
        }
        float * row     = a.har + (f0 + f) * 2 * a.bins;
        row[b]          = static_cast<float>(hypot(re, im));
        row[a.bins + b] = static_cast<float>(atan2(im, re));
    }
}

bool contiguous_f32(const shp_tensor * t) {
    return well_formed(t) && t->type == SHP_TYPE_F32 && contiguous(*t) && reinterpret_cast<uintptr_t>(t->data) % 4 == 0;
}

}  // namespace
}  // namespace shp

using namespace shp;

extern "C" shp_status_t shp_harmonic_source(const shp_tensor * f0,
                                            const shp_tensor * merge_weight,
                                            float              merge_bias,
                                            const shp_tensor * rand_ini,
                                            const shp_tensor * noise,
                                            int32_t            sampling_rate,
                                            int32_t            upsample_scale,
                                            float              sine_amp,
                                            float              noise_std,
                                            float              voiced_threshold,
                                            int32_t            n_fft,
                                            int32_t            hop,
                                            shp_tensor *       excitation,
                                            shp_tensor *       har,
                                            shp_stream_t       stream) {
    if (!contiguous_f32(f0) || !contiguous_f32(merge_weight) || !contiguous_f32(rand_ini) || !contiguous_f32(noise) ||
        !contiguous_f32(excitation) || !contiguous_f32(har)) {
        return SHP_ERR_INVALID_ARG;
    }
    const int64_t L = nelements(*f0), H = nelements(*merge_weight);
    if (sampling_rate < 1 || upsample_scale < 1 || n_fft < 2 || n_fft % 2 != 0 || hop < 1 || nelements(*rand_ini) != H) {
        return SHP_ERR_INVALID_ARG;
    }
    const int64_t U = L * upsample_scale, bins = n_fft / 2 + 1, frames = U / hop + 1;
    // one sample cannot be reflect-padded (the host code's reflection loop
    // would not end)
    if (U < 2 || noise->ne[0] != H || nelements(*noise) != U * H || nelements(*excitation) != U || har->ne[0] != 2 * bins ||
        nelements(*har) != frames * 2 * bins) {
        return SHP_ERR_INVALID_ARG;
    }
    // the kernel limits; the spectrum's memory stages the L*H coarse phases
    if (H > kSrcMaxH || n_fft > kSrcMaxNfft || L * H > frames * 2 * bins || U > INT32_MAX ||
        frames * bins > INT32_MAX) {
        return SHP_ERR_UNSUPPORTED;
    }
    const shp_tensor * ins[] = { f0, merge_weight, rand_ini, noise };
    for (const shp_tensor * t : ins) {
        if (spans_overlap(*t, *excitation) || spans_overlap(*t, *har)) {
            return SHP_ERR_UNSUPPORTED;
        }
    }
    if (spans_overlap(*excitation, *har)) {
        return SHP_ERR_UNSUPPORTED;
    }
    if (dry_run()) {
        return SHP_OK;
    }
    SourceArgs a{};
    a.f0        = static_cast<const float *>(f0->data);
    a.mw        = static_cast<const float *>(merge_weight->data);
    a.ri        = static_cast<const float *>(rand_ini->data);
    a.noise     = static_cast<const float *>(noise->data);
    a.exc       = static_cast<float *>(excitation->data);
    a.har       = static_cast<float *>(har->data);
    a.L         = L;
    a.U         = U;
    a.frames    = frames;
    a.bias      = merge_bias;
    a.amp       = sine_amp;
    a.noise_std = noise_std;
    a.threshold = voiced_threshold;
    a.rate      = static_cast<float>(sampling_rate);
    a.H         = static_cast<int32_t>(H);
    a.scale     = upsample_scale;
    a.nfft      = n_fft;
    a.hop       = hop;
    a.bins      = static_cast<int32_t>(bins);
    a.fpb       = static_cast<int32_t>(kSrcStftBlock / bins);
    a.fH        = make_fastdiv(static_cast<uint32_t>(H));
    a.fscale    = make_fastdiv(static_cast<uint32_t>(upsample_scale));
    a.fnfft     = make_fastdiv(static_cast<uint32_t>(n_fft));
    a.fbins     = make_fastdiv(static_cast<uint32_t>(bins));
    const hipStream_t st = as_stream(stream);
    hipLaunchKernelGGL(k_source_phase, dim3(1), dim3(kSrcPhaseBlock),
                       static_cast<size_t>(H * source_stride(static_cast<int>(H))) * sizeof(float), st, a);
    shp_status_t s = launch_status();
    if (s != SHP_OK) {
        return s;
    }
    hipLaunchKernelGGL(k_source_excite, dim3(static_cast<unsigned>((U + 255) / 256)), dim3(256), 0, st, a);
    s = launch_status();
    if (s != SHP_OK) {
        return s;
    }
    const size_t lds = static_cast<size_t>(bins * n_fft) * sizeof(double2) + static_cast<size_t>((a.fpb + 1) * n_fft) * sizeof(float);
    hipLaunchKernelGGL(k_source_stft, dim3(static_cast<unsigned>((frames + a.fpb - 1) / a.fpb)), dim3(kSrcStftBlock), lds, st, a);
    return launch_status();
}
