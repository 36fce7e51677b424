// The Qwen3-TTS speaker encoder's log-mel front end for gfx950
// (qwen3-tts/mel.cpp:63-299, compute_log_mel; the reference runs it on the
// host before the ECAPA graph): PCM to [mel_bins, frames] log energies.
//
// The arithmetic is the host code's, stage for stage: the frame's reflect-
// padded samples times the periodic Hann window, an in-place radix-2 transform
// whose butterflies multiply and add in double and round their two results to
// f32 per stage, the amplitudes sqrt(re^2 + im^2 + 1e-9) (double, rounded),
// and per mel bin the filterbank-weighted sum in double in frequency order and
// log(max(energy, 1e-5)). It differs from the host code's in these: one of a
// butterfly's two products is fused with their sum (a rounding of the double
// fewer; the two apart: 4-10 % of the time), and the device's double cos, sin,
// sqrt and log replace the host library's; sqrt is correctly rounded on both.
// Every form below gives a frame the same bits.
//
// A block has 1, 2 or 4 transform waves and kMelScan more:
//   - a transform wave runs whole frames (one at n_fft 1024, more of a shorter
//     transform, so that every lane has work): every lane loads 16 samples at
//     their bit-reversed places straight from memory, runs four stages on them
//     in registers, and two more register passes (four and two stages at n_fft
//     1024) exchange through LDS within the wave, with no barrier;
//   - meanwhile the other waves read the filterbank once for the block's
//     frames and note which float4 of each mel bin's weights are not all zero: a
//     Slaney filter covers a few of the 513 frequencies (1,000 nonzero weights
//     of 65,664), and a zero weight adds nothing to a sum of finite amplitudes;
//   - after a barrier every thread forms amplitudes, and after another a lane
//     per (bin, frame) sums its bin's span in frequency order. A frame with an
//     amplitude that is not finite sums every frequency, since 0 * inf is NaN
//     in the host code's sum.
// Bound by one block's latency at a clip's few hundred blocks (one a CU): of
// its 25,000 cycles the transform takes 12,500 (5,120 f64 butterflies a wave),
// the filterbank read beside it 13,000, the amplitudes 2,800, the mel sums and
// logs 4,200. Measured on MI355X at the production parameters: a 10-second clip
// (937 frames) 52.1 -> 12.2 us, one second 40.4 -> 10.9, 20 seconds 93.7 -> 23.0
// (n_fft 512, hop 160, 80 bins, 10 s: 24.9 -> 11.7; n_fft 2048, hop 512: 54.1 ->
// 32.2), against a 256-thread block per frame with a barrier per stage, n_fft - 1
// twiddles evaluated per block and every lane reading a whole filterbank row.
// Slower here: the stages' roundings on the bits of the double instead of by
// conversion (20.4 us), the span of each filter by LDS minima (16-20 us: lanes of
// one row meet on one address), and straight-line code beyond a few KB anywhere,
// since every launch fetches it afresh.
//
// shp_mel_filterbank is the Slaney filterbank the transform is weighted with
// (mel.cpp:96-170), computed on the host once per model.

#include <cmath>
#include <vector>

#include "shp_internal.hpp"

namespace shp {
namespace {

constexpr double kMelPi      = 3.14159265358979323846;
constexpr int    kMelMaxNfft = 2048;

constexpr int    kMelWaves   = 4;    // transform waves per block (one at n_fft 2048: 64 KB of LDS)
constexpr int    kMelScan    = 8;    // waves that scan the filterbank
constexpr int    kMelBins    = 256;  // mel bins whose masks are held at a time
constexpr int    kMelPerWave = 8;    // frames of a short transform a wave takes at most

constexpr int    kMelUnmasked  = 32;     // n_fft up to which every frequency is summed: no more than four float4 a filter
constexpr int    kMelFrameNfft = 256;    // the block-per-frame form's n_fft,
constexpr int    kMelFrameMost = 2048;   // frames (its blocks of one round: eight a CU)
constexpr int    kMelFrameWork = 98304;  // and samples at most

struct MelArgs {
    const float * pcm;
    const float * fb;  // [bins][n_fft/2 + 1]
    float *       y;   // [frames][bins]
    int64_t       ns;
    int64_t       frames;
    FastDiv       fnf;  // n_fft/2 + 1
    int32_t       nfft;
    int32_t       log2n;
    int32_t       hop;
    int32_t       win;
    int32_t       pad;
    int32_t       bins;
    int32_t       lfw;  // log2 of the frames a transform wave takes
    int32_t       masked;  // the filters' spans are found first
    int64_t       block0;  // the launch's first block
};

// LDS place of transform element i: one element of padding per 16 spreads the
// strided register passes over the banks.
__device__ __forceinline__ int mel_at(int i) {
    return i + (i >> 4);
}

__host__ __device__ __forceinline__ int mel_frame_elems(int n) {
    return n + n / 16;
}

// 64-bit words of a filter row's mask: a bit per float4 of its n/2 + 1 weights
// (those past the last float4 have none).
__host__ __device__ __forceinline__ int mel_words(int n) {
    return (n / 8 + kWave - 1) / kWave;
}

// Orders a wave's LDS accesses across its lanes (LDS serves one wave's
// accesses in order, so this only stops the compiler from moving them).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// SN stages of the transform, from stage length 2 << lh, on the 2^SN elements
// v[j] at base + (j << lh); k0 = base mod (1 << lh). tw[k] is the twiddle of
// the last stage's offset k; a shorter stage's offset k is that of k times the
// ratio of the lengths, bit for bit (a power of two scales the angle exactly).
template <int SN, bool FIRST>
__device__ __forceinline__ void mel_stages(float2 (&v)[1 << SN], const double2 * tw, int k0, int lh, int log2n) {
#pragma unroll
    for (int st = 0; st < SN; ++st) {
        const int shift = log2n - 1 - (lh + st);
#pragma unroll
        for (int j = 0; j < (1 << SN); ++j) {
            if ((j >> st) & 1) {
                continue;
            }
            const int    jb = j + (1 << st);
            const float2 b  = v[jb], a = v[j];
            if (FIRST && st == 0) {
                // twiddle (1, -0) on real inputs: an f32 sum and difference (a
                // double sum of two f32 rounded to f32 is their f32 sum), and
                // an imaginary part of 0, or NaN where the sample is infinite
                const float xi = b.x * -0.0f + 0.0f;
                v[jb]          = make_float2(a.x - b.x, 0.0f - xi);
                v[j]           = make_float2(a.x + b.x, 0.0f + xi);
                continue;
            }
            const double2 t  = tw[(k0 + ((j & ((1 << st) - 1)) << lh)) << shift];
            const double  br = b.x, bi = b.y;
            const double  xr = fma(br, t.x, -(bi * t.y));
            const double  xi = fma(br, t.y, bi * t.x);
            const double  ar = a.x, ai = a.y;
            v[jb] = make_float2(static_cast<float>(ar - xr), static_cast<float>(ai - xi));
            v[j]  = make_float2(static_cast<float>(ar + xr), static_cast<float>(ai + xi));
        }
    }
}

// A later pass: SN stages in place on the wave's frames' elements in LDS.
template <int SN>
__device__ __forceinline__ void mel_pass(float2 * d, const double2 * tw, int lane, int lh, int log2n, int live) {
    const int lg = log2n - SN;
    for (int t = lane; t < live << lg; t += kWave) {
        const int g    = t & ((1 << lg) - 1);
        const int k0   = g & ((1 << lh) - 1);
        const int base = ((g >> lh) << (lh + SN)) + k0;
        float2 *  df   = d + (t >> lg) * mel_frame_elems(1 << log2n);
        float2    v[1 << SN];
#pragma unroll
        for (int j = 0; j < (1 << SN); ++j) {
            v[j] = df[mel_at(base + (j << lh))];
        }
        mel_stages<SN, false>(v, tw, k0, lh, log2n);
#pragma unroll
        for (int j = 0; j < (1 << SN); ++j) {
            df[mel_at(base + (j << lh))] = v[j];
        }
    }
    wave_lds_sync();
}

// The first pass: SN stages on the windowed samples, read at their bit-reversed
// places (element 2^SN g + j is sample rev(j) * n / 2^SN + rev(g)).
template <int SN>
__device__ __forceinline__ void mel_first(float2 * d, const double2 * tw, const float * win, const MelArgs & a, int64_t f,
                                          int lane, int live) {
    const int log2n = a.log2n, lg = log2n - SN;
    for (int t = lane; t < live << lg; t += kWave) {
        const int     g     = t & ((1 << lg) - 1);
        const int64_t start = (f + (t >> lg)) * a.hop - a.pad;
        // (a shift by 32 - 0 is none: with one group g is 0)
        const int rg = lg > 0 ? static_cast<int>(__brev(static_cast<unsigned>(g)) >> (32 - lg)) : 0;
        float     x[1 << SN];
#pragma unroll
        for (int j = 0; j < (1 << SN); ++j) {
            const int rj = static_cast<int>(__brev(static_cast<unsigned>(j)) >> (32 - SN));
            // the padded signal at frame start + i: reflect-padded by `pad`
            const int64_t p = start + (rj << lg) + rg;
            x[j]            = a.pcm[p < 0 ? -p : (p < a.ns ? p : 2 * a.ns - 2 - p)];
        }
        float2 v[1 << SN];
#pragma unroll
        for (int j = 0; j < (1 << SN); ++j) {
            const int rj = static_cast<int>(__brev(static_cast<unsigned>(j)) >> (32 - SN));
            v[j]         = make_float2(x[j] * win[(rj << lg) + rg], 0.0f);
        }
        mel_stages<SN, true>(v, tw, 0, 0, log2n);
        float2 * df = d + (t >> lg) * mel_frame_elems(1 << log2n);
#pragma unroll
        for (int j = 0; j < (1 << SN); ++j) {
            df[mel_at((g << SN) + j)] = v[j];
        }
    }
    wave_lds_sync();
}

// The transforms of `live` frames from frame f on, by one wave.
__device__ __forceinline__ void mel_transform(float2 * d, const double2 * tw, const float * win, const MelArgs & a,
                                              int64_t f, int lane, int live) {
    int lh = a.log2n < 4 ? a.log2n : 4;
    if (lh == 4) {
        mel_first<4>(d, tw, win, a, f, lane, live);
    } else if (lh == 3) {
        mel_first<3>(d, tw, win, a, f, lane, live);
    } else if (lh == 2) {
        mel_first<2>(d, tw, win, a, f, lane, live);
    } else if (lh == 1) {
        mel_first<1>(d, tw, win, a, f, lane, live);
    } else {  // one sample a frame: its own transform
        if (lane < live) {
            d[lane * mel_frame_elems(1)] = make_float2(a.pcm[(f + lane) * a.hop] * win[0], 0.0f);
        }
        wave_lds_sync();
    }
    for (; a.log2n - lh >= 4; lh += 4) {
        mel_pass<4>(d, tw, lane, lh, a.log2n, live);
    }
    if (a.log2n - lh == 3) {
        mel_pass<3>(d, tw, lane, lh, a.log2n, live);
    } else if (a.log2n - lh == 2) {
        mel_pass<2>(d, tw, lane, lh, a.log2n, live);
    } else if (a.log2n - lh == 1) {
        mel_pass<1>(d, tw, lane, lh, a.log2n, live);
    }
}

// For each of nb filter rows, which of its float4 hold a weight that is not
// zero (a NaN is not): bit q % 64 of word q / 64, `words` words a row. By
// kMelScan waves, kMelRows rows at a time each, 128 float4 of each row.
constexpr int kMelRows = 8;

__device__ __forceinline__ void mel_masks(const float * rows, int nb, int nf, int words, int scan, int lane, uint64_t * s_mask) {
    const int n4 = nf / 4;
    for (int r0 = scan * kMelRows; r0 < nb; r0 += kMelScan * kMelRows) {
        for (int c = 0; c < words; c += 2) {
            const int q0 = c * kWave + lane, q1 = q0 + kWave;
            f32x4     w[kMelRows][2];
#pragma unroll
            for (int u = 0; u < kMelRows; ++u) {
                // (a row past the last is the last again, written again)
                const float * row = rows + static_cast<int64_t>(r0 + u < nb ? r0 + u : nb - 1) * nf;
                w[u][0]           = ld4u(row + (q0 < n4 ? q0 : 0) * 4);
                w[u][1]           = ld4u(row + (q1 < n4 ? q1 : 0) * 4);
            }
#pragma unroll
            for (int u = 0; u < kMelRows; ++u) {
                uint64_t * out = s_mask + (r0 + u < nb ? r0 + u : nb - 1) * words + c;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t bits = (__float_as_uint(w[u][h].x) | __float_as_uint(w[u][h].y)) |
                                          (__float_as_uint(w[u][h].z) | __float_as_uint(w[u][h].w));
                    const uint64_t any = __ballot(((bits & 0x7fffffffu) != 0u) & ((h == 0 ? q0 : q1) < n4));
                    if (c + h < words) {
                        out[h] = any;
                    }
                }
            }
        }
    }
}

template <int WAVES> __global__ __launch_bounds__((WAVES + kMelScan) * kWave) void k_log_mel(const MelArgs a) {
    constexpr int kThreads = (WAVES + kMelScan) * kWave;
    // [n/2] twiddles, the bins' masks, the frames' elements, the window, the
    // amplitudes, the frames' flags
    extern __shared__ double2 s_tw[];
    const int     n    = a.nfft;
    const int     nf   = n / 2 + 1;
    const int     tid  = static_cast<int>(threadIdx.x);
    const int     lane = tid % kWave;
    const int     wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int     fpb  = WAVES << a.lfw;
    uint64_t *    s_mask = reinterpret_cast<uint64_t *>(s_tw + n / 2);
    const int     words  = a.masked != 0 ? mel_words(n) : 0;
    float2 *      s_d    = reinterpret_cast<float2 *>(s_mask + kMelBins * words);
    float *       s_win = reinterpret_cast<float *>(s_d + fpb * mel_frame_elems(n));
    float *       s_mag = s_win + n;
    int *         s_bad = reinterpret_cast<int *>(s_mag + fpb * nf);
    const int64_t f0    = (a.block0 + blockIdx.x) * fpb;
    const int     nfr   = static_cast<int>(a.frames - f0 < fpb ? a.frames - f0 : fpb);  // the block's frames

    for (int k = tid; k < n / 2; k += kThreads) {
        const double angle = -2.0 * kMelPi / static_cast<double>(n);
        double       sn, cs;
        sincos(angle * static_cast<double>(k), &sn, &cs);
        s_tw[k] = double2{ cs, sn };
        if (a.win == n) {  // (n > 1: the loop does not run for n == 1)
            // cos(2 pi k / n) is the twiddle's, bit for bit, and half a turn on its negative
            s_win[k]         = static_cast<float>(0.5 - 0.5 * cs);
            s_win[n / 2 + k] = static_cast<float>(0.5 + 0.5 * cs);
        }
    }
    if (a.win != n || n == 1) {
        const int wpl = (n - a.win) / 2;
        for (int i = tid; i < n; i += kThreads) {
            float w = 0.0f;
            if (i >= wpl && i < wpl + a.win) {
                const double phase = 2.0 * kMelPi * static_cast<double>(i - wpl) / static_cast<double>(a.win);
                w                  = static_cast<float>(0.5 - 0.5 * cos(phase));
            }
            s_win[i] = w;
        }
    }
    if (tid < fpb) {
        s_bad[tid] = 0;
    }
    __syncthreads();
    if (wave < WAVES) {
        const int first = wave << a.lfw;
        const int live  = nfr - first < (1 << a.lfw) ? nfr - first : 1 << a.lfw;  // not above 0: none
        float2 *  d     = s_d + first * mel_frame_elems(n);
        if (live > 0) {
            mel_transform(d, s_tw, s_win, a, f0 + first, lane, live);
        }
    }
    for (int b0 = 0; b0 < a.bins; b0 += kMelBins) {
        const int     nb   = a.bins - b0 < kMelBins ? a.bins - b0 : kMelBins;
        const float * rows = a.fb + static_cast<int64_t>(b0) * nf;
        if (b0 != 0) {
            __syncthreads();  // the masks of the bins before have been used
        }
        if (wave >= WAVES && a.masked != 0) {
            mel_masks(rows, nb, nf, words, wave - WAVES, lane, s_mask);
        }
        __syncthreads();
        if (b0 == 0) {
#pragma unroll 3
            for (int t = tid; t < nfr * nf; t += kThreads) {
                const int    f = static_cast<int>(fastdiv(static_cast<uint32_t>(t), a.fnf));
                const float2 z = s_d[f * mel_frame_elems(n) + mel_at(t - f * nf)];
                const double sq = static_cast<double>(z.x) * static_cast<double>(z.x) +
                                  static_cast<double>(z.y) * static_cast<double>(z.y);
                const float m = static_cast<float>(sqrt(sq + 1e-9));
                s_mag[t]      = m;
                if (!(m <= 3.402823466e38f)) {
                    s_bad[f] = 1;
                }
            }
            __syncthreads();
        }
        // a lane per (frame, bin): consecutive lanes on consecutive bins
        for (int t = tid; t < nfr * nb; t += kThreads) {
            const int     f   = t / nb;
            const int     b   = t - f * nb;
            const float * row = rows + static_cast<int64_t>(b) * nf;
            const float * mag = s_mag + f * nf;
            int           lo = nf / 4, hi = 0;
            for (int i = 0; i < words; ++i) {
                const uint64_t any = s_mask[b * words + i];
                if (any != 0u) {
                    lo = lo < nf / 4 ? lo : i * kWave + __ffsll(static_cast<unsigned long long>(any)) - 1;
                    hi = i * kWave + 64 - __clzll(static_cast<long long>(any));
                }
            }
            const bool every = s_bad[f] != 0 || words == 0;
            lo               = every ? 0 : lo;
            hi               = every ? nf / 4 : hi;
            double        e = 0.0;
            // the product of two f32 is exact in double: one rounding either way
#pragma unroll 4
            for (int q = lo; q < hi; ++q) {
                const f32x4 w = ld4u(row + q * 4);
                e = fma(static_cast<double>(w.x), static_cast<double>(mag[q * 4]), e);
                e = fma(static_cast<double>(w.y), static_cast<double>(mag[q * 4 + 1]), e);
                e = fma(static_cast<double>(w.z), static_cast<double>(mag[q * 4 + 2]), e);
                e = fma(static_cast<double>(w.w), static_cast<double>(mag[q * 4 + 3]), e);
            }
            for (int k = nf / 4 * 4; k < nf; ++k) {  // the Nyquist frequency, in no float4
                e = fma(static_cast<double>(row[k]), static_cast<double>(mag[k]), e);
            }
            a.y[(f0 + f) * a.bins + b0 + b] = static_cast<float>(log(e < 1e-5 ? 1e-5 : e));  // std::max(e, 1e-5)
        }
    }
}

// A block per frame, all its lanes on one stage at a time and a lane per mel bin
// over every frequency: short transforms of few frames, which leave k_log_mel's
// waves a few lanes of work each and a long chain (n_fft 64, hop 16, 80 bins: 250
// frames 4.8 us against 6.3, 1500 frames 7.0 against 7.4, 3750 frames 13.5 against
// 9.1; MI355X, cold).
__global__ __launch_bounds__(256) void k_log_mel_frame(const MelArgs a) {
    extern __shared__ double2 s_tw[];  // [nfft - 1] twiddles, then re, im (f32), then amplitudes
    float *       s_re  = reinterpret_cast<float *>(s_tw + (a.nfft - 1));
    float *       s_im  = s_re + a.nfft;
    float *       s_mag = s_im + a.nfft;
    const int     tid   = static_cast<int>(threadIdx.x);
    const int64_t f     = blockIdx.x;
    const int     n     = a.nfft;
    const int     nf    = n / 2 + 1;
    // twiddle idx = len/2 - 1 + k for stage length len and butterfly offset k
    for (int idx = tid; idx < n - 1; idx += 256) {
        const int    half  = 1 << (31 - __clz(idx + 1));  // len / 2
        const int    len   = half * 2;
        const int    k     = idx - (half - 1);
        const double angle = -2.0 * kMelPi / static_cast<double>(len);
        double       sn, cs;
        sincos(angle * static_cast<double>(k), &sn, &cs);
        s_tw[idx] = double2{ cs, sn };
    }
    const int wpl = (n - a.win) / 2;
    for (int i = tid; i < n; i += 256) {
        // the padded signal at frame start + i: reflect-padded by `pad`
        const int64_t p = f * a.hop + i;
        float         x;
        if (p < a.pad) {
            x = a.pcm[a.pad - p];
        } else if (p < a.pad + a.ns) {
            x = a.pcm[p - a.pad];
        } else {
            x = a.pcm[a.ns - 2 - (p - a.pad - a.ns)];
        }
        float w = 0.0f;
        if (i >= wpl && i < wpl + a.win) {
            const double phase = 2.0 * kMelPi * static_cast<double>(i - wpl) / static_cast<double>(a.win);
            w                  = static_cast<float>(0.5 - 0.5 * cos(phase));
        }
        const int r = static_cast<int>(__brev(static_cast<unsigned>(i)) >> (32 - a.log2n));
        s_re[r]     = x * w;
        s_im[r]     = 0.0f;
    }
    __syncthreads();
    for (int half = 1; half < n; half *= 2) {
        for (int t = tid; t < n / 2; t += 256) {
            const int     k   = t & (half - 1);
            const int     ia  = (t - k) * 2 + k;  // start + k, start = (t / half) * 2 * half
            const int     ib  = ia + half;
            const double2 tw  = s_tw[half - 1 + k];
            const double  br  = s_re[ib], bi = s_im[ib];
            const double  xr  = fma(br, tw.x, -(bi * tw.y));
            const double  xi  = fma(br, tw.y, bi * tw.x);
            const double  ar  = s_re[ia];
            const double  ai  = s_im[ia];
            s_re[ib]          = static_cast<float>(ar - xr);
            s_im[ib]          = static_cast<float>(ai - xi);
            s_re[ia]          = static_cast<float>(ar + xr);
            s_im[ia]          = static_cast<float>(ai + xi);
        }
        __syncthreads();
    }
    for (int k = tid; k < nf; k += 256) {
        const double sq = static_cast<double>(s_re[k]) * static_cast<double>(s_re[k]) +
                          static_cast<double>(s_im[k]) * static_cast<double>(s_im[k]);
        s_mag[k]        = static_cast<float>(sqrt(sq + 1e-9));
    }
    __syncthreads();
    for (int b = tid; b < a.bins; b += 256) {
        const float * row = a.fb + static_cast<int64_t>(b) * nf;
        double        e   = 0.0;
        for (int k = 0; k < nf; ++k) {
            e += static_cast<double>(row[k]) * static_cast<double>(s_mag[k]);
        }
        a.y[f * a.bins + b] = static_cast<float>(log(e < 1e-5 ? 1e-5 : e));  // std::max(e, 1e-5)
    }
}

template <int WAVES> shp_status_t launch_mel(const MelArgs & a, hipStream_t stream) {
    const int    n   = a.nfft, nf = n / 2 + 1;
    const int    fpb = WAVES << a.lfw;
    const size_t lds = static_cast<size_t>(n / 2) * sizeof(double2) + static_cast<size_t>(fpb) * mel_frame_elems(n) * sizeof(float2) +
                       static_cast<size_t>(n + fpb * nf) * sizeof(float) + static_cast<size_t>(a.masked != 0 ? kMelBins * mel_words(n) : 0) * sizeof(uint64_t) +
                       static_cast<size_t>(fpb) * sizeof(int);
    constexpr int kThreads = (WAVES + kMelScan) * kWave;
    return in_launches((a.frames + fpb - 1) / fpb, kThreads, [&](int64_t first, dim3 grid) {
        MelArgs part = a;
        part.block0  = first;
        hipLaunchKernelGGL((k_log_mel<WAVES>), grid, dim3(kThreads), lds, stream, part);
    });
}

double slaney_step() {
    return std::log(6.4) / 27.0;
}

double hz_to_mel(double hz) {
    const double min_log_mel = 1000.0 / (200.0 / 3.0);
    return hz >= 1000.0 ? min_log_mel + std::log(hz / 1000.0) / slaney_step() : hz / (200.0 / 3.0);
}

double mel_to_hz(double mel) {
    const double min_log_mel = 1000.0 / (200.0 / 3.0);
    return mel >= min_log_mel ? 1000.0 * std::exp(slaney_step() * (mel - min_log_mel)) : (200.0 / 3.0) * mel;
}

bool pow2(int64_t v) {
    return v > 0 && (v & (v - 1)) == 0;
}

}  // namespace
}  // namespace shp

using namespace shp;

extern "C" shp_status_t shp_mel_filterbank(int32_t sample_rate, int32_t n_fft, int32_t mel_bins, float fmin, float fmax,
                                           float * out) {
    if (out == nullptr || sample_rate < 1 || n_fft < 2 || mel_bins < 1) {
        return SHP_ERR_INVALID_ARG;
    }
    const int64_t       nf = n_fft / 2 + 1;
    std::vector<double> edges(static_cast<size_t>(mel_bins) + 2);
    const double        lo = hz_to_mel(static_cast<double>(fmin)), hi = hz_to_mel(static_cast<double>(fmax));
    for (size_t i = 0; i < edges.size(); ++i) {
        edges[i] = mel_to_hz(lo + (hi - lo) * static_cast<double>(i) / static_cast<double>(mel_bins + 1));
    }
    for (int64_t b = 0; b < mel_bins; ++b) {
        const double enorm = 2.0 / (edges[b + 2] - edges[b]);
        for (int64_t k = 0; k < nf; ++k) {
            const double hz    = static_cast<double>(k) * static_cast<double>(sample_rate) / static_cast<double>(n_fft);
            const double lower = (hz - edges[b]) / (edges[b + 1] - edges[b]);
            const double upper = (edges[b + 2] - hz) / (edges[b + 2] - edges[b + 1]);
            const double v     = upper < lower ? upper : lower;  // std::min(lower, upper)
            out[b * nf + k]    = static_cast<float>((0.0 < v ? v : 0.0) * enorm);
        }
    }
    return SHP_OK;
}

extern "C" shp_status_t shp_log_mel(const shp_tensor * pcm,
                                    const shp_tensor * filterbank,
                                    int32_t            n_fft,
                                    int32_t            hop,
                                    int32_t            win_length,
                                    shp_tensor *       mel,
                                    shp_stream_t       stream) {
    if (!well_formed(pcm) || !well_formed(filterbank) || !well_formed(mel)) {
        return SHP_ERR_INVALID_ARG;
    }
    if (pcm->type != SHP_TYPE_F32 || filterbank->type != SHP_TYPE_F32 || mel->type != SHP_TYPE_F32 ||
        !contiguous(*pcm) || !contiguous(*filterbank) || !contiguous(*mel)) {
        return SHP_ERR_UNSUPPORTED;
    }
    if (!pow2(n_fft) || hop < 1 || win_length < 1 || win_length > n_fft || hop > n_fft) {
        return SHP_ERR_INVALID_ARG;
    }
    const int64_t ns   = nelements(*pcm);
    const int64_t pad  = (n_fft - hop) / 2;
    const int64_t plen = ns + 2 * pad;
    const int64_t bins = filterbank->ne[1];
    // upstream's reflect pad needs more samples than the pad
    if (ns <= pad || plen < n_fft || filterbank->ne[0] != n_fft / 2 + 1 || nelements(*filterbank) != bins * (n_fft / 2 + 1)) {
        return SHP_ERR_INVALID_ARG;
    }
    const int64_t frames = 1 + (plen - n_fft) / hop;
    if (mel->ne[0] != bins || nelements(*mel) != bins * frames) {
        return SHP_ERR_INVALID_ARG;
    }
    if (n_fft > kMelMaxNfft || frames > INT32_MAX) {
        return SHP_ERR_UNSUPPORTED;
    }
    if (spans_overlap(*pcm, *mel) || spans_overlap(*filterbank, *mel)) {
        return SHP_ERR_UNSUPPORTED;
    }
    if (dry_run()) {
        return SHP_OK;
    }
    MelArgs a{};
    a.pcm    = static_cast<const float *>(pcm->data);
    a.fb     = static_cast<const float *>(filterbank->data);
    a.y      = static_cast<float *>(mel->data);
    a.ns     = ns;
    a.frames = frames;
    a.nfft   = n_fft;
    a.log2n  = 31 - __builtin_clz(static_cast<unsigned>(n_fft));
    a.hop    = hop;
    a.win    = win_length;
    a.pad    = static_cast<int32_t>(pad);
    a.bins   = static_cast<int32_t>(bins);
    a.fnf    = make_fastdiv(static_cast<uint32_t>(n_fft / 2 + 1));
    if (n_fft > 1 && n_fft <= kMelFrameNfft && frames <= kMelFrameMost && n_fft * frames <= kMelFrameWork) {
        const size_t lds = static_cast<size_t>(n_fft - 1) * sizeof(double2) + static_cast<size_t>(2 * n_fft + n_fft / 2 + 1) * sizeof(float);
        hipLaunchKernelGGL(k_log_mel_frame, dim3(static_cast<unsigned>(frames)), dim3(256), lds, as_stream(stream), a);
        return launch_status();
    }
    a.masked = n_fft > kMelUnmasked;
    // The fewest frames a block that leave one block a CU, more of a short
    // transform to a wave (16 samples a lane: a wave takes 1024 of them) before
    // more waves (four waves' elements and tables are 58 KB of LDS at n_fft 1024).
    // n_fft 1024, hop 256, 80 bins: 234 frames one a block 10.3 us, four 11.6; 937
    // frames 35 and 12.2. n_fft 64, 128 bins: 1500 frames in eights 9.4, in 32s 14.7.
    int most = 0;
    while ((n_fft << (most + 1)) <= 1024 && (2 << most) <= kMelPerWave) {
        ++most;
    }
    const int waves = n_fft <= 1024 ? kMelWaves : 1;
    int       fpb   = 1;
    while (fpb < waves << most && (frames + fpb - 1) / fpb > 256) {
        fpb *= 2;
    }
    while (a.lfw < most && (2 << a.lfw) <= fpb) {
        ++a.lfw;
    }
    switch (fpb >> a.lfw) {
        case 1:
            return launch_mel<1>(a, as_stream(stream));
        case 2:
            return launch_mel<2>(a, as_stream(stream));
        default:
            return launch_mel<kMelWaves>(a, as_stream(stream));
    }
}
