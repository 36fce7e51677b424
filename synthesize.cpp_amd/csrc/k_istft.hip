// Kokoro's inverse short-time transform for gfx950 (kokoro/decoder-host.cpp:
// 28-100; the host runs it on the generator's output at kokoro/model.cpp:1056,
// after copying the spectrum off the device): from frames of n_fft/2 + 1
// log-magnitudes and as many raw phases, the waveform, in double as the host
// code computes it.
//
// One block per run of output samples:
//   1. the twiddles cos/sin(2 pi k / n_fft) and the complex bins of every frame
//      its samples overlap -- exp(log-magnitude) * (cos, sin)(sin(raw phase))
//      -- are formed once each into LDS;
//   2. a lane per (frame, s <= n_fft/2) takes the real inverse DFT at the
//      mirrored samples s and n_fft - s together: with A the cosine and B the
//      sine part, they are A - B and A + B (bin 0 and the Nyquist bin once, the
//      others twice, over n_fft); windowed, into LDS;
//   3. each lane's output samples t, at position P = t + n_fft/2, sum the
//      windowed values of the frames f with f*hop <= P < f*hop + n_fft and their
//      squared window values, in frame order; the output is the quotient rounded
//      to f32, or 0 where the envelope is below 1e-11.
// The window is the periodic Hann window rounded to f32, the value the host
// code tabulates. The turn of bin b at sample s is taken from the twiddle of
// (b*s) mod n_fft, A and B are summed apart, each product fused with its sum,
// and the division by n_fft is a product with its reciprocal: the host computes
// cos(2 pi b s / n_fft) of the unreduced product, one sum and its quotient, which
// differ in the last bits of the double. (k_istft_direct keeps the one sum and
// the division.)
//
// Bound by the f64 arithmetic and its latency (an exp, a sine and a sincos per
// bin); every sample taking its frames' whole DFT read each bin n_fft times from
// LDS. Measured on MI355X at n_fft 20, hop 5, 5 seconds (24001 frames) 9.9 -> 7.0
// us, 20 seconds 22.8 -> 16.4; n_fft 256, hop 64, 2000 frames 44.9 -> 31.9, against
// k_istft_direct.

#include <cmath>
#include <numeric>

#include "shp_internal.hpp"

namespace shp {
namespace {

constexpr int    kIstftBlock  = 512;
constexpr int    kIstftDirect = 256;
constexpr size_t kIstftLds   = 48 * 1024;  // bytes of LDS a block may take
constexpr double kIstftPi    = 3.14159265358979323846;

struct IstftArgs {
    const char * spec;
    int64_t      snb1;    // bytes between frames
    float *      y;
    int64_t      frames;
    int64_t      kept;    // output samples, (frames - 1) * hop
    int32_t      nfft;
    int32_t      hop;
    int32_t      bins;
    int32_t      bt;      // output samples per block
    int32_t      nf_max;  // frames a block's samples overlap, at most
    int32_t      pad;
    FastDiv      fhop;
    FastDiv      fbins;
    int64_t      block0;  // the launch's first block
};

__global__ __launch_bounds__(kIstftBlock) void k_istft(const IstftArgs a) {
    extern __shared__ double2 sm[];  // [nfft] twiddles, [nf][bins] frame bins, [nfft] window, [nf][nfft] windowed samples
    double2 *     tw   = sm;
    double2 *     fb   = sm + a.nfft;
    double *      win  = reinterpret_cast<double *>(fb + a.nf_max * a.bins);
    double *      vw   = win + a.nfft;
    const int     tid  = static_cast<int>(threadIdx.x);
    const int64_t t0   = (a.block0 + blockIdx.x) * a.bt;
    const int     nt   = static_cast<int>(a.kept - t0 < a.bt ? a.kept - t0 : a.bt);
    const int     half = a.nfft / 2;
    // frames overlapping positions [t0 + half, t0 + nt - 1 + half]
    const int64_t p0  = t0 + half;
    const int64_t flo = p0 < a.nfft ? 0 : static_cast<int64_t>(fastdiv(static_cast<uint32_t>(p0 - a.nfft), a.fhop)) + 1;
    int64_t       fhi = fastdiv(static_cast<uint32_t>(p0 + nt - 1), a.fhop);
    fhi               = fhi > a.frames - 1 ? a.frames - 1 : fhi;
    const int nf      = static_cast<int>(fhi - flo + 1);  // <= nf_max (host-checked bound); 0 in a gap between frames
    for (int k = tid; k < a.nfft; k += kIstftBlock) {
        const double turn = 2.0 * kIstftPi * static_cast<double>(k) / static_cast<double>(a.nfft);
        double       sn, cs;
        sincos(turn, &sn, &cs);
        tw[k]  = double2{ cs, sn };
        win[k] = static_cast<double>(static_cast<float>(0.5 * (1.0 - cs)));
    }
    for (int i = tid; i < nf * a.bins; i += kIstftBlock) {
        const int     f   = static_cast<int>(fastdiv(static_cast<uint32_t>(i), a.fbins));
        const int     b   = i - f * a.bins;
        const float * row = reinterpret_cast<const float *>(a.spec + (flo + f) * a.snb1);
        const double  mag = exp(static_cast<double>(row[b]));
        const double  ang = sin(static_cast<double>(row[a.bins + b]));
        double        sn, cs;
        sincos(ang, &sn, &cs);
        fb[i] = double2{ mag * cs, mag * sn };
    }
    __syncthreads();
    const double scale = 1.0 / static_cast<double>(a.nfft);
    for (int i = tid; i < nf * a.bins; i += kIstftBlock) {
        const int       f  = static_cast<int>(fastdiv(static_cast<uint32_t>(i), a.fbins));
        const int       s  = i - f * a.bins;
        const double2 * bf = fb + f * a.bins;
        double          A = 0.0, B = 0.0;
        int             k = s;  // (b * s) mod nfft
        for (int b = 1; b < a.bins - 1; ++b) {
            const double2 c = tw[k];
            const double2 z = bf[b];
            A               = fma(z.x, c.x, A);
            B               = fma(z.y, c.y, B);
            k += s;
            k = k >= a.nfft ? k - a.nfft : k;
        }
        const double2 z0 = bf[0], zn = bf[half], cn = tw[(s & 1) != 0 ? half : 0];
        A = fma(2.0, A, fma(zn.x, cn.x, z0.x * tw[0].x));
        B = fma(2.0, B, fma(zn.y, cn.y, z0.y * tw[0].y));
        vw[f * a.nfft + s] = (A - B) * scale * win[s];
        if (s != 0 && s != half) {
            vw[f * a.nfft + a.nfft - s] = (A + B) * scale * win[a.nfft - s];
        }
    }
    __syncthreads();
    const int off = static_cast<int>(p0 - flo * a.hop);  // the first sample's position from frame flo on
    for (int t = tid; t < nt; t += kIstftBlock) {
        const int P  = off + t;
        const int fa = P < a.nfft ? 0 : static_cast<int>(fastdiv(static_cast<uint32_t>(P - a.nfft), a.fhop)) + 1;
        int       fz = P < 0 ? -1 : static_cast<int>(fastdiv(static_cast<uint32_t>(P), a.fhop));
        fz           = fz > nf - 1 ? nf - 1 : fz;
        double acc = 0.0, env = 0.0;
        for (int f = fa; f <= fz; ++f) {
            const int s = P - f * a.hop;
            acc += vw[f * a.nfft + s];
            env += win[s] * win[s];
        }
        a.y[t0 + t] = fabs(env) < static_cast<double>(1e-11f) ? 0.0f : static_cast<float>(acc / env);
    }
}

// Windows too long for their hop to hold a block's windowed frames as well:
// each lane's samples take the whole DFT of their frames from the bins.
__device__ __forceinline__ int64_t floor_div(int64_t a, int64_t b) {
    return a >= 0 ? a / b : -((-a + b - 1) / b);
}

__global__ __launch_bounds__(kIstftDirect) void k_istft_direct(const IstftArgs a) {
    extern __shared__ double2 sm[];  // [nfft] twiddles, then [nf][bins] frame bins
    double2 *     tw   = sm;
    double2 *     fb   = sm + a.nfft;
    const int     tid  = static_cast<int>(threadIdx.x);
    const int64_t t0   = (a.block0 + blockIdx.x) * a.bt;
    const int64_t t1   = t0 + a.bt < a.kept ? t0 + a.bt : a.kept;
    const int     half = a.nfft / 2;
    // frames overlapping positions [t0 + half, t1 - 1 + half]
    int64_t       flo  = floor_div(t0 + half - (a.nfft - 1) + a.hop - 1, a.hop);
    flo                = flo < 0 ? 0 : flo;
    int64_t fhi        = (t1 - 1 + half) / a.hop;
    fhi                = fhi > a.frames - 1 ? a.frames - 1 : fhi;
    const int nf       = static_cast<int>(fhi - flo + 1);  // <= nf_max (host-checked bound)
    for (int k = tid; k < a.nfft; k += kIstftDirect) {
        const double turn = 2.0 * kIstftPi * static_cast<double>(k) / static_cast<double>(a.nfft);
        double       sn, cs;
        sincos(turn, &sn, &cs);
        tw[k] = double2{ cs, sn };
    }
    for (int i = tid; i < nf * a.bins; i += kIstftDirect) {
        const int     f   = i / a.bins;
        const int     b   = i - f * a.bins;
        const float * row = reinterpret_cast<const float *>(a.spec + (flo + f) * a.snb1);
        const double  mag = exp(static_cast<double>(row[b]));
        const double  ang = sin(static_cast<double>(row[a.bins + b]));
        double        sn, cs;
        sincos(ang, &sn, &cs);
        fb[i] = double2{ mag * cs, mag * sn };
    }
    __syncthreads();
    for (int64_t t = t0 + tid; t < t1; t += kIstftDirect) {
        const int64_t P  = t + half;
        int64_t       fa = floor_div(P - (a.nfft - 1) + a.hop - 1, a.hop);
        fa               = fa < flo ? flo : fa;
        int64_t fz       = P / a.hop;
        fz               = fz > fhi ? fhi : fz;
        double acc = 0.0, env = 0.0;
        for (int64_t f = fa; f <= fz; ++f) {
            const int       s   = static_cast<int>(P - f * a.hop);
            const double2 * bf  = fb + (f - flo) * a.bins;
            double          v   = 0.0;
            int             k   = 0;  // (b * s) mod nfft
            for (int b = 0; b < a.bins; ++b) {
                const double  w  = (b == 0 || b == a.bins - 1) ? 1.0 : 2.0;
                const double2 c  = tw[k];
                const double2 z  = bf[b];
                v += w * (z.x * c.x - z.y * c.y);
                k += s;
                k = k >= a.nfft ? k - a.nfft : k;
            }
            v                 = v / static_cast<double>(a.nfft);
            const double  win = static_cast<double>(static_cast<float>(0.5 * (1.0 - tw[s].x)));
            acc += v * win;
            env += win * win;
        }
        a.y[t] = fabs(env) < static_cast<double>(1e-11f) ? 0.0f : static_cast<float>(acc / env);
    }
}

// The kernel and the output samples per block of one call: the least estimated
// time among k_istft at 64 to 512 samples a block (or as many whole hops as make
// one round of its lanes) and k_istft_direct at the most samples that the LDS
// budget holds. Forming each mirrored pair of a frame's samples once is ahead
// while the chip has room, or where a block's samples are many against its
// frames' overlap with its neighbours', which every block transforms again; at
// n_fft 400, hop 100 the budget holds 64 samples a block, whose six frames are
// 3.3 times the work of taking each sample's four (20 s of 24 kHz, MI355X: 560 us
// against 187; but 30,000 samples 47 against 56). The estimate is in f64 operations a
// lane, its weights fitted to 1,871 measured calls (n_fft 20 to 800, hops of an
// eighth to all of it, 1,500 to 1,920,000 samples): its pick is 0.8 % from the
// fastest form on average, and at most 1.13 of k_istft_direct's time.
struct IstftForm {
    int64_t nfft, hop, kept, bins;
    int64_t bt     = 0;  // 0: windows too long for their hop
    bool    direct = true;

    IstftForm(int64_t n, int64_t h, int64_t samples) : nfft(n), hop(h), kept(samples), bins(n / 2 + 1) {
        for (int64_t cand : { 256, 128, 64 }) {
            if (lds(cand, true) <= kIstftLds) {
                bt = cand;
                break;
            }
        }
        if (bt == 0) {
            return;
        }
        int64_t       least = cost(bt, true);
        const int64_t whole = (kIstftBlock / bins - (nfft + hop - 1) / hop) * hop;
        for (int64_t cand : { int64_t{ 64 }, int64_t{ 128 }, int64_t{ 256 }, int64_t{ 512 }, whole }) {
            if (cand < 64 || cand > 512 || lds(cand, false) > kIstftLds) {
                continue;
            }
            const int64_t c = cost(cand, false);
            if (c < least) {
                least  = c;
                bt     = cand;
                direct = false;
            }
        }
    }

    // Frames that `samples` consecutive samples overlap, at most.
    int64_t frames_of(int64_t samples) const { return (samples - 1 + nfft - 1) / hop + 2; }

    size_t lds(int64_t samples, bool whole_dft) const {
        const int64_t nf = frames_of(samples);
        return static_cast<size_t>(nf * bins + nfft) * sizeof(double2) +
               (whole_dft ? size_t{ 0 } : static_cast<size_t>(nf * nfft + nfft) * sizeof(double));
    }

    int64_t cost(int64_t samples, bool whole_dft) const {
        const int64_t lanes = whole_dft ? kIstftDirect : kIstftBlock;
        const int64_t all   = kept / hop + 1;
        const int64_t align = std::gcd(std::gcd(samples, hop), nfft / 2);  // of every block's first position to a frame's
        const int64_t upto  = (samples + nfft - align + hop - 1) / hop;
        const int64_t items = (upto < all ? upto : all) * bins;
        const int64_t round = (items + lanes - 1) / lanes, turns = (samples + lanes - 1) / lanes;
        // a bin formed, and a term of a mirrored pair's sums: per round of the
        // lanes and, for what the waves share, per item
        const int64_t block = whole_dft ? 547 + round * 47 + items * 74 / lanes + turns * nfft * bins * 16 / hop :
                                          148 + round * (47 + bins * 6) + items * (74 + bins * 6) / lanes + turns * nfft * 2 / hop;
        // a CU's blocks share its f64 units, which eight waves fill
        const int64_t percu = ((kept + samples - 1) / samples + 255) / 256;
        const int64_t busy  = percu * (lanes / kWave) / 8;
        return block * (busy > 1 ? busy : 1);
    }
};

}  // namespace
}  // namespace shp

using namespace shp;

extern "C" shp_status_t shp_inverse_stft(const shp_tensor * spectrum,
                                         int32_t            n_fft,
                                         int32_t            hop,
                                         shp_tensor *       audio,
                                         shp_stream_t       stream) {
    if (!well_formed(spectrum) || !well_formed(audio) || n_fft < 2 || n_fft % 2 != 0 || hop <= 0) {
        return SHP_ERR_INVALID_ARG;
    }
    if (spectrum->type != SHP_TYPE_F32 || audio->type != SHP_TYPE_F32) {
        return SHP_ERR_UNSUPPORTED;
    }
    const int64_t frames = spectrum->ne[1];
    if (spectrum->ne[0] != n_fft + 2 || spectrum->ne[2] != 1 || spectrum->ne[3] != 1 || frames < 2 ||
        audio->ne[0] != (frames - 1) * hop || audio->ne[1] != 1 || audio->ne[2] != 1 || audio->ne[3] != 1) {
        return SHP_ERR_INVALID_ARG;
    }
    if (spans_overlap(*spectrum, *audio) || frames > INT32_MAX || audio->ne[0] > INT32_MAX) {
        return SHP_ERR_UNSUPPORTED;
    }
    const IstftForm form{ n_fft, hop, audio->ne[0] };
    if (form.bt == 0) {
        return SHP_ERR_UNSUPPORTED;  // windows too long for their hop to stage a block's frames
    }
    if (dry_run()) {
        return SHP_OK;
    }
    IstftArgs a{};
    a.spec       = static_cast<const char *>(spectrum->data);
    a.snb1       = static_cast<int64_t>(spectrum->nb[1]);
    a.y          = static_cast<float *>(audio->data);
    a.frames     = frames;
    a.kept       = audio->ne[0];
    a.nfft       = n_fft;
    a.hop        = hop;
    a.bins       = static_cast<int32_t>(form.bins);
    a.bt         = static_cast<int32_t>(form.bt);
    a.nf_max     = static_cast<int32_t>(form.frames_of(form.bt));
    a.fhop       = make_fastdiv(static_cast<uint32_t>(hop));
    a.fbins      = make_fastdiv(static_cast<uint32_t>(form.bins));
    const size_t  lds    = form.lds(form.bt, form.direct);
    const int64_t blocks = (a.kept + form.bt - 1) / form.bt;
    const int     block  = form.direct ? kIstftDirect : kIstftBlock;
    return in_launches(blocks, block, [&](int64_t first, dim3 grid) {
        a.block0 = first;
        hipLaunchKernelGGL(form.direct ? k_istft_direct : k_istft, grid, dim3(block), lds, as_stream(stream), a);
    });
}
