// ggml_im2col, 1-D (is_2D = false), for gfx950: the column matrix every
// convolution of the vocoders, codecs and speech encoders feeds its GEMM
// (vits/waveform-decoder.cpp:104, vits/operations.cpp:40,103,
// kokoro/operations.cpp:76, omnivoice/codec.cpp:114,
// omnivoice/reference-encoder.cpp:190, qwen3-tts/codec.cpp:96,129,
// qwen3-tts/speaker-encoder.cpp:174, qwen3-tts/codec-encoder.cpp:359).
//
//   x [IW, IC, N] (F32)  ->  y [IC*K, OW, N] (F32 or F16)
//   y[n][ow][ic*K + k] = x[n][ic][ow*s0 + k*d0 - p0], 0 outside [0, IW)
//
// A pure gather: every output is one input element (or 0), rounded to nearest
// even for an F16 y, so the result is bit-exact. The write of K copies of the
// input is the traffic (HBM-bound).
//
// One block per tile of OWT output positions x ICT channels of one batch
// entry (no loop: a block's stores never wait at a barrier):
//   1. the tile's input window (ICT channel rows of (OWT-1)*s0 + (K-1)*d0 + 1
//      samples, zeros past the input's ends) goes to LDS, consecutive lanes on
//      consecutive addresses, four values a lane (by_value's calls: one): along time
//      for a time-contiguous x, along channels for a channel-contiguous x (the
//      transposed view of a channel-major activation, so the ggml_cont the
//      reference puts in front of im2col is not needed). Value by value, behind
//      a leaky-ReLU that has just written x (MI355X, both launches): K = 3
//      [128,131072] 75.3 -> 72.5 us, [256,4136] 10.4 -> 9.1; K = 7 d = 3 F16
//      [128,131072] 101 -> 89.7;
//   2. the tile's outputs are written in y's order, V values (16 bytes) per
//      store. The LDS offsets of the values a store takes repeat with a short
//      period -- one position's run of ICT*K values, or for a tile of every
//      channel (one contiguous range of y) lcm(IC*K, V) values -- so each tile
//      first tabulates one period's offsets in LDS; a store is then one table
//      read, V window reads and running sums, with no division.
// Both phases step their indices by running sums: the kernel is bound by its
// stores, not by address arithmetic (per-value divisions held an earlier form
// to ~65 % of HBM peak at [128,131072], K = 3). A replay over inputs that no
// kernel rewrites reads them from the Infinity Cache (the stores bypass it):
// the figures below are such replays' and compare tiles, but an input fresh
// from its producer comes from HBM, at 5.4 TB/s with the writes.

#include "shp_internal.hpp"

namespace shp {
namespace {

constexpr int kIm2colBlock = 256;
constexpr int kIm2colLds   = 4480;   // floats of LDS window per block at most (17.5 KB; with the table, 8 blocks per CU)
constexpr int kIm2colBatch = 8;      // window loads a lane issues before its LDS writes
constexpr int kIm2colQuads = 4;      // the same for float4 loads
constexpr int kIm2colTab   = 1024;   // int16 LDS offsets of the store table (one period)

// Tile shape: ict channels; at least owt positions, or enough for `elems`
// outputs; fewer positions when the window passes kIm2colLds. Measured on
// MI355X over K = 3 / 7 / 11, dilations 1-5, [128,131072] and [512,8192],
// F32 and F16 columns, both input layouts (% of HBM peak at [128,131072];
// the same-run copy reaches 75 %):
//   - runs shorter than a 128-byte line per position (ict*K*esize) cost
//     2-3x (8 channels: 21-38 %);
//   - time-contiguous x, F32, K <= 4: 16 x 64 (4096 outputs) 76 %, against
//     69 % for 32 x 128;
//   - time-contiguous x otherwise: 32 x 64, K = 11 d = 5 75 % (66-68 % for
//     16 or 64 channels, or 128 positions); F16 K = 7: 32 x 128 69 %;
//   - channel-contiguous x: 32 x 128, 76 % (63 % for 16 channels);
//   - one channel (the depthwise form): 4096 outputs 63 %, 8192 56 %.
struct TileRule {
    int ict;
    int owt;
    int elems;
};

inline TileRule tile_rule(bool chfast, bool f16, int64_t ic, int64_t k) {
    if (ic == 1) {
        return { 1, 64, 4096 };
    }
    if (chfast) {
        return { 32, 128, 8192 };
    }
    if (!f16 && k <= 4) {
        return { 16, 64, 4096 };
    }
    return f16 ? TileRule{ 32, 128, 8192 } : TileRule{ 32, 64, 8192 };
}

// How a block reads its window: value by value (any strides), or four samples of
// a channel (time-contiguous x) or four channels of a sample (channel-contiguous)
// per load.
enum Im2colWalk { kWalkValues = 0, kWalkTime = 1, kWalkChannels = 2 };

struct Im2colArgs {
    const char * x;
    char *       y;
    int64_t      xnb0;  // byte strides of x: time, channel, batch
    int64_t      xnb1;
    int64_t      xnb2;
    int64_t      iw;    // IW
    int64_t      ic;    // IC
    int64_t      ow;    // OW
    int64_t      row;   // IC*K: y values per (n, ow)
    int32_t      k;
    int32_t      s0;
    int32_t      p0;
    int32_t      d0;
    int32_t      ict;   // tile extents
    int32_t      owt;
    int32_t      wt;    // window samples of a full tile
    int32_t      wtp;   // LDS row stride (wt, odd)
    FastDiv      tic;   // channel tiles
    FastDiv      tow;   // position tiles
    FastDiv      kdiv;  // K
    FastDiv      rdiv;  // IC*K
    FastDiv      segf;  // ICT*K: a full channel tile's run per position
    FastDiv      segl;  // the last channel tile's run
    // window walk: ns rows of nf values (time-contiguous x: ICT channel rows of
    // wt samples; channel-contiguous x: wt sample rows of ICT channels); lane
    // tid starts at (tid / nf, tid % nf) and steps 256 values at a time
    FastDiv      fdiv;  // nf
    int32_t      ns;
    int32_t      ds;    // 256 / nf
    int32_t      df;    // 256 % nf
    int32_t      nbs;   // x byte strides of a row and of a value of the walk
    int32_t      nbf;
    int32_t      ls;    // LDS strides of the same
    int32_t      lf;
    int32_t      pad;
};

// V consecutive values of y from index e (e % V == 0 for V > 1), nontemporal.
template <int V, bool F16> __device__ __forceinline__ void put(char * y, int64_t e, const float (&v)[V]) {
    if constexpr (F16) {
        typedef _Float16 hv __attribute__((ext_vector_type(V)));
        hv h;
#pragma unroll
        for (int i = 0; i < V; ++i) {
            h[i] = static_cast<_Float16>(v[i]);
        }
        if constexpr (V == 1) {
            __builtin_nontemporal_store(h[0], reinterpret_cast<_Float16 *>(y) + e);
        } else {
            __builtin_nontemporal_store(h, reinterpret_cast<hv *>(y) + e / V);
        }
    } else {
        if constexpr (V == 1) {
            __builtin_nontemporal_store(v[0], reinterpret_cast<float *>(y) + e);
        } else {
            typedef float fv __attribute__((ext_vector_type(V)));
            fv f;
#pragma unroll
            for (int i = 0; i < V; ++i) {
                f[i] = v[i];
            }
            __builtin_nontemporal_store(f, reinterpret_cast<fv *>(y) + e / V);
        }
    }
}

// LDS offset of value f of the tile, whose values run (position, channel, tap)
// with rd.d values per position.
__device__ __forceinline__ int tap_offset(const Im2colArgs & a, uint32_t f, const FastDiv & rd) {
    const uint32_t owl = fastdiv(f, rd);
    const uint32_t j   = f - owl * rd.d;
    const uint32_t icl = fastdiv(j, a.kdiv);
    return static_cast<int>(icl) * a.wtp + static_cast<int>(owl) * a.s0 + static_cast<int>(j - icl * a.kdiv.d) * a.d0;
}

// FLAT: the tile holds every channel (ICT == IC): its outputs are one range of
// y, written in V-value stores between scalar ends (table period lcm(row, V)
// values). Otherwise each position has a run of ICT*K values, a multiple of V,
// starting V-aligned (table period: one run). V == 1: no table, one value per
// lane and step, located by division (layouts the others cannot take).
template <bool FLAT, int V, bool F16, int WALK>
__global__ __launch_bounds__(kIm2colBlock) void k_im2col(const Im2colArgs a) {
    typedef int16_t         tv __attribute__((ext_vector_type(V > 1 ? V : 2)));  // one store's offsets
    extern __shared__ f32x4 lds4[];
    float *                 lds = reinterpret_cast<float *>(lds4);
    __shared__ tv           tabv[V > 1 ? kIm2colTab / V : 1];
    int16_t *               tab = reinterpret_cast<int16_t *>(tabv);
    const int               tid = static_cast<int>(threadIdx.x);
    const uint32_t          t   = blockIdx.x;
    const uint32_t          q   = fastdiv(t, a.tic);
    const uint32_t          n   = fastdiv(q, a.tow);
    const int64_t           ic0 = static_cast<int64_t>(t - q * a.tic.d) * a.ict;
    const int64_t           ow0 = static_cast<int64_t>(q - n * a.tow.d) * a.owt;
    const int               nic = static_cast<int>(a.ic - ic0 < a.ict ? a.ic - ic0 : a.ict);
    const int               now = static_cast<int>(a.ow - ow0 < a.owt ? a.ow - ow0 : a.owt);
    const int64_t           iw0 = ow0 * a.s0 - a.p0;
    // the window's first sample (may lie before x: only in-range samples are read)
    const char *            xw  = a.x + static_cast<int64_t>(n) * a.xnb2 + ic0 * a.xnb1 + iw0 * a.xnb0;
    const int               wlo = static_cast<int>(iw0 < 0 ? -iw0 : 0);                      // first sample in x
    const int               whi = static_cast<int>(a.iw - iw0 < a.wt ? a.iw - iw0 : a.wt);  // past the last
    // 1. the window, by running sums; zeros outside [wlo, whi) and for
    //    channels past IC (never read). (Offsets past the walk's end wrap,
    //    unused.)
    const int nf = static_cast<int>(a.fdiv.d);
    int       s  = static_cast<int>(fastdiv(static_cast<uint32_t>(tid), a.fdiv));
    int       f  = tid - s * nf;
    uint32_t  ox = static_cast<uint32_t>(s) * a.nbs + static_cast<uint32_t>(f) * a.nbf;
    int       ol = s * a.ls + f * a.lf;
    const uint32_t sx = static_cast<uint32_t>(a.ds) * a.nbs + static_cast<uint32_t>(a.df) * a.nbf;
    const uint32_t cx = static_cast<uint32_t>(a.nbs) - static_cast<uint32_t>(nf) * a.nbf;
    const int      sl = a.ds * a.ls + a.df * a.lf, cl = a.ls - nf * a.lf;
    auto           step = [&]() {
        s += a.ds;
        f += a.df;
        ox += sx;
        ol += sl;
        if (f >= nf) {
            f -= nf;
            ++s;
            ox += cx;
            ol += cl;
        }
    };
    if constexpr (WALK == kWalkValues) {
        while (s < a.ns) {
            float v[kIm2colBatch];
            int   at[kIm2colBatch];
#pragma unroll
            for (int u = 0; u < kIm2colBatch; ++u) {
                at[u] = s < a.ns ? ol : -1;
                v[u]  = 0.0f;
                if (s < a.ns && s < nic && f >= wlo && f < whi) {
                    v[u] = *reinterpret_cast<const float *>(xw + ox);
                }
                step();
            }
#pragma unroll
            for (int u = 0; u < kIm2colBatch; ++u) {
                if (at[u] >= 0) {
                    lds[at[u]] = v[u];
                }
            }
        }
    } else {
        // four at a time from any 4-byte boundary: whole where the row goes on
        // in memory (past the window's last sample too: its row of LDS has room)
        const int most = WALK == kWalkTime ? static_cast<int>(a.iw - iw0 < a.wt + 4 ? a.iw - iw0 : a.wt + 4) : nic;
        const int from = WALK == kWalkTime ? wlo : 0;
        while (s < a.ns) {
            f32x4 v[kIm2colQuads];
            int   at[kIm2colQuads], ch[kIm2colQuads];
#pragma unroll
            for (int u = 0; u < kIm2colQuads; ++u) {
                at[u]         = s < a.ns ? ol : -1;
                ch[u]         = f * 4;
                v[u]          = splat4(0.0f);
                const bool in = s < a.ns && (WALK == kWalkTime ? s < nic : (s >= wlo && s < whi));
                if (in && f * 4 >= from && f * 4 + 4 <= most) {
                    v[u] = ld4u(reinterpret_cast<const float *>(xw + ox));
                } else if (in) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (f * 4 + e >= from && f * 4 + e < most) {
                            v[u][e] = reinterpret_cast<const float *>(xw + ox)[e];
                        }
                    }
                }
                step();
            }
#pragma unroll
            for (int u = 0; u < kIm2colQuads; ++u) {
                if (at[u] >= 0) {
                    if constexpr (WALK == kWalkTime) {
                        *reinterpret_cast<f32x4 *>(lds + at[u]) = v[u];
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            if (ch[u] + e < a.ict) {
                                lds[at[u] + e * a.wtp] = v[u][e];
                            }
                        }
                    }
                }
            }
        }
    }
    const int64_t ybase = (static_cast<int64_t>(n) * a.ow + ow0) * a.row + ic0 * a.k;  // first value's index
    const FastDiv sd    = nic == a.ict ? a.segf : a.segl;                              // run per position
    // the store pattern (V > 1): FLAT ranges start V-aligned after `head`
    // scalar values; P stores per period, covering cpos positions and cst
    // values of y
    int64_t       len  = 0;
    int           head = 0;
    int           P = 1, cpos = 1;
    int64_t       cst  = 0;
    int64_t       nvec = 0;
    if constexpr (V > 1) {
        if constexpr (FLAT) {
            len              = static_cast<int64_t>(now) * a.row;
            const int head0  = static_cast<int>((V - ybase % V) % V);
            head             = static_cast<int>(head0 < len ? head0 : len);
            const int64_t rw = a.row;
            const int     g  = rw % V == 0 ? V : (rw % (V / 2) == 0 ? V / 2 : (rw % 2 == 0 ? 2 : 1));  // gcd(row, V)
            P                = static_cast<int>(rw / g);  // lcm(row, V) / V
            cpos             = V / g;                     // lcm(row, V) / row
            cst              = static_cast<int64_t>(P) * V;
            nvec             = (len - head) / V;
            for (int r = tid; r < P * V; r += kIm2colBlock) {
                tab[r] = static_cast<int16_t>(tap_offset(a, static_cast<uint32_t>(head + r), a.rdiv));
            }
        } else {
            const int seg = static_cast<int>(sd.d);
            P             = seg / V;
            cst           = a.row;
            nvec          = static_cast<int64_t>(now) * P;
            for (int r = tid; r < seg; r += kIm2colBlock) {
                const uint32_t icl = fastdiv(static_cast<uint32_t>(r), a.kdiv);
                tab[r]             = static_cast<int16_t>(static_cast<int>(icl) * a.wtp +
                                                          (r - static_cast<int>(icl * a.kdiv.d)) * a.d0);
            }
        }
    }
    __syncthreads();
    // 2. the outputs, in y's order
    if constexpr (V == 1) {
        const FastDiv rd   = FLAT ? a.rdiv : sd;
        const int64_t nval = static_cast<int64_t>(now) * rd.d;
        for (int64_t f = tid; f < nval; f += kIm2colBlock) {
            const uint32_t owl   = fastdiv(static_cast<uint32_t>(f), rd);
            const float    v1[1] = { lds[tap_offset(a, static_cast<uint32_t>(f), rd)] };
            put<1, F16>(a.y, ybase + static_cast<int64_t>(owl) * a.row + (static_cast<uint32_t>(f) - owl * rd.d), v1);
        }
    } else {
        if constexpr (FLAT) {
            // the scalar ends of the range
            const int64_t tail = head + nvec * V;
            if (tid < head) {
                const float v1[1] = { lds[tap_offset(a, static_cast<uint32_t>(tid), a.rdiv)] };
                put<1, F16>(a.y, ybase + tid, v1);
            }
            if (tail + tid < len) {
                const float v1[1] = { lds[tap_offset(a, static_cast<uint32_t>(tail + tid), a.rdiv)] };
                put<1, F16>(a.y, ybase + tail + tid, v1);
            }
        }
        // store vi: period c = vi / P, entry r = vi % P, by running sums (the
        // block's 256 lanes step 256 stores: dc periods and dr entries)
        int           c      = tid / P;
        int           r      = tid - c * P;
        const int     dc     = kIm2colBlock / P, dr = kIm2colBlock % P;
        const int     lstep  = cpos * a.s0;  // window offset per period
        int           lb     = c * lstep;
        int64_t       ye     = ybase + head + static_cast<int64_t>(c) * cst + static_cast<int64_t>(r) * V;
        const int64_t ystep  = static_cast<int64_t>(dc) * cst + static_cast<int64_t>(dr) * V;
        const int64_t ycarry = cst - static_cast<int64_t>(P) * V;
        for (int64_t vi = tid; vi < nvec; vi += kIm2colBlock) {
            const tv o = tabv[r];  // one LDS read for the V offsets
            float    vals[V];
#pragma unroll
            for (int e = 0; e < V; ++e) {
                vals[e] = lds[lb + o[e]];
            }
            put<V, F16>(a.y, ye, vals);
            r += dr;
            lb += dc * lstep;
            ye += ystep;
            if (r >= P) {
                r -= P;
                lb += lstep;
                ye += ycarry;
            }
        }
    }
}

template <bool FLAT, int V, bool F16>
void launch_form(const Im2colArgs & a, int walk, unsigned grid, size_t shmem, hipStream_t s) {
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(kIm2colBlock), shmem, s, a); };
    walk == kWalkTime     ? go(k_im2col<FLAT, V, F16, kWalkTime>) :
    walk == kWalkChannels ? go(k_im2col<FLAT, V, F16, kWalkChannels>) : go(k_im2col<FLAT, V, F16, kWalkValues>);
}

inline int64_t window(int64_t owt, int64_t s0, int64_t k, int64_t d0) {
    return (owt - 1) * s0 + (k - 1) * d0 + 1;
}

// LDS row stride of a window of w samples: odd, which spreads a column of the
// window over the banks; for rows written 16 bytes at a time, an odd number of
// float4, which spreads 16 channels' taps over all of them.
inline int64_t padded(int64_t w, bool quads) {
    return quads ? ((w + 3) / 4 | 1) * 4 : w | 1;
}

// The most of a wave's 64 lanes that read one LDS bank for the first value of
// their stores (the others' counts are alike), at a row stride of wtp.
int bank_depth(const Im2colArgs & a, int v, int64_t wtp) {
    uint8_t depth[64] = {};
    int     most = 0, ch = 0, tap = 0, pos = 0;
    for (int l = 0; l < kWave; ++l) {
        uint8_t & n = depth[(ch * wtp + static_cast<int64_t>(tap) * a.d0 + static_cast<int64_t>(pos) * a.s0) & 63];
        most        = ++n > most ? n : most;
        for (tap += v; tap >= a.k; tap -= a.k) {
            ch  = ch + 1 < a.ict ? ch + 1 : 0;
            pos = ch == 0 ? pos + 1 : pos;
        }
    }
    return most;
}

// Whether F16 columns of a time-contiguous x read the window by value all the
// same. Eight LDS reads a store make them sensitive to bank conflicts, and at some
// tap distances the quads' row stride has them: K = 3 with d = 3 or 5, six lanes a
// bank against two at the odd stride. And few columns a sample leave the launch to
// its loads where x is between the L2s' size and the memory's. Both launches
// behind a leaky-ReLU that has just written x, by four and by value (MI355X, cold):
// K = 3 d = 5 [512,4000] 14.4 us and 11.5, im2col alone 8.4 and 7.0; K = 3 [256,4000]
// 10.8 and 9.8, alone 6.2 and 6.5; [64,65536] 20.0 and 16.6, alone 10.5 and 9.7; but
// K = 11 [256,4000] 13.6 and 14.2, alone 8.4 and 10.7, K = 3 [256,1000] alone 5.7 and
// 6.2, and F32 K = 3 [256,4000] 7.9 and 8.1, alone 4.7 and 5.0.
bool by_value(const Im2colArgs & a, int64_t n) {
    const int64_t values = n * a.ic * a.iw;
    if (a.ict < 32) {  // tiles of fewer channels: by four in all of these
        return false;
    }
    if (bank_depth(a, 8, padded(a.wt, true)) >= 3 * bank_depth(a, 8, padded(a.wt, false))) {
        return true;
    }
    return a.k <= 4 * static_cast<int64_t>(a.s0) && values < (int64_t{ 1 } << 23) && n * a.ow * a.row >= (int64_t{ 3 } << 20);
}

inline int64_t gcd64(int64_t a, int64_t b) {
    while (b != 0) {
        const int64_t r = a % b;
        a               = b;
        b               = r;
    }
    return a;
}

}  // namespace

// ggml_calc_conv_output_size with C's truncating division; < 1: no output.
int64_t im2col_out_len(int64_t iw, int64_t k, int64_t s0, int64_t p0, int64_t d0) {
    return (iw + 2 * p0 - d0 * (k - 1) - 1) / s0 + 1;
}

// The launch plan. chfast: x's channel stride is 4 bytes and its time stride is
// not (the transposed view of a channel-major activation).
struct Im2colPlan {
    Im2colArgs args{};
    bool       flat   = false;
    int        v      = 1;   // values per store: 1, 4 (F32 or F16) or 8 (F16)
    bool       f16    = false;
    bool       chfast = false;
    int        walk   = kWalkValues;
    unsigned   grid   = 0;   // one block per tile
    size_t     shmem  = 0;
};

shp_status_t plan_im2col(const shp_tensor * kernel, const shp_tensor * x, int32_t s0, int32_t p0, int32_t d0,
                         const shp_tensor * y, Im2colPlan & pl) {
    if (kernel == nullptr || x == nullptr || y == nullptr || x->data == nullptr || x->reserved != 0 ||
        kernel->reserved != 0) {
        return SHP_ERR_INVALID_ARG;
    }
    for (int d = 0; d < 4; ++d) {
        if (kernel->ne[d] < 1 || x->ne[d] < 1) {
            return SHP_ERR_INVALID_ARG;
        }
    }
    if (s0 < 1 || d0 < 1 || p0 < 0) {
        return SHP_ERR_INVALID_ARG;
    }
    if (x->type != SHP_TYPE_F32) {
        return SHP_ERR_UNSUPPORTED;
    }
    // ggml_im2col (1-D): the kernel's channel extent is x's; x has no 4th dim
    if (kernel->ne[1] != x->ne[1] || x->ne[3] != 1) {
        return SHP_ERR_INVALID_ARG;
    }
    if (reinterpret_cast<uintptr_t>(x->data) % 4 != 0 || x->nb[0] % 4 != 0 || x->nb[1] % 4 != 0 ||
        x->nb[2] % 4 != 0) {
        return SHP_ERR_UNSUPPORTED;
    }
    const int64_t K = kernel->ne[0], IW = x->ne[0], IC = x->ne[1], N = x->ne[2];
    if (K > INT32_MAX / 4 || static_cast<int64_t>(d0) * (K - 1) > INT32_MAX / 4) {
        return SHP_ERR_UNSUPPORTED;
    }
    const int64_t OW = im2col_out_len(IW, K, s0, p0, d0);
    if (OW < 1) {
        return SHP_ERR_INVALID_ARG;
    }
    if (!well_formed(y) || !contiguous(*y)) {
        return SHP_ERR_INVALID_ARG;
    }
    if (y->type != SHP_TYPE_F32 && y->type != SHP_TYPE_F16) {
        return SHP_ERR_UNSUPPORTED;
    }
    if (y->ne[0] != IC * K || y->ne[1] != OW || y->ne[2] != N || y->ne[3] != 1) {
        return SHP_ERR_INVALID_ARG;
    }
    if (spans_overlap(*x, *y)) {
        return SHP_ERR_UNSUPPORTED;
    }
    // tile: ICT channels, OWT positions, the window in LDS: as many positions
    // as wanted and fit (window + 1 for the odd row stride <= kIm2colLds /
    // ICT), fewer channels when not one position fits
    const int64_t  nb0 = static_cast<int64_t>(x->nb[0]), nb1 = static_cast<int64_t>(x->nb[1]);
    pl.chfast          = nb1 == 4 && nb0 != 4 && IC > 1;
    pl.f16             = y->type == SHP_TYPE_F16;
    const TileRule rule = tile_rule(pl.chfast, pl.f16, IC, K);
    int64_t        ict  = IC < rule.ict ? IC : rule.ict;
    int64_t owt = 0;
    for (;; ict = (ict + 1) / 2) {
        const int64_t room = kIm2colLds / ict - 1 - (K - 1) * d0 - 1;  // (owt - 1) * s0 at most
        owt                = room < 0 ? 0 : room / s0 + 1;
        if (owt >= 1 || ict == 1) {
            break;
        }
    }
    if (owt < 1) {
        return SHP_ERR_UNSUPPORTED;  // one channel's receptive field alone passes the window
    }
    const int64_t want = rule.elems / (ict * K) > rule.owt ? rule.elems / (ict * K) : rule.owt;
    owt                = owt < want ? owt : want;
    owt                = owt < OW ? owt : OW;
    const int64_t tic = (IC + ict - 1) / ict, tow = (OW + owt - 1) / owt;
    if (IC * K > INT32_MAX || OW > INT32_MAX || N > INT32_MAX || tic * tow * N > INT32_MAX) {
        return SHP_ERR_UNSUPPORTED;
    }
    const int64_t wt = window(owt, s0, K, d0);
    // the window walk's byte offsets are 32-bit
    if ((ict - 1) * nb1 + (wt - 1) * nb0 + kIm2colBlock * (nb0 + nb1) > INT32_MAX) {
        return SHP_ERR_UNSUPPORTED;
    }
    const int64_t last = IC - (tic - 1) * ict;  // channels of the last channel tile
    Im2colArgs &  a    = pl.args;
    a.x                = static_cast<const char *>(x->data);
    a.y                = static_cast<char *>(y->data);
    a.xnb0             = nb0;
    a.xnb1             = nb1;
    a.xnb2             = static_cast<int64_t>(x->nb[2]);
    a.iw               = IW;
    a.ic               = IC;
    a.ow               = OW;
    a.row              = IC * K;
    a.k                = static_cast<int32_t>(K);
    a.s0               = s0;
    a.p0               = p0;
    a.d0               = d0;
    a.ict              = static_cast<int32_t>(ict);
    a.owt              = static_cast<int32_t>(owt);
    a.wt               = static_cast<int32_t>(wt);
    pl.walk            = pl.chfast ? kWalkChannels : (nb0 == 4 && !(pl.f16 && by_value(a, N)) ? kWalkTime : kWalkValues);
    a.wtp              = static_cast<int32_t>(padded(wt, pl.walk == kWalkTime));
    a.tic              = make_fastdiv(static_cast<uint32_t>(tic));
    a.tow              = make_fastdiv(static_cast<uint32_t>(tow));
    a.kdiv             = make_fastdiv(static_cast<uint32_t>(K));
    a.rdiv             = make_fastdiv(static_cast<uint32_t>(IC * K));
    a.segf             = make_fastdiv(static_cast<uint32_t>(ict * K));
    a.segl             = make_fastdiv(static_cast<uint32_t>(last * K));
    const int64_t per  = pl.walk == kWalkValues ? 1 : 4;  // values per load
    const int64_t nf   = ((pl.chfast ? ict : wt) + per - 1) / per;
    a.fdiv             = make_fastdiv(static_cast<uint32_t>(nf));
    a.ns               = static_cast<int32_t>(pl.chfast ? wt : ict);
    a.ds               = static_cast<int32_t>(kIm2colBlock / nf);
    a.df               = static_cast<int32_t>(kIm2colBlock % nf);
    a.nbs              = static_cast<int32_t>(pl.chfast ? nb0 : nb1);
    a.nbf              = static_cast<int32_t>((pl.chfast ? nb1 : nb0) * per);
    a.ls               = pl.chfast ? 1 : a.wtp;
    a.lf               = static_cast<int32_t>((pl.chfast ? a.wtp : 1) * per);
    // Stores of 16 bytes where the layout allows (8 values of F16, 4 of F32),
    // else 8 bytes of F16, else one value. One table period must fit.
    const size_t    esz   = pl.f16 ? 2 : 4;
    const uintptr_t yaddr = reinterpret_cast<uintptr_t>(y->data);
    pl.flat               = ict == IC;
    pl.v                  = 1;
    for (int v : { pl.f16 ? 8 : 4, 4 }) {
        const bool    aligned = yaddr % (v * esz) == 0;
        const bool    runs    = (IC * K) % v == 0 && (ict * K) % v == 0;
        const int64_t per     = pl.flat ? IC * K * v / gcd64(IC * K, v) : ict * K;  // table entries
        if (aligned && (pl.flat || runs) && per <= kIm2colTab) {
            pl.v = v;
            break;
        }
    }
    pl.grid  = static_cast<unsigned>(tic * tow * N);
    pl.shmem = static_cast<size_t>(ict * a.wtp) * sizeof(float);
    return SHP_OK;
}

shp_status_t launch_im2col(const Im2colPlan & pl, hipStream_t s) {
    const Im2colArgs & a = pl.args;
    const int          c = pl.walk;
    if (pl.f16) {
        if (pl.flat) {
            pl.v == 8 ? launch_form<true, 8, true>(a, c, pl.grid, pl.shmem, s) :
            pl.v == 4 ? launch_form<true, 4, true>(a, c, pl.grid, pl.shmem, s) :
                        launch_form<true, 1, true>(a, c, pl.grid, pl.shmem, s);
        } else {
            pl.v == 8 ? launch_form<false, 8, true>(a, c, pl.grid, pl.shmem, s) :
            pl.v == 4 ? launch_form<false, 4, true>(a, c, pl.grid, pl.shmem, s) :
                        launch_form<false, 1, true>(a, c, pl.grid, pl.shmem, s);
        }
    } else if (pl.flat) {
        pl.v == 4 ? launch_form<true, 4, false>(a, c, pl.grid, pl.shmem, s) :
                    launch_form<true, 1, false>(a, c, pl.grid, pl.shmem, s);
    } else {
        pl.v == 4 ? launch_form<false, 4, false>(a, c, pl.grid, pl.shmem, s) :
                    launch_form<false, 1, false>(a, c, pl.grid, pl.shmem, s);
    }
    return launch_status();
}

}  // namespace shp

using namespace shp;

extern "C" shp_status_t shp_im2col(const shp_tensor * kernel, const shp_tensor * x, int32_t s0, int32_t p0, int32_t d0,
                                   shp_tensor * y, shp_stream_t stream) {
    Im2colPlan         pl;
    const shp_status_t st = plan_im2col(kernel, x, s0, p0, d0, y, pl);
    if (st != SHP_OK || dry_run()) {
        return st;
    }
    return launch_im2col(pl, as_stream(stream));
}
