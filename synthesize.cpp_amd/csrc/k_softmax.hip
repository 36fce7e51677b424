// ggml_soft_max_ext(a, mask, scale, max_bias = 0) for gfx950: the attention
// softmax of src/arch/qwen3-tts/operations.cpp:131-133 (scores over the cached
// keys, scaled by 1/sqrt(head_dim), causal mask).
//
// Per row, in ggml-CPU's rounding order:
//   w_i  = x_i*scale + 1*mask_i          (f32; the slope is 1 without ALiBi)
//   m    = max_i w_i
//   v_i  = exp(w_i - m)                  (f32 difference, exp rounded to f32)
//   sum  = sum_i (double) v_i            (double)
//   y_i  = v_i * (float)(1/sum)          (the reciprocal in double, rounded to f32)
// The exp is shp_expf.hpp's table-driven exp, within ~2^-44 before its f32
// rounding: it differs from the correctly rounded exp on 19 of the 2^32 f32
// inputs, glibc's expf (the CPU's) on 170,648. The double sum is added in a
// different order than the CPU's loop, which moves the f32 reciprocal only
// when the sum lies within ~1e-16 of a rounding boundary. A row holding a NaN
// or +inf (or only -inf) comes out NaN, as on the CPU: the max is then NaN or
// inf, or the NaN reaches the sum.
//
// Launch shapes: rows of up to 16384 scores are held in the registers of 1 to
// 16 waves, a float4 from any 4-byte boundary at a time (a prompt of an odd
// length has odd rows): one wave per row (wave-level reductions only: no LDS,
// no barrier) where the rows fill the chip, more where they are few or long
// (the decode step's 16 rows, a short prefill). Longer rows take one block and
// three passes over the row; rows of up to 128 scores, and odd ones up to 512 of
// which there are not many, a wave and an element per lane at a time.

#include <cmath>

#include "shp_expf.hpp"
#include "shp_internal.hpp"

namespace shp {
namespace {

struct SoftMaxArgs {
    const float * x;
    RowMap        xm;
    const float * mask;  // null: no mask
    int64_t       mnb1;
    int64_t       mnb2;
    int64_t       mnb3;
    int64_t       mne2;  // mask heads (broadcast: head i2 reads mask head i2 % mne2)
    int64_t       mne3;
    float *       y;
    RowMap        ym;
    int64_t       nrows;
    int64_t       ne1;   // rows per head
    int64_t       ne2;   // heads
    int32_t       ne0;
    float         scale;
    // Every row index and mask extent below 2^32: the mask row's indices come
    // from multiply-shift divisions (FastDiv) instead of 64-bit divisions.
    int32_t       mfast;
    int32_t       pad;
    int64_t       block0;  // the launch's first block
    int64_t       n_past;  // causal form: element i of row r is masked when i > n_past + r % ne1
    FastDiv       fne1;
    FastDiv       fne2;
    FastDiv       fmne2;
    FastDiv       fmne3;
};

// Mask forms: none, a mask tensor added to the scaled scores, or the causal
// mask of ggml_diag_mask_inf in front of the softmax (the masked scores
// replaced by -inf before the scale, as the two nodes compute them: a masked
// +inf or NaN score drops out instead of turning the row into NaN).
enum MaskKind { kMaskNone = 0, kMaskTensor = 1, kMaskCausal = 2 };

constexpr int kSoftMaxRegs  = 16384;  // widest row held in registers
constexpr int kSoftMaxBlock = 1024;   // threads per longer row

// Mask row of score row r = (i1, i2, i3): ggml's i11 = i1, i12 = i2 % ne12,
// i13 = i3 % ne13.
__device__ __forceinline__ const float * mask_row(const SoftMaxArgs & a, int64_t r) {
    if (a.mfast) {
        const uint32_t q  = fastdiv(static_cast<uint32_t>(r), a.fne1);
        const uint32_t i1 = static_cast<uint32_t>(r) - q * a.fne1.d;
        const uint32_t i3 = fastdiv(q, a.fne2);
        const uint32_t i2 = q - i3 * a.fne2.d;
        return reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.mask) + i1 * a.mnb1 +
                                               fastmod(i2, a.fmne2) * a.mnb2 + fastmod(i3, a.fmne3) * a.mnb3);
    }
    const int64_t i1 = r % a.ne1;
    const int64_t q  = r / a.ne1;
    const int64_t i2 = q % a.ne2;
    const int64_t i3 = q / a.ne2;
    return reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.mask) + i1 * a.mnb1 +
                                           (i2 % a.mne2) * a.mnb2 + (i3 % a.mne3) * a.mnb3);
}

// The causal form's last unmasked element of row r: n_past + i1.
__device__ __forceinline__ int64_t causal_lim(const SoftMaxArgs & a, int64_t r) {
    if (a.mfast) {
        return a.n_past + fastmod(static_cast<uint32_t>(r), a.fne1);
    }
    return a.n_past + r % a.ne1;
}

// The kernel arguments a softmax wave needs before its first load.
template <int MK> __device__ __forceinline__ void softmax_args_in_sgprs(const SoftMaxArgs & a) {
    args_in_sgprs(a.x, a.xm.flat, a.xm.rs, a.y, a.ym.flat, a.ym.rs, a.nrows, a.ne0, a.scale);
    if constexpr (MK == kMaskTensor) {
        args_in_sgprs(a.mask, a.mfast, a.fne1.d, a.fne1.m, a.fne1.l, a.fne2.d, a.fne2.m, a.fne2.l, a.fmne2.d,
                      a.fmne2.m, a.fmne2.l, a.fmne3.d, a.fmne3.m, a.fmne3.l, a.mnb1, a.mnb2, a.mnb3);
    }
}

// One wave per row of up to 64 K scores (K at most 8), element lane + 64k in
// register k: a short row's lane then has one or two exps in its chain, not a
// float4's four (a decode step's 16 rows of 38: 1.71 us, 2.04 by float4).
template <int K, int MK> __global__ __launch_bounds__(256) void k_soft_max_wave(const SoftMaxArgs a) {
    constexpr bool MASK = MK == kMaskTensor;
    __shared__ double s_tab[256 / kWave][64];
    softmax_args_in_sgprs<MK>(a);
    const int     lane = threadIdx.x % kWave;
    const int64_t r    = (a.block0 + blockIdx.x) * (256 / kWave) +
                      __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    if (r >= a.nrows) {
        return;  // whole wave
    }
    const float * xr = reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.x) + row_offset(a.xm, r));
    float *       yr = reinterpret_cast<float *>(reinterpret_cast<char *>(a.y) + row_offset(a.ym, r));
    const float * mr  = MASK ? mask_row(a, r) : nullptr;
    const int64_t lim = MK == kMaskCausal ? causal_lim(a, r) : 0;
    float         w[K];
    float         mk[K];
    // The exp table's entry is loaded with the row. Loads are unconditional
    // (a lane past the row re-reads element 0) and out-of-row values are
    // zeroed by selects afterwards: a guarded load becomes a branch with a
    // wait of its own.
    const double entry = exp_table_entry(lane);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = lane + kWave * k;
        w[k]        = xr[i < a.ne0 ? i : 0];
        mk[k]       = MASK ? mr[i < a.ne0 ? i : 0] : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const bool in = lane + kWave * k < a.ne0;
        w[k]          = in ? w[k] : 0.0f;
        mk[k]         = in ? mk[k] : 0.0f;
    }
    const double * tab = wave_exp_table(s_tab, lane, entry);
    float          mx  = -INFINITY;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = lane + kWave * k;
        w[k]        = w[k] * a.scale;
        if constexpr (MASK) {
            w[k] = w[k] + mk[k];
        }
        if constexpr (MK == kMaskCausal) {
            w[k] = i > lim ? -INFINITY : w[k];
        }
        mx = i < a.ne0 ? fmaxf(mx, w[k]) : mx;
    }
    mx         = wave_max(mx);
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = lane + kWave * k;
        w[k]        = exp_f32_lds(w[k] - mx, tab);
        sum += i < a.ne0 ? static_cast<double>(w[k]) : 0.0;
    }
    sum             = group_sum<kWave>(sum);
    const float inv = static_cast<float>(1.0 / sum);
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = lane + kWave * k;
        if (i < a.ne0) {
            yr[i] = w[k] * inv;
        }
    }
}

// Rows of at least four scores, WPR waves per row: lane q of the row's 64*WPR
// lanes holds chunks q + 64*WPR*k in registers k (k < K4). Chunk c is the four
// scores from 4c on; the row's last chunk, where fewer are left, the row's last
// four, whose first ones belong to the chunk before (left out of the sum here,
// and stored twice with the same value).
// The scores are read and the probabilities written once per launch, so both
// stream with the nontemporal hint (the mask, shared by heads, stays
// cacheable): 21 % faster than plain loads and stores at [512,512,16] on
// MI355X (9.65 -> 7.58 us). The causal form does not read a chunk that the mask
// hides, nor take its exps. Measured on MI355X (cold) against a wave per row with
// 4-byte accesses for odd rows and a 256-thread block of three passes past 2048:
// 16 heads of 1021 x 1021 31.0 -> 27.0 us, with a mask 35.4 -> 31.7, causal 30.2 ->
// 23.8; 16 rows of 4000 9.6 -> 3.3, 16 x 16 rows of 4096 15.8 -> 4.7, 8 x 64 of
// 12000 66 -> 14; 1024 x 1024 with aligned rows unchanged (26.2). Slower for 1021:
// two or four waves a row (30.1, 33.8). With a mask, blocks of one position's
// four heads, to share its row: 30.8, but 28.1 against 26.8 at 1024.
// WPR > 1 spreads the few long rows of a decode or short prefill over more
// waves; the row's waves then combine their max and sum through LDS, in wave
// order.
// ODD: the row is no whole number of chunks.
template <int WPR, int K4, int MK, bool ODD, int BLOCK = (WPR > 4 ? WPR * kWave : 256)>
__global__ __launch_bounds__(BLOCK) void k_soft_max_rows4(const SoftMaxArgs a) {
    constexpr bool MASK   = MK == kMaskTensor;
    constexpr int  kLanes = kWave * WPR;
    __shared__ float  s_max[BLOCK / kWave];
    __shared__ double s_sum[BLOCK / kWave];
    __shared__ double s_tab[BLOCK / kWave][64];
    softmax_args_in_sgprs<MK>(a);
    const int     lane = threadIdx.x % kWave;
    const int     q    = threadIdx.x % kLanes;
    const int     wv   = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    const int     slot = wv / WPR;  // row of this block
    const int64_t r    = (a.block0 + blockIdx.x) * (BLOCK / kLanes) + slot;
    const bool    live = r < a.nrows;
    if (WPR == 1 && !live) {
        return;  // whole wave; the one-wave form has no barrier
    }
    const int64_t rr = live ? r : 0;
    const float * xr = reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.x) + row_offset(a.xm, rr));
    float *       yr = reinterpret_cast<float *>(reinterpret_cast<char *>(a.y) + row_offset(a.ym, rr));
    const float * mr = MASK ? mask_row(a, rr) : nullptr;
    const int64_t lim  = MK == kMaskCausal ? causal_lim(a, rr) : 0;
    const int     nc   = live ? (a.ne0 + 3) / 4 : 0;
    const int     last = a.ne0 - 4;  // the last chunk's first score
    auto          first = [last](int c) { return ODD && c * 4 > last ? last : c * 4; };  // of chunk c
    f32x4         w[K4];
    f32x4         mk[K4];
    // The exp table's entry is loaded with the row, so it is not a round trip
    // of its own. Loads are unconditional (a lane past the row re-reads chunk
    // 0 of row rr), zeroed by selects afterwards: a guarded load becomes a
    // branch with a wait of its own.
    const double entry = exp_table_entry(lane);
#pragma unroll
    for (int k = 0; k < K4; ++k) {
        const int c = q + kLanes * k;
        const int i = c < nc ? first(c) : 0;
        if constexpr (MK == kMaskCausal) {
            w[k] = splat4(-INFINITY);
            if (i <= lim) {
                w[k] = ld_stream4u(xr + i);
            }
        } else {
            w[k] = ld_stream4u(xr + i);
        }
        mk[k] = MASK ? ld4u(mr + i) : splat4(0.0f);
    }
#pragma unroll
    for (int k = 0; k < K4; ++k) {
        const bool in = q + kLanes * k < nc;
        w[k]          = in ? w[k] : splat4(0.0f);
        mk[k]         = in ? mk[k] : splat4(0.0f);
    }
    const double * tab = wave_exp_table(s_tab, lane, entry);
    float          mx  = -INFINITY;
#pragma unroll
    for (int k = 0; k < K4; ++k) {
        const int c = q + kLanes * k;
        w[k]        = f32x4{ w[k].x * a.scale, w[k].y * a.scale, w[k].z * a.scale, w[k].w * a.scale };
        if constexpr (MASK) {
            w[k] = f32x4{ w[k].x + mk[k].x, w[k].y + mk[k].y, w[k].z + mk[k].z, w[k].w + mk[k].w };
        }
        if constexpr (MK == kMaskCausal) {
            const int64_t i = first(c);
            w[k]            = f32x4{ i > lim ? -INFINITY : w[k].x, i + 1 > lim ? -INFINITY : w[k].y,
                                     i + 2 > lim ? -INFINITY : w[k].z, i + 3 > lim ? -INFINITY : w[k].w };
        }
        const float m4 = fmaxf(fmaxf(w[k].x, w[k].y), fmaxf(w[k].z, w[k].w));
        mx             = c < nc ? fmaxf(mx, m4) : mx;
    }
    mx = wave_max(mx);
    if constexpr (WPR > 1) {
        if (lane == 0) {
            s_max[wv] = mx;
        }
        __syncthreads();
        mx = s_max[slot * WPR];
#pragma unroll
        for (int j = 1; j < WPR; ++j) {
            mx = fmaxf(mx, s_max[slot * WPR + j]);
        }
    }
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < K4; ++k) {
        const int c = q + kLanes * k;
        if (MK == kMaskCausal && kLanes * k * 4 > lim + 3 && mx > -INFINITY) {
            // the row's chunks from here on are all hidden, the scores a last chunk shares
            // with the one before it included: e^-inf (an infinite or NaN
            // maximum takes the exps)
            w[k] = splat4(0.0f);
            continue;
        }
        w[k] = f32x4{ exp_f32_lds(w[k].x - mx, tab), exp_f32_lds(w[k].y - mx, tab), exp_f32_lds(w[k].z - mx, tab),
                      exp_f32_lds(w[k].w - mx, tab) };
        // the last chunk's scores that are the chunk before's
        const int    twice = ODD ? c * 4 - last : 0;
        const double s4    = (static_cast<double>(twice > 0 ? 0.0f : w[k].x) + static_cast<double>(twice > 1 ? 0.0f : w[k].y)) +
                          (static_cast<double>(twice > 2 ? 0.0f : w[k].z) + static_cast<double>(w[k].w));
        sum += c < nc ? s4 : 0.0;
    }
    sum = group_sum<kWave>(sum);
    if constexpr (WPR > 1) {
        if (lane == 0) {
            s_sum[wv] = sum;
        }
        __syncthreads();
        sum = s_sum[slot * WPR];
#pragma unroll
        for (int j = 1; j < WPR; ++j) {
            sum += s_sum[slot * WPR + j];
        }
    }
    const float inv = static_cast<float>(1.0 / sum);
#pragma unroll
    for (int k = 0; k < K4; ++k) {
        const int c = q + kLanes * k;
        if (c < nc) {
            st_stream4u(yr + first(c),
                        f32x4{ w[k].x * inv, w[k].y * inv, w[k].z * inv, w[k].w * inv });
        }
    }
}

// One block per row too long for registers, three passes: the max, the sum,
// the scaled exps; chunks as above.
template <int MK>
__device__ __forceinline__ f32x4 sm_w4(const SoftMaxArgs & a, const float * xr, const float * mr, int64_t lim, int i) {
    f32x4 w;
    if constexpr (MK == kMaskCausal) {
        w = i <= lim ? ld4u(xr + i) : splat4(-INFINITY);
    } else {
        w = ld4u(xr + i);
    }
    w = f32x4{ w.x * a.scale, w.y * a.scale, w.z * a.scale, w.w * a.scale };
    if constexpr (MK == kMaskTensor) {
        const f32x4 m = ld4u(mr + i);
        w             = f32x4{ w.x + m.x, w.y + m.y, w.z + m.z, w.w + m.w };
    }
    if constexpr (MK == kMaskCausal) {
        w = f32x4{ i > lim ? -INFINITY : w.x, i + 1 > lim ? -INFINITY : w.y, i + 2 > lim ? -INFINITY : w.z,
                   i + 3 > lim ? -INFINITY : w.w };
    }
    return w;
}

template <int MK> __global__ __launch_bounds__(kSoftMaxBlock) void k_soft_max_block(const SoftMaxArgs a) {
    constexpr bool MASK   = MK == kMaskTensor;
    constexpr int  kWaves = kSoftMaxBlock / kWave;
    __shared__ float  s_max[kWaves];
    __shared__ double s_sum[kWaves];
    __shared__ double s_tab[kWaves][64];
    const int64_t  r    = a.block0 + blockIdx.x;
    const int      lane = threadIdx.x % kWave;
    const int      wv   = threadIdx.x / kWave;
    const float *  xr   = reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.x) + row_offset(a.xm, r));
    float *        yr   = reinterpret_cast<float *>(reinterpret_cast<char *>(a.y) + row_offset(a.ym, r));
    const float *  mr   = MASK ? mask_row(a, r) : nullptr;
    const int64_t  lim  = MK == kMaskCausal ? causal_lim(a, r) : 0;
    const int      nc   = (a.ne0 + 3) / 4, last = a.ne0 - 4;
    const double * tab  = wave_exp_table(s_tab, lane, exp_table_entry(lane));

    float mx = -INFINITY;
#pragma unroll 2
    for (int c = threadIdx.x; c < nc; c += kSoftMaxBlock) {
        const f32x4 w = sm_w4<MK>(a, xr, mr, lim, c * 4 < last ? c * 4 : last);
        mx            = fmaxf(mx, fmaxf(fmaxf(w.x, w.y), fmaxf(w.z, w.w)));
    }
    mx = wave_max(mx);
    if (lane == 0) {
        s_max[wv] = mx;
    }
    __syncthreads();
    mx = s_max[0];
#pragma unroll
    for (int j = 1; j < kWaves; ++j) {
        mx = fmaxf(mx, s_max[j]);
    }

    double sum = 0.0;
#pragma unroll 2
    for (int c = threadIdx.x; c < nc; c += kSoftMaxBlock) {
        const f32x4 w     = sm_w4<MK>(a, xr, mr, lim, c * 4 < last ? c * 4 : last);
        const int   twice = c * 4 - last;
        const float e0 = exp_f32_lds(w.x - mx, tab), e1 = exp_f32_lds(w.y - mx, tab), e2 = exp_f32_lds(w.z - mx, tab);
        sum += (static_cast<double>(twice > 0 ? 0.0f : e0) + static_cast<double>(twice > 1 ? 0.0f : e1)) +
               (static_cast<double>(twice > 2 ? 0.0f : e2) + static_cast<double>(exp_f32_lds(w.w - mx, tab)));
    }
    sum = group_sum<kWave>(sum);
    if (lane == 0) {
        s_sum[wv] = sum;
    }
    __syncthreads();
    sum = s_sum[0];
#pragma unroll
    for (int j = 1; j < kWaves; ++j) {
        sum += s_sum[j];
    }
    const float inv = static_cast<float>(1.0 / sum);
    // Each score is written by the chunk that owns it (the last chunk's shared
    // ones by the chunk before), which has read it: in place, nothing reads a
    // written score but the last chunk, read ahead of the barrier.
    const int   tail  = nc - 1;
    const bool  owner = static_cast<int>(threadIdx.x) == tail % kSoftMaxBlock;
    const f32x4 wt    = owner ? sm_w4<MK>(a, xr, mr, lim, last) : splat4(0.0f);
    __syncthreads();
#pragma unroll 2
    for (int c = threadIdx.x; c < tail; c += kSoftMaxBlock) {
        const f32x4 w = sm_w4<MK>(a, xr, mr, lim, c * 4);
        st_stream4u(yr + c * 4, f32x4{ exp_f32_lds(w.x - mx, tab) * inv, exp_f32_lds(w.y - mx, tab) * inv,
                                       exp_f32_lds(w.z - mx, tab) * inv, exp_f32_lds(w.w - mx, tab) * inv });
    }
    if (owner) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (last + e >= tail * 4) {
                yr[last + e] = exp_f32_lds(wt[e] - mx, tab) * inv;
            }
        }
    }
}

// Rows of 257 to 512 float4 in one wave (launch_rows4).
inline bool one_wave(int64_t nrows, int nc, bool mask) {
    return nrows > (nc > 400 ? 2688 : 4608) && nrows <= (mask ? 3328 : 6144);
}

// The forms' rule reads the row count and length, and whether a mask tensor is
// added, so that the causal launch adds a row in the order that the softmax alone
// does: diag_mask_inf and soft_max_ext come out bit for bit the same in one launch.
template <int MK, bool ODD, class Go> shp_status_t launch_rows4(const SoftMaxArgs & a, const Go & go) {
    const int nc = (a.ne0 + 3) / 4;
    if (nc <= 64) {
        return go(k_soft_max_rows4<1, 1, MK, ODD>, 4, 256);
    }
    // Few rows (under 8 waves per CU at one wave per row): 2, 4 or 16 waves per
    // row. The decode step's 16 rows of 512 take one wave each (2.30 us
    // against 2.36 us with two waves and their LDS combine, MI355X), in
    // one-wave blocks: each row on its own CU (2.12 -> 1.99 us warm; the
    // 28-layer decode graph's layer with the softmax 9.62 -> 9.45 us). Rows
    // of 513-1023 scores: four waves, odd ones below 1024 rows (16 of 601: 2.85
    // us, one wave 3.2, two 3.0; 1024: 4.6, 4.2, 4.4), whole ones up to 64.
    if (a.nrows < 2048 && nc >= 128) {
        if (nc >= 256) {
            if (a.nrows <= 256 && nc > 512) {
                return nc <= 1024 ? go(k_soft_max_rows4<16, 1, MK, ODD>, 1, 1024) :
                       nc <= 2048 ? go(k_soft_max_rows4<16, 2, MK, ODD>, 1, 1024) :
                                    go(k_soft_max_rows4<16, 4, MK, ODD>, 1, 1024);
            }
            return nc <= 256  ? go(k_soft_max_rows4<4, 1, MK, ODD>, 1, 256) :
                   nc <= 512  ? go(k_soft_max_rows4<4, 2, MK, ODD>, 1, 256) :
                   nc <= 1024 ? go(k_soft_max_rows4<4, 4, MK, ODD>, 1, 256) :
                   nc <= 2048 ? go(k_soft_max_rows4<4, 8, MK, ODD>, 1, 256) :
                                go(k_soft_max_rows4<16, 4, MK, ODD>, 1, 1024);
        }
        if (nc > 128 && a.nrows < (ODD ? 1024 : 65)) {
            return go(k_soft_max_rows4<4, 1, MK, ODD>, 1, 256);
        }
        if (!ODD && a.nrows > 64) {
            return nc <= 128 ? go(k_soft_max_rows4<2, 1, MK, ODD>, 2, 256) : go(k_soft_max_rows4<2, 2, MK, ODD>, 2, 256);
        }
    }
    if (nc <= 128) {
        // a decode step's few rows: one one-wave block per row
        return a.nrows <= 64 ? go(k_soft_max_rows4<1, 2, MK, ODD, kWave>, 1, kWave) :
                               go(k_soft_max_rows4<1, 2, MK, ODD>, 4, 256);
    }
    // Many rows: one wave up to 1024 scores, two up to 2048 (8 heads of 2000 x
    // 2000, one wave / two / four: no mask 46.3 us / 44.5 / 45.1, with a mask 57.1
    // / 49.8 / 50.4, causal 39.6 / 35.8 / 40.2; 16 of 1100 x 1100: 36.5 / 38.5 /
    // 41.8, 41.7 / 40.4 / 45.2, 26.4 / 26.8 / 32.8), but one where two waves a
    // row begin a second round of the chip that one does not, until the rounds even
    // out: rows past 1600 scores from some 2700, shorter ones from 4600 (no mask and
    // causal, one wave / two: 2560 x 1800 9.6 / 8.3 and 10.3 / 9.1, 3072 x 2000 10.2 /
    // 13.4 and 11.3 / 10.7, 4096 x 2000 12.7 / 14.0 and 13.0 / 13.7, 5120 x 1200 12.4 / 12.5
    // and 10.9 / 12.5, 8192 x 2000 25.6 / 24.6 and 25.5 / 24.3; with a mask 3072 x 2000
    // 11.1 / 12.8, 5120 x 1800 18.4 / 17.8).
    if (nc > 256 && nc <= 512 && one_wave(a.nrows, nc, MK == kMaskTensor)) {
        return go(k_soft_max_rows4<1, 8, MK, ODD>, 4, 256);
    }
    return nc <= 256  ? go(k_soft_max_rows4<1, 4, MK, ODD>, 4, 256) :
           nc <= 512  ? go(k_soft_max_rows4<2, 4, MK, ODD>, 2, 256) :
           nc <= 1024 ? go(k_soft_max_rows4<4, 4, MK, ODD>, 1, 256) :
           nc <= 2048 ? go(k_soft_max_rows4<4, 8, MK, ODD>, 1, 256) : go(k_soft_max_rows4<16, 4, MK, ODD>, 1, 1024);
}

// Up to 128 scores, and odd rows up to 512 where a wave each leaves the chip
// room, an element per lane at a time: the last float4 of an odd row costs a
// lane four exps for its one to three scores (16 rows of 301, MI355X: 2.53 us,
// 2.82 by float4; 1024: 3.0 and 3.6; 2048: 3.6 and 4.1; but 16384: 13.0 and
// 12.2; of 511, 2048: 4.3 and 4.4, 4096: 6.9 and 5.7).
inline bool by_elements(const SoftMaxArgs & a) {
    return a.ne0 <= 2 * kWave || (a.ne0 % 4 != 0 && a.ne0 <= 8 * kWave && a.nrows <= (a.ne0 <= 5 * kWave ? 4096 : 2048));
}

template <int MK> shp_status_t launch_soft_max(const SoftMaxArgs & a, hipStream_t stream) {
    if (dry_run()) {
        return SHP_OK;
    }
    auto go = [&](auto kernel, int rows_per_block, int block) {
        return in_launches((a.nrows + rows_per_block - 1) / rows_per_block, block, [&](int64_t first, dim3 grid) {
            SoftMaxArgs part = a;
            part.block0      = first;
            hipLaunchKernelGGL(kernel, grid, dim3(block), 0, stream, part);
        });
    };
    if (by_elements(a)) {
        return a.ne0 <= 1 * kWave ? go(k_soft_max_wave<1, MK>, 4, 256) :
               a.ne0 <= 2 * kWave ? go(k_soft_max_wave<2, MK>, 4, 256) :
               a.ne0 <= 3 * kWave ? go(k_soft_max_wave<3, MK>, 4, 256) :
               a.ne0 <= 4 * kWave ? go(k_soft_max_wave<4, MK>, 4, 256) :
               a.ne0 <= 6 * kWave ? go(k_soft_max_wave<6, MK>, 4, 256) : go(k_soft_max_wave<8, MK>, 4, 256);
    }
    if (a.ne0 > kSoftMaxRegs) {
        return go(k_soft_max_block<MK>, 1, kSoftMaxBlock);
    }
    return a.ne0 % 4 == 0 ? launch_rows4<MK, false>(a, go) : launch_rows4<MK, true>(a, go);
}

}  // namespace
}  // namespace shp

using namespace shp;

extern "C" shp_status_t shp_soft_max_ext(const shp_tensor * a,
                                         const shp_tensor * mask,
                                         float              scale,
                                         float              max_bias,
                                         shp_tensor *       y,
                                         shp_stream_t       stream) {
    if (!well_formed(a) || !well_formed(y) || (mask != nullptr && !well_formed(mask))) {
        return SHP_ERR_INVALID_ARG;
    }
    if (a->type != SHP_TYPE_F32 || y->type != SHP_TYPE_F32 || (mask != nullptr && mask->type != SHP_TYPE_F32)) {
        return SHP_ERR_UNSUPPORTED;
    }
    if (max_bias != 0.0f) {
        return SHP_ERR_UNSUPPORTED;  // ALiBi slopes: not on this path
    }
    if (!same_shape(*a, *y) || a->ne[0] > INT32_MAX || nrows(*a) > INT32_MAX) {
        return SHP_ERR_INVALID_ARG;
    }
    // ggml_soft_max_ext's mask contract: same row length, at least as many
    // rows, heads and batches broadcast by whole repeats.
    if (mask != nullptr && (mask->ne[0] != a->ne[0] || mask->ne[1] < a->ne[1] || a->ne[2] % mask->ne[2] != 0 ||
                            a->ne[3] % mask->ne[3] != 0)) {
        return SHP_ERR_INVALID_ARG;
    }
    SoftMaxArgs g{};
    g.x     = static_cast<const float *>(a->data);
    g.xm    = make_rowmap(*a);
    g.y     = static_cast<float *>(y->data);
    g.ym    = make_rowmap(*y);
    g.nrows = nrows(*a);
    g.ne1   = a->ne[1];
    g.ne2   = a->ne[2];
    g.ne0   = static_cast<int32_t>(a->ne[0]);
    g.scale = scale;
    if (mask != nullptr) {
        g.mask = static_cast<const float *>(mask->data);
        g.mnb1 = static_cast<int64_t>(mask->nb[1]);
        g.mnb2 = static_cast<int64_t>(mask->nb[2]);
        g.mnb3 = static_cast<int64_t>(mask->nb[3]);
        g.mne2 = mask->ne[2];
        g.mne3 = mask->ne[3];
        constexpr int64_t kU32 = int64_t{ UINT32_MAX };
        g.mfast = g.nrows <= kU32 && g.ne1 <= kU32 && g.ne2 <= kU32 && g.mne2 <= kU32 && g.mne3 <= kU32;
        if (g.mfast) {
            g.fne1  = make_fastdiv(static_cast<uint32_t>(g.ne1));
            g.fne2  = make_fastdiv(static_cast<uint32_t>(g.ne2));
            g.fmne2 = make_fastdiv(static_cast<uint32_t>(g.mne2));
            g.fmne3 = make_fastdiv(static_cast<uint32_t>(g.mne3));
        }
    }
    return mask != nullptr ? launch_soft_max<kMaskTensor>(g, as_stream(stream))
                           : launch_soft_max<kMaskNone>(g, as_stream(stream));
}

// ggml_diag_mask_inf(x, n_past): every element past n_past + its row's index
// in the matrix (i0 > n_past + i1) becomes -inf, the rest copied.
struct DiagMaskArgs {
    const float * x;
    RowMap        xm;
    float *       y;
    RowMap        ym;
    int64_t       n_past;
    int64_t       ne1;
    int64_t       total;  // rows x ne0
    FastDiv       fne0;
    FastDiv       fne1;
};

__global__ __launch_bounds__(256) void k_diag_mask_inf(const DiagMaskArgs a) {
    const int64_t step = static_cast<int64_t>(gridDim.x) * 256;
    for (int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; t < a.total; t += step) {
        const uint32_t r  = fastdiv(static_cast<uint32_t>(t), a.fne0);
        const uint32_t i0 = static_cast<uint32_t>(t) - r * a.fne0.d;
        const uint32_t i1 = fastmod(r, a.fne1);
        const float *  xr = reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.x) + row_offset(a.xm, r));
        float *        yr = reinterpret_cast<float *>(reinterpret_cast<char *>(a.y) + row_offset(a.ym, r));
        yr[i0]            = static_cast<int64_t>(i0) > a.n_past + i1 ? -INFINITY : xr[i0];
    }
}

extern "C" shp_status_t shp_diag_mask_inf(const shp_tensor * x, int32_t n_past, shp_tensor * y, shp_stream_t stream) {
    if (!well_formed(x) || !well_formed(y) || n_past < 0) {
        return SHP_ERR_INVALID_ARG;
    }
    if (x->type != SHP_TYPE_F32 || y->type != SHP_TYPE_F32) {
        return SHP_ERR_UNSUPPORTED;
    }
    if (!same_shape(*x, *y) || nelements(*x) > INT32_MAX) {
        return SHP_ERR_INVALID_ARG;
    }
    const bool in_place = x->data == y->data && x->nb[1] == y->nb[1] && x->nb[2] == y->nb[2] && x->nb[3] == y->nb[3];
    if (!in_place && spans_overlap(*x, *y)) {
        return SHP_ERR_UNSUPPORTED;
    }
    if (dry_run()) {
        return SHP_OK;
    }
    DiagMaskArgs g{};
    g.x                  = static_cast<const float *>(x->data);
    g.xm                 = make_rowmap(*x);
    g.y                  = static_cast<float *>(y->data);
    g.ym                 = make_rowmap(*y);
    g.n_past             = n_past;
    g.ne1                = x->ne[1];
    g.total              = nelements(*x);
    g.fne0               = make_fastdiv(static_cast<uint32_t>(x->ne[0]));
    g.fne1               = make_fastdiv(static_cast<uint32_t>(x->ne[1]));
    const int64_t blocks = (g.total + 255) / 256;
    hipLaunchKernelGGL(k_diag_mask_inf, dim3(static_cast<unsigned>(blocks < (1 << 20) ? blocks : (1 << 20))),
                       dim3(256), 0, as_stream(stream), g);
    return launch_status();
}

extern "C" shp_status_t shp_soft_max_causal(const shp_tensor * a,
                                            int32_t            n_past,
                                            float              scale,
                                            shp_tensor *       y,
                                            shp_stream_t       stream) {
    if (!well_formed(a) || !well_formed(y) || n_past < 0) {
        return SHP_ERR_INVALID_ARG;
    }
    if (a->type != SHP_TYPE_F32 || y->type != SHP_TYPE_F32) {
        return SHP_ERR_UNSUPPORTED;
    }
    // -inf times the scale is -inf only for a positive finite scale
    if (!(scale > 0.0f) || !(scale < INFINITY)) {
        return SHP_ERR_UNSUPPORTED;
    }
    if (!same_shape(*a, *y) || a->ne[0] > INT32_MAX || nrows(*a) > INT32_MAX) {
        return SHP_ERR_INVALID_ARG;
    }
    SoftMaxArgs g{};
    g.x      = static_cast<const float *>(a->data);
    g.xm     = make_rowmap(*a);
    g.y      = static_cast<float *>(y->data);
    g.ym     = make_rowmap(*y);
    g.nrows  = nrows(*a);
    g.ne1    = a->ne[1];
    g.ne2    = a->ne[2];
    g.ne0    = static_cast<int32_t>(a->ne[0]);
    g.scale  = scale;
    g.n_past = n_past;
    g.mfast  = 1;  // rows below 2^31
    g.fne1   = make_fastdiv(static_cast<uint32_t>(g.ne1));
    return launch_soft_max<kMaskCausal>(g, as_stream(stream));
}
