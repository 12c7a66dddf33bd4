// mfma.h -- matrix-core (MFMA) variant of the fused six-output Gaussian filter.
//
// The direct FP32 filter needs about 16 r + 6 vector operations per output
// pixel for the six outputs (262 at radius 16), which makes it VALU-bound at
// a quarter of the HBM roofline.  Here both passes run on the matrix cores as
// banded matrix products, and the vector units only split, scale and store.
//
// Strip: one wave64 filters 16 centre rows x 64 centre columns (4 blocks of
// 16 columns); a workgroup holds 4 strips, one above the other or two by two
// (MFMA_WYS), whose halo rows meet in L1 or in a window of the input in LDS.
// With RC the radius class (8 or 16; lobes zero-padded to it) and K = 16 + 2 RC:
//   vertical pass, per field block b (16 input columns starting at
//   x0 - RC + 16 b) and lobe l:
//       F^T (16 cols x 16 rows) = X^T (16 cols x K input rows) * T_l^T (K x 16)
//   horizontal pass, per output block o (16 columns starting at x0 + 16 o):
//       O^T (16 cols x 16 rows) = T_h^T (16 x K field cols) * F^T (K x 16 rows)
//   with T the band matrices of the lobes.  The vertical product's
//   accumulator layout (lane l: row l % 16, columns 4 (l / 16) .. +3) is
//   exactly the layout the horizontal product wants for its B operand when
//   the K index of the band matrix is permuted to match, so fields never
//   leave registers.
// Precision: matrix operands are f16.  A float v is scaled by a power of two
// and split as hi = f16(v), lo = f16(v - hi); the products hi*hi + hi*lo +
// lo*hi carry about 22 significant bits (the dropped lo*lo term and the
// split residual are each below 2^-22 relative), summed in FP32.  Scales
// (all powers of two): taps of lobe l by mp[l] (largest tap in [2^5, 2^6),
// MFMA_TAP_EXP); the input of each strip by mq times a factor putting its
// largest magnitude in [2^12, 2^13) (u8 input: the factor for 255, 2^5,
// whatever the strip holds), mq <= 1 / (L1 norm * mp) of every lobe,
// so that the vertical fields stay below 2^13 and no operand leaves the f16
// range; each output is multiplied back by mu[k] / (the strip's factor).
// Where lo falls below f16's normal range (2^-14) it keeps an absolute
// 2^-25 instead of 11 more bits, so the error of an output is bounded by
// about 2^-25 (L1 / X + n tapmax / T) times the strip's largest input, with
// X and T the scaled input and tap peaks; the tap peak of 2^6 balances the
// two terms (a peak of 2^12 left the inputs at a quarter and their lo
// halves subnormal below half the strip's largest value: 20x the error on
// an image whose strips mix 0..255 data with values of 10^6).
// A strip whose input holds a NaN or an Inf, or whose largest magnitude the
// scale cannot bring into range, is filtered by the FP32 form, and so is every
// strip where a tap is not finite or a lobe so small that its scale overflows
// (mfma_strip_fp32), which reaches exactly the outputs whose window holds
// a non-finite input, as the reference's tap sums do.
#pragma once

#include "sepfir.h"
#include "batch.h"

#include <algorithm>
#include <type_traits>

namespace tucu {

typedef _Float16 v4f16 __attribute__((ext_vector_type(4)));
typedef _Float16 v8f16 __attribute__((ext_vector_type(8)));

constexpr int MSTRIP_W = 64;              // centre columns per strip
constexpr int MNB      = MSTRIP_W / 16;   // output blocks per strip
constexpr int MWAVES   = 4;               // strips (waves) per workgroup
constexpr int MOPITCH  = MSTRIP_W + 4;    // row pitch (floats) of a wave's output staging area
constexpr int MT4      = 112;             // tap-run table entries per lobe
constexpr int MBASE    = 64;              // run t starts with tap t - MBASE
constexpr int MHP      = MT4 - 16;        // entries of the horizontal pair table
constexpr int MINVALID = int(0x80000000u);   // buffer offset past any image: loads return 0
constexpr int MFMA_TAP_EXP = 6;           // largest scaled tap of each lobe in [2^5, 2^6)

template <int RC> struct MGeo {
    static constexpr bool K48 = RC == 16;                 // K = 48 (two 32-entry slices), else 32
    static constexpr int  KV  = 16 + 2 * RC;              // input rows per strip
    static constexpr int  NVB = MNB + (K48 ? 2 : 1);      // field blocks per strip
    static constexpr int  NLD = K48 ? 12 : 8;             // input values per lane per block
};

#ifdef TUCU_TIMELINE
// Phase timeline of the one-round six-output launch (radius class 16, float
// in and out), in a build made for it (make timeline; read by
// tucuda_amd/timeline.py): lane 0 of each wave writes the 100 MHz real-time
// counter into slot i of its row of tucu_timeline at each phase -- 0 start,
// 10 strip loads issued, 11 operand tables copied, 1 barrier passed, 2
// input scaled and split, 3 + k output k stored, 9 end.  The default build
// has none of it.
constexpr int TL_SLOTS = 12;
constexpr int TL_WAVES = 2048;
static __device__ uint64_t tucu_timeline[TL_WAVES * TL_SLOTS];
__device__ __forceinline__ void tl_stamp(int i)
{
    const uint64_t t = __builtin_amdgcn_s_memrealtime();
    const unsigned w = blockIdx.x * MWAVES + (threadIdx.x >> 6);
    if ((threadIdx.x & 63) == 0 && w < unsigned(TL_WAVES)) tucu_timeline[w * TL_SLOTS + i] = t;
}
#endif

// Per-lane operand runs, in LDS: run[(part * 3 + l) * MT4 + t] holds taps
// t - MBASE .. t - MBASE + 3 of lobe l, times mp[l], as four f16 (part 0 the high
// half, part 1 the low half).  Tap o is the weight of the input at offset o
// (row or column) from the centre, zero beyond the lobe: symmetric lobes (0,
// 2) weigh both sides c[|o|]; the antisymmetric lobe 1 weighs the upper /
// left side +c[k] and the lower / right side -c[k] (FIRFilter.h:66-176 pairs
// them the same way).  A lane's operand is one or two runs, so it loads
// with 8-byte LDS reads and needs no conversion.
// ONE: of a one-output launch, the runs of the vertical taps (lobe 0) and the
// pairs of the horizontal ones (lobe 1) only: 6 KB instead of 16, which leave a
// CU's LDS to four workgroups of a tile loop with 16-bit input instead of three
// and shorten the copy.
template <bool ONE> struct alignas(16) MfmaTabsOf {
    static constexpr int NL = ONE ? 1 : 3;
    v4f16 run[2 * NL * MT4];
    v8f16 hpair[2 * NL * MHP]; // horizontal operands: runs t and t + 16 side by side
    float lobe[ONE ? 68 : 66]; // staging: cv[l][k] at 17 l + k (GAUSS), tv / th at 33 l + o + 16 (TAPS)
    float tap[ONE ? 2 : 3][MT4 + 4];   // staging: tap o of lobe l times mp[l] at [l][o + MBASE]

    static __device__ __forceinline__ int run_at(int part, int l) { return (part * NL + (ONE ? 0 : l)) * MT4; }
    static __device__ __forceinline__ int pair_at(int part, int l) { return (part * NL + (ONE ? 0 : l)) * MHP; }
};
using MfmaTabs = MfmaTabsOf<false>;             // the layout of tables in device memory
template <int MODE> using ModeTabs = MfmaTabsOf<MODE == MODE_TAPS>;

// f(std::integral_constant<int, I>) for I = 0 .. N-1, unrolled.
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// Tap o of lobe l from the staged lobe words (MfmaTabs::lobe).  MODE_GAUSS:
// the three lobes of the Gaussian (centre-indexed cv[l]).  MODE_TAPS (one
// output of FIRFilter2 or of general taps): table 0 holds the vertical taps,
// table 1 the horizontal ones, both as full taps with tap o at index o + 16
// of tv / th.
template <int MODE>
__device__ __forceinline__ float mfma_tap_lds(const ModeTabs<MODE>& T, int l, int o)
{
    const int k = o < 0 ? -o : o;
    if (k > 16) return 0.f;
    if constexpr (MODE == MODE_TAPS) {
        return l < 2 ? T.lobe[33 * l + o + 16] : 0.f;
    } else {
        const float c = T.lobe[17 * l + k];
        return l != 1 ? c : o == 0 ? 0.f : o < 0 ? c : -c;
    }
}

template <int MODE> constexpr int mfma_nlobes() { return MODE == MODE_TAPS ? 2 : 3; }

// Builds the operand tables of one job in LDS.  Every thread of the
// workgroup calls it (it holds a barrier); the caller puts another barrier
// between it and the first use of T.  The lobe words are read with scalar
// loads (their own counter, so vector loads issued before the call, such as
// a strip's input, stay in flight) and written to LDS by one lane; every
// entry is then built from LDS.
template <int MODE = MODE_GAUSS, class A>
__device__ __forceinline__ void mfma_build_tabs(const A& a, ModeTabs<MODE>& T)
{
    constexpr int NL = mfma_nlobes<MODE>();
    constexpr int NW = MODE == MODE_TAPS ? 66 : 51;
    if (threadIdx.x == 0) {
        static_for<0, NW>([&](auto ic) {
            constexpr int i = ic;
            if constexpr (MODE == MODE_TAPS) T.lobe[i] = i < 33 ? a.tv[i] : a.th[i - 33];
            else                             T.lobe[i] = a.cv[i / 17][i % 17];
        });
    }
    const float mp0 = a.mp[0], mp1 = a.mp[1], mp2 = a.mp[2];
    __syncthreads();
    constexpr int NT4 = MT4 + 4;
    for (int e = threadIdx.x; e < NL * NT4; e += blockDim.x) {
        const int l = e / NT4, t = e - l * NT4;
        T.tap[l][t] = mfma_tap_lds<MODE>(T, l, t - MBASE) * (l == 0 ? mp0 : l == 1 ? mp1 : mp2);
    }
    __syncthreads();
    // runs (vertical operands: taps t - MBASE .. +3) and pairs of runs 16
    // apart (horizontal operands)
    for (int e = threadIdx.x; e < NL * (MT4 + MHP); e += blockDim.x) {
        const bool pair = e >= NL * MT4;
        const int ee = pair ? e - NL * MT4 : e;
        const int n = pair ? MHP : MT4;
        const int l = ee / n, t = ee - l * n;
        if (MODE == MODE_TAPS && l != int(pair)) continue;
        v8f16 hi, lo;
#pragma unroll
        for (int i = 0; i < 8; ++i) {               // taps t .. t + 3, then (pairs) t + 16 .. t + 19
            const float c = i < 4 || pair ? T.tap[l][t + (i < 4 ? i : 12 + i)] : 0.f;
            const _Float16 h = _Float16(c);
            hi[i] = h;
            lo[i] = _Float16(c - float(h));
        }
        if (pair) {
            T.hpair[T.pair_at(0, l) + t] = hi;
            T.hpair[T.pair_at(1, l) + t] = lo;
        } else {
            T.run[T.run_at(0, l) + t] = __builtin_shufflevector(hi, hi, 0, 1, 2, 3);
            T.run[T.run_at(1, l) + t] = __builtin_shufflevector(lo, lo, 0, 1, 2, 3);
        }
    }
}

// The operand tables of a launch in LDS: copied from a.tabs, where the
// host has built them once for these lobes (the same values, bit for bit:
// mfma_host_tabs restates mfma_build_tabs), else built here.  Every thread
// of the workgroup calls it; the caller puts a barrier between it and the
// first use of T.  (Building them took 2-3 us of a 1080p launch.)
template <int MODE = MODE_GAUSS, class A>
__device__ __forceinline__ void mfma_get_tabs(const A& a, ModeTabs<MODE>& T)
{
    if (a.tabs) {                               // uniform
        const gptr<const v4f32> src = reinterpret_cast<gptr<const v4f32>>(reinterpret_cast<uintptr_t>(a.tabs));
        v4f32* const dst = reinterpret_cast<v4f32*>(&T);
        if constexpr (MODE == MODE_TAPS) {
            // run (part 0, 1; lobe 0), pair (part 0, 1; lobe 1), lobe words: 16-byte words of either layout
            constexpr int RN = MT4 / 2, HN = MHP, LN = 17, H0 = 2 * 3 * RN, L0 = H0 + 2 * 3 * HN;
            static_assert(offsetof(MfmaTabs, hpair) == 16 * H0 && offsetof(MfmaTabs, lobe) == 16 * L0);
            static_assert(offsetof(ModeTabs<MODE>, hpair) == 32 * RN && offsetof(ModeTabs<MODE>, lobe) == 32 * (RN + HN));
            for (int i = threadIdx.x; i < 2 * (RN + HN) + LN; i += blockDim.x) {
                const int h = i - 2 * RN, l = h - 2 * HN;
                dst[i] = src[l >= 0 ? L0 + l : h >= HN ? H0 + 4 * HN + (h - HN) : h >= 0 ? H0 + HN + h :
                             i >= RN ? 3 * RN + (i - RN) : i];
            }
        } else {
            for (int i = threadIdx.x; i < int(sizeof(MfmaTabs) / 16); i += blockDim.x) dst[i] = src[i];
        }
    } else {
        mfma_build_tabs<MODE>(a, T);
    }
}

__device__ __forceinline__ v8f16 cat8(v4f16 a, v4f16 b)
{
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}

// v of the lane that DPP control CTRL selects (within rows of 16 lanes).
template <int CTRL> __device__ __forceinline__ float dpp_f32(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// Largest v over the wave (every lane active), in every lane, NaN if a lane
// holds one: DPP within each row of 16 lanes (quad swaps, half-row and row
// mirrors), then the four row results read as scalars.  (Six ds_bpermute
// rounds, each waiting for the LDS, did the same with a longer dependent
// chain.)
__device__ __forceinline__ float wave_max(float v)
{
    const auto mx = [](float a, float b) { return __builtin_elementwise_maximum(a, b); };
    v = mx(v, dpp_f32<0xb1>(v));                // quad_perm [1, 0, 3, 2]
    v = mx(v, dpp_f32<0x4e>(v));                // quad_perm [2, 3, 0, 1]
    v = mx(v, dpp_f32<0x141>(v));               // row_half_mirror
    v = mx(v, dpp_f32<0x140>(v));               // row_mirror
    const float a = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 0));
    const float b = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 16));
    const float c = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 32));
    const float d = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 48));
    return mx(mx(a, b), mx(c, d));
}

// A wave's output staging area: 16 rows of 64 pixels in the output's type,
// the row pitch a multiple of 16 bytes that spreads the rows over the banks;
// a store instruction takes 16 bytes a lane, RPI rows.
template <class OUT> struct MStage {
    static constexpr int ES    = int(sizeof(OUT));
    static constexpr int PITCH = MSTRIP_W * ES + 16;
    static constexpr int EPL   = 16 / ES;                   // pixels per lane
    static constexpr int LPR   = MSTRIP_W / EPL;            // lanes per row
    static constexpr int RPI   = 64 / LPR;
    static constexpr int NI    = 16 / RPI;                  // store instructions per output
    static_assert(PITCH <= MOPITCH * 4, "staging area too narrow");
};

typedef v4u32 v4u32u __attribute__((aligned(1), may_alias));

// Stores a strip of float rows that do not start at 128-byte lines, 4 rows an
// instruction (16 lanes of 16 bytes each), rows pitch bytes apart in the output
// from base, PITCH in LDS from src (the lane's first chunk, c bytes into row
// r0): the chunks of whole lines streaming, those of the lines that the strip
// shares with its neighbours by ordinary stores, which L2 merges.  Where the row
// starts at a 16-byte boundary (3001 x 4004 packed f32 six outputs): all
// streamed, a shared line is written to memory in parts, 142 us; all ordinary,
// whole lines stay dirty in L2 until they are evicted, 100; so split 62, as rows
// of whole lines take.  Elsewhere the two chunks at the ends of a whole line
// reach into the next and go out ordinarily, so that most of that line is
// streamed and the rest merges: 3001 x 4003 101 us ordinary, 74 so.
template <int PITCH>
__device__ __forceinline__ void
store_rows(__amdgpu_buffer_rsrc_t r, uintptr_t base, const char* src, int r0, int c, int pitch)
{
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int at = (r0 + 4 * i) * pitch;
        const uint32_t seg = uint32_t(base) + uint32_t(at);                     // low bits of the row's address
        const int f0 = int(-seg & 127u), f1 = 256 - int((seg + 256) & 127u);    // the whole lines of the row
        const bool whole = c >= f0 && c + 16 <= f1;
        const v4u32 q = *reinterpret_cast<const v4u32_any*>(src + 4 * i * PITCH);
        __builtin_amdgcn_raw_buffer_store_b128(q, r, whole ? at + c : MINVALID, 0, CPOL_NT);
        __builtin_amdgcn_raw_buffer_store_b128(q, r, whole ? MINVALID : at + c, 0, 0);
    }
}

// Input values of field block b for lane (g, m), float input: column x0 - RC +
// 16 b + m, rows y0 - RC + 8 g + j (j < 8) and, for K = 48, y0 - RC + 32 +
// 4 g + j (j < 4).  INSIDE: every pixel of the strip's window lies in the
// image (row offsets as scalar offsets); otherwise pixels outside the image
// read as 0 by the buffer's range check.
template <int RC, bool INSIDE, class A>
__device__ __forceinline__ void
mfma_load_block(const A& a, __amdgpu_buffer_rsrc_t rsrc, int y0, int x0, int b, int g, int m, float* v)
{
    constexpr int NLD = MGeo<RC>::NLD;
    constexpr int es = int(sizeof(float));
    const int col = x0 - RC + 16 * b + m;
    const int sb = a.in_stride_b;
    const int r0 = y0 - RC + 8 * g;            // first row of entries 0 .. 7
    const int r1 = y0 - RC + 32 + 4 * g;       // first row of entries 8 .. 11
    if constexpr (INSIDE) {
        const int v0 = r0 * sb + col * es, v1 = r1 * sb + col * es;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = Px<float>::ld(rsrc, v0, j * sb);
        if constexpr (MGeo<RC>::K48) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[8 + j] = Px<float>::ld(rsrc, v1, j * sb);
        }
    } else {
        const bool colok = unsigned(col) < unsigned(a.ncol);
#pragma unroll
        for (int j = 0; j < NLD; ++j) {
            const int row = j < 8 ? r0 + j : r1 + (j - 8);
            const bool ok = colok && unsigned(row) < unsigned(a.nrow);
            v[j] = Px<float>::ld(rsrc, ok ? row * sb + col * es : MINVALID, 0);
        }
    }
}

// The same for 16-bit input, in 32-bit registers as stored, of one-output
// strips of radius class 8 (see MFMA_DIRECT).  Windows inside the image load
// at uniform row bases plus a 32-bit lane offset: the zero-extending form, so
// that no mask right after the loads makes the wave wait for them.  At the
// image's edge the same loads at clamped addresses, and 0 outside.
template <bool INSIDE, class A>
__device__ __forceinline__ void mfma_load_block16(const A& a, int y0, int x0, int b, int g, int m, uint32_t* v)
{
    constexpr int RC = 8;
    const int col = x0 - RC + 16 * b + m, sb = a.in_stride_b;
    const char* const in = static_cast<const char*>(a.in);
    const auto ld = [](const char* row, uint32_t off) -> uint32_t {
        return *reinterpret_cast<gptr<const uint16_t>>(reinterpret_cast<uintptr_t>(row) + off);
    };
    if constexpr (INSIDE) {
        const uint32_t off = uint32_t(8 * g * sb + 2 * col);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = ld(in + int64_t(y0 - RC + j) * sb, off);
    } else {
        const bool colok = unsigned(col) < unsigned(a.ncol);
        const uint32_t off = uint32_t(2 * min(max(col, 0), a.ncol - 1));
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int row = y0 - RC + 8 * g + j;
            const uint32_t x = ld(in + int64_t(min(max(row, 0), a.nrow - 1)) * sb, off);
            v[j] = colok && unsigned(row) < unsigned(a.nrow) ? x : 0u;
        }
    }
}

// ------------------------------------------------------------ input window
// u8, f16 and bf16 input reaches the strips through LDS: the workgroup loads
// the window of its tile (SY strips down by SX across, and the radius class
// around them) once, as stored, with 16-byte loads, and each strip reads its
// matrix operands from there with the transposing LDS reads (ds_read_b64_tr:
// within 16 lanes, lane i supplies the address of 8 bytes and receives column
// i of the 4 rows of 16-bit or 8 rows of 8-bit elements they cover), which
// hand each lane the 8 rows of one column that a vertical product takes as
// its K entries.  One load per pixel and lane (40 or 72 per strip, each
// touching four rows for 64 or 128 bytes) kept the address units busy for a
// fifth of a launch, held 40 - 72 registers, and read the rows that
// neighbouring strips share once per strip.
// Pixels outside the image are 0 in the window.
template <int RC, int SY, int SX, class IN>
struct MWin {
    static constexpr int ES    = int(sizeof(IN));
    static constexpr int ROWS  = 16 * SY + 2 * RC;
    static constexpr int COLS  = 16 * (MNB * SX + MGeo<RC>::NVB - MNB);
    static constexpr int PITCH = COLS * ES;                 // bytes, a multiple of 16
    static constexpr int CPR   = PITCH / 16;                // 16-byte chunks per row
    static constexpr int NC    = ROWS * CPR;
    static constexpr int NT_   = 64 * SY * SX;              // threads of the workgroup
    static constexpr int N     = (NC + NT_ - 1) / NT_;      // chunks per thread
    static constexpr int EPC   = 16 / ES;                   // elements per chunk
    // u8 at radius class 16: the 8-row transposing reads of the last 16 rows
    // take 4 rows more than they use
    static constexpr int BYTES = PITCH * (ROWS + (ES == 1 && MGeo<RC>::K48 ? 4 : 0));
};

// v shifted by d elements of ES bytes: result element j = element j + d of v,
// 0 where that lies outside.
template <int ES> __device__ __forceinline__ v4u32 shift_chunk(v4u32 v, int d)
{
    uint64_t lo = uint64_t(v[1]) << 32 | v[0], hi = uint64_t(v[3]) << 32 | v[2];
    const int r = max(d, 0) * (8 * ES), l = max(-d, 0) * (8 * ES);   // at most one is nonzero
    // right, then left, by 64 and by the rest (x << 1 << (63 - k) is x <<
    // (64 - k), and 0 for k = 0)
    const int r1 = r & 63, l1 = l & 63;
    const uint64_t a0 = r >= 64 ? hi : lo, a1 = r >= 64 ? 0 : hi;
    lo = a0 >> r1 | a1 << 1 << (63 - r1);
    hi = a1 >> r1;
    const uint64_t b1 = l >= 64 ? lo : hi, b0 = l >= 64 ? 0 : lo;
    hi = b1 << l1 | b0 >> 1 >> (63 - l1);
    lo = b0 << l1;
    const bool in = r < 128 && l < 128;
    return in ? v4u32{uint32_t(lo), uint32_t(lo >> 32), uint32_t(hi), uint32_t(hi >> 32)} : v4u32{0, 0, 0, 0};
}

// Issues the loads of the window whose tile's first strip is at (y0, x0);
// every thread (tid) of the workgroup calls it, the chunks arrive in v.
template <int RC, int SY, int SX, class IN, class A>
__device__ __forceinline__ void mwin_load(const A& a, int tid, int y0, int x0, v4u32* v)
{
    using W = MWin<RC, SY, SX, IN>;
    const int yw = y0 - RC, xw = x0 - RC, sb = a.in_stride_b;
    const char* const in = static_cast<const char*>(a.in);
    const bool inside = yw >= 0 && yw + W::ROWS <= a.nrow && xw >= 0 && xw + W::COLS <= a.ncol;   // uniform
    if (inside) {
        const char* const base = in + int64_t(yw) * sb + xw * W::ES;
#pragma unroll
        for (int i = 0; i < W::N; ++i) {
            const int c = min(tid + i * W::NT_, W::NC - 1);
            const int r = c / W::CPR, q = c - r * W::CPR;
            v[i] = *reinterpret_cast<gptr<const v4u32u>>(reinterpret_cast<uintptr_t>(base + uint32_t(r * sb + 16 * q)));
        }
        return;
    }
    // Rows and chunks clamped into the image, then moved to their place: a
    // chunk that straddles an edge keeps the pixels inside.
    const bool narrow = a.ncol < W::EPC;                    // uniform: no whole chunk in a row
    const auto at = [&](int i, int& row, int& col, int& cc) {
        const int c = min(tid + i * W::NT_, W::NC - 1);
        const int r = c / W::CPR, q = c - r * W::CPR;
        row = yw + r;
        col = xw + W::EPC * q;
        cc = min(max(col, 0), max(a.ncol - W::EPC, 0));
        return reinterpret_cast<uintptr_t>(in + int64_t(min(max(row, 0), a.nrow - 1)) * sb);
    };
    int row, col, cc;
    if (!narrow) {
#pragma unroll
        for (int i = 0; i < W::N; ++i) {
            const uintptr_t line = at(i, row, col, cc);
            v[i] = *reinterpret_cast<gptr<const v4u32u>>(line + uintptr_t(cc * W::ES));
        }
    } else {                                                // byte by byte
#pragma unroll
        for (int i = 0; i < W::N; ++i) {
            const gptr<const uint8_t> p = reinterpret_cast<gptr<const uint8_t>>(at(i, row, col, cc));
            uint64_t lo = 0, hi = 0;
#pragma unroll 1
            for (int j = 0; j < a.ncol * W::ES; ++j) {
                const uint64_t x = uint64_t(p[j]) << (8 * (j & 7));
                lo |= j < 8 ? x : 0;
                hi |= j < 8 ? 0 : x;
            }
            v[i] = v4u32{uint32_t(lo), uint32_t(lo >> 32), uint32_t(hi), uint32_t(hi >> 32)};
        }
    }
#pragma unroll
    for (int i = 0; i < W::N; ++i) {
        (void)at(i, row, col, cc);
        const v4u32 x = shift_chunk<W::ES>(v[i], col - cc);
        v[i] = unsigned(row) < unsigned(a.nrow) ? x : v4u32{0, 0, 0, 0};
    }
}

// Writes the loaded chunks into the workgroup's window in LDS.
template <int RC, int SY, int SX, class IN>
__device__ __forceinline__ void mwin_store(int tid, char* win, const v4u32* v)
{
    using W = MWin<RC, SY, SX, IN>;
#pragma unroll
    for (int i = 0; i < W::N; ++i)
        *reinterpret_cast<v4u32*>(win + 16 * min(tid + i * W::NT_, W::NC - 1)) = v[i];
}

// A barrier that orders the workgroup's LDS accesses only: loads from and
// stores to memory stay in flight across it.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <class T> using lptr = T __attribute__((address_space(3)))*;   // LDS
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef int v2i32 __attribute__((ext_vector_type(2)));

// f16 hi / lo split of 4 floats times s.
__device__ __forceinline__ void split4(float v0, float v1, float v2, float v3, float s, v4f16& hi, v4f16& lo)
{
    const v4f32 x = {v0 * s, v1 * s, v2 * s, v3 * s};
    hi = __builtin_convertvector(x, v4f16);
    lo = __builtin_convertvector(x - __builtin_convertvector(hi, v4f32), v4f16);
}

// Entries 4 O .. 4 O + 7 of a field vector: field blocks O and O + 1.
template <int O, class V>
__device__ __forceinline__ v8f16 pair8(const V& f)
{
    return __builtin_shufflevector(f, f, 4 * O, 4 * O + 1, 4 * O + 2, 4 * O + 3,
                                   4 * O + 4, 4 * O + 5, 4 * O + 6, 4 * O + 7);
}

// Field blocks 2 P and 2 P + 1 (pairs that do not overlap).
template <int P, class V>
__device__ __forceinline__ v8f16 pairP(const V& f)
{
    return pair8<2 * P>(f);
}

// ------------------------------------------------------------------------
// FP32 form of one strip, for input the split-f16 products cannot carry:
// non-finite values (a band product multiplies every input of a block by
// every band entry, zeros included, so one NaN or Inf would reach all 16 x
// 16 outputs of its block window, and Inf - Inf in the hi / lo split turns
// Inf into NaN), or a strip whose largest magnitude lies outside the range
// its power-of-two scale covers.  Each output is summed over exactly the
// taps of its lobes -- the true radius, zero taps inside it included, none
// beyond it, no centre tap for an antisymmetric lobe, paired as
// FIRFilter.h:66-176 pairs them -- so a NaN or an Inf reaches exactly the
// outputs whose window holds it, with the sign the reference's sums give.
// Vertical pass first, one half strip (32 output columns, 32 + 2 RC field
// columns) at a time through the wave's staging area.  Kept out of line so
// that the matrix-core path's register allocation and schedule are its own.

// Tap sum over w(-R) .. w(R) around w(0) of a lobe of radius r <= R whose
// tap at distance k is c(k) on the upper / left side: symmetric: sum_k c(k)
// (w(-k) + w(k)) + c(0) w(0); antisymmetric: sum_k c(k) (w(-k) - w(k));
// outermost tap first.  Taps beyond r are skipped, never multiplied.
template <int R, class C, class W>
__device__ __forceinline__ float fp32_paired(const C& c, int r, bool sym, const W& w)
{
    float acc = 0.f;
#pragma unroll
    for (int k = R; k >= 1; --k) {
        const float lo = w(-k), hi = w(k);
        const float s = sym ? lo + hi : lo - hi;
        acc = k <= r ? (k == r ? c(k) * s : __builtin_fmaf(c(k), s, acc)) : acc;
    }
    return sym ? __builtin_fmaf(c(0), w(0), acc) : acc;
}

// General taps t(o), o = -r .. r, top / left tap first.
template <int R, class C, class W>
__device__ __forceinline__ float fp32_taps(const C& t, int r, const W& w)
{
    float acc = 0.f;
#pragma unroll
    for (int o = -R; o <= R; ++o) {
        const int k = o < 0 ? -o : o;
        acc = k <= r ? (o == -r ? t(o) * w(o) : __builtin_fmaf(t(o), w(o), acc)) : acc;
    }
    return acc;
}

// The taps come from the lobe words staged in LDS (MfmaTabs::lobe): MODE_GAUSS
// c_l(k) at 17 l + k; MODE_TAPS the full vertical taps at 16 + o and the
// horizontal ones at 33 + 16 + o, which for FIRFilter2 lobes (sgnv, sgnh
// nonzero) are c(k) on the upper / left side.
template <int RC, class IN, class OUT, int MODE>
__device__ __forceinline__ void
mfma_strip_fp32(ConstArgs& a, int y0, int x0, const ModeTabs<MODE>& T, float* stage, unsigned mask)
{
    constexpr bool ONE = MODE == MODE_TAPS;
    constexpr int NFC = 32 + 2 * RC;            // field columns per half strip
    static_assert(NFC <= MOPITCH, "staging area too narrow");
    // Values the compiler cannot see through: nothing of this rarely taken
    // path is computed ahead of it (in a tile loop, such hoisted values would
    // hold registers across the matrix-core path).
    int lane = threadIdx.x & 63;
    y0 = __builtin_amdgcn_readfirstlane(y0);
    x0 = __builtin_amdgcn_readfirstlane(x0);
    mask = __builtin_amdgcn_readfirstlane(mask);
    asm volatile("" : "+v"(lane), "+s"(y0), "+s"(x0), "+s"(mask));
    const int es = int(sizeof(IN));
    const int sb = a.in_stride_b;
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.in), short(0), int(a.in_bytes), BUF_DWORD3);
    constexpr int HL[6] = {ONE ? 1 : 0, 1, 0, 2, 1, 0};   // horizontal lobe of output k (TAPS: table 1)
    constexpr int VL[6] = {0, 0, 1, 0, 1, 2};             // vertical lobe of output k
    const unsigned fneed[3] = {ONE ? 1u : mask & 0x0bu, ONE ? 0u : mask & 0x14u, ONE ? 0u : mask & 0x20u};
    const float* const lw = T.lobe;

#pragma unroll 1
    for (int l = 0; l < 3; ++l) {
        if (!fneed[l]) continue;
#pragma unroll 1
        for (int q = 0; q < 2; ++q) {
            // vertical pass: lane = field column x0 + 32 q - RC + lane, rows y0 .. y0 + 15;
            // one row at a time, its window loaded again (L2-resident), so that
            // this rarely taken path stays small in registers
            const int col = x0 + 32 * q - RC + lane;
            if (lane < NFC) {
                const bool colok = unsigned(col) < unsigned(a.ncol);
#pragma unroll 1
                for (int i = 0; i < 16; ++i) {
                    const auto win = [&](int d) {
                        const int row = y0 + i + d;
                        const bool ok = colok && unsigned(row) < unsigned(a.nrow);
                        return Px<IN>::ld(rsrc, ok ? row * sb + col * es : MINVALID, 0);
                    };
                    float f;
                    if constexpr (ONE) {
                        f = a.sgnv != 0.f ? fp32_paired<RC>([&](int k) { return lw[16 - k]; }, a.r[0], a.sgnv > 0.f, win)
                                          : fp32_taps<RC>([&](int o) { return lw[16 + o]; }, a.r[0], win);
                    } else {
                        f = fp32_paired<RC>([&](int k) { return lw[17 * l + k]; }, a.r[l], l != 1, win);
                    }
                    stage[i * MOPITCH + lane] = f;
                }
            }
            __builtin_amdgcn_wave_barrier();
            // horizontal pass: lane = output column x0 + 32 q + (lane & 31), rows (lane >> 5) * 8 + 0 .. 7
            const int j = lane & 31, i0 = (lane >> 5) * 8;
            const int x = x0 + 32 * q + j;
#pragma unroll 1
            for (int k = 0; k < (ONE ? 1 : 6); ++k) {
                if (VL[k] != l || !(mask >> k & 1u)) continue;
                const int h = HL[k];
                const int rv = ONE ? a.r[0] : a.r[VL[k]], rh = ONE ? a.r[1] : a.r[h];
#pragma unroll 1
                for (int i = 0; i < 8; ++i) {
                    const float* srow = stage + (i0 + i) * MOPITCH + RC + j;
                    const auto win = [&](int d) { return srow[d]; };
                    float v;
                    if constexpr (ONE) {
                        v = a.sgnh != 0.f ? fp32_paired<RC>([&](int kk) { return lw[49 - kk]; }, a.r[1], a.sgnh > 0.f, win)
                                          : fp32_taps<RC>([&](int o) { return lw[49 + o]; }, a.r[1], win);
                    } else {
                        v = fp32_paired<RC>([&](int kk) { return lw[17 * h + kk]; }, a.r[h], h != 1, win);
                    }
                    const int y = y0 + i0 + i;
                    if (y >= rv && y < a.nrow - rv && x >= rh && x < a.ncol - rh) {
                        const gptr<OUT> p = reinterpret_cast<gptr<OUT>>(
                            a.obase[k] + uintptr_t(int64_t(y) * a.ostride[k] + x) * sizeof(OUT));
                        Px<OUT>::st(p, v);
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// The arguments behind a pointer the compiler cannot see through, so that it
// reads those of the rarely taken FP32 form there, and not before the strip
// code, where they would hold 40 scalar registers: a job's in device memory,
// or the kernel's own (every matrix-core kernel's first argument).
__device__ __forceinline__ ConstArgs& opaque_args(ConstArgs& a)
{
    const uintptr_t p = (uintptr_t)&a;
    uint32_t lo = __builtin_amdgcn_readfirstlane(uint32_t(p)), hi = __builtin_amdgcn_readfirstlane(uint32_t(p >> 32));
    asm volatile("" : "+s"(lo), "+s"(hi));
    return *(ConstArgs*)(uintptr_t(hi) << 32 | lo);
}
__device__ __forceinline__ ConstArgs& opaque_args(const SepArgs&)
{
    uintptr_t p = (uintptr_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(ConstArgs*)p;
}

#define TUCU_MFMA(A_, B_, C_) __builtin_amdgcn_mfma_f32_16x16x32_f16((A_), (B_), (C_), 0, 0, 0)

// A strip's float input, as loaded: field block b, entry j
// (mfma_load_block's order); radius class 8 uses blocks 0 .. 4 and entries
// 0 .. 7.
using MfmaRaw = float[6][12];
using MfmaRaw16 = uint32_t[MGeo<8>::NVB][8];    // of 16-bit input (mfma_load_block16)

// A strip's matrix operands of the vertical pass, and its scale.
// xh / xl: entries 0 .. 7 (rows 8 g + j), high and low halves; xt (K = 48):
// entries 8 .. 11 (rows 32 + 4 g + j), high then low halves, so that one
// product with the high taps twice covers both halves of those rows.
// Inputs exact in f16 have no low half: xt then holds the high halves
// twice, and one product with the high and the low taps side by side
// covers both tap halves (one product per block instead of two).
struct MfmaOps {
    v8f16 xh[6], xl[6], xt[6];  // field blocks; radius class 8 uses 0 .. 4
    float inv_s;                // undoes the strip's scale
    bool  redo;                 // the products cannot carry the input: the FP32 form filters the strip
};

// Register budget of the kernels: three waves per SIMD (the one-round and
// batched float kernels need 160 - 169 registers; 64 batched 1080p images f32
// 12.2 us each against 13.0 at two waves).  The single-image tile loop of
// float input keeps two: inlined in a loop the strip code needs more registers.
constexpr int MFMA_WAVES_PER_SIMD = 3;

// The single-image tile loop (large images): the float strip code inlined in
// a loop needs more registers than the one-round kernels, two waves per SIMD
// (the one-output mode needs fewer, but at three or four it spills);
// narrow input, which holds no float values and prefetches the next window
// in at most 36 registers, takes three at radius class 16 (four by itself
// where it needs 128 registers or fewer).  Six outputs u8 -> f32 at radius class
// 8 are scheduled for two, though their 109 registers admit four: more of a
// strip's work then overlaps (3840 x 2160 43.6 -> 42.6 us, 4032 x 3000 62.6 ->
// 61.4, 4608 x 3456 81.3 -> 79.7).
template <int RC, class IN, class OUT, int MODE>
constexpr bool MFMA_LOOP_TWO = MODE == MODE_GAUSS && RC == 8 && sizeof(IN) == 1 && sizeof(OUT) == 4;
template <int RC, class IN, class OUT, int MODE>
constexpr int MFMA_LOOP_WAVES = sizeof(IN) == 4 || MFMA_LOOP_TWO<RC, IN, OUT, MODE> ? 2 : 3;
template <int RC, class IN, class OUT, int MODE>
constexpr int MFMA_LOOP_WAVES_MAX = MFMA_LOOP_TWO<RC, IN, OUT, MODE> ? 2 : 8;

// Strips of the tile loop that load their 16-bit input themselves, without the
// window in LDS: one output of radius class 8 is too little work per tile to
// cover the window's way through LDS and its two barriers (4096 x 4096 17 x 17
// taps bf16 22.5 -> 18.9 us, f16 21.4 -> 18.3; 16 columns more per strip, at
// radius class 16, are loaded faster by the workgroup: 52 us so, 30 by the
// window; u8 halves the window's bytes).
template <int RC, class IN, int MODE>
constexpr bool MFMA_DIRECT = MODE == MODE_TAPS && RC == 8 && sizeof(IN) == 2;

// Issues the loads of the float strip at (y0, x0); the values arrive in raw.
// FRESH: the lane index is opaque to the compiler (a caller's loop then
// recomputes what derives from it in each pass instead of holding it).
template <int RC, bool FRESH = false, class A>
__device__ __forceinline__ void mfma_load(const A& a, int y0, int x0, MfmaRaw& raw)
{
    using G = MGeo<RC>;
    int lane = threadIdx.x & 63;
    if constexpr (FRESH) asm volatile("" : "+v"(lane));
    const int g = lane >> 4, m = lane & 15;
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.in), short(0), int(a.in_bytes), BUF_DWORD3);
    // One test for the whole window (y0, x0 are wave-uniform): with a test
    // per block, the compiler makes each block's edge path wait for the
    // loads of the blocks before it.
    const bool inside = y0 - RC >= 0 && y0 - RC + G::KV <= a.nrow &&
                        x0 - RC >= 0 && x0 - RC + 16 * G::NVB <= a.ncol;
    if (inside) {
#pragma unroll
        for (int b = 0; b < G::NVB; ++b) mfma_load_block<RC, true>(a, rsrc, y0, x0, b, g, m, raw[b]);
    } else {
#pragma unroll
        for (int b = 0; b < G::NVB; ++b) mfma_load_block<RC, false>(a, rsrc, y0, x0, b, g, m, raw[b]);
    }
    if constexpr (!G::K48) {
#pragma unroll
        for (int b = 0; b < G::NVB; ++b) raw[b][8] = raw[b][9] = raw[b][10] = raw[b][11] = 0;
    }
}

// The same of a 16-bit strip, radius class 8.
template <class A> __device__ __forceinline__ void mfma_load16(const A& a, int y0, int x0, MfmaRaw16& raw)
{
    using G = MGeo<8>;
    const int lane = threadIdx.x & 63, g = lane >> 4, m = lane & 15;
    const bool inside = y0 >= 8 && y0 - 8 + G::KV <= a.nrow && x0 >= 8 && x0 - 8 + 16 * G::NVB <= a.ncol;   // uniform
    if (inside) {
#pragma unroll
        for (int b = 0; b < G::NVB; ++b) mfma_load_block16<true>(a, y0, x0, b, g, m, raw[b]);
    } else {
#pragma unroll
        for (int b = 0; b < G::NVB; ++b) mfma_load_block16<false>(a, y0, x0, b, g, m, raw[b]);
    }
}

// Power-of-two scale of a strip whose largest magnitude (over the wave) is
// mx: the exponent ex puts it in [2^12, 2^13).  Strips whose largest magnitude
// is below 2^-87 or above 2^113 are out of the scale's reach (their scaled
// values would lose precision or overflow f16), and strips with a NaN or an
// Inf (mx is then one) would spread it: the FP32 form filters them, and every
// strip of a launch whose taps have no scale (xmax).
__device__ __forceinline__ int mfma_scale_exp(float mx, float xmax, bool& redo)
{
    int ex;
    (void)frexpf(mx, &ex);                      // mx < 2^ex
    ex = 13 - ex;
    redo = ex < -100 || ex > 100 || !(mx <= xmax);
    return ex;
}

// The operands of a float strip from its loaded values.
template <int RC, class A>
__device__ __forceinline__ void mfma_ops_raw(const A& a, const MfmaRaw& raw, MfmaOps& p)
{
    using G = MGeo<RC>;
    float mx = 0.f;
#pragma unroll
    for (int b = 0; b < G::NVB; ++b)
#pragma unroll
        for (int j = 0; j < G::NLD; ++j) mx = __builtin_elementwise_maximum(mx, fabsf(raw[b][j]));   // keeps a NaN
    const int ex = mfma_scale_exp(wave_max(mx), a.xmax, p.redo);
    const float s = ldexpf(a.mq, ex);
    p.inv_s = ldexpf(1.f, -ex);
#pragma unroll
    for (int b = 0; b < G::NVB; ++b) {
        v4f16 h0, l0, h1, l1;
        const float* const r = raw[b];
        split4(r[0], r[1], r[2], r[3], s, h0, l0);
        split4(r[4], r[5], r[6], r[7], s, h1, l1);
        p.xh[b] = cat8(h0, h1);
        p.xl[b] = cat8(l0, l1);
        if constexpr (G::K48) {
            v4f16 h2, l2;
            split4(r[8], r[9], r[10], r[11], s, h2, l2);
            p.xt[b] = cat8(h2, l2);
        }
    }
}

// Two 16-bit values as stored times s, in f16 (round to nearest even): the
// multiplication and the conversion in one mixed-precision FMA each.
template <class IN> __device__ __forceinline__ v2f16 scale_pair(uint32_t w, float s, float zero)
{
    float lo, hi;
    if constexpr (std::is_same_v<IN, bf16_t>) {
        lo = __uint_as_float(w << 16);
        hi = __uint_as_float(w & 0xffff0000u);
    } else {
        const v2f16 h = __builtin_bit_cast(v2f16, w);
        lo = float(h[0]);
        hi = float(h[1]);
    }
    return v2f16{_Float16(__builtin_fmaf(lo, s, zero)), _Float16(__builtin_fmaf(hi, s, zero))};
}

// The operands of a 16-bit strip of radius class 8 from its loaded values.
template <class IN, class A>
__device__ __forceinline__ void mfma_ops_raw16(const A& a, const MfmaRaw16& raw, MfmaOps& p)
{
    constexpr int NVB = MGeo<8>::NVB;
    const auto value = [](uint32_t v) -> float {
        if constexpr (std::is_same_v<IN, f16_t>) return float(__builtin_bit_cast(_Float16, uint16_t(v)));
        else                                     return __uint_as_float(v << 16);
    };
    float mx = 0.f;
#pragma unroll
    for (int b = 0; b < NVB; ++b)
#pragma unroll
        for (int j = 0; j < 8; ++j) mx = __builtin_elementwise_maximum(mx, fabsf(value(raw[b][j])));     // keeps a NaN
    const int ex = mfma_scale_exp(wave_max(mx), a.xmax, p.redo);
    const float s = ldexpf(a.mq, ex);
    p.inv_s = ldexpf(1.f, -ex);
    float zero = 0.f;                           // opaque: x s + 0 stays one mixed-precision FMA
    asm("" : "+v"(zero));
#pragma unroll
    for (int b = 0; b < NVB; ++b)
#pragma unroll
        for (int j = 0; j < 8; ++j) p.xh[b][j] = _Float16(__builtin_fmaf(value(raw[b][j]), s, zero));
}

// Two u8 values (bytes I, I + 1 of w) as f16 times s, exactly: with M = 1024 s
// a power of two in f16's normal range, M's bits with x (< 256) in the low
// mantissa bits are the f16 M + x s, and subtracting M leaves x s.  mb = M's
// bits in both halves (the low byte of each is 0), nm = -M in both halves.
template <int I> __device__ __forceinline__ v2f16 u8pair_f16(uint32_t w, uint32_t mb, v2f16 nm)
{
    // v_perm selector: bytes 0 - 3 of the second source, 4 - 7 of the first
    constexpr uint32_t sel = uint32_t(I) | 5u << 8 | uint32_t(I + 1) << 16 | 7u << 24;
    return __builtin_bit_cast(v2f16, __builtin_amdgcn_perm(mb, w, sel)) + nm;
}

// The operands of a narrow strip from the window in LDS (row pitch PITCH
// bytes); win is the window's byte at the first row and column of the strip's
// own window.
template <int RC, class IN, int PITCH, class A>
__device__ __forceinline__ void mfma_ops_win(const A& a, const char* win, int lane, MfmaOps& p)
{
    using G = MGeo<RC>;
    constexpr int NVB = G::NVB;
    const int g = lane >> 4, i = lane & 15;
    if constexpr (std::is_same_v<IN, uint8_t>) {
        // The scale of 255 (2^5) whatever the strip holds: every byte times
        // 2^5 mq is exact in f16, and the error bound, relative to 255, stays
        // that of the brightest strip.  s lies in [2^-7, 2^5] (mq in
        // [2^-12, 1]), so M = 1024 s is a normal f16.
        constexpr int ex = 5;
        p.redo = false;
        p.inv_s = ldexpf(1.f, -ex);
        const _Float16 M = _Float16(1024.f * ldexpf(a.mq, ex));
        const uint32_t mb = uint32_t(__builtin_bit_cast(uint16_t, M)) * 0x10001u;
        const v2f16 nm = {-M, -M};
        const char* const w0 = win + (8 * g + i / 2) * PITCH + 8 * (i % 2);
        const char* const w1 = win + (32 + 4 * g + i / 2) * PITCH + 8 * (i % 2);
#pragma unroll
        for (int b = 0; b < NVB; ++b) {
            const v2i32 d = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lptr<v2i32>)(w0 + 16 * b));
            const v2f16 p0 = u8pair_f16<0>(d[0], mb, nm), p1 = u8pair_f16<2>(d[0], mb, nm);
            const v2f16 p2 = u8pair_f16<0>(d[1], mb, nm), p3 = u8pair_f16<2>(d[1], mb, nm);
            p.xh[b] = v8f16{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
            if constexpr (G::K48) {
                const v2i32 e = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lptr<v2i32>)(w1 + 16 * b));
                const v2f16 p4 = u8pair_f16<0>(e[0], mb, nm), p5 = u8pair_f16<2>(e[0], mb, nm);
                p.xt[b] = v8f16{p4[0], p4[1], p5[0], p5[1], p4[0], p4[1], p5[0], p5[1]};
            }
        }
    } else {
        constexpr int NP = G::NLD / 2;          // pairs of rows per lane and block
        typedef uint32_t v2u __attribute__((ext_vector_type(2)));
        uint32_t d[NVB][NP];
        const char* const w0 = win + (8 * g + i / 4) * PITCH + 8 * (i % 4);
        const char* const w1 = win + (32 + 4 * g + i / 4) * PITCH + 8 * (i % 4);
        const auto rd = [](const char* q) {
            return __builtin_bit_cast(v2u, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lptr<v4i16>)q));
        };
#pragma unroll
        for (int b = 0; b < NVB; ++b) {
            const v2u x = rd(w0 + 32 * b), y = rd(w0 + 32 * b + 4 * PITCH);
            d[b][0] = x[0]; d[b][1] = x[1]; d[b][2] = y[0]; d[b][3] = y[1];
            if constexpr (G::K48) {
                const v2u z = rd(w1 + 32 * b);
                d[b][4] = z[0]; d[b][5] = z[1];
            }
        }
        // largest magnitude, a NaN if there is one
        float mx = 0.f;
        if constexpr (std::is_same_v<IN, bf16_t>) {
            // the upper value of a pair with the lower one's bits below its
            // own: they change neither its exponent nor what is not finite,
            // except that of an upper 0 they leave a denormal below bfloat16's
            // smallest (of 0 and -0.0: 2^-134), taken for 0 below
#pragma unroll
            for (int b = 0; b < NVB; ++b)
#pragma unroll
                for (int j = 0; j < NP; ++j)
                    mx = __builtin_elementwise_maximum(
                        __builtin_elementwise_maximum(mx, fabsf(__uint_as_float(d[b][j] << 16))),
                        fabsf(__uint_as_float(d[b][j])));
        } else {
            v2f16 m2 = {0, 0};
#pragma unroll
            for (int b = 0; b < NVB; ++b)
#pragma unroll
                for (int j = 0; j < NP; ++j) {
                    const v2f16 h = __builtin_bit_cast(v2f16, d[b][j]);
                    m2 = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m2, h), -h);
                }
            mx = __builtin_elementwise_maximum(float(m2[0]), float(m2[1]));
        }
        mx = wave_max(mx);
        if constexpr (std::is_same_v<IN, bf16_t>) mx = mx < 0x1p-133f ? 0.f : mx;
        const int ex = mfma_scale_exp(mx, a.xmax, p.redo);
        const float s = ldexpf(a.mq, ex);
        p.inv_s = ldexpf(1.f, -ex);
        float zero = 0.f;                       // opaque: x s + 0 stays one mixed-precision FMA
        asm("" : "+v"(zero));
#pragma unroll
        for (int b = 0; b < NVB; ++b) {
            v2f16 h[NP];
#pragma unroll
            for (int j = 0; j < NP; ++j) h[j] = scale_pair<IN>(d[b][j], s, zero);
            p.xh[b] = v8f16{h[0][0], h[0][1], h[1][0], h[1][1], h[2][0], h[2][1], h[3][0], h[3][1]};
            if constexpr (G::K48)
                p.xt[b] = v8f16{h[4][0], h[4][1], h[5][0], h[5][1], h[4][0], h[4][1], h[5][0], h[5][1]};
        }
    }
}

// One strip: centre rows y0 .. y0+15, centre columns x0 .. x0+63, its
// operands in p.  T holds the operand runs (mfma_build_tabs), stage is the
// wave's output staging area.  Every lane of the wave calls it.
// before_store() runs once, before the strip's first stores: a tile loop
// waits there for the next window's loads.  The wait counter of a wave
// covers loads and stores in order, so after this tile's stores it would
// wait for them too; there it covers only the previous tile's.
//
// Operand layouts (lane = 16 g + m; m is also the row / output column n):
//   vertical, block b, K32 slice: A = input rows y0 - RC + 8 g + j (j < 8)
//     of column x0 - RC + 16 b + m; B = taps of offsets 8 g + j - RC - n.
//   vertical, K48 second slice: A = rows 32 + 4 g .. +3 of the lane's
//     input, high halves then low halves; B = taps of offsets
//     32 + 4 g + j - RC - n twice (high taps: both halves of the input in
//     one product), or once and then zeros (low taps x high input).
//   horizontal, K32 (radius class 8), output block o: B = field blocks o,
//     o + 1 (lane holds columns 4 g .. 4 g + 3 of each, window columns
//     4 g + j and 16 + 4 g + j); A = taps of offsets (window column) - RC - m.
//   horizontal, K48: two K32 slices over the fixed pairs P_(o/2) and
//     P_(o/2 + 1) of field blocks (2 p, 2 p + 1); A = taps as above, shifted
//     by d = 32 p - 16 o (zero for the block outside the window).
template <int RC, class IN, class OUT, int MODE = MODE_GAUSS, int CPOL = CPOL_NT, bool FRESH = false, class A, class S, class H>
__device__ __forceinline__ void
mfma_filter(const A& a, int y0, int x0, const MfmaOps& p, const ModeTabs<MODE>& T, float* stage, S&& sink, unsigned mask,
            H&& before_store)
{
    constexpr bool ONE = MODE == MODE_TAPS;     // one field (table 0), one output (table 1 across)
    using G = MGeo<RC>;
    constexpr int NVB = G::NVB;
    constexpr bool XLO = sizeof(IN) == 4;       // f16 / bf16 / u8 inputs are exact in one f16
    constexpr int NF = 4 * NVB;                 // field entries per lane
    typedef _Float16 vfield __attribute__((ext_vector_type(NF)));
    int lane = threadIdx.x & 63;
    if constexpr (FRESH) asm volatile("" : "+v"(lane));    // as for mfma_load
    const int g = lane >> 4, m = lane & 15;
    const v4f16 z4 = {0, 0, 0, 0};
    constexpr bool CHECK = !std::is_same_v<IN, uint8_t> && MODE != MODE_ICIA;   // u8 input is always in range
    const float inv_s = p.inv_s;

    // --------------------------------------------------- vertical pass
    // fh[l] / fl[l]: entries 4 b .. 4 b + 3 = field l at row y0 + n, columns
    // x0 - RC + 16 b + 4 g .. +3 (the accumulator layout), split in f16.
    // One lobe at a time, the chains of the field blocks interleaved.
    // 1.0 in a register whose value the compiler does not see: v * one - hi
    // then stays one v_fma_mix (v - hi alone would be a convert, a subtract
    // and another convert)
    float one = 1.f;
    asm("" : "+v"(one));
    auto vpass = [&](int l, vfield& fh, vfield& fl) {
        const int t1 = MBASE + 8 * g - RC - m;
        const v8f16 ch1 = cat8(T.run[T.run_at(0, l) + t1], T.run[T.run_at(0, l) + t1 + 4]);
        const v8f16 cl1 = cat8(T.run[T.run_at(1, l) + t1], T.run[T.run_at(1, l) + t1 + 4]);
        v8f16 cht, clt;
        if constexpr (G::K48) {                 // rows 32 + 4 g + j: high taps for both halves
            const int t2 = MBASE + 32 + 4 * g - RC - m;
            const v4f16 th = T.run[T.run_at(0, l) + t2];
            const v4f16 tl = T.run[T.run_at(1, l) + t2];
            cht = XLO ? cat8(th, th) : cat8(th, tl);
            clt = cat8(tl, z4);
        }
        v4f32 acc[NVB];
#pragma unroll
        for (int b = 0; b < NVB; ++b) acc[b] = v4f32{0.f, 0.f, 0.f, 0.f};
        // smaller products first
        if constexpr (XLO) {
#pragma unroll
            for (int b = 0; b < NVB; ++b) acc[b] = TUCU_MFMA(p.xl[b], ch1, acc[b]);
        }
#pragma unroll
        for (int b = 0; b < NVB; ++b) acc[b] = TUCU_MFMA(p.xh[b], cl1, acc[b]);
        if constexpr (G::K48) {
            if constexpr (XLO) {
#pragma unroll
                for (int b = 0; b < NVB; ++b) acc[b] = TUCU_MFMA(p.xt[b], clt, acc[b]);   // hi x lo taps
            }
            // XLO: (hi + lo) x hi taps; otherwise hi x (hi + lo taps)
#pragma unroll
            for (int b = 0; b < NVB; ++b) acc[b] = TUCU_MFMA(p.xt[b], cht, acc[b]);
        }
#pragma unroll
        for (int b = 0; b < NVB; ++b) acc[b] = TUCU_MFMA(p.xh[b], ch1, acc[b]);
#pragma unroll
        for (int b = 0; b < NVB; ++b) {
            const v4f16 h = __builtin_convertvector(acc[b], v4f16);
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                const v2f16 lo = {_Float16(__builtin_fmaf(acc[b][i], one, -float(h[i]))),
                                  _Float16(__builtin_fmaf(acc[b][i + 1], one, -float(h[i + 1])))};
                fh[4 * b + i] = h[i]; fh[4 * b + i + 1] = h[i + 1];
                fl[4 * b + i] = lo[0]; fl[4 * b + i + 1] = lo[1];
            }
        }
        // Radius class 8 reads overlapping pairs of blocks: as one register
        // tuple the field is used in place (as separate values the compiler
        // copies every second pair).
        if constexpr (!G::K48) {
            typedef uint32_t vregs __attribute__((ext_vector_type(NF / 2)));
            vregs r = __builtin_bit_cast(vregs, fh), q = __builtin_bit_cast(vregs, fl);
            asm("" : "+v"(r), "+v"(q));
            fh = __builtin_bit_cast(vfield, r);
            fl = __builtin_bit_cast(vfield, q);
        }
    };

    // ------------------------------------------------- horizontal pass
    const bool fast = y0 >= a.fy0 && y0 + 16 <= a.fy1 && x0 >= a.fx0 && x0 + MSTRIP_W <= a.fx1;
    constexpr int NOUT  = ONE ? 1 : 6;
    constexpr int HL[6] = {ONE ? 1 : 0, 1, 0, 2, 1, 0};   // horizontal table of output k
    constexpr int VL[6] = {0, 0, 1, 0, 1, 2};             // vertical field of output k
    bool hooked = false;                        // uniform
    const auto hook = [&] {
        if (!hooked) before_store();
        hooked = true;
    };
    auto hpass = [&](int l, int k, const vfield& fh, const vfield& fl) {
        const int h = HL[k], v = VL[k];
        v4f32 acc[MNB];
#pragma unroll
        for (int o = 0; o < MNB; ++o) acc[o] = v4f32{0.f, 0.f, 0.f, 0.f};
        if constexpr (G::K48) {
            // Fixed pairs of field blocks P_p = (2 p, 2 p + 1), so that no
            // two B operands overlap: output block o takes P_(o/2) and
            // P_(o/2 + 1), whose columns lie d = 32 p - 16 o from its own
            // (d in {-16, 0, 16, 32}; taps beyond the lobe are zero).
            v8f16 ah[4], al[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = MBASE + 16 * i - 16 + 4 * g - RC - m;
                ah[i] = T.hpair[T.pair_at(0, h) + t];
                al[i] = T.hpair[T.pair_at(1, h) + t];
            }
            // smaller products first, as in the vertical pass
            static_for<0, MNB>([&](auto oc) { constexpr int o = oc, p = o / 2, i = (o & 1) ? 0 : 1;
                acc[o] = TUCU_MFMA(al[i], pairP<p>(fh), acc[o]); });
            static_for<0, MNB>([&](auto oc) { constexpr int o = oc, p = o / 2, i = (o & 1) ? 0 : 1;
                acc[o] = TUCU_MFMA(ah[i], pairP<p>(fl), acc[o]); });
            static_for<0, MNB>([&](auto oc) { constexpr int o = oc, p = o / 2 + 1, i = (o & 1) ? 2 : 3;
                acc[o] = TUCU_MFMA(al[i], pairP<p>(fh), acc[o]); });
            static_for<0, MNB>([&](auto oc) { constexpr int o = oc, p = o / 2 + 1, i = (o & 1) ? 2 : 3;
                acc[o] = TUCU_MFMA(ah[i], pairP<p>(fl), acc[o]); });
            static_for<0, MNB>([&](auto oc) { constexpr int o = oc, p = o / 2 + 1, i = (o & 1) ? 2 : 3;
                acc[o] = TUCU_MFMA(ah[i], pairP<p>(fh), acc[o]); });
            static_for<0, MNB>([&](auto oc) { constexpr int o = oc, p = o / 2, i = (o & 1) ? 0 : 1;
                acc[o] = TUCU_MFMA(ah[i], pairP<p>(fh), acc[o]); });
        } else {
            const int t1 = MBASE + 4 * g - RC - m;
            const v8f16 ch1 = T.hpair[T.pair_at(0, h) + t1];
            const v8f16 cl1 = T.hpair[T.pair_at(1, h) + t1];
            static_for<0, MNB>([&](auto oc) { constexpr int o = oc; acc[o] = TUCU_MFMA(cl1, pair8<o>(fh), acc[o]); });
            static_for<0, MNB>([&](auto oc) { constexpr int o = oc; acc[o] = TUCU_MFMA(ch1, pair8<o>(fl), acc[o]); });
            static_for<0, MNB>([&](auto oc) { constexpr int o = oc; acc[o] = TUCU_MFMA(ch1, pair8<o>(fh), acc[o]); });
        }
        const float u = a.mu[k] * inv_s;
        if constexpr (MODE == MODE_ICIA) {      // the gradient stays on chip
            sink(k, acc, u);
            return;
        }
        // Through the wave's LDS staging area, in the output's type, so that
        // each store writes RPI rows x 64 contiguous pixels, 16 bytes a lane
        // (from the accumulators a store would write 16 rows x 16 pixels).
        using ST = MStage<OUT>;
        char* const sb = reinterpret_cast<char*>(stage);
#pragma unroll
        for (int o = 0; o < MNB; ++o) {
            const v4f32 r = acc[o] * u;
            Px<OUT>::pack4(sb + m * ST::PITCH + (16 * o + 4 * g) * ST::ES, r[0], r[1], r[2], r[3]);
        }
        if (k == (l == 0 ? 0 : l == 1 ? 2 : 5)) hook();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        const int r0 = lane / ST::LPR, c0 = lane % ST::LPR * ST::EPL;
        const char* const src = sb + r0 * ST::PITCH + c0 * ST::ES;
        // Buffer stores carry the cache policy: rows from the strip's first row
        // (a uniform base), lane offsets in 32 bits (the host keeps 16 rows of
        // every output within 2^31 bytes).  No scalar offset: after a 16-byte
        // store with one the compiler lets the next vector instruction
        // overwrite the data, and some lanes then stored the new value.
        // At the edge of the valid region a lane whose chunk lies outside takes an
        // offset past the buffer, which drops its store; where the edge lies
        // within a chunk, moved chunks need no store of single pixels (1291 x
        // 1192 f32 six outputs, radius 16: 15.0 us with the pieces of a cut chunk
        // stored one by one, 13.3 so; 823 x 519 11.4 -> 9.1, bf16 9.9 -> 8.0).
        // A tile loop takes the strips inside the valid region first, without
        // these conditions, and reads what the others need from the arguments
        // there and then (held through the loop it spilled 38 scalar registers
        // more: 3840 x 2160 u8 -> f32 42.4 us, 41.8 so; f32 52.6 against 51.7,
        // 2560 x 1440 radius 12 29.4 against 28.4, 4096 x 4096 9 x 9 taps 35.8
        // against 34.9).
        // Where the edge lies within a line, the strip writes a part of it:
        // streamed, that part goes to memory by itself, stored ordinarily it
        // stays in L2 until the kernel ends.  In the tile loops a float strip
        // streams the chunks of its whole lines and stores those of a line that is
        // cut ordinarily (six outputs f32, 3840 x 2160 radius 4: all streamed 47.2
        // us, all ordinary 42.8, so 42.8; 4096 x 4096 91, 94, 83; 2560 x 1440, no
        // buffer in a cache, 24.4, 26.4, 24.6; 64 mixed images 272, 278, 257),
        // except that f32 -> f32 of radius class 16 streams halves too (3000 x 1500
        // radius 16, no buffer in a cache, 29.0 us so, 32.2 ordinarily).  A
        // one-round launch streams the strips whose lines are whole or cut in half
        // and, at radius class 16, lack the last 16 bytes alone (1080p radius 4, 16
        // bytes cut at the left, streaming against ordinary 14.4 against 12.6 us,
        // the last 16 at the right alone 13.2 against 12.3; radius 16, half a line,
        // 14.1 against 14.8, 1292 x 1192 the last 16 bytes 11.6 against 12.7; line by
        // line as the loops VGA radius 4 7.9 against 7.4).  16-bit strips stream it wherever no chunk is cut
        // (1080p bf16 radius 16, a quarter line, 11.1 us, ordinary 11.9), and so
        // do 8-bit ones, whose rows of 64 bytes are half lines throughout (u8 ->
        // u8 1080p radius 16 9.0 us, ordinary and tile by tile along the rows
        // 10.4; 4096 x 4096 17 x 9 taps 15.2, 18.2).
        // Rows that do not start at 128-byte lines take ordinary stores where
        // strips meet in a line (store_rows) or, where no line lies within a
        // strip's row or in a one-round launch, throughout (one-round 1080 x
        // 1923 f32 16.6 us, split 20.9).
        constexpr bool LOOP = CPOL == CPOL_NT, ROWS = ST::ES == 4 && LOOP;
        const auto rsrc_of = [](uintptr_t base) {
            return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(base), short(0), 0x7fffffff, BUF_DWORD3);
        };
        // the strip's chunks through a buffer at base, those where valid(i) holds
        const auto chunks = [&](auto cp, uintptr_t base, int pitch, const auto& valid) {
            constexpr int CP = cp;
            const __amdgpu_buffer_rsrc_t orsrc = rsrc_of(base);
            const int off = r0 * pitch + c0 * ST::ES;
#pragma unroll
            for (int i = 0; i < ST::NI; ++i)
                __builtin_amdgcn_raw_buffer_store_b128(
                    *reinterpret_cast<const v4u32_any*>(src + i * ST::RPI * ST::PITCH), orsrc,
                    valid(i) ? off + i * ST::RPI * pitch : MINVALID, 0, CP);
        };
        const auto streaming = std::integral_constant<int, CPOL>{};
        const auto ordinary = std::integral_constant<int, 0>{};
        // any strip, with c the launch's arguments
        const auto edge = [&](const auto& c) {
            const int64_t pitch64 = int64_t(c.ostride[k]) * ST::ES;
            const int pitch = int(pitch64);         // wraps only where c.far keeps it unused
            const uintptr_t base = c.obase[k] + uintptr_t(y0 * pitch64 + int64_t(x0) * ST::ES);
            const int rv = c.r[v], rh = c.r[h];
            const bool buf = (ST::ES == 4 || c.aligned) && !c.far;
            // the valid columns of the strip: [e0, e1)
            const int e0 = max(rh - x0, 0), e1 = min(c.ncol - rh - x0, MSTRIP_W);
            const bool cut = ((e0 | e1) & (ST::EPL - 1)) != 0;      // uniform: an edge lies within a chunk
            const int yv = y0 + r0 - rv, rows = c.nrow - 2 * rv;    // row step i is valid: yv + RPI i in [0, rows)
            const int b0 = e0 * ST::ES, b1 = e1 * ST::ES;           // the strip's part of its lines
            // the lane's chunk lies in a line that the strip writes whole
            const auto in_whole = [&] {
                const int cb = c0 * ST::ES;
                return cb >= ((b0 + 127) & ~127) && cb + 16 <= (b1 & ~127);
            };
            // A chunk that an edge cuts is moved inside, where it overlaps its
            // neighbour, with the same values.  (What a branch needs is computed
            // in it: shared, it is held in scalar registers, 294 spilled in the
            // f32 tile loop of radius class 8, 160 so, 121 with the arguments read
            // here.)
            if constexpr (ST::ES == 4) {
                if (buf && cut && e1 - e0 >= ST::EPL) {
                    const int cs = min(max(c0, e0), e1 - ST::EPL);
                    const bool in = c0 + ST::EPL > e0 && c0 < e1;
                    const __amdgpu_buffer_rsrc_t orsrc = rsrc_of(base);
                    const int off = r0 * pitch + cs * ST::ES;
                    const auto moved = [&](auto cp, bool at) {
                        constexpr int CP = cp;
#pragma unroll
                        for (int i = 0; i < ST::NI; ++i)
                            __builtin_amdgcn_raw_buffer_store_b128(
                                *reinterpret_cast<const v4u32u*>(src + i * ST::RPI * ST::PITCH + (cs - c0) * ST::ES), orsrc,
                                at && unsigned(yv + i * ST::RPI) < unsigned(rows) ? off + i * ST::RPI * pitch : MINVALID, 0,
                                CP);
                    };
                    if (LOOP && c.lines) {
                        const bool wl = in_whole();
                        moved(streaming, in && wl);
                        moved(ordinary, in && !wl);
                    } else {
                        moved(ordinary, in);
                    }
                    return;
                }
            }
            if (buf && !cut) {
                const auto valid = [&](int i) {
                    return c0 >= e0 && c0 < e1 && unsigned(yv + i * ST::RPI) < unsigned(rows);
                };
                const bool stream = ST::ES < 4 ? true
                                    : LOOP     ? ((b0 | b1) & (RC == 16 && sizeof(IN) == 4 ? 63 : 127)) == 0
                                               : (b0 & 63) == 0 && ((b1 & 63) == 0 || (RC == 16 && (b1 & 127) >= 112));
                if (c.lines && stream) {
                    chunks(streaming, base, pitch, valid);
                } else if (ROWS && c.lines) {
                    const bool wl = in_whole();
                    chunks(streaming, base, pitch, [&](int i) { return wl && valid(i); });
                    chunks(ordinary, base, pitch, [&](int i) { return !wl && valid(i); });
                } else {
                    chunks(ordinary, base, pitch, valid);
                }
            } else if (e1 - e0 >= ST::EPL) {
                // an edge within a chunk of 16-bit or 8-bit pixels, rows of them
                // that are not aligned to four, rows too far apart: plain addresses
                const int cs = min(max(c0, e0), e1 - ST::EPL);
                const bool in = c0 + ST::EPL > e0 && c0 < e1;
#pragma unroll
                for (int i = 0; i < ST::NI; ++i)
                    if (in && unsigned(yv + i * ST::RPI) < unsigned(rows))
                        *reinterpret_cast<gptr<v4u32u>>(base + uintptr_t((i * ST::RPI + r0) * pitch64 + cs * ST::ES)) =
                            *reinterpret_cast<const v4u32u*>(src + i * ST::RPI * ST::PITCH + (cs - c0) * ST::ES);
            } else {
                // less than a chunk: a lane a pixel (six outputs of radius 4, 1291 x
                // 1192 bf16 9.1 us, 823 x 519 f32 7.9; with the pixels of a row stored
                // one after the other 11.0 and 10.1)
                using T = std::conditional_t<ST::ES == 4, u32_any, std::conditional_t<ST::ES == 2, u16_any, uint8_t>>;
                const int x = e0 + lane % ST::EPL, q = lane / ST::EPL;
#pragma unroll
                for (int i = 0; i < 16; i += 64 / ST::EPL)
                    if (x < e1 && unsigned(y0 + q + i - rv) < unsigned(rows))
                        *reinterpret_cast<gptr<T>>(base + uintptr_t((q + i) * pitch64 + x * ST::ES)) =
                            *reinterpret_cast<const T*>(sb + (q + i) * ST::PITCH + x * ST::ES);
            }
        };
        if constexpr (LOOP) {
            if (fast && (ST::ES == 4 || a.aligned) && !a.far) {
                const int pitch = a.ostride[k] * ST::ES;
                const uintptr_t base = a.obase[k] + uintptr_t(int64_t(y0) * pitch + int64_t(x0) * ST::ES);
                const auto all = [](int) { return true; };
                if (a.lines)             chunks(streaming, base, pitch, all);
                else if constexpr (ROWS) store_rows<ST::PITCH>(rsrc_of(base), base, src, r0, c0 * ST::ES, pitch);
                else                     chunks(ordinary, base, pitch, all);
            } else {
                edge(opaque_args(a));
            }
        } else {
            edge(a);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
#ifdef TUCU_TIMELINE
        if constexpr (CPOL == CPOL_NT_WT && MODE == MODE_GAUSS && RC == 16 && std::is_same_v<IN, float> &&
                      std::is_same_v<OUT, float>)
            tl_stamp(3 + k);
#endif
    };

    // One field at a time, each followed by the outputs it feeds, so that
    // the first stores leave after a third of the vertical work.
    const unsigned fneed[3] = {ONE ? 1u : mask & 0x0bu, ONE ? 0u : mask & 0x14u, ONE ? 0u : mask & 0x20u};
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        if (!fneed[l]) continue;
        vfield fh, fl;
        vpass(l, fh, fl);
        if (!(mask >> (l == 0 ? 0 : l == 1 ? 2 : 5) & 1u)) hook();   // else in the field's first output
#pragma unroll
        for (int k = 0; k < NOUT; ++k)
            if (VL[k] == l && (mask >> k & 1u)) hpass(l, k, fh, fl);
    }
    // Rare: the products could not carry this strip's input.  Its outputs are
    // written again by the FP32 form, after the stores above have completed.
    if constexpr (CHECK) {
        if (p.redo) {                           // wave-uniform
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            mfma_strip_fp32<RC, IN, OUT, MODE>(opaque_args(a), y0, x0, T, stage, mask);
        }
    }
}

// The same without a sink, for the outputs of a.mask (every mode that
// writes its outputs).
template <int RC, class IN, class OUT, int MODE = MODE_GAUSS, int CPOL = CPOL_NT, bool FRESH = false, class A, class H>
__device__ __forceinline__ void
mfma_filter(const A& a, int y0, int x0, const MfmaOps& p, const ModeTabs<MODE>& T, float* stage, H&& before_store)
{
    mfma_filter<RC, IN, OUT, MODE, CPOL, FRESH>(a, y0, x0, p, T, stage, 0, a.mask, before_store);
}
#undef TUCU_MFMA

// Workgroup tiles (strip-major: tile = tx * tiles_y + ty) hold WY strips
// down by 4 / WY across, i.e. 16 WY rows x 256 / WY columns.  Every shape
// filters the same 16 x 64 strips (at rows cy0 + 16 i, columns cx0 + 64 j),
// so the shape changes no result.
struct TilePos {
    int ty, tx;                 // first row and column of the tile
    int y0, x0;                 // first row and column of this wave's strip
    bool live;                  // the strip lies in the region
};

template <int WY, int NW = MWAVES, class A>
__device__ __forceinline__ TilePos mfma_tile_pos(const A& a, int tile)
{
    constexpr int WX = NW / WY;
    const int tx = tile / a.tiles_y;
    const int ty = tile - tx * a.tiles_y;
    const int w  = int(threadIdx.x) >> 6;
    // wave-uniform, and held in scalar registers so that every test on the
    // strip's position is a scalar branch: a divergent if / else around the
    // loads makes the compiler wait for the loads already in flight before
    // the other side's address arithmetic
    TilePos p;
    p.ty = __builtin_amdgcn_readfirstlane(a.cy0 + ty * (16 * WY));
    p.tx = __builtin_amdgcn_readfirstlane(a.cx0 + tx * (MSTRIP_W * WX));
    p.y0 = __builtin_amdgcn_readfirstlane(p.ty + 16 * (w / WX));
    p.x0 = __builtin_amdgcn_readfirstlane(p.tx + MSTRIP_W * (w % WX));
    p.live = p.y0 < a.cy1 && p.x0 < a.cx1;
    return p;
}

// The operands of a strip of the tile whose window, laid out for radius class
// WC >= RC, is in LDS at win.
template <int RC, int SY, int SX, class IN, bool FRESH = false, int WC = RC, class A>
__device__ __forceinline__ void mfma_ops_tile(const A& a, const char* win, MfmaOps& p)
{
    using W = MWin<WC, SY, SX, IN>;
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    int lane = threadIdx.x & 63;
    if constexpr (FRESH) asm volatile("" : "+v"(lane));    // as for mfma_load
    mfma_ops_win<RC, IN, W::PITCH>(a, win + (16 * (w / SX) + WC - RC) * W::PITCH + (MSTRIP_W * (w % SX) + WC - RC) * W::ES,
                                    lane, p);
}

// First tile of XCD x's range when ntiles tiles are shared by grid
// workgroups: ranges proportional to the workgroups each XCD receives, so
// that with as many workgroups as tiles every workgroup takes exactly one.
__device__ __forceinline__ int mfma_share_lo(int ntiles, int grid, int x)
{
    const int q = grid / QN, r = grid - q * QN;
    return int(int64_t(ntiles) * (q * x + min(x, r)) / grid);
}

// Reads, in one round of scalar loads, every kernel argument a strip's
// loads depend on.  Left to itself the compiler reads each where it is first
// used, behind branches that need the one before: six dependent round trips
// to the argument block before a wave could issue its first input load
// (1080p six outputs: 2 % of the launch).
template <class A>
__device__ __forceinline__ void mfma_args_early(const A& a)
{
    const int grid = int(gridDim.x);
    const int ty = a.tiles_y, cy0 = a.cy0, cy1 = a.cy1, cx0 = a.cx0, cx1 = a.cx1;
    const int nr = a.nrow, nc = a.ncol, sb = a.in_stride_b;
    const uint32_t nb = a.in_bytes;
    const void* const in = a.in;
    const void* const tabs = a.tabs;
    asm volatile("" ::"s"(grid), "s"(ty), "s"(cy0), "s"(cy1), "s"(cx0), "s"(cx1), "s"(nr), "s"(nc), "s"(sb), "s"(nb),
                 "s"(in), "s"(tabs));
}

// One image, one workgroup per tile (images with no more tiles than
// resident workgroups, such as 1080p).
template <int RC, int WY, class IN, class OUT, int MODE = MODE_GAUSS>
__global__ void __launch_bounds__(64 * MWAVES) __attribute__((amdgpu_waves_per_eu(MFMA_WAVES_PER_SIMD)))
sepfir_mfma_kernel(const SepArgs a)
{
    __shared__ ModeTabs<MODE> T;
    __shared__ v4f32 stage4[MWAVES * 16 * MOPITCH / 4];
#ifdef TUCU_TIMELINE
    constexpr bool TL = MODE == MODE_GAUSS && RC == 16 && std::is_same_v<IN, float> && std::is_same_v<OUT, float>;
    const auto stamp = [](int i) {
        if constexpr (TL) {
            __builtin_amdgcn_sched_barrier(0);
            tl_stamp(i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#else
    const auto stamp = [](int) {};
#endif
    stamp(0);
    mfma_args_early(a);
    float* const stage = reinterpret_cast<float*>(stage4) + (threadIdx.x >> 6) * 16 * MOPITCH;
    const TilePos t = mfma_tile_pos<WY>(a, xcd_remap(blockIdx.x, gridDim.x));
    MfmaOps p;
    if constexpr (sizeof(IN) < 4) {
        using W = MWin<RC, WY, MWAVES / WY, IN>;
        __shared__ v4u32 win4[W::BYTES / 16];
        char* const win = reinterpret_cast<char*>(win4);
        v4u32 v[W::N];
        const int tid = int(threadIdx.x);
        mwin_load<RC, WY, MWAVES / WY, IN>(a, tid, t.ty, t.tx, v);    // in flight while the tables are copied
        mfma_get_tabs<MODE>(a, T);
        mwin_store<RC, WY, MWAVES / WY, IN>(tid, win, v);
        __syncthreads();
        if (!t.live) return;
        mfma_ops_tile<RC, WY, MWAVES / WY, IN>(a, win, p);
    } else {
        MfmaRaw raw;
        if (t.live) mfma_load<RC>(a, t.y0, t.x0, raw);    // in flight while the tables are built
        stamp(10);
        mfma_get_tabs<MODE>(a, T);
        stamp(11);
        __syncthreads();
        stamp(1);
        if (!t.live) return;
        mfma_ops_raw<RC>(a, raw, p);
        stamp(2);
    }
    // one round of workgroups: outputs written through L2 (CPOL_NT_WT)
    mfma_filter<RC, IN, OUT, MODE, CPOL_NT_WT>(a, t.y0, t.x0, p, T, stage, [] {});
    stamp(9);
}

// One large image: a grid of the resident workgroups; each builds the tap
// tables once and filters a static share of the tiles: the tile list
// (strip-major, so consecutive tiles are vertically adjacent) is cut into one
// contiguous range per XCD, and the workgroups of XCD x take the tiles of
// range x in turn, so neighbouring tiles, which read the same halo rows, run
// at the same time on one L2.  The tables are read-only after the build and
// each wave has its own staging area, so the tiles need no barrier between
// them.  (A 4096 x 4096 FIRFilter2 launch: 21.5 us against 25.5 us with one
// workgroup per tile, which rebuilds the tables 4096 times.)
template <int RC, int WY, class IN, class OUT, int MODE = MODE_GAUSS>
__global__ void __launch_bounds__(64 * MWAVES) __attribute__((amdgpu_waves_per_eu(MFMA_LOOP_WAVES<RC, IN, OUT, MODE>, MFMA_LOOP_WAVES_MAX<RC, IN, OUT, MODE>)))
sepfir_mfma_loop_kernel(const SepArgs a, int ntiles)
{
    __shared__ ModeTabs<MODE> T;
    __shared__ v4f32 stage4[MWAVES * 16 * MOPITCH / 4];
    mfma_args_early(a);
    const int grid = int(gridDim.x), b = int(blockIdx.x);
    const int x = b % QN, step = (grid - x + QN - 1) / QN;           // workgroups on this XCD
    const int hi = mfma_share_lo(ntiles, grid, x + 1);
    int t = mfma_share_lo(ntiles, grid, x) + b / QN;
    float* const stage = reinterpret_cast<float*>(stage4) + (threadIdx.x >> 6) * 16 * MOPITCH;
    if (t >= hi) return;                            // uniform over the workgroup
    // The six-output strip code takes its lane index afresh in each tile: left to
    // itself the compiler computes the lane-derived offsets once, before the loop,
    // and holds them through it (3840 x 2160 six outputs f32 1 % faster).  The
    // one-output loop does so for 16-bit input at radius class 16 alone (4096 x
    // 4096 bf16 29.4 against 31.4 us): u8 runs 3-7 % slower so.
    constexpr bool FRESH = MODE == MODE_GAUSS || (sizeof(IN) == 2 && RC == 16);
    // The next window goes into LDS before the tile's first stores, so that the
    // wait for its loads is not one for the stores too.
    // Output rows that do not start at 128-byte lines: the tiles row by row, so
    // that tiles which meet in a line run at about the same time and L2 merges
    // their parts of it (3001 x 4003 packed, radius 16: bf16 66 -> 58 us, f32 91
    // -> 87 against tiles of 16 x 256 pixels in strip-major order).
    const int nx = a.lines ? 0 : ntiles / a.tiles_y;
    const auto place = [&](int i) { return mfma_tile_pos<WY>(a, nx ? i % nx * a.tiles_y + i / nx : i); };
    TilePos pos = place(t);
    if constexpr (MFMA_DIRECT<RC, IN, MODE>) {
        MfmaRaw16 raw;
        if (pos.live) mfma_load16(a, pos.y0, pos.x0, raw);      // in flight while the tables are built
        mfma_get_tabs<MODE>(a, T);
        __syncthreads();
        while (t < hi) {                            // uniform over the workgroup
            if (pos.live) {
                MfmaOps p;
                mfma_ops_raw16<IN>(a, raw, p);
                mfma_filter<RC, IN, OUT, MODE, CPOL_NT, FRESH>(a, pos.y0, pos.x0, p, T, stage, [] {});
            }
            t += step;
            if (t >= hi) break;
            pos = place(t);
            if (pos.live) mfma_load16(a, pos.y0, pos.x0, raw);
        }
    } else if constexpr (sizeof(IN) < 4) {
        using W = MWin<RC, WY, MWAVES / WY, IN>;
        __shared__ v4u32 win4[W::BYTES / 16];
        char* const win = reinterpret_cast<char*>(win4);
        v4u32 v[W::N];
        int tid = int(threadIdx.x);
        mwin_load<RC, WY, MWAVES / WY, IN>(a, tid, pos.ty, pos.tx, v);    // in flight while the tables are copied
        mfma_get_tabs<MODE>(a, T);
        mwin_store<RC, WY, MWAVES / WY, IN>(tid, win, v);
        for (;;) {
            if constexpr (FRESH) asm volatile("" : "+v"(tid));
            lds_barrier();                          // the window (at first also the tables) is complete
            MfmaOps p;
            if (pos.live) mfma_ops_tile<RC, WY, MWAVES / WY, IN, FRESH>(a, win, p);
            lds_barrier();                          // every wave has its operands: the window may be overwritten
            const TilePos now = pos;
            t += step;
            const bool more = t < hi;
            if (more) {                             // the next window's loads run under this tile's work
                pos = place(t);
                mwin_load<RC, WY, MWAVES / WY, IN>(a, tid, pos.ty, pos.tx, v);
            }
            const auto next = [&] { if (more) mwin_store<RC, WY, MWAVES / WY, IN>(tid, win, v); };
            if (now.live)
                mfma_filter<RC, IN, OUT, MODE, CPOL_NT, FRESH>(a, now.y0, now.x0, p, T, stage, next);
            else
                next();
            if (!more) break;
        }
    } else {
        MfmaRaw raw;
        if (pos.live) mfma_load<RC>(a, pos.y0, pos.x0, raw);    // in flight while the tables are built
        mfma_get_tabs<MODE>(a, T);
        __syncthreads();
        while (t < hi) {                            // uniform over the workgroup
            if (pos.live) {
                MfmaOps p;
                mfma_ops_raw<RC>(a, raw, p);
                mfma_filter<RC, IN, OUT, MODE, CPOL_NT, FRESH>(a, pos.y0, pos.x0, p, T, stage, [] {});
            }
            t += step;
            if (t >= hi) break;
            pos = place(t);
            if (pos.live) mfma_load<RC, FRESH>(a, pos.y0, pos.x0, raw);
        }
    }
}

inline int mfma_cus()
{
    int dev = 0, ncu = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    return std::max(1, ncu);
}

// Workgroups resident at once on the whole GPU for this instantiation.
template <class K>
int mfma_resident(K kernel)
{
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kernel), 64 * MWAVES, 0)
            != hipSuccess || per_cu < 1)
        per_cu = 1;
    return mfma_cus() * per_cu;
}

// Workgroups of a tile loop over n tiles, at most resident of them: the
// fewest per CU that take no more rounds (2560 x 1440 u8 -> f32 six outputs,
// radius 16: 22.5 us, 24.9 with all that fit).  (Six outputs f32 -> f32,
// radius class 8, with two per CU where the last of at most three rounds of three
// is half empty: 3840 x 2160 51.9 us against 49.4 with three, 2000 x 4096 52.0
// against 49.5, 3000 x 1500 30.3 against 29.0.)
inline int mfma_loop_grid(int n, int resident)
{
    static const int ncu = mfma_cus();
    const int64_t rounds = (int64_t(n) + resident - 1) / resident;
    const int64_t per_cu = (n + rounds * ncu - 1) / (rounds * ncu);
    return int(std::min<int64_t>({int64_t(n), int64_t(resident), per_cu * ncu}));
}

// The most workgroups per CU of a tile loop.  One output of u8 input at radius
// class 8 has registers for four or five and is bound by memory: with three,
// 4096 x 4096 17 x 9 taps u8 -> f16 take 14.9 us against 16.0, -> u8 15.4 against
// 16.0, 3840 x 2160 17 x 17 -> f32 10.4 against 10.7.
template <int RC, class IN, int MODE>
constexpr int MFMA_LOOP_PER_CU = MODE == MODE_TAPS && RC == 8 && sizeof(IN) == 1 ? 3 : 8;

// One image in the region of a: one workgroup per WYR-shaped tile where they
// fit the resident workgroups, else the tile loop with WYL, whose tile count
// nblocks and tiles_y the call brings.  (One-output launches, MODE_TAPS, WYR =
// 1 x 4 strips and WYL = 2 x 2: 1080p 17 x 17 lobes 7.0 us against 7.3 with 2 x
// 2, the 4096^2 u8 launches 3-7 % slower with 1 x 4.)
template <int RC, int WYR, int WYL, class IN, class OUT, int MODE = MODE_GAUSS>
hipError_t launch_sepfir_mfma(const SepArgs& a, int nblocks, hipStream_t s)
{
    static const int loop = std::min(mfma_resident(sepfir_mfma_loop_kernel<RC, WYL, IN, OUT, MODE>),
                                     mfma_cus() * MFMA_LOOP_PER_CU<RC, IN, MODE>);
    static const int one = MODE == MODE_TAPS ? mfma_resident(sepfir_mfma_kernel<RC, WYR, IN, OUT, MODE>) : loop;
    constexpr int H = 16 * WYR, W = MSTRIP_W * (MWAVES / WYR);
    SepArgs r = a;
    r.tiles_y = (a.cy1 - a.cy0 + H - 1) / H;
    const int64_t n = int64_t((a.cx1 - a.cx0 + W - 1) / W) * r.tiles_y;
    if (n <= one)
        hipLaunchKernelGGL((sepfir_mfma_kernel<RC, WYR, IN, OUT, MODE>), dim3(int(n)), dim3(64 * MWAVES), 0, s, r);
    else
        hipLaunchKernelGGL((sepfir_mfma_loop_kernel<RC, WYL, IN, OUT, MODE>), dim3(mfma_loop_grid(nblocks, loop)),
                           dim3(64 * MWAVES), 0, s, a, nblocks);
    return hipGetLastError();
}

// Matrix-core variant of batch_kernel: the same tile queue; the tap
// tables in LDS are rebuilt when the job changes (tiles of a job are
// contiguous in the list).  Tiles hold SY x SX strips, one per wave (SY = SX
// = 1: one-wave workgroups, each with its own tables).
// Float input: each tile is loaded, filtered and stored in turn.
template <int SY, int SX, class IN, class OUT>
__device__ __forceinline__ void
batch_mfma_float(const SepArgs* __restrict__ jobs_, const BatchTile* __restrict__ tiles, int ntiles,
                 int* __restrict__ counter, MfmaTabs& T, float* stage, int& next)
{
    ConstArgs* const jobs = (ConstArgs*)(uintptr_t)jobs_;
    int cur = -1;
    TileQueue q;
    int ti = q.first(ntiles);
    for (;;) {
        if (threadIdx.x == 0)          // the answer is read after this tile
            next = q.grab(counter, ntiles);
        if (ti >= 0) {
            const BatchTile e = tiles[ti];
            ConstArgs& a = jobs[e.job];
            if (int(e.job) != cur) {   // uniform over the workgroup
                mfma_build_tabs(a, T);
                cur = int(e.job);
                __syncthreads();
            }
            const TilePos t = mfma_tile_pos<SY, SY * SX>(a, int(e.tile));
            if (t.live) {
                MfmaRaw raw;
                const auto strip = [&](auto rc) {
                    constexpr int RC = rc;
                    MfmaOps p;
                    mfma_load<RC>(a, t.y0, t.x0, raw);
                    mfma_ops_raw<RC>(a, raw, p);
                    mfma_filter<RC, IN, OUT>(a, t.y0, t.x0, p, T, stage, [] {});
                };
                if (a.rt <= 8) strip(std::integral_constant<int, 8>{});
                else           strip(std::integral_constant<int, 16>{});
            }
        }
        __syncthreads();               // T reuse; `next` was written before this barrier
        ti = __builtin_amdgcn_readfirstlane(next);
        __syncthreads();               // all have read `next` before thread 0 writes it again
        if (ti >= ntiles) break;
    }
}

// Narrow input: the window of the next tile is loaded (into registers) while
// the current one is filtered, so the queue is asked two tiles ahead; its
// answer is looked at after the tile's work.
template <int SY, int SX, class IN, class OUT>
__device__ __forceinline__ void
batch_mfma_narrow(const SepArgs* __restrict__ jobs_, const BatchTile* __restrict__ tiles, int ntiles,
                  int* __restrict__ counter, MfmaTabs& T, float* stage, int& next, char* win)
{
    ConstArgs* const jobs = (ConstArgs*)(uintptr_t)jobs_;
    v4u32 v[MWin<16, SY, SX, IN>::N];
    int tid = int(threadIdx.x);
    int job = 0;                       // of the tile whose window is in v, then in LDS
    TilePos t{};
    // one window layout for both radius classes
    const auto load = [&](int i) {
        job = __builtin_amdgcn_readfirstlane(int(tiles[i].job));
        ConstArgs& a = jobs[job];
        t = mfma_tile_pos<SY, SY * SX>(a, __builtin_amdgcn_readfirstlane(int(tiles[i].tile)));
        mwin_load<16, SY, SX, IN>(a, tid, t.ty, t.tx, v);
    };
    int cur = -1;
    TileQueue q;
    const int first = q.first(ntiles);
    if (threadIdx.x == 0) next = q.grab(counter, ntiles);
    if (first >= 0) {
        load(first);
        mwin_store<16, SY, SX, IN>(tid, win, v);
    }
    for (;;) {                         // everything but v, tid and raw is uniform over the workgroup
        asm volatile("" : "+v"(tid));  // what derives from it is computed in each tile, not held through the loop
        job = __builtin_amdgcn_readfirstlane(job);
        ConstArgs& a = jobs[job];
        if (job != cur) {
            lds_barrier();             // no wave reads the old tables any more
            mfma_build_tabs(a, T);
            cur = job;
        }
        lds_barrier();                 // the window, the tables and `next` are written
        const int nt = __builtin_amdgcn_readfirstlane(next);
        const TilePos now = t;
        const bool small = a.rt <= 8;
        MfmaOps p;
        if (now.live) {
            if (small) mfma_ops_tile<8, SY, SX, IN, true, 16>(a, win, p);
            else       mfma_ops_tile<16, SY, SX, IN, true>(a, win, p);
        }
        lds_barrier();                 // the window and `next` have been read
        int raw = 0;
        if (nt < ntiles) {
            if (threadIdx.x == 0) raw = q.ask(counter);
            load(nt);
        }
        const auto after = [&] { if (nt < ntiles) mwin_store<16, SY, SX, IN>(tid, win, v); };
        if (!now.live)  after();
        else if (small) mfma_filter<8, IN, OUT, MODE_GAUSS, CPOL_NT, true>(a, now.y0, now.x0, p, T, stage, after);
        else            mfma_filter<16, IN, OUT, MODE_GAUSS, CPOL_NT, true>(a, now.y0, now.x0, p, T, stage, after);
        if (nt >= ntiles) break;
        if (threadIdx.x == 0) next = q.answer(counter, ntiles, raw);
    }
}

template <int SY, int SX, class IN, class OUT>
__global__ void __launch_bounds__(64 * SY * SX)
__attribute__((amdgpu_waves_per_eu(SY * SX == 1 ? 2 : MFMA_WAVES_PER_SIMD)))   // one-wave: LDS allows no more
batch_mfma_kernel(const SepArgs* __restrict__ jobs, const BatchTile* __restrict__ tiles, int ntiles,
                  int* __restrict__ counter)
{
    __shared__ MfmaTabs T;
    __shared__ v4f32 stage4[SY * SX * 16 * MOPITCH / 4];
    __shared__ int next;
    float* const stage = reinterpret_cast<float*>(stage4) + (threadIdx.x >> 6) * 16 * MOPITCH;
    if constexpr (sizeof(IN) == 4) {
        batch_mfma_float<SY, SX, IN, OUT>(jobs, tiles, ntiles, counter, T, stage, next);
    } else {
        __shared__ v4u32 win4[MWin<16, SY, SX, IN>::BYTES / 16];
        batch_mfma_narrow<SY, SX, IN, OUT>(jobs, tiles, ntiles, counter, T, stage, next, reinterpret_cast<char*>(win4));
    }
}

template <int SY, int SX, class IN, class OUT>
hipError_t launch_batch_mfma(const SepArgs* jobs, const BatchTile* tiles, int ntiles, int* counter,
                             int grid, hipStream_t s)
{
    hipLaunchKernelGGL(reset_queue<>, dim3(1), dim3(64), 0, s, counter, grid);
    hipLaunchKernelGGL((batch_mfma_kernel<SY, SX, IN, OUT>), dim3(grid), dim3(64 * SY * SX), 0, s, jobs, tiles, ntiles,
                       counter);
    return hipGetLastError();
}

// Workgroup shapes: WY = 1, 2, 4 strips down (tile rows 16, 32, 64).
constexpr int MFMA_RADII[2] = {8, 16};
constexpr int NMWY = 3;
constexpr int MFMA_WYS[NMWY] = {1, 2, 4};
// Default shapes (indices into MFMA_WYS), measured: the six-output kernels
// 1 x 4 strips, 64 x 64 pixels (1080p f32 / bf16 / f16 2.5-4 % faster than
// 2 x 2, 3840 x 2160 3 %: the strips of a workgroup share their vertical
// halo rows in L1); the one-output FIR / general-taps tile loop 2 x 2, 32 x
// 128 (the 4096^2 u8 launches 2.5-7 % slower with 1 x 4), its one-round
// launches 1 x 4 (launch_sepfir_mfma); the ICIA pass 1 x 4 (1080p f32 sigma 3
// projective 8 %, 3840 x 2160 u8 1-3 % faster, 1080p sigma 2 2 % slower).
constexpr int MFMA_WY_DEFAULT = 2;
constexpr int MFMA_WY_ONE = 1;
constexpr int MFMA_WY_ICIA = 2;

extern KernelEntry g_gauss_mfma_table[2][NMWY][4][4];
extern KernelEntry g_fir_mfma_table[2][4][4];       // MODE_TAPS, default shape: [radius class][in][out]

}   // namespace tucu
