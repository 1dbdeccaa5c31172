// The decoder's convolutions on the bf16 matrix cores without giving up F32
// (the three-way split of Henry, Tang and Heinecke, "Leveraging the bfloat16
// Artificial Intelligence Datatype For Higher-Precision Computations", 2019):
// every F32 operand v of 2^-110 and up is the exact sum of three bf16 values,
// hi + mid + lo (each the round-to-nearest bf16 of what the ones before leave; 8
// + 8 + 8 significand bits), and a product a * b is
//   hi hi + (hi mid + mid hi) + mid mid + (hi lo + lo hi)
// in F32 accumulators of v_mfma_f32_32x32x16_bf16. Of the products left out, mid
// lo and lo mid are below 2^-25 |a b| each and below 2^-24 together, about the F32
// rounding of a single product. The five small products have accumulators of
// their own, so the large sum rounds once per 16 terms (the F32 MFMA: once per
// 4): against float64 the results lie 1.5 to 3.2 times closer than the F32
// launches' on sums of four terms and more (512 channels, k = 7: 2.0e-7 against
// 5.4e-7 in the 2-norm); shorter ones stay with those.
//
// What bounds it: the matrix pipe's power. Six bf16 MFMAs take the place of
// work that costs 16 times their cycles in F32, 417 TFLOP/s of F32 sums at the
// nominal clock; MFMAs alone on random data hold 1.82 PFLOP/s (the clock falls),
// 303 TFLOP/s of sums. 512 channels x 60000, k = 7: 2.1 ms and 104 TFLOP/s with
// the F32 MFMA, 0.95 ms and 231 TFLOP/s here. The weights' way from L2 is 22 %
// of the time and the staging 16 % (timed with each left out).
//
// As an implicit GEMM: rows R (output channels; for a transposed convolution
// channel times stride phase, R = co * stride + r, so that one lane's
// neighbouring rows are neighbouring output samples), columns = samples, K =
// input channels times taps in steps of 16 channels of one tap.
// - Weights: a pack launch splits them once per call into the caller's
//   workspace in fragment order ([32 rows][16 channels][tap][plane][lane] of 16
//   bytes); a wave loads its fragments from L2 into registers, one K step
//   ahead, and no weight passes through LDS. It also evaluates the SnakeBeta
//   parameters (three floats a channel).
// - Input: a chunk's columns (halo included) are loaded, SnakeBeta applied and
//   split once per workgroup into LDS as [plane][8 channels][column], so that a
//   B fragment of any tap is one conflict-free 16-byte read at a column offset.
//   Double buffered; the staging of the next chunk runs between the MFMAs.
// - A workgroup is 8 waves of 32 rows x 128 columns (4 in the residual units of
//   128 channels), two waves a SIMD. Waves of 64 x 64 load every weight twice
//   per workgroup: 0.94 of the speed; one wave a SIMD with 64 x 128: 0.87; four
//   waves a workgroup, two workgroups a CU (twice the staging): 0.92.
//
// Infinities and NaN: the first part carries them, the others are NaN then. The
// hi hi sums have accumulators of their own, so where one is not finite it is
// the output as it stands: an infinite or NaN operand makes it what the F32 sum
// is, and what the small products did does not matter (a decode of 252 frames, all
// of it NaN in the end: 10.6 ms with the look through the tiles' inputs, 7.1 ms for
// an ordinary one; F32 launches 15.9 and 13.5 ms). What that does not cover
// is summed again in plain F32, by the workgroup whose tile it is (f32_needed):
// sums that are not finite where a finite product may overflow (its parts'
// products overflow apart, or only the first does) or an operand is so small
// that its first part may be zero, and tiles of operands so small that the parts
// lose bits (bf16's smallest is 2^-133). 20 to 40 times the tile's time.
#include "conv_x3.hpp"

#include "snake_math.hpp"

#include <algorithm>
#include <type_traits>

namespace levo_hip {
namespace {

constexpr int kThreads = 256;
constexpr int kUnit = 128;  // channels of a fused residual unit
constexpr int kCI = 16;     // input channels per K step
constexpr int kMaxHalo = 64;  // (taps - 1) * dilation: k = 7 up to dilation 10
constexpr int kNT = 128;      // columns per workgroup
constexpr int kUnitItems = 6 * (kUnit / kCI) * 64;  // half a unit's h: [16 channels][plane][8 channels][column]
constexpr int kUnitInfoItems = kUnit * 24 / 16;     // unit_row per channel

template <int KW, bool FUSE>
struct x3_shape {
    static constexpr int WAVES = FUSE ? 4 : 8;           // of 32 rows each
    static constexpr int ROWS = 32 * WAVES;
    static constexpr int THREADS = 64 * WAVES;
    static constexpr int CG = KW <= 2 ? 2 : 1;           // 16-channel groups per chunk
    static constexpr int CI = 16 * CG;                   // input channels per chunk
    static constexpr int KS = CG * KW;                   // K steps per chunk
    static constexpr bool HALO = KW > 2;
    static constexpr int OUT = KW == 2 ? kNT - 1 : kNT;  // columns kept: k = 2 gives up one for its halo
    // Columns of a staged row in LDS: fixed, so that planes and column groups
    // are immediate offsets.
    static constexpr int W = kNT + (KW == 1 ? 0 : KW == 2 ? 8 : kMaxHalo);
    static constexpr int GROUP = 6 * W;                  // 16-byte items of a channel group: [plane][8 channels][column]
    static constexpr int BUF = CG * GROUP;
    // Pairs of channels staged per thread and chunk: main columns, then halo.
    static constexpr int MAIN = 16 * CG / WAVES;
    static constexpr int PAIRS = MAIN + (HALO ? 8 / WAVES : 0);
    // LDS: two buffers of a chunk, over them what the epilogue needs; then the
    // words of tile_state
    static constexpr int STATE = FUSE ? std::max(2 * BUF, kUnitItems + kUnitInfoItems) : 2 * BUF;
    static constexpr int LDS_ITEMS = STATE + 2;
};

typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef float f32x16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));

struct x3_kernel_params {
    x3_conv c;
    const u32x4 * w;         // packed fragments
    const uint32_t * w_range;  // [32-row tiles][channel groups]: value_range of the weights
    const snake_param * pre;   // [channel groups * 16] (c.snake)
    const snake_param * post;  // [c_out] (c.post_alpha_log)
    int32_t rows;            // c_out * stride
    int32_t chunks;
    int32_t tiles_x, tiles;  // column tiles; column tiles times row tiles
    int32_t splits;
    float * part;            // splits > 1: partial sums [split][row][part_pitch]
    int64_t part_slice, part_pitch;
    // the k = 1 convolution of a residual unit (unit_tail)
    const u32x4 * w1;
    const uint32_t * w1_range;
    const float * w1_raw;
    const float * bias1;
};

__device__ __forceinline__ uint32_t pack2(bf16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ float lo_f32(uint32_t v) { return __builtin_bit_cast(float, v << 16); }
__device__ __forceinline__ float hi_f32(uint32_t v) { return __builtin_bit_cast(float, v & 0xffff0000u); }

// Two values into their three bf16 parts. An infinity or NaN is its first part,
// the other two are NaN.
__device__ __forceinline__ void split2(float a, float b, uint32_t (&o)[3]) {
    o[0] = pack2(__builtin_convertvector(f32x2v{a, b}, bf16x2));
    a -= lo_f32(o[0]);
    b -= hi_f32(o[0]);
    o[1] = pack2(__builtin_convertvector(f32x2v{a, b}, bf16x2));
    a -= lo_f32(o[1]);
    b -= hi_f32(o[1]);
    o[2] = pack2(__builtin_convertvector(f32x2v{a, b}, bf16x2));
}

template <int N>
__device__ __forceinline__ void split_n(const float (&v)[N], uint32_t (&o)[3][N / 2]) {
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        uint32_t t[3];
        split2(v[2 * i], v[2 * i + 1], t);
        o[0][i] = t[0];
        o[1][i] = t[1];
        o[2][i] = t[2];
    }
}

// The range of some values: the bits of the largest finite |v|, with kHasTiny
// where a value other than zero is below 2^-100.
constexpr uint32_t kHasTiny = 0x80000000u;
constexpr uint32_t kInfBits = 0x7f800000u;
constexpr float kTinyBelow = 0x1p-100f;

__device__ __forceinline__ uint32_t join_ranges(uint32_t a, uint32_t b) {
    return std::max(a & ~kHasTiny, b & ~kHasTiny) | ((a | b) & kHasTiny);
}

__device__ __forceinline__ uint32_t value_range(float v) {
    const float m = __builtin_fabsf(v);
    const uint32_t b = __builtin_bit_cast(uint32_t, m);
    return b >= kInfBits ? 0 : b | (m != 0.0f && m < kTinyBelow ? kHasTiny : 0);
}

__device__ __forceinline__ uint32_t wave_range(uint32_t r) {
#pragma unroll
    for (int n = 32; n >= 1; n >>= 1) r = join_ranges(r, __shfl_xor(r, n));
    return r;
}

__device__ __forceinline__ float param_at(const void * p, int32_t f16, int i) {
    return f16 ? h2f(static_cast<const uint16_t *>(p)[i]) : static_cast<const float *>(p)[i];
}

// Parameters of a wave-uniform channel by scalar loads: the pack launch wrote
// them, nothing does during this one.
__device__ __forceinline__ snake_param scalar_param(const snake_param * p, int i) {
    const auto * f = (const __attribute__((address_space(4))) float *)(reinterpret_cast<uintptr_t>(p + i));
    return snake_param{f[0], f[1], f[2]};
}

// ---- weights into fragment order ---------------------------------------------------
//
// A block per (32-row tile, 16-channel group), a thread per (tap, lane): eight
// weights, three 16-byte stores. The blocks after the last one evaluate SnakeBeta parameters.
// With w1 (a residual unit's k = 1 weights, 128 x 128) KW of its (32-row tile,
// 16-channel group) pairs are a block's.
// Returns the range of the lane's weights.
__device__ __forceinline__ uint32_t pack_item(const float * src, int ci_left, int ci_step, u32x4 * dst, int lane) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = i < ci_left ? src[i * ci_step] : 0.0f;
    uint32_t o[3][4];
    split_n<8>(v, o);
#pragma unroll
    for (int p = 0; p < 3; ++p) dst[64 * p + lane] = u32x4{o[p][0], o[p][1], o[p][2], o[p][3]};
    uint32_t range = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) range = join_ranges(range, value_range(v[i]));
    return range;
}

template <int KW>
__global__ __launch_bounds__(64 * KW) void x3_pack_kernel(const x3_conv c, u32x4 * w, uint32_t * w_range,
                                                          snake_param * pre, snake_param * post, int rows, int groups,
                                                          int row_tiles, const float * w1, u32x4 * w1_packed,
                                                          uint32_t * w1_range) {
    __shared__ uint32_t tap_range[KW];
    int b = static_cast<int>(blockIdx.x);
    const int tid = static_cast<int>(threadIdx.x);
    const int tap = tid >> 6;
    const int lane = tid & 63;
    if (b < row_tiles * groups) {
        const int rt = b / groups;
        const int row = rt * 32 + (lane & 31);
        const int ci = (b - rt * groups) * kCI + 8 * (lane >> 5);
        const int co = row / c.stride;
        const float * src = c.w + ((static_cast<int64_t>(row - co * c.stride) * c.c_out + co) * c.c_in + ci) * KW + tap;
        const uint32_t range =
                wave_range(pack_item(src, row < rows ? c.c_in - ci : 0, KW, w + (static_cast<int64_t>(b) * KW + tap) * 192, lane));
        if (lane == 0) tap_range[tap] = range;
        __syncthreads();
        if (tid == 0) {
            uint32_t all = 0;
#pragma unroll
            for (int k = 0; k < KW; ++k) all = join_ranges(all, tap_range[k]);
            w_range[b] = all;
        }
        return;
    }
    b -= row_tiles * groups;
    if (w1 != nullptr) {
        constexpr int kItems = kUnit / 32 * (kUnit / kCI);
        if (b < (kItems + KW - 1) / KW) {
            const int item = b * KW + tap;
            if (item >= kItems) return;
            const int row = item / (kUnit / kCI) * 32 + (lane & 31);
            const int ci = item % (kUnit / kCI) * kCI + 8 * (lane >> 5);
            const float * src = w1 + row * kUnit + ci;
            uint32_t range = wave_range(pack_item(src, 8, 1, w1_packed + item * 192, lane));
            // one that is not finite counts as the largest here: the tiles are summed in F32
            bool finite = true;
#pragma unroll
            for (int i = 0; i < 8; ++i) finite &= __builtin_fabsf(src[i]) < __builtin_inff();
            if (__ballot(!finite) != 0) range = kInfBits;
            if (lane == 0) w1_range[item] = range;
            return;
        }
        b -= (kItems + KW - 1) / KW;
    }
    const int n_pre = c.snake ? groups * kCI : 0;
    int e = b * 64 * KW + tid;
    if (e < n_pre) {
        // channels past c_in stage zeros
        pre[e] = e < c.c_in ? make_snake_param(param_at(c.alpha_log, c.param_f16, e), param_at(c.beta_log, c.param_f16, e))
                            : snake_param{0.0f, 1.0f, 1.0f};
        return;
    }
    e -= n_pre;
    if (c.post_alpha_log && e < c.c_out)
        post[e] = make_snake_param(param_at(c.post_alpha_log, c.param_f16, e), param_at(c.post_beta_log, c.param_f16, e));
}

// ---- the convolution -----------------------------------------------------------------

__device__ __forceinline__ f32x16v mfma(const u32x4 & a, const u32x4 & b, const f32x16v & c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// acc_0 += A * B_0, acc_1 += A * B_1, the small products into lo_0 and lo_1; the
// sums alternate so that no MFMA waits for the one before it.
__device__ __forceinline__ void mfma_x3(const u32x4 (&a)[3], const u32x4 (&b)[2][3], f32x16v & acc0, f32x16v & acc1,
                                        f32x16v & lo0, f32x16v & lo1) {
    constexpr int kA[5] = {2, 1, 1, 0, 0};
    constexpr int kB[5] = {0, 0, 1, 1, 2};
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        lo0 = mfma(a[kA[s]], b[0][kB[s]], lo0);
        lo1 = mfma(a[kA[s]], b[1][kB[s]], lo1);
    }
    acc0 = mfma(a[0], b[0][0], acc0);
    acc1 = mfma(a[0], b[1][0], acc1);
}

// Row of accumulator item u of a 32 x 32 tile, in lane half hl.
__device__ __forceinline__ int acc_row(int u, int hl) { return (u & 3) + 8 * (u >> 2) + 4 * hl; }

// acc += lo; where acc, the sum of the products of the operands' first parts,
// is not finite it is the sum as it stands. `bad` turns NaN where a sum is not
// finite.
__device__ __forceinline__ void join_sums(f32x16v & acc, const f32x16v & lo, float & bad) {
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const float sum = acc[u] + lo[u];
        acc[u] = __builtin_fabsf(acc[u]) < __builtin_inff() ? sum : acc[u];
        bad = __builtin_fmaf(acc[u], 0.0f, bad);
    }
}

// What a workgroup has seen of its sums and operands; each wave's go into
// tile_state::seen. "Ordinary" is large enough for a product with an ordinary
// one of the other side to keep its bits.
enum : uint32_t {
    kSumNotFinite = 1,
    kInputNonzero = 2, kInputOrdinary = 4,
    kWeightNonzero = 8, kWeightOrdinary = 16,
    kMidNonzero = 32, kMidOrdinary = 64,  // a residual unit's h
    kWeight1Nonzero = 128, kWeight1Ordinary = 256,
};
constexpr float kOrdinaryInput = 0x1p-60f;
constexpr float kOrdinaryWeight = 0x1p-40f;

struct tile_state {
    uint32_t seen;
    // ranges over the tile (f32_needed)
    uint32_t w, x, x_bound, x_infinite;
    uint32_t mid, w1;
    uint32_t pad;
};
static_assert(sizeof(tile_state) == 32, "two items of LDS");

__device__ __forceinline__ uint32_t seen_if(bool lane_has, uint32_t bit) { return __ballot(lane_has) != 0 ? bit : 0; }

__device__ __forceinline__ bool worth_a_look(uint32_t seen) {
    auto small = [&](uint32_t a, uint32_t a_ordinary, uint32_t b, uint32_t b_ordinary) {
        return (seen & a) && (seen & b) && !((seen & a_ordinary) && (seen & b_ordinary));
    };
    return (seen & kSumNotFinite) || small(kInputNonzero, kInputOrdinary, kWeightNonzero, kWeightOrdinary) ||
           small(kMidNonzero, kMidOrdinary, kWeight1Nonzero, kWeight1Ordinary);
}

// Whether sums of n products of values up to a and b may overflow, or the values
// or products be too small for their parts.
__device__ __forceinline__ bool out_of_split_range(float a_bound, float a, float b, float n) {
    const bool large = a_bound >= 0x1p126f || b >= 0x1p126f || a_bound * b * n >= 0x1p126f;
    const bool small = a > 0.0f && b > 0.0f && (a < 0x1p-90f || b < 0x1p-90f || a * b < 0x1p-100f);
    return large || small;
}

// The channel and phase of a row, its bias and output SnakeBeta, kept in LDS
// for the epilogue.
struct row_info {
    float bias;
    snake_param post;
    int32_t co;
    int32_t r;
};

// bias, residual, SnakeBeta and store of one output.
__device__ __forceinline__ float finish_value(const x3_conv & c, float v, const row_info & ri, float res) {
    if (c.bias) v = v + ri.bias;
    if (c.residual) v = res + v;
    if (c.post_alpha_log) v = snake(v, ri.post);
    return v;
}

// The sums of rows row .. row + 3 at one column in plain F32, for tiles with
// infinities or NaN: short code, since what is inlined here costs the kernel's
// own loop registers (a staged form of it 8 % of its speed).
template <int KW>
__device__ __forceinline__ void plain_sums(const x3_kernel_params & p, int row, int64_t col, int ci0, int ci1, float (&s)[4]) {
    const x3_conv & c = p.c;
    const float * w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        s[r] = 0.0f;
        const int rr = std::min(row + r, p.rows - 1);
        const int co = rr / c.stride;
        w[r] = c.w + (static_cast<int64_t>(rr - co * c.stride) * c.c_out + co) * c.c_in * KW;
    }
#pragma unroll 1
    for (int ci = ci0; ci < ci1; ++ci) {
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const int64_t t = col + static_cast<int64_t>(k) * c.dil - c.pad;
            float v = t >= 0 && t < c.t_in ? c.x[ci * c.x_pitch + t] : 0.0f;
            if (c.snake) v = snake(v, p.pre[ci]);
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] = __builtin_fmaf(w[r][ci * KW + k], v, s[r]);
        }
    }
}

// Whether a tile worth a look has to be summed in plain F32: looks through its
// inputs (columns col0 .. of kNT and the halo; SnakeBeta adds up to 1 / beta)
// and the ranges of its weights. Every thread of the workgroup calls it and
// gets the same answer.
template <int KW, int THREADS>
__device__ __forceinline__ bool f32_needed(const x3_kernel_params & p, tile_state * state, int rt0, int row_tiles,
                                           int64_t col0, int chunk0, int chunk1) {
    constexpr int CG = KW <= 2 ? 2 : 1;
    const x3_conv & c = p.c;
    const int tid = static_cast<int>(threadIdx.x);
    uint32_t wr = 0;
    for (int e = tid; e < row_tiles * (chunk1 - chunk0) * CG; e += THREADS) {
        const int rt = rt0 + e % row_tiles;
        if (rt * 32 < p.rows) wr = join_ranges(wr, p.w_range[rt * p.chunks * CG + chunk0 * CG + e / row_tiles]);
    }
    uint32_t xr = 0, infinite = 0;
    float bound = 0.0f;
    const int span = kNT + (KW - 1) * c.dil;
    const int ci0 = chunk0 * kCI * CG, ci1 = std::min(chunk1 * kCI * CG, c.c_in);
#pragma unroll 1
    for (int col = tid % 64; col < span; col += 64) {
        const int64_t t = col0 - c.pad + col;
        if (t < 0 || t >= c.t_in) continue;
#pragma unroll 4
        for (int ci = ci0 + tid / 64; ci < ci1; ci += THREADS / 64) {
            const float v = __builtin_fabsf(c.x[ci * c.x_pitch + t]);
            xr = join_ranges(xr, value_range(v));
            infinite |= v == __builtin_inff();
            const float b = c.snake ? v + __builtin_fmaxf(p.pre[ci].rbeta, 0.0f) : v;
            if (v < __builtin_inff()) bound = __builtin_fmaxf(bound, b);
        }
    }
    atomicMax(&state->w, wr & ~kHasTiny);
    atomicMax(&state->x, xr & ~kHasTiny);
    atomicMax(&state->x_bound, __builtin_bit_cast(uint32_t, bound));
    atomicOr(&state->x_infinite, (infinite ? 1u : 0u) | (xr & kHasTiny ? 2u : 0u) | (wr & kHasTiny ? 4u : 0u));
    __syncthreads();
    const uint32_t odd = state->x_infinite;
    // an infinity times a value whose first part may be zero (one of the weights
    // times a tiny input, or the other way)
    if ((state->seen & kSumNotFinite) && ((odd & 2) || (odd & 5) == 5)) return true;
    return out_of_split_range(__builtin_bit_cast(float, state->x_bound), __builtin_bit_cast(float, state->x),
                              __builtin_bit_cast(float, state->w), static_cast<float>((ci1 - ci0) * KW));
}

// The k = 1 half of a residual unit of 128 channels, in the k = 7 launch: a
// workgroup holds every channel of its 128 columns. h = acc + bias goes through
// the post SnakeBeta, split, into LDS (in two halves of 64 columns, so that two
// workgroups share a CU) as the B operand of the k = 1 weights, which come from
// L2 like the others; the result + bias + the unit's input is the output. A tile
// whose sums or operands ask for it (f32_needed, the same for h and the k = 1
// weights) is summed again in plain F32 over what was stored.
struct unit_row {
    float bias0, bias1;
    snake_param post;
    float pad;
};
static_assert(sizeof(unit_row) * kUnit == kUnitInfoItems * 16, "unit_row fills its items");

__device__ __forceinline__ void unit_tail(const x3_kernel_params & p, u32x4 * lds, const f32x16v (&acc)[kNT / 32],
                                          tile_state * state, uint32_t seen, int64_t t0) {
    const x3_conv & c = p.c;
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31;
    const int hl = lane >> 5;
    float bad = 0.0f, largest = 0.0f;
    unit_row * info = reinterpret_cast<unit_row *>(lds + kUnitItems);
    if (tid < kUnit) info[tid] = unit_row{c.bias ? c.bias[tid] : 0.0f, p.bias1 ? p.bias1[tid] : 0.0f, p.post[tid], 0.0f};
    const char * wp = reinterpret_cast<const char *>(p.w1) + static_cast<int64_t>(wave) * (kUnit / kCI) * 3072;
    auto run_half = [&](auto which) __attribute__((always_inline)) {
        constexpr int half = decltype(which)::value;
        // the unit's input and the first weights arrive during the SnakeBetas
        float res[2][16];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int64_t t = std::min(t0 + 64 * half + 32 * j + n, c.cols - 1);
#pragma unroll
            for (int u = 0; u < 16; ++u) res[j][u] = c.x[(32 * wave + acc_row(u, hl)) * c.x_pitch + t];
        }
        u32x4 a[2][3];
#pragma unroll
        for (int s = 0; s < 3; ++s) a[0][s] = *reinterpret_cast<const u32x4 *>(wp + 16 * lane + 1024 * s);
        __syncthreads();  // info is there; the first half's fragments are read
        auto store_h = [&](bool exact, bool & slow) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int u = 0; u < 16; u += 4) {
                    float v[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const unit_row & ri = info[32 * wave + acc_row(u + q, hl)];
                        float h = acc[2 * half + j][u + q];
                        if (c.bias) h = h + ri.bias0;
                        v[q] = exact ? snake(h, ri.post) : snake_reduced(h, ri.post, slow);
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) largest = __builtin_fmaxf(largest, __builtin_fabsf(v[q]));
                    uint32_t o[3][2];
                    split_n<4>(v, o);
                    // rows 32 wave + 8 (u / 4) + 4 hl ..: half an item of channel group row / 8
                    const int item = (2 * wave + u / 8) * 6 * 64 + ((u >> 2) & 1) * 64 + 32 * j + n;
#pragma unroll
                    for (int s = 0; s < 3; ++s)
                        reinterpret_cast<u32x2v *>(lds + item + s * 128)[hl] = u32x2v{o[s][0], o[s][1]};
                }
        };
        bool slow = false;
        const float before = largest;
        store_h(false, slow);
        if (slow) {  // rare: arguments beyond the reduced sine's range
            largest = before;
            store_h(true, slow);
        }
        __syncthreads();
        f32x16v out[2], lo[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                out[j][u] = 0.0f;
                lo[j][u] = 0.0f;
            }
#pragma unroll
        for (int st = 0; st < kUnit / kCI; ++st) {
            if (st + 1 < kUnit / kCI) {
#pragma unroll
                for (int s = 0; s < 3; ++s)
                    a[(st + 1) & 1][s] = *reinterpret_cast<const u32x4 *>(wp + (st + 1) * 3072 + 16 * lane + 1024 * s);
            }
            u32x4 b[2][3];
#pragma unroll
            for (int s = 0; s < 6; ++s) b[s / 3][s % 3] = lds[st * 6 * 64 + (s % 3) * 128 + hl * 64 + 32 * (s / 3) + n];
            mfma_x3(a[st & 1], b, out[0], out[1], lo[0], lo[1]);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int64_t t = t0 + 64 * half + 32 * j + n;
            if (t >= c.cols) continue;
            join_sums(out[j], lo[j], bad);
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const int row = 32 * wave + acc_row(u, hl);
                float v = out[j][u];
                if (p.bias1) v = v + info[row].bias1;
                c.y[row * c.y_pitch + t] = res[j][u] + v;
            }
        }
    };
    run_half(std::integral_constant<int, 0>{});
    run_half(std::integral_constant<int, 1>{});
    seen |= seen_if(bad != 0.0f, kSumNotFinite) | seen_if(largest > 0.0f, kMidNonzero) |
            seen_if(largest >= kOrdinaryInput, kMidOrdinary);
    if (lane == 0) atomicOr(&state->seen, seen);
    __syncthreads();
    if (!worth_a_look(state->seen)) return;
    atomicMax(&state->mid, __builtin_bit_cast(uint32_t, largest));
    if (tid < kUnit / 32 * (kUnit / kCI)) atomicMax(&state->w1, p.w1_range[tid] & ~kHasTiny);
    if (!f32_needed<7, kThreads>(p, state, 0, kUnit / 32, t0, 0, p.chunks) &&
        !out_of_split_range(__builtin_bit_cast(float, state->mid), __builtin_bit_cast(float, state->mid),
                            __builtin_bit_cast(float, state->w1), kUnit))
        return;
    // plain F32, 32 columns of h at a time
    float * hs = reinterpret_cast<float *>(lds);
#pragma unroll 1
    for (int c0 = 0; c0 < kNT; c0 += 32) {
        const int col = c0 + tid % 32;
        const int64_t t = std::min(t0 + col, c.cols - 1);
#pragma unroll 1
        for (int r = 4 * (tid / 32); r < kUnit; r += 32) {
            float h[4];
            plain_sums<7>(p, r, t, 0, c.c_in, h);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (c.bias) h[q] = h[q] + info[r + q].bias0;
                hs[(r + q) * 32 + tid % 32] = snake(h[q], info[r + q].post);
            }
        }
        __syncthreads();
#pragma unroll 1
        for (int r = tid / 32; r < kUnit; r += 8) {
            float s = 0.0f;
#pragma unroll 4
            for (int ci = 0; ci < kUnit; ++ci) s = __builtin_fmaf(p.w1_raw[r * kUnit + ci], hs[ci * 32 + tid % 32], s);
            if (p.bias1) s = s + info[r].bias1;
            if (t0 + col < c.cols) c.y[r * c.y_pitch + t] = c.x[r * c.x_pitch + t] + s;
        }
        __syncthreads();
    }
}

template <int KW, bool SNAKE, bool FUSE>
__global__ __launch_bounds__((x3_shape<KW, FUSE>::THREADS), 2) void x3_conv_kernel(const x3_kernel_params p) {
    using S = x3_shape<KW, FUSE>;
    const x3_conv & c = p.c;
    // XCD j takes the j-th run of consecutive tiles (a run is one row tile's
    // columns, or part of them: its weights stay in that XCD's L2), each
    // tile's splits back to back
    const int lin = static_cast<int>(blockIdx.x);
    const int run = (p.tiles + 7) >> 3;
    const int tile = (lin & 7) * run + (lin >> 3) / p.splits;
    const int split = (lin >> 3) % p.splits;
    if (tile >= p.tiles || (lin >> 3) >= run * p.splits) return;
    const int row0 = (tile / p.tiles_x) * S::ROWS;
    const int64_t t0 = static_cast<int64_t>(tile % p.tiles_x) * S::OUT;
    const int c_begin = static_cast<int>(static_cast<int64_t>(split) * p.chunks / p.splits);
    const int c_end = static_cast<int>(static_cast<int64_t>(split + 1) * p.chunks / p.splits);

    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];

    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31;
    const int hl = lane >> 5;

    tile_state * state = reinterpret_cast<tile_state *>(lds + S::STATE);
    if (tid < static_cast<int>(sizeof(tile_state) / 4)) reinterpret_cast<uint32_t *>(state)[tid] = 0;
    uint32_t seen = 0;  // the wave's
    {
        uint32_t wr = 0, wr1 = 0;
        const int g_begin = c_begin * S::CG;
        const int n_ranges = S::WAVES * (c_end - c_begin) * S::CG;
        for (int e = tid; e < n_ranges; e += S::THREADS) {
            const int rt = row0 / 32 + e % S::WAVES;
            if (rt * 32 < p.rows) wr = join_ranges(wr, p.w_range[rt * p.chunks * S::CG + g_begin + e / S::WAVES]);
        }
        if (FUSE && tid < kUnit / 32 * (kUnit / kCI)) wr1 = p.w1_range[tid];
        auto at_least = [](uint32_t r, float v) { return (r & ~kHasTiny) >= __builtin_bit_cast(uint32_t, v); };
        seen = seen_if(wr != 0, kWeightNonzero) | seen_if(at_least(wr, kOrdinaryWeight), kWeightOrdinary);
        if (FUSE) seen |= seen_if(wr1 != 0, kWeight1Nonzero) | seen_if(at_least(wr1, kOrdinaryWeight), kWeight1Ordinary);
    }
    float largest = 0.0f;  // |input| staged by the thread

    // Staging: waves deal the columns, channel halves and groups of a chunk
    // among them, in pairs of channels; the eight channels of a column's item
    // are kg's. The loads are unconditional (clamped) and masked where they are
    // staged, so that nothing waits for them before the MFMAs.
    const int kg = wave & 1;
    const int tb = static_cast<int>(t0) - c.pad;  // sample of column 0 (launches keep to 2^28)
    const int t_last = static_cast<int>(c.t_in) - 1;
    float xr[S::PAIRS][2];
    auto pair_place = [&](int m, int l, int & u, int & col, int & ch) {
        if (m < S::MAIN) {
            // wave bit 1: column half; bit 2 (eight waves): the channel group, or half of the channels
            col = (wave & 2) * 32 + l;
            u = S::CG == 2 ? (S::WAVES == 8 ? wave >> 2 : m / 4) : 0;
            ch = S::WAVES == 8 && S::CG == 1 ? 4 * (wave >> 2) + 2 * m : 2 * (m & 3);
        } else {
            u = 0;
            col = kNT + l;
            ch = S::WAVES == 8 ? 2 * (wave >> 1) : 4 * (wave >> 1) + 2 * (m - S::MAIN);
        }
    };
    auto load_x = [&](int chunk) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < S::PAIRS; ++m) {
            int l = lane;
            if (m == 0 || m == S::MAIN) asm volatile("" : "+v"(l));  // a fresh 32-bit offset from a uniform row: nothing to keep in registers
            int u, col, ch;
            pair_place(m, l, u, col, ch);
            const uint32_t off = 4u * static_cast<uint32_t>(std::min(std::max(tb + col, 0), t_last));
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int ci = std::min(chunk * S::CI + 16 * u + 8 * kg + ch + q, c.c_in - 1);
                const float * row = c.x + static_cast<int64_t>(ci) * c.x_pitch;
                xr[m][q] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(row) + off);
            }
        }
    };
    // Pair m through SnakeBeta, in three planes; the second of two neighbouring
    // pairs stores both pairs' eight bytes in each plane.
    auto stage_pair = [&](int chunk, int buf, int m, bool exact, uint32_t (&o)[3][2],
                          bool & slow) __attribute__((always_inline)) {
        int u, col, ch;
        pair_place(m, lane, u, col, ch);
        const int ci = chunk * S::CI + 16 * u + 8 * kg + ch;
        const int t = tb + col;
        const bool inside = t >= 0 && t <= t_last;
        float v[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            v[q] = inside && ci + q < c.c_in ? xr[m][q] : 0.0f;
            if (SNAKE) {
                const snake_param sp = scalar_param(p.pre, ci + q);
                v[q] = exact ? snake(v[q], sp) : snake_reduced(v[q], sp, slow);
            }
        }
        largest = __builtin_fmaxf(__builtin_fmaxf(largest, __builtin_fabsf(v[0])), __builtin_fabsf(v[1]));
        uint32_t w[3];
        split2(v[0], v[1], w);
        u32x4 * item = lds + buf * S::BUF + u * S::GROUP + kg * S::W + col;
        if (S::WAVES == 8 && m >= S::MAIN) {  // a single halo pair
#pragma unroll
            for (int s = 0; s < 3; ++s) reinterpret_cast<uint32_t *>(item + s * 2 * S::W)[ch >> 1] = w[s];
            return;
        }
#pragma unroll
        for (int s = 0; s < 3; ++s) o[s][m & 1] = w[s];
        if (m & 1) {
#pragma unroll
            for (int s = 0; s < 3; ++s) reinterpret_cast<u32x2v *>(item + s * 2 * S::W)[ch >> 2] = u32x2v{o[s][0], o[s][1]};
        }
    };
    auto stage_all = [&](int chunk, int buf) __attribute__((always_inline)) {
        uint32_t o[3][2];
        bool slow = false;
#pragma unroll
        for (int m = 0; m < S::PAIRS; ++m) stage_pair(chunk, buf, m, true, o, slow);
    };

    // weight fragments: rows 32 * wave of the tile; a K step is 3072 bytes
    // after the one before. Row tiles past the last are clamped (computed and
    // dropped).
    const int rt_last = (p.rows + 31) / 32 - 1;
    const int64_t rt_bytes = static_cast<int64_t>(p.chunks) * S::KS * 3072;
    const char * wp = reinterpret_cast<const char *>(p.w) + std::min(row0 / 32 + wave, rt_last) * rt_bytes +
                      static_cast<int64_t>(c_begin) * S::KS * 3072;
    u32x4 a[2][3];
    auto load_a = [&](u32x4 (&d)[3], int step) {
        uint32_t off = 16u * lane;
        asm volatile("" : "+v"(off));  // uniform base plus 32-bit lane offset: no 64-bit address registers
#pragma unroll
        for (int s = 0; s < 3; ++s)
            d[s] = *reinterpret_cast<const u32x4 *>(wp + static_cast<int64_t>(step) * 3072 + off + 1024 * s);
    };

    constexpr int NJ = kNT / 32;
    f32x16v acc[NJ], lo[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            acc[j][u] = 0.0f;
            lo[j][u] = 0.0f;
        }

    load_a(a[0], 0);
    load_x(c_begin);
    stage_all(c_begin, 0);
    __syncthreads();

    const int steps = (c_end - c_begin) * S::KS;
    // Group g of a chunk is K step g / 2 on half of the columns. Step
    // n + 1's weights, the next group's fragments and the next chunk's inputs
    // are asked for ahead of the MFMAs; the next chunk's channel pairs are
    // staged in the last groups, between the MFMAs (the scheduling barriers
    // keep all that so). An odd number of steps takes two chunks a turn, as the
    // steps alternate between two register sets.
    constexpr int kGroups = 2 * S::KS;
    constexpr int kPairs = S::PAIRS;
    constexpr int kFirst = std::max(kGroups / 2, kGroups - kPairs);
    constexpr int kSpan = kGroups - kFirst;
    constexpr int kValu = (SNAKE ? 7 : 4) * ((kPairs + kSpan - 1) / kSpan);  // per MFMA
    constexpr int kTurn = S::KS & 1 ? 2 : 1;
    int step = 0;
    for (int turn = c_begin; turn < c_end; turn += kTurn) {
#pragma unroll
        for (int half = 0; half < kTurn; ++half) {
            const int chunk = turn + half;
            if (chunk >= c_end) break;
            const int buf = (chunk - c_begin) & 1;
            const bool more = chunk + 1 < c_end;
            const int next = more ? chunk + 1 : chunk;  // past the last: staged again, not read
            const u32x4 * bp = lds + buf * S::BUF + hl * S::W + n;
            u32x4 b[2][2][3];
            uint32_t o[3][2];
            bool slow = false;
#pragma unroll
            for (int s = 0; s < 6; ++s) b[0][s / 3][s % 3] = bp[(s % 3) * 2 * S::W + 32 * (s / 3)];
#pragma unroll
            for (int g = 0; g < kGroups; ++g) {
                const int st = g / 2;
                const int j = g % 2;
                const int cur = (half * S::KS + st) & 1;
                if (j == 0) load_a(a[cur ^ 1], std::min(step + st + 1, steps - 1));
                if (g == 0) {
                    __builtin_amdgcn_sched_barrier(0);  // behind the weights, which are waited for first
                    load_x(next);
                }
                if (g + 1 < kGroups) {
                    const int st1 = (g + 1) / 2;
#pragma unroll
                    for (int s = 0; s < 6; ++s)
                        b[(g + 1) & 1][s / 3][s % 3] = bp[(st1 / KW) * S::GROUP + (s % 3) * 2 * S::W + 64 * ((g + 1) % 2) +
                                                          32 * (s / 3) + (st1 % KW) * c.dil];
                }
                __builtin_amdgcn_sched_barrier(0);
                mfma_x3(a[cur], b[g & 1], acc[2 * j], acc[2 * j + 1], lo[2 * j], lo[2 * j + 1]);
                if (g >= kFirst) {
                    const int m0 = (g - kFirst) * kPairs / kSpan, m1 = (g + 1 - kFirst) * kPairs / kSpan;
#pragma unroll
                    for (int m = m0; m < m1; ++m) stage_pair(next, buf ^ 1, m, false, o, slow);
#pragma unroll
                    for (int q = 0; q < 12; ++q) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            step += S::KS;
            if (SNAKE && slow) stage_all(next, buf ^ 1);  // rare: arguments beyond the reduced sine's range
            __syncthreads();
        }
    }

    // ---- epilogue
    {
        float bad = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            // k = 2 reads past what it stages for the columns it drops
            float tile_bad = 0.0f;
            join_sums(acc[j], lo[j], tile_bad);
            if (32 * (j + 1) <= S::OUT || 32 * j + n < S::OUT) bad += tile_bad;
        }
        seen |= seen_if(bad != 0.0f, kSumNotFinite) | seen_if(largest > 0.0f, kInputNonzero) |
                seen_if(largest >= kOrdinaryInput, kInputOrdinary);
    }
    if constexpr (FUSE) {
        unit_tail(p, lds, acc, state, seen, t0);
    } else {
        // every residual load before any store (y may be the residual), and all
        // of them at once: one trip to memory (clamped, masked at the store)
        float res[NJ][16];
        const bool add = KW != 2 && c.residual != nullptr && p.splits == 1;
        if (add) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int64_t t = std::min(t0 + 32 * j + n, c.cols - 1);
#pragma unroll
                for (int u = 0; u < 16; ++u)
                    res[j][u] = c.residual[std::min(row0 + 32 * wave + acc_row(u, hl), p.rows - 1) * c.r_pitch + t];
            }
        }
        row_info * info = reinterpret_cast<row_info *>(lds);
        if (lane == 0) atomicOr(&state->seen, seen);
        __syncthreads();
        const bool redo = worth_a_look(state->seen) &&
                          f32_needed<KW, S::THREADS>(p, state, row0 / 32, S::WAVES, t0, c_begin, c_end);
        if (tid < S::ROWS) {
            const int row = std::min(row0 + tid, p.rows - 1);
            row_info ri{};
            ri.co = row / c.stride;
            ri.r = row - ri.co * c.stride;
            if (c.bias) ri.bias = c.bias[ri.co];
            if (c.post_alpha_log) ri.post = p.post[ri.co];
            info[tid] = ri;
        }
        __syncthreads();
        if (p.splits > 1) {
            float * part = p.part + split * p.part_slice;
            if (redo) {
#pragma unroll 1
                for (int e = tid; e < S::ROWS / 4 * S::OUT; e += S::THREADS) {
                    const int row = row0 + 4 * (e / S::OUT);
                    const int64_t t = t0 + e % S::OUT;
                    if (row >= p.rows || t >= c.cols) continue;
                    float s[4];
                    plain_sums<KW>(p, row, t, c_begin * S::CI, std::min(c_end * S::CI, c.c_in), s);
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (row + r < p.rows) part[(row + r) * p.part_pitch + t] = s[r];
                }
                return;
            }
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                    const int col = 32 * j + n;
                    const int64_t t = t0 + col;
#pragma unroll
                    for (int u = 0; u < 16; ++u) {
                        const int row = row0 + 32 * wave + acc_row(u, hl);
                        if (row < p.rows && col < S::OUT && t < c.cols) part[row * p.part_pitch + t] = acc[j][u];
                    }
                }
            return;
        }
        if (redo) {
#pragma unroll 1
            for (int e = tid; e < S::ROWS / 4 * S::OUT; e += S::THREADS) {
                const int row = row0 + 4 * (e / S::OUT);
                const int64_t t = t0 + e % S::OUT;
                if (row >= p.rows || t >= c.cols) continue;
                float s[4];
                plain_sums<KW>(p, row, t, 0, c.c_in, s);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (row + r >= p.rows) break;
                    const row_info ri = info[row - row0 + r];
                    const int64_t o = t * c.stride + ri.r + c.o_base;
                    if (o < 0 || o >= c.y_len) continue;
                    const float res = c.residual ? c.residual[ri.co * c.r_pitch + o] : 0.0f;
                    c.y[ri.co * c.y_pitch + o] = finish_value(c, s[r], ri, res);
                }
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
                const int col = 32 * j + n;
                    const int64_t t = t0 + col;
                if (KW == 2) {
                    // transposed: a lane's four consecutive rows are
                    // neighbouring phases (and channels)
                    auto put = [&](int u, auto width) {
                        constexpr int kN = decltype(width)::value;
                        typedef float vec __attribute__((ext_vector_type(kN), aligned(4)));
                        const int rl = 32 * wave + acc_row(u, hl);
                        const row_info & ri = info[rl];
                        const int64_t o = t * c.stride + ri.r + c.o_base;
                        if (row0 + rl >= p.rows || col >= S::OUT || t >= c.cols) return;
                        float * dst = c.y + ri.co * c.y_pitch + o;
                        vec v;
#pragma unroll
                        for (int q = 0; q < kN; ++q) v[q] = c.bias ? acc[j][u + q] + ri.bias : acc[j][u + q];
                        if (o >= 0 && o + kN <= c.y_len) {
                            *reinterpret_cast<vec *>(dst) = v;
                        } else {
#pragma unroll
                            for (int q = 0; q < kN; ++q)
                                if (o + q >= 0 && o + q < c.y_len) dst[q] = v[q];
                        }
                    };
                    if (c.stride % 4 == 0) {
#pragma unroll
                        for (int u = 0; u < 16; u += 4) put(u, std::integral_constant<int, 4>{});
                    } else if (c.stride % 2 == 0) {
#pragma unroll
                        for (int u = 0; u < 16; u += 2) put(u, std::integral_constant<int, 2>{});
                    } else {
#pragma unroll
                        for (int u = 0; u < 16; ++u) {
                            const int rl = 32 * wave + acc_row(u, hl);
                            const row_info & ri = info[rl];
                            const int64_t o = t * c.stride + ri.r + c.o_base;
                            if (row0 + rl < p.rows && col < S::OUT && t < c.cols && o >= 0 && o < c.y_len)
                                c.y[ri.co * c.y_pitch + o] = c.bias ? acc[j][u] + ri.bias : acc[j][u];
                        }
                    }
                } else {
                    float v[16];
#pragma unroll
                    for (int u = 0; u < 16; ++u) {
                        v[u] = acc[j][u];
                        if (c.bias) v[u] = v[u] + info[32 * wave + acc_row(u, hl)].bias;
                        if (add) v[u] = res[j][u] + v[u];
                    }
                    if (c.post_alpha_log) {
                        float sv[16];
                        bool slow = false;
#pragma unroll
                        for (int u = 0; u < 16; ++u) sv[u] = snake_reduced(v[u], info[32 * wave + acc_row(u, hl)].post, slow);
                        if (slow) {
#pragma unroll
                            for (int u = 0; u < 16; ++u) sv[u] = snake(v[u], info[32 * wave + acc_row(u, hl)].post);
                        }
#pragma unroll
                        for (int u = 0; u < 16; ++u) v[u] = sv[u];
                    }
#pragma unroll
                    for (int u = 0; u < 16; ++u) {
                        const int64_t row = row0 + 32 * wave + acc_row(u, hl);
                        if (t < c.cols && row < p.rows) c.y[row * c.y_pitch + t] = v[u];
                    }
                }
            }
    }
}

// The split launch's partial sums in split order, then the epilogue's steps.
__global__ __launch_bounds__(kThreads) void x3_combine_kernel(const x3_kernel_params p) {
    const x3_conv & c = p.c;
    const int64_t e = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (e >= c.y_len * c.c_out) return;
    const int co = static_cast<int>(e / c.y_len);
    const int64_t o = e - co * c.y_len;
    const int64_t u = o - c.o_base;
    const int64_t q = u / c.stride;
    const int64_t row = static_cast<int64_t>(co) * c.stride + (u - q * c.stride);
    const float * src = p.part + row * p.part_pitch + q;
    float v = src[0];
#pragma unroll 4
    for (int z = 1; z < p.splits; ++z) v = v + src[z * p.part_slice];
    row_info ri{};
    if (c.bias) ri.bias = c.bias[co];
    if (c.post_alpha_log) ri.post = p.post[co];
    c.y[co * c.y_pitch + o] = finish_value(c, v, ri, c.residual ? c.residual[co * c.r_pitch + o] : 0.0f);
}


struct x3_layout {
    int64_t rows, row_tiles, chunks, groups;
    int64_t frag_bytes, flag_bytes, pre_bytes, post_bytes;
    int64_t bytes() const { return frag_bytes + flag_bytes + pre_bytes + post_bytes; }
};

int64_t round16(int64_t n) { return (n + 15) / 16 * 16; }

x3_layout layout_of(const x3_conv & c, int kw) {
    x3_layout l;
    l.rows = static_cast<int64_t>(c.c_out) * c.stride;
    l.row_tiles = ceil_div(l.rows, 32);
    const int64_t cg = kw <= 2 ? 2 : 1;  // x3_shape<kw>::CG
    l.chunks = ceil_div(c.c_in, kCI * cg);
    l.groups = l.chunks * cg;
    l.frag_bytes = l.row_tiles * l.groups * kw * 3072;
    l.flag_bytes = round16(4 * l.row_tiles * l.groups);
    l.pre_bytes = c.snake ? round16(l.groups * kCI * static_cast<int64_t>(sizeof(snake_param))) : 0;
    l.post_bytes = c.post_alpha_log ? round16(c.c_out * static_cast<int64_t>(sizeof(snake_param))) : 0;
    return l;
}

// A residual unit's k = 1 weights in fragment order.
constexpr int64_t kUnitFragBytes = kUnit / 32 * (kUnit / kCI) * 3072;

// Fewer multiply-adds than this (8 us at the F32 launches' 100 TFLOP/s) are not
// worth the pack launch of about 5 us; nor are those of a residual unit, one
// launch in F32 too, below twice as many.
constexpr int64_t kMinMacs = 400'000'000;
constexpr int64_t kMinUnitMacs = 800'000'000;

// Microseconds of a launch with `splits` splits: rounds of one workgroup a CU
// at 0.075 us per K value (measured with every CU busy: 512 channels x 60000,
// k = 7: 3.7 rounds of K = 3584 in 0.94 ms), plus the partial sums' way through
// memory.
double plan_us(int64_t tiles, int64_t k, int splits, double part_mb, int cus) {
    const double tile_us = 0.075 * (static_cast<double>(k) / splits) + 6.0;
    const double combine = splits > 1 ? 4.0 + 2.0 * splits * part_mb / 5.0 : 0.0;
    return static_cast<double>(ceil_div(tiles * splits, cus)) * tile_us + combine;
}

// The number of splits (each of at least four chunks, as many as the partial
// sums' space holds) that plan_us puts first, and its time.
int pick_splits(const x3_conv & c, const x3_layout & l, int64_t tiles, int64_t k, int64_t part_floats, double & best_us) {
    const int cus = std::max(1, device_cu_count());
    const int64_t slice = l.rows * ((c.cols + 3) / 4 * 4);
    int best = 1;
    best_us = plan_us(tiles, k, 1, 0.0, cus);
    for (int s = 2; s <= 8 && l.chunks / s >= 4 && s * slice <= part_floats; ++s) {
        const double us = plan_us(tiles, k, s, 4.0e-6 * static_cast<double>(slice), cus);
        if (us < best_us) {
            best_us = us;
            best = s;
        }
    }
    return best;
}

template <int KW, bool SNAKE, bool FUSE>
int launch_kernel(const x3_kernel_params & p, hipStream_t st, const char * what) {
    using S = x3_shape<KW, FUSE>;
    static_assert(S::ROWS * sizeof(row_info) <= sizeof(u32x4) * S::STATE, "the epilogue's rows fit the buffers");
    const size_t lds = sizeof(u32x4) * S::LDS_ITEMS;
    const void * fn = reinterpret_cast<const void *>(&x3_conv_kernel<KW, SNAKE, FUSE>);
    if (const int rc = allow_dynamic_lds(fn, 80 * 1024, what); rc != LEVO_HIP_OK) return rc;
    const uint32_t grid = static_cast<uint32_t>(ceil_div(p.tiles, 8) * 8 * p.splits);
    x3_conv_kernel<KW, SNAKE, FUSE><<<grid, S::THREADS, lds, st>>>(p);
    return launch_status(what);
}

// The pack launch; fills the parameters' pointers into `pack`.
template <int KW, bool FUSE>
int launch_pack(x3_kernel_params & p, const x3_conv & c, const x3_layout & l, char * pack, const float * w1,
                hipStream_t st, const char * what) {
    p.c = c;
    u32x4 * frag = reinterpret_cast<u32x4 *>(pack);
    uint32_t * flags = reinterpret_cast<uint32_t *>(pack += l.frag_bytes);
    snake_param * pre = reinterpret_cast<snake_param *>(pack += l.flag_bytes);
    snake_param * post = reinterpret_cast<snake_param *>(pack += l.pre_bytes);
    u32x4 * frag1 = reinterpret_cast<u32x4 *>(pack += l.post_bytes);
    uint32_t * flags1 = reinterpret_cast<uint32_t *>(pack + kUnitFragBytes);
    p.w = frag;
    p.w_range = flags;
    p.pre = pre;
    p.post = post;
    p.rows = static_cast<int32_t>(l.rows);
    p.chunks = static_cast<int32_t>(l.chunks);
    p.w1 = frag1;
    p.w1_range = flags1;
    p.w1_raw = w1;
    const int64_t tx = ceil_div(c.cols, x3_shape<KW, FUSE>::OUT);
    p.tiles_x = static_cast<int32_t>(tx);
    p.tiles = static_cast<int32_t>(tx * ceil_div(l.rows, x3_shape<KW, FUSE>::ROWS));
    p.splits = 1;
    const int64_t params = (c.snake ? l.groups * kCI : 0) + (c.post_alpha_log ? c.c_out : 0);
    const int64_t blocks = l.row_tiles * l.groups + (w1 ? ceil_div(kUnit / 32 * (kUnit / kCI), KW) : 0) + ceil_div(params, 64 * KW);
    x3_pack_kernel<KW><<<static_cast<uint32_t>(blocks), 64 * KW, 0, st>>>(
            c, frag, flags, pre, post, p.rows, static_cast<int>(l.groups), static_cast<int>(l.row_tiles), w1, frag1, flags1);
    return launch_status(what);
}

template <int KW>
int launch_conv(const x3_conv & c, const x3_layout & l, char * pack, float * part, int64_t part_floats, hipStream_t st,
                const char * what) {
    x3_kernel_params p{};
    if (const int rc = launch_pack<KW, false>(p, c, l, pack, nullptr, st, what); rc != LEVO_HIP_OK) return rc;
    double us;
    p.splits = pick_splits(c, l, p.tiles, l.groups * kCI * KW, part_floats, us);
    p.part = part;
    p.part_pitch = (c.cols + 3) / 4 * 4;
    p.part_slice = l.rows * p.part_pitch;
    const int rc = c.snake ? launch_kernel<KW, true, false>(p, st, what) : launch_kernel<KW, false, false>(p, st, what);
    if (rc != LEVO_HIP_OK || p.splits == 1) return rc;
    x3_combine_kernel<<<static_cast<uint32_t>(ceil_div(c.y_len * c.c_out, kThreads)), kThreads, 0, st>>>(p);
    return launch_status(what);
}

}  // namespace

int64_t x3_pack_bytes(const x3_conv & c, int kw) {
    if (kw != 1 && kw != 2 && kw != 3 && kw != 7) return -1;
    if (static_cast<int64_t>(c.dil) * (kw - 1) > kMaxHalo) return -1;
    if (static_cast<int64_t>(c.c_out) * c.stride <= 128) return -1;
    // sums of one to three terms: a product's own rounding counts, and the F32 launch's is the smaller (2.53e-8
    // against 2.60e-8 of the result for one term; 4.0e-8 against 2.7e-8 for four)
    if (static_cast<int64_t>(c.c_in) * kw < 4) return -1;
    if (c.c_out > (1 << 16) || c.c_in > (1 << 16) || c.cols >= (int64_t{1} << 28)) return -1;
    const double macs = static_cast<double>(c.c_out) * c.stride * c.c_in * kw * static_cast<double>(c.cols);
    if (macs < kMinMacs) return -1;
    return layout_of(c, kw).bytes();
}

// Fitted like the F32 launches' estimate (snake_conv.hip): rounds of one
// workgroup a CU on the fullest XCD, the partial sums' way through memory, the
// pack launch; split weights that the 256 MB last-level cache cannot hold with
// what they are made from come from memory again.
double x3_us(const x3_conv & c, int kw, int64_t part_floats) {
    const x3_layout l = layout_of(c, kw);
    const int64_t tiles = ceil_div(c.cols, kw == 2 ? kNT - 1 : kNT) * ceil_div(l.rows, 256);
    double us;
    const int splits = pick_splits(c, l, tiles, l.groups * kCI * kw, part_floats, us);
    const double k_us = kw == 1 ? 0.087 : kw == 2 ? 0.067 : kw == 3 ? 0.061 : 0.050;
    const double share = static_cast<double>(ceil_div(l.chunks, splits) * (l.groups / l.chunks) * kCI * kw);
    const double rounds = static_cast<double>(ceil_div(ceil_div(tiles, 8) * splits, 32));
    const double part_mb = splits > 1 ? 4.0e-6 * static_cast<double>(splits * l.rows * ((c.cols + 3) / 4 * 4)) : 0.0;
    const double frag_mb = 1.0e-6 * static_cast<double>(l.frag_bytes);
    return (kw == 2 ? 6.0 : 3.0) + rounds * (k_us * share + 11.0) + 0.4 * part_mb + (frag_mb < 128.0 ? 0.43 : 0.6) * frag_mb;
}

int launch_x3(const x3_conv & c, int kw, void * pack, float * part, int64_t part_floats, hipStream_t st,
              const char * what) {
    const x3_layout l = layout_of(c, kw);
    char * base = static_cast<char *>(pack);
    switch (kw) {
        case 1: return launch_conv<1>(c, l, base, part, part_floats, st, what);
        case 2: return launch_conv<2>(c, l, base, part, part_floats, st, what);
        case 3: return launch_conv<3>(c, l, base, part, part_floats, st, what);
        default: return launch_conv<7>(c, l, base, part, part_floats, st, what);
    }
}

int64_t x3_unit_pack_bytes(const x3_conv & c) {
    if (c.c_in != kUnit || c.c_out != kUnit || c.stride != 1 || !c.snake || !c.post_alpha_log || c.residual ||
        static_cast<int64_t>(c.dil) * 6 > kMaxHalo || c.cols >= (int64_t{1} << 28) ||
        c.cols * kUnit * kUnit * 8 < kMinUnitMacs)
        return -1;
    return layout_of(c, 7).bytes() + kUnitFragBytes + round16(4 * (kUnit / 32) * (kUnit / kCI));
}

int launch_x3_unit(const x3_conv & c, const float * w1, const float * bias1, void * pack, hipStream_t st,
                   const char * what) {
    const x3_layout l = layout_of(c, 7);
    x3_kernel_params p{};
    if (const int rc = launch_pack<7, true>(p, c, l, static_cast<char *>(pack), w1, st, what); rc != LEVO_HIP_OK) return rc;
    p.bias1 = bias1;
    return launch_kernel<7, true, true>(p, st, what);
}

}  // namespace levo_hip
