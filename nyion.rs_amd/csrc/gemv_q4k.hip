// gemv_q4k.hip — Q4_K weight products (gfx950), the projection step either
// side of decode attention.
//
// The reference computes out[r] = sum_j W[r][j] x[j] with W in GGUF Q4_K
// blocks of 256 weights (swamp-kernels/src/fused_gemv_q4k.rs:59-99 dispatch,
// scalar semantics 395-448): a 144-byte block of f16 d, f16 dmin, 12 bytes of
// 6-bit scales/mins (unpack 30-43) and 128 nibble bytes, where byte i of qs
// pair p holds element 64p+i (low nibble, sub-block 2p) and element 64p+32+i
// (high nibble, sub-block 2p+1).  The weight is (d*scale)*q - (dmin*min).
//
// Arithmetic.  Every product runs on v_mfma_f32_16x16x32_f16, inputs as the
// 16 rows of A and weight rows as the 16 columns of B, with operands that
// hold the f32 product exactly but for the last bit of x:
//  * scale * (q - z), at most 945 in magnitude, is exact in binary16, so the
//    block's d multiplies one f32 sum per block; scale * z and dmin * min
//    multiply the sums of x per sub-block.  z = round(dmin * min / (d * scale))
//    makes these operands about as small as the weights (z = 0 throughout: 1.5
//    times the error), and zero where a weight is zero: a value of x that no
//    weight takes up, however large, costs the others nothing (a fixed z = 8
//    under min = 0 put 2e-5 of the output's norm in it for a value of 2^10);
//  * each input's 256 values of a block are scaled by the power of two that
//    brings their largest magnitude into [2^14, 2^15) and split into two
//    binary16 terms, x = hi + lo 2^-11, which hold it to within 2^-23 of x or
//    2^-50 of the block's largest, whichever is more (2^-45 for the sums of x
//    per sub-block, which are split likewise); hi and lo have an accumulator
//    each (lo added to hi's doubled the error).
// A block's value for one (row, input) is a chain of eight K steps, and an
// output is the sum of kSumWays sums of its blocks' values, whichever kernel,
// tile or wavefront computed them: single, multi-matrix and batched calls
// give the same bits.  Against float64 the outputs are off by 1.5e-7 to 1.8e-7
// of their norm for N(0, 1) inputs (512 to 14336 columns; f32 FMAs in runs of
// 16 were 1.5e-7 to 2.2e-7), and as much beside a value 2^28 times the others
// that meets zero weights.
//
// Two kernels.  gemv_split_kernel (up to eight inputs): the wavefronts of a
// workgroup take the blocks of 16 rows among them, each converting the inputs
// of its own blocks into LDS once for all the rows the workgroup walks.
// gemv_tile_kernel (more): the wavefronts take different rows and walk the
// blocks together over inputs converted once per workgroup.
//
// What bounds them.  Up to eight inputs, HBM and the chain in front of it: a
// wavefront's 16 rows x 256 weights are 2304 bytes, 125 VALU instructions (143
// with eight inputs) and 10 MFMAs, where a convert and an FMA per weight and
// input were 300 instructions for the first input alone; 14336 x 4096 with
// eight inputs keeps the VALU 64 % and the matrix cores 7 % busy.  Many inputs,
// VALU and matrix cores in turn: 5632 x 2048 with 509 inputs 65 % and 31 %.
// f32 FMAs and now, us: 14336 x 4096, one input 12.8 and 9.7, eight inputs 65.7
// and 14.6; 5632 x 2048, 509 inputs 1319 and 39.8.
#include "gemv.hpp"

#include <limits.h>

#include <algorithm>

namespace nyion {

constexpr int kSplitMaxInputs = 8;  // of gemv_split_kernel: hi and lo rows of one MFMA

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ halfx2 as_half2(uint32_t w) { return __builtin_bit_cast(halfx2, w); }
__device__ __forceinline__ uint32_t as_word(halfx2 h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ halfx8 as_half8(u32x4 w) { return __builtin_bit_cast(halfx8, w); }
__device__ __forceinline__ halfx2 splat2(_Float16 h) { return halfx2{h, h}; }

// The high bytes of two halves 1024 + n, n < 256
constexpr uint32_t kHalf1024 = 0x64006400u;

// What the low terms of x count: they are kept 2^11 times larger, so that
// they are normal binary16 numbers wherever the high terms are.
constexpr float kLowTerm = 1.f / 2048;

// ---------------------------------------------------------------------------
// Weights.  Lane (n, g) of a wavefront (n = lane & 15 the row, g = lane >> 4)
// holds 64 weights of its row's block, eight for each K step s = 0..7, as the
// two runs of four x values at x_offset(s, g) and kRunGap further on, each in
// the order 0, 2, 1, 3.
// ---------------------------------------------------------------------------

struct Q4k {
    static constexpr int kBlockBytes = kQ4kBlockBytes;
    static constexpr int kRunGap = 32;  // x distance from the low run to the high run
    // the block's 16-byte header and nibble bytes 32g..32g+31: sub-blocks 2g
    // (low nibbles) and 2g+1 (high nibbles)
    struct Raw {
        u32x4 hdr, qa, qb;
    };
    // Factors and offsets of the two sub-blocks for the low nibbles' and the
    // high nibbles' weights; scale * offset and the mins as operands of the
    // sums of x (the mins also for their low terms); d and dmin.
    struct Scales {
        halfx2 s_lo, o_lo, s_hi, o_hi;
        uint32_t offsets, mins, mins_low;
        float d, dmin;
    };
    __device__ static int x_offset(int s, int g) { return 64 * g + 4 * s; }
    __device__ __forceinline__ static void load(const uint8_t* bp, int g, Raw& r) {
        r.hdr = *(const u32x4*)bp;
        r.qa = *(const u32x4*)(bp + 16 + 32 * g);
        r.qb = *(const u32x4*)(bp + 32 + 32 * g);
    }
    // unpack_scales_q4k for sub-blocks 2g and 2g+1, two bytes at a time: the
    // 6-bit fields of sub-blocks 0-3 are whole bytes, those of 4-7 a nibble
    // and two bits (masks, so that the lanes do not part)
    __device__ __forceinline__ static void scales(const Raw& r, int g, Scales& c) {
        const int k = 16 * (g & 1);
        const uint32_t whole = g < 2 ? 0x3f3fu : 0u, nib = g < 2 ? 0u : 0x0f0fu, two = g < 2 ? 0u : 0x3030u;
        const uint32_t a = r.hdr.y >> k, b = r.hdr.z >> k, e = r.hdr.w >> k;
        const uint32_t sc = (a & whole) | (e & nib) | ((a >> 2) & two);
        const uint32_t mn = (b & whole) | ((e >> 4) & nib) | ((b >> 2) & two);
        // bytes 0 and 1 as the low bytes of two halves 1024 + n
        const halfx2 s = as_half2(__builtin_amdgcn_perm(kHalf1024, sc, 0x07010700u)) - splat2(1024);
        const halfx2 m = as_half2(__builtin_amdgcn_perm(kHalf1024, mn, 0x07010700u)) - splat2(1024);
        const float d = f16_bits_to_f32(r.hdr.x), dmin = f16_bits_to_f32(r.hdr.x >> 16);
        // z = dmin * min / (d * scale) to the nearest integer within 0 .. 15
        // (any would do: quotients of zeros, infinities and NaNs end in there too)
        halfx2 z = m * halfx2{(_Float16)__builtin_amdgcn_rcph(s.x), (_Float16)__builtin_amdgcn_rcph(s.y)} *
                   splat2((_Float16)(dmin * __builtin_amdgcn_rcpf(d)));
        z = __builtin_elementwise_min(__builtin_elementwise_max(z, splat2(0)), splat2(15));
        z = (z + splat2(1024)) - splat2(1024);
        const halfx2 sz = s * z;
        // nibbles masked in place are the binary16 denormals q 2^-24 (low) and
        // q 2^-20 (high)
        c.s_lo = splat2(s.x) * splat2(1024);
        c.s_hi = splat2(s.y) * splat2(64);
        c.o_lo = splat2(sz.x) * splat2((_Float16)(-1.0 / 16384));
        c.o_hi = splat2(sz.y) * splat2((_Float16)(-1.0 / 16384));
        c.offsets = as_word(sz * splat2((_Float16)(1.0 / 512)));
        c.mins = as_word(m);
        c.mins_low = as_word(m * splat2((_Float16)kLowTerm));
        c.d = d * 16384.f;
        c.dmin = dmin * 32.f;
    }
    // scale * (q - z) * 2^-14, exact
    __device__ __forceinline__ static halfx8 weights(const Raw& r, const Scales& c, int s) {
        const uint32_t q = s < 4 ? r.qa[s] : r.qb[s - 4];
        const uint32_t o = q >> 8;
        const u32x4 v = {as_word(__builtin_elementwise_fma(as_half2(q & 0x000f000fu), c.s_lo, c.o_lo)),
                         as_word(__builtin_elementwise_fma(as_half2(o & 0x000f000fu), c.s_lo, c.o_lo)),
                         as_word(__builtin_elementwise_fma(as_half2(q & 0x00f000f0u), c.s_hi, c.o_hi)),
                         as_word(__builtin_elementwise_fma(as_half2(o & 0x00f000f0u), c.s_hi, c.o_hi))};
        return as_half8(v);
    }
    // The block's value of one (row, input), of the scaled input, from its
    // sums: acc of scale * q * 2^-14 and accm of min * sum(x) / 32.
    __device__ __forceinline__ static float value(const Scales& c, float acc, float accm) {
        return __builtin_fmaf(-c.dmin, accm, c.d * acc);
    }
};

// ---------------------------------------------------------------------------
// Inputs
// ---------------------------------------------------------------------------

// The value of the lane that DPP control CTRL names (all lanes active).
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float add_dpp(float x) {
    return x + __uint_as_float(dpp<CTRL>(__float_as_uint(x)));
}

// Max over the 32 lanes of a half wavefront, in every lane (as integers:
// the bits of magnitudes).
__device__ __forceinline__ uint32_t max_half_wave(uint32_t x) {
    x = max(x, dpp<0xb1>(x));   // quad_perm [1,0,3,2]
    x = max(x, dpp<0x4e>(x));   // quad_perm [2,3,0,1]
    x = max(x, dpp<0x141>(x));  // row_half_mirror
    x = max(x, dpp<0x140>(x));  // row_mirror
    const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(x, x, false, false));
    return max(r.x, r.y);
}

// One lane's share of an input's block: step s, group g (s = lane & 7,
// g = lane >> 3 & 3; a half wavefront does one input's block).
struct XShare {
    float4 lo, hi;
};

__device__ __forceinline__ XShare load_x(const float* xb, int s, int g) {
    const float* p = xb + Q4k::x_offset(s, g);
    return XShare{*(const float4*)p, *(const float4*)(p + Q4k::kRunGap)};
}

// The two binary16 terms of the share (operand words of step s, group g),
// the block's 1 / scale, and, in the lanes with s = 0, the two terms of the
// sums of x over sub-blocks 2g and 2g+1 (times 2^-5: the sum of 32 values
// stays in range).  An infinity leaves a NaN in lo, so that it makes every
// output of its input NaN, as a NaN does.
struct XTerms {
    u32x4 hi, lo;
    uint32_t sum_hi, sum_lo;
    float inv;
};

// a and b as two binary16 terms each, a = hi + lo * kLowTerm.  The high term
// is converted back to be subtracted, so that the low one also holds what a
// denormal high term leaves (kept out of v_fma_mix, which issues at a quarter
// of the rate of a subtraction).
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& hi, uint32_t& lo) {
    hi = as_word(halfx2{(_Float16)a, (_Float16)b});
    asm("" : "+v"(hi));
    float ha = (float)as_half2(hi).x, hb = (float)as_half2(hi).y;
    asm("" : "+v"(ha));
    asm("" : "+v"(hb));
    lo = as_word(halfx2{(_Float16)((a - ha) * (1.f / kLowTerm)), (_Float16)((b - hb) * (1.f / kLowTerm))});
}

__device__ __forceinline__ XTerms split_x(const XShare& x) {
    const float u[8] = {x.lo.x, x.lo.z, x.lo.y, x.lo.w, x.hi.x, x.hi.z, x.hi.y, x.hi.w};
    // the largest magnitude (a NaN's bits are larger than any other's)
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) m = max(m, __float_as_uint(u[i]) & 0x7fffffffu);
    m = max_half_wave(m);
    // exponent at least 15, so that 1 / scale is a normal number
    const uint32_t e = max(m >> 23, 15u);
    const float scale = __uint_as_float((268u - e) << 23);
    XTerms t;
    t.inv = __uint_as_float((e - 14u) << 23);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t h, l;
        split_pair(u[2 * i] * scale, u[2 * i + 1] * scale, h, l);
        t.hi[i] = h;
        t.lo[i] = l;
    }
    float s0 = (u[0] + u[1]) + (u[2] + u[3]), s1 = (u[4] + u[5]) + (u[6] + u[7]);
    s0 = add_dpp<0xb1>(s0);
    s1 = add_dpp<0xb1>(s1);
    s0 = add_dpp<0x4e>(s0);
    s1 = add_dpp<0x4e>(s1);
    s0 = add_dpp<0x141>(s0);
    s1 = add_dpp<0x141>(s1);
    const float sum_scale = scale * 0.03125f;
    split_pair(s0 * sum_scale, s1 * sum_scale, t.sum_hi, t.sum_lo);
    return t;
}

// x + kLowTerm times the value of x 32 lanes on, in the lower half of the
// wavefront.
__device__ __forceinline__ float add_low_rows(float x) {
    const u32x2 r = __builtin_bit_cast(
        u32x2, __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false));
    return __builtin_fmaf(__uint_as_float(r.y), kLowTerm, __uint_as_float(r.x));
}

// An output is the sum of kSumWays sums, in order, of the values of the
// blocks k, k + kSumWays, ...
constexpr int kSumWays = 4;

// The sum of a quad's values in order, in its first lane (the quad's lanes
// all active).
__device__ __forceinline__ float sum_quad(float x) {
    const uint32_t v = __float_as_uint(x);
    x += __uint_as_float(dpp<0x55>(v));  // quad_perm [1,1,1,1]
    x += __uint_as_float(dpp<0xaa>(v));  // quad_perm [2,2,2,2]
    return x + __uint_as_float(dpp<0xff>(v));
}

__device__ __forceinline__ floatx4 mfma(const halfx8& a, const halfx8& b, const floatx4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Operands of the products with a word or two per lane on either side (the
// sums of x per sub-block): the other words stay zero in their registers.  (The
// K = 16 form, of half the words, gave wrong sums behind a K = 32 chain into
// the same accumulator with this compiler.)
__device__ __forceinline__ u32x4 zero_words() {
    u32x4 w = {0, 0, 0, 0};
    asm("" : "+v"(w));
    return w;
}

// ---------------------------------------------------------------------------
// Few inputs: the wavefronts of a workgroup split the blocks of 16 rows
// ---------------------------------------------------------------------------

struct GemvMat {
    const uint8_t* w;  // [rows][nb * block bytes]
    float* out;        // [n_inputs][out_stride]
    int rows;
    int unit0;  // its first unit (INT_MAX: no such matrix)
};

struct GemvSplitArgs {
    GemvMat mat[kGemvMaxMats];
    int units;       // of all matrices
    int full, rest;  // groups of blocks per wavefront, one more for the first `rest`
    int waves;       // of a workgroup that multiply
    int converters;  // of a workgroup that convert the inputs (SHARED)
    const float* x;  // [n_inputs][x_stride]
    long long x_stride;
    long long out_stride;
    int nb;        // blocks per row
    int n_inputs;  // 1..kSplitMaxInputs
};

// LDS of a workgroup for B inputs: per block (of the row, or of a step of
// each wavefront where the row's would not fit) the operands [step 8][g 4]
// [term 2][input] of 16 bytes, the sums [g 4][term 2][input] words and
// 1 / scale [input]; then two buffers of the blocks' values [block][input]
// [row].
__host__ __device__ constexpr int split_block_bytes(int B) { return (B * (1024 + 32 + 4) + 15) & ~15; }
__host__ __device__ constexpr int split_lds_bytes(int blocks, int nb, int B, int R) {
    return blocks * split_block_bytes(B) + 2 * nb * B * R * 4;
}

// A unit is R rows of one matrix; the 16 columns of an MFMA are its rows in
// 16 / R consecutive blocks, and the 16 rows of A the two terms of up to
// R / 2 inputs for each of these blocks (the products of a block's weights
// with another block's inputs are not used).
//
// The inputs are converted once per workgroup, each wavefront's blocks by
// itself or (SHARED: workgroups of one unit) all blocks by those that multiply
// and more that only convert; or (EACH_STEP, for rows whose operands would not
// fit the LDS) by each wavefront for each of its steps.
template <int B, int R, bool EACH_STEP, bool SHARED>
__global__ __launch_bounds__(1024) void gemv_split_kernel(GemvSplitArgs a) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int KB = 16 / R;  // blocks per step
    constexpr int BP = R / 2;   // rows of A per block and term
    static_assert(B <= BP, "inputs of a step");
    const int lane = threadIdx.x & 63;
    const int kp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int P = a.waves;
    const int n = lane & 15, g = lane >> 4;
    const int nb = a.nb, last_in = a.n_inputs - 1;
    const int npass = a.full + (kp < a.rest);  // this wavefront's groups kp, kp + P, ... of KB blocks
    const int first = (int)blockIdx.x, stride = (int)gridDim.x;  // units first, first + stride, ...
    const int U = a.units;
    const long long row_bytes = (long long)nb * Q4k::kBlockBytes;
    constexpr int kBlk = split_block_bytes(B);
    float* vals = (float*)(lds + (EACH_STEP ? P * KB : nb) * kBlk);
    const int row_n = n % R, blk_n = n / R;  // this lane's row of the unit and block of the group

    // the matrix of unit u, selected in scalar registers: an indexed load of
    // the arguments is one more round trip ahead of the weights, and of the
    // outputs behind the sums
    auto mat_of = [&](int u) __attribute__((always_inline)) {
        GemvMat m = a.mat[0];
#pragma unroll
        for (int i = 1; i < kGemvMaxMats; i++) {
            const uint8_t* const w = a.mat[i].w;
            float* const out = a.mat[i].out;
            const int rows = a.mat[i].rows, unit0 = a.mat[i].unit0;
            const bool in = u >= unit0;
            m.w = in ? w : m.w;
            m.out = in ? out : m.out;
            m.rows = in ? rows : m.rows;
            m.unit0 = in ? unit0 : m.unit0;
        }
        return m;
    };
    // rows past the matrix repeat its last, blocks past the row its last
    auto load_w = [&](int u, int pass, Q4k::Raw& r) __attribute__((always_inline)) {
        const GemvMat m = mat_of(u);
        const int row = min((u - m.unit0) * R + row_n, m.rows - 1);
        const int b = min((kp + P * pass) * KB + blk_n, nb - 1);
        Q4k::load(m.w + row * row_bytes + (long long)b * Q4k::kBlockBytes, g, r);
    };

    // inputs, two (block, input) pairs at a time, one per half wavefront
    // (inputs past the last repeat it, and an odd last pair is done twice)
    const int s = lane & 7, gx = (lane >> 3) & 3, half = lane >> 5;
    auto load_pair = [&](int b, int in) __attribute__((always_inline)) {
        const float* x = B == 1 ? a.x : a.x + min(in, last_in) * a.x_stride;
        return load_x(x + (long long)b * kKqBlockElems, s, gx);
    };
    auto store_pair = [&](const XShare& xs, uint8_t* base, int in) __attribute__((always_inline)) {
        const XTerms t = split_x(xs);
        const int at = (s * 4 + gx) * 2 * B + in;
        *(u32x4*)(base + at * 16) = t.hi;
        *(u32x4*)(base + (at + B) * 16) = t.lo;
        if (s == 0) {
            *(uint32_t*)(base + 1024 * B + (gx * 2 * B + in) * 4) = t.sum_hi;
            *(uint32_t*)(base + 1024 * B + ((gx * 2 + 1) * B + in) * 4) = t.sum_lo;
        }
        if (s == 0 && gx == 0) *(float*)(base + 1056 * B + in * 4) = t.inv;
    };
    // the pairs of one step
    constexpr int kPairs = KB * B, kShares = (kPairs + 1) / 2;
    XShare xs[kShares];
    auto load_step_x = [&](int pass) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kShares; i++) {
            const int c = min(2 * i + half, kPairs - 1);
            xs[i] = load_pair(min((kp + P * pass) * KB + c / B, nb - 1), c % B);
        }
    };
    Q4k::Raw raw[2];
    uint8_t* own = lds + kp * KB * kBlk;  // EACH_STEP: this wavefront's blocks
    if constexpr (EACH_STEP) {
        load_step_x(0);
        load_w(first, 0, raw[0]);
    } else if constexpr (SHARED) {
        // all blocks' pairs among all wavefronts; the fence as below
        auto item = [&](int i) __attribute__((always_inline)) { return (unsigned)min(2 * i + half, nb * B - 1); };
        const int items = (nb * B + 1) / 2, di = a.converters;
        auto load_at = [&](int i) __attribute__((always_inline)) {
            const unsigned c = item(i);
            return load_pair(c / B, c % B);
        };
        XShare cur = load_at(kp), next;
        if (kp + di < items) next = load_at(kp + di);
        asm volatile("" ::: "memory");
        if (kp < P) load_w(first, 0, raw[0]);
        for (int i = kp;;) {
            const unsigned c = item(i);
            store_pair(cur, lds + c / B * kBlk, c % B);
            if ((i += di) >= items) break;
            cur = next;
            if (i + di < items) next = load_at(i + di);
        }
        __syncthreads();
        if (kp >= P) {
            __syncthreads();  // the unit's
            return;
        }
    } else {
        // all of this wavefront's blocks; the first weights are requested
        // behind the loads of the first pairs and ahead of their conversion.
        // The fence holds them there: loads return in order, and with the
        // weights first the conversion began only when they had come from HBM
        // (88 launches of 256 to 11264 rows, replayed: 493 -> 414 us with the
        // matrices and passes below out of the way too)
        const int pairs = npass * kPairs;
        auto block_of = [&](unsigned c) __attribute__((always_inline)) {
            const unsigned k = c / B;
            return min((kp + P * (int)(k / KB)) * KB + (int)(k % KB), nb - 1);
        };
        auto load_at = [&](int i) __attribute__((always_inline)) {
            const int c = min(i, pairs - 1);
            return load_pair(block_of(c), c % B);
        };
        auto store_at = [&](const XShare& x, int i) __attribute__((always_inline)) {
            const int c = min(i + half, pairs - 1);
            store_pair(x, lds + block_of(c) * kBlk, c % B);
        };
        XShare cur = load_at(half), next;
        if (pairs > 2) next = load_at(2 + half);
        asm volatile("" ::: "memory");
        load_w(first, 0, raw[0]);
        store_at(cur, 0);
        for (int i = 2; i < pairs; i += 2) {
            cur = next;
            if (i + 2 < pairs) next = load_at(i + 2 + half);
            store_at(cur, i);
        }
    }

    // row n of A: term n / 8, block (n & 7) / BP of the group, input
    // (n & 7) % BP (past the inputs the last again)
    const int blk_a = (n & 7) / BP;
    const int ta = (n >> 3) * B + min((n & 7) % BP, B - 1);
    const uint8_t* op0 = (EACH_STEP ? own : lds) + (g * 2 * B + ta) * 16;
    const uint8_t* sum0 = (EACH_STEP ? own : lds) + 1024 * B + (g * 2 * B + ta) * 4;
    // Row 4g + r of the result: that row of A.  This lane's block and input
    // t are row blk_n * BP + t (hi), and 32 lanes on its lo: lane group
    // (blk_n * BP + t) / 4, register (blk_n * BP + t) % 4.
    constexpr int kRegs = B < 4 ? B : 4;         // inputs of a lane's registers
    const int g_out = blk_n * BP / 4;            // first lane group of this lane's block
    const int t0 = BP > 4 ? 4 * (g - g_out) : 0;  // its first input here
    const bool out_lane = g >= g_out && t0 < B && g < (BP > 4 ? 2 : g_out + 1);
    const bool upper = BP < 4 && (blk_n & 1);    // its registers start at 2
    const float* inv0 = (const float*)((EACH_STEP ? own : lds) + 1056 * B) + (out_lane ? t0 : 0);

    // one (unit, pass) of this wavefront; returns with the next step's
    // weights requested
    int u = first, pass = 0, par = 0;
    u32x4 word_a = zero_words(), word_b = zero_words(), word_c = zero_words();
    auto step = [&](Q4k::Raw& cur, Q4k::Raw& nxt) __attribute__((always_inline)) {
        const bool more = pass + 1 < npass;
        if constexpr (EACH_STEP) {
            // over the last step's operands: a wavefront's LDS operations
            // complete in order
#pragma unroll
            for (int i = 0; i < kShares; i++) {
                const int c = min(2 * i + half, kPairs - 1);
                store_pair(xs[i], own + c / B * kBlk, c % B);
            }
            load_step_x(more ? pass + 1 : 0);
        }
        if (more || u + stride < U) load_w(more ? u : u + stride, more ? pass + 1 : 0, nxt);
        const int b0 = (kp + P * pass) * KB;
        const int off = (EACH_STEP ? blk_a : min(b0 + blk_a, nb - 1)) * kBlk;
        Q4k::Scales sc;
        Q4k::scales(cur, g, sc);
        floatx4 acc = {0.f, 0.f, 0.f, 0.f}, accm = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < 8; st++) {
            const halfx8 xv = as_half8(*(const u32x4*)(op0 + off + st * 128 * B));
            acc = mfma(xv, Q4k::weights(cur, sc, st), acc);
        }
        // the offsets' term as the weights' (hi and lo rows); the mins' with both
        // terms of the sums of x, as two words, into the rows of hi: two products
        // one after the other were off by 4 % more (1.7e-7) and took 1.5 % longer
        // (14336 x 4096, eight inputs)
        word_a.x = *(const uint32_t*)(sum0 + off);
        word_a.y = 0;
        word_b.x = sc.offsets;
        acc = mfma(as_half8(word_a), as_half8(word_b), acc);
        word_a.y = *(const uint32_t*)(sum0 + off + 4 * B);
        word_c.x = sc.mins;
        word_c.y = sc.mins_low;
        accm = mfma(as_half8(word_a), as_half8(word_c), accm);
        float v[kRegs];
#pragma unroll
        for (int r = 0; r < kRegs; r++) {
            float full = add_low_rows(acc[r]), m = accm[r];
            if constexpr (BP < 4) {
                const float full2 = add_low_rows(acc[r + 2]);
                full = upper ? full2 : full;
                m = upper ? accm[r + 2] : m;
            }
            v[r] = Q4k::value(sc, full, m);
        }
        const int b = b0 + blk_n;
        if (out_lane && b < nb) {
            const float* inv = inv0 + (EACH_STEP ? blk_n : b) * (kBlk / 4);
#pragma unroll
            for (int r = 0; r < kRegs; r++) vals[((par * nb + b) * B + t0 + r) * R + row_n] = v[r] * inv[r];
        }
        if (++pass < npass) return;
        pass = 0;
        __syncthreads();  // the buffers alternate, so one barrier per unit suffices
        // one thread per output and sum, the four of an output in a quad (4096
        // x 14336 11.9 -> 11.7 us against one thread per output)
        for (int t = threadIdx.x; t < R * B * kSumWays; t += 64 * P) {
            const int o = t / kSumWays;
            const float* w = vals + par * nb * B * R + o;
            float sum = 0.f;
#pragma unroll 4
            for (int i = t % kSumWays; i < nb; i += kSumWays) sum += w[i * B * R];
            sum = sum_quad(sum);
            const GemvMat m = mat_of(u);
            const int row = (u - m.unit0) * R + o % R;
            if (t % kSumWays == 0 && row < m.rows && o / R <= last_in) m.out[o / R * a.out_stride + row] = sum;
        }
        par ^= 1;
        u += stride;
    };
    while (u < U) {
        step(raw[0], raw[1]);
        if (u >= U) break;
        step(raw[1], raw[0]);
    }
}

// ---------------------------------------------------------------------------
// Many inputs: the wavefronts of a workgroup take different rows
// ---------------------------------------------------------------------------

struct GemvTileArgs {
    const uint8_t* w;
    float* out;
    const float* x;
    long long x_stride, out_stride;
    int rows, nb, n_inputs;
    int in_tiles;  // workgroups across the inputs
};

// The operands of one block's inputs in LDS.
template <int MT>
struct TileX {
    // [input tile][term][step][g * 16 + input]; a step's row is one slot longer,
    // so that the eight steps of a group, stored by consecutive lanes, fall on
    // different banks
    u32x4 x[MT][2][8][65];
    uint32_t sums[MT][2][4][16];  // [input tile][term][g][input]
    float inv[16 * MT];
};

// LDS of a gemv_tile workgroup: two buffers of operands per K group, and a
// float per thread and output (the sums that are done).
template <int RW, int KS, int RT, int MT>
constexpr int tile_lds_bytes() {
    return KS * 2 * (int)sizeof(TileX<MT>) + RW * KS * 64 * RT * MT * 16;
}

// A workgroup of KS groups of RW wavefronts: RW*RT*16 rows x MT*16 inputs.
// Group k takes the sums k, k + KS, ... of kSumWays.
template <int RW, int KS, int RT, int MT, int WPS>
__global__ __launch_bounds__(64 * RW * KS, WPS) void gemv_tile_kernel(GemvTileArgs a) {
    static_assert(KS == 1 || KS == kSumWays, "a group's sums");
    constexpr int TM = 16 * MT;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int kg = wave / RW;
    TileX<MT>* xb = (TileX<MT>*)lds + 2 * kg;
    floatx4* done = (floatx4*)(lds + KS * 2 * sizeof(TileX<MT>));  // [output register group][thread]
    const int n = lane & 15, g = lane >> 4;
    const int nb = a.nb;
    const int in0 = ((int)blockIdx.x % a.in_tiles) * TM;
    const int row0 = ((int)blockIdx.x / a.in_tiles) * (RW * RT * 16) + (wave % RW) * RT * 16;
    const long long row_bytes = (long long)nb * Q4k::kBlockBytes;
    const uint8_t* wp[RT];
#pragma unroll
    for (int i = 0; i < RT; i++) wp[i] = a.w + min(row0 + 16 * i + n, a.rows - 1) * row_bytes;

    u32x4 word_h = zero_words(), word_l = zero_words(), word_w = zero_words(), word_m = zero_words();
    floatx4 total[RT][MT];  // the sum in progress
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < MT; j++) total[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // conversion: half wavefront h of the group takes inputs h, h + 2 RW, ...
    const int s = lane & 7, gx = (lane >> 3) & 3;
    const int h = ((int)threadIdx.x >> 5) % (2 * RW);
    constexpr int kShares = (TM + 2 * RW - 1) / (2 * RW);
    XShare xv[kShares];
    auto load_xs = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kShares; i++) {
            const int t = min(in0 + h + 2 * RW * i, a.n_inputs - 1);
            xv[i] = load_x(a.x + t * a.x_stride + (long long)b * kKqBlockElems, s, gx);
        }
    };
    auto convert = [&](TileX<MT>& to) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kShares; i++) {
            const XTerms t = split_x(xv[i]);
            const int in = h + 2 * RW * i, m = in & 15, j = in >> 4;
            if (TM % (2 * RW) && in >= TM) continue;
            const int slot = gx * 16 + m;
            to.x[j][0][s][slot] = t.hi;
            to.x[j][1][s][slot] = t.lo;
            if (s == 0) {
                to.sums[j][0][gx][m] = t.sum_hi;
                to.sums[j][1][gx][m] = t.sum_lo;
            }
            if (s == 0 && gx == 0) to.inv[in] = t.inv;
        }
    };
    // the group's blocks in order: those of sum kg, then (KS = 1) of the next;
    // past the last nb, which may be b + kSumWays as well: a sum's end is told
    // by b alone
    auto next_of = [&](int b) __attribute__((always_inline)) {
        if (b + kSumWays < nb) return b + kSumWays;
        const int k = b % kSumWays + 1;
        return KS == 1 && k < min(kSumWays, nb) ? k : nb;
    };
    const int steps = KS == 1 ? nb : (nb + KS - 1) / KS;  // of the longest group; barriers are common to all

    int b = min(kg, nb);
    Q4k::Raw cur[RT];
    load_xs(min(b, nb - 1));
#pragma unroll
    for (int i = 0; i < RT; i++) Q4k::load(wp[i] + (long long)min(b, nb - 1) * Q4k::kBlockBytes, g, cur[i]);
    convert(xb[0]);
    __syncthreads();

    for (int q = 0; q < steps; q++) {
        const TileX<MT>& X = xb[q & 1];
        const int b1 = b < nb ? next_of(b) : nb;
        const int bl = min(b1, nb - 1);  // past the last block its loads repeat one and are not used
        load_xs(bl);                     // converted at the end of this step
        if (KS == 1 || b < nb) {
            Q4k::Scales sc[RT];
#pragma unroll
            for (int i = 0; i < RT; i++) Q4k::scales(cur[i], g, sc[i]);
            floatx4 hi[RT][MT], lo[RT][MT];
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int j = 0; j < MT; j++) hi[i][j] = lo[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < 8; st++) {
                halfx8 w[RT];
#pragma unroll
                for (int i = 0; i < RT; i++) w[i] = Q4k::weights(cur[i], sc[i], st);
#pragma unroll
                for (int j = 0; j < MT; j++) {
                    const halfx8 xh = as_half8(X.x[j][0][st][lane]), xl = as_half8(X.x[j][1][st][lane]);
#pragma unroll
                    for (int i = 0; i < RT; i++) hi[i][j] = mfma(xh, w[i], hi[i][j]);
#pragma unroll
                    for (int i = 0; i < RT; i++) lo[i][j] = mfma(xl, w[i], lo[i][j]);
                }
            }
            // the next block's weights take the registers of this one's
#pragma unroll
            for (int i = 0; i < RT; i++) Q4k::load(wp[i] + (long long)bl * Q4k::kBlockBytes, g, cur[i]);
#pragma unroll
            for (int j = 0; j < MT; j++) {
                const floatx4 inv = *(const floatx4*)&X.inv[16 * j + 4 * g];
                word_h.x = X.sums[j][0][g][n];
                word_h.y = word_l.x = X.sums[j][1][g][n];
#pragma unroll
                for (int i = 0; i < RT; i++) {
                    word_w.x = sc[i].offsets;
                    hi[i][j] = mfma(as_half8(word_h), as_half8(word_w), hi[i][j]);
                    lo[i][j] = mfma(as_half8(word_l), as_half8(word_w), lo[i][j]);
                    word_m.x = sc[i].mins;
                    word_m.y = sc[i].mins_low;
                    const floatx4 m = mfma(as_half8(word_h), as_half8(word_m), floatx4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        total[i][j][r] = __builtin_fmaf(
                            Q4k::value(sc[i], __builtin_fmaf(lo[i][j][r], kLowTerm, hi[i][j][r]), m[r]), inv[r],
                            total[i][j][r]);
                }
            }
        }
        if (KS == 1 && b + kSumWays >= nb) {  // a sum is done (uniform)
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int j = 0; j < MT; j++) {
                    floatx4& d = done[(i * MT + j) * (64 * RW * KS) + threadIdx.x];
                    d = b % kSumWays ? d + total[i][j] : total[i][j];
                    total[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
                }
        }
        // the other buffer was last read before the barrier that ended the
        // previous step
        convert(xb[(q + 1) & 1]);
        b = b1;
        __syncthreads();
    }
    if constexpr (KS > 1) {
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int j = 0; j < MT; j++) done[(i * MT + j) * (64 * RW * KS) + threadIdx.x] = total[i][j];
        __syncthreads();
        if (kg > 0) return;
    }
#pragma unroll
    for (int i = 0; i < RT; i++) {
        const int row = row0 + 16 * i + n;
        if (row >= a.rows) continue;
#pragma unroll
        for (int j = 0; j < MT; j++) {
            const floatx4* d = done + (i * MT + j) * (64 * RW * KS) + threadIdx.x;
            floatx4 v = d[0];
#pragma unroll
            for (int k = 1; k < KS; k++) v += d[k * 64 * RW];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int t = in0 + 16 * j + 4 * g + r;
                if (t < a.n_inputs) a.out[t * a.out_stride + row] = v[r];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Dispatch
// ---------------------------------------------------------------------------

constexpr int kLdsPerCu = 160 * 1024;

// Allows a kernel the whole LDS of a CU (once per device).
template <class K>
static void allow_lds(std::atomic<int>* cache, K kernel, int lds) {
    if (lds > 64 * 1024)
        per_device_value(
            cache,
            [&] {
                return hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           kLdsPerCu) == hipSuccess;
            },
            0);
}

static int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }

// Wavefronts of a workgroup: with several inputs as many as there are block
// groups, up to 16, since they share the conversion of the inputs.  With one
// input the conversion is short and more, smaller workgroups on a CU keep
// more of them out of step with each other's barriers: as few wavefronts as
// leave two per SIMD and pass in the launch's units, four at least (28672 x
// 4096 Q4_K 17.6 us with 16, 14.9 with 4; 14336 x 4096 10.9 with 16, 9.7 with 8).  The groups are then dealt
// out in equal passes.
static int split_waves(int groups, int units, int B) {
    const int most = B > 1 ? 16 : std::min(16, std::max(4, ceil_div(8192, units)));
    return ceil_div(groups, ceil_div(groups, most));
}

// A launch's shape: wavefronts and LDS of a workgroup (0: not for this
// kernel), and whether the inputs are converted for each step.
struct SplitShape {
    int waves, lds;
    bool each_step;
};
static SplitShape split_shape(int nb, int units, int B, int R) {
    const int groups = ceil_div(nb, 16 / R);
    int waves = split_waves(groups, units, B);
    if (split_lds_bytes(nb, nb, B, R) <= kLdsPerCu) return {waves, split_lds_bytes(nb, nb, B, R), false};
    const int block = 16 / R * split_block_bytes(B);
    const int most = (kLdsPerCu - split_lds_bytes(0, nb, B, R)) / block;
    if (most < 4) return {0, 0, false};
    waves = ceil_div(groups, ceil_div(groups, std::min(16, most)));
    return {waves, split_lds_bytes(16 / R * waves, nb, B, R), true};
}

template <int B, int R>
static int launch_split_br(GemvSplitArgs& a, int cus, hipStream_t st) {
    int units = 0;
    for (int m = 0; m < kGemvMaxMats; m++) {
        a.mat[m].unit0 = a.mat[m].rows > 0 ? units : INT_MAX;
        units += ceil_div(a.mat[m].rows, R);
    }
    a.units = units;
    const SplitShape sh = split_shape(a.nb, units, B, R);
    const int groups = ceil_div(a.nb, 16 / R);
    a.waves = sh.waves;
    a.full = groups / sh.waves;
    a.rest = groups % sh.waves;
    // Where a workgroup has one unit and no SIMD more than one wavefront that
    // multiplies, the conversion is most of the launch, and more wavefronts
    // share it: four inputs of 2048, 256 rows 4.7 -> 4.0 us, 2048 rows 5.2 ->
    // 4.6, two inputs 3.7 -> 3.5.  With eight that multiply (1024 x 4096, four
    // inputs) 6.2 -> 6.3.
    a.converters = sh.waves;
    if (B > 1 && !sh.each_step && units <= cus && sh.waves <= 4)
        a.converters = std::max(sh.waves, std::min(16, ceil_div(a.nb * B, 2)));
    const bool shared = a.converters > sh.waves;
    // resident workgroups: four or (one input) five wavefronts per SIMD
    const int cap = std::max(1, std::min((B > 1 ? 16 : 20) / sh.waves, kLdsPerCu / sh.lds)) * cus;
    static std::atomic<int> allowed[3][kMaxDevices];
    auto kernel = sh.each_step ? gemv_split_kernel<B, R, true, false> : gemv_split_kernel<B, R, false, false>;
    if (shared) kernel = gemv_split_kernel<B, R, false, (B > 1)>;
    allow_lds(allowed[shared ? 2 : sh.each_step], kernel, sh.lds);
    hipLaunchKernelGGL(kernel, dim3(std::min(units, cap)), dim3(64 * a.converters), sh.lds, st, a);
    return check_launch("gemv q4k");
}

// Rows per unit: 16, or 8 with two blocks per step where units of 16 would
// leave CUs without one (2048 x 2048 3.8 -> 3.2 us, 2048 x 5632
// 5.3 -> 4.5 us in a graph of such calls; four rows and four blocks gained
// nothing over that at 256 rows).
template <int B>
static int launch_split_b(GemvSplitArgs& a, int rows, int cus, hipStream_t st) {
    if constexpr (B <= 4)
        if (rows <= 16 * cus - 16) return launch_split_br<B, 8>(a, cus, st);
    return launch_split_br<B, 16>(a, cus, st);
}

// Inputs that a gemv_split launch computes for n: what the registers and the
// LDS are laid out for.
static int padded_inputs(int n) { return n <= 2 ? n : n <= 4 ? 4 : 8; }
static bool split_fits(int nb, int n) {
    return n <= kSplitMaxInputs && split_shape(nb, 1, padded_inputs(n), 16).waves > 0;
}

static int launch_split(GemvSplitArgs& a, int rows, hipStream_t st) {
    const int cus = device_cu_count();
    switch (padded_inputs(a.n_inputs)) {
        case 1: return launch_split_b<1>(a, rows, cus, st);
        case 2: return launch_split_b<2>(a, rows, cus, st);
        case 4: return launch_split_b<4>(a, rows, cus, st);
        default: return launch_split_b<8>(a, rows, cus, st);
    }
}

template <int RW, int KS, int RT, int MT, int WPS>
static int launch_tile(GemvTileArgs& a, hipStream_t st) {
    a.in_tiles = ceil_div(a.n_inputs, 16 * MT);
    const int row_tiles = ceil_div(a.rows, RW * RT * 16);
    constexpr int lds = tile_lds_bytes<RW, KS, RT, MT>();
    static_assert(lds <= kLdsPerCu, "LDS of a workgroup");
    static std::atomic<int> allowed[kMaxDevices];
    allow_lds(allowed, gemv_tile_kernel<RW, KS, RT, MT, WPS>, lds);
    hipLaunchKernelGGL((gemv_tile_kernel<RW, KS, RT, MT, WPS>), dim3((unsigned)(row_tiles * a.in_tiles)),
                       dim3(64 * RW * KS), lds, st, a);
    return check_launch("gemv q4k");
}

// The tile: rows x inputs, and in how many K groups.  A larger tile converts
// and unpacks less per product, a smaller one and K groups fill more CUs.  A
// launch takes about blocks x max(alone, round x workgroups per CU) us; the
// two figures are what one workgroup on a
// CU took per block and what each took of a launch of many, from 256 x 2048
// with 20 inputs up to 5632 x 2048 with 509.  Us in the order below: 5632 x
// 2048, 509 inputs 175, 101, 72.6, 62.4, 59.2, 42.0; 14336 x 4096, 12 inputs
// 27.3, 16.9, 23.5, 40.4, 53.2, 68.7; 2048 x 2048, 33 inputs 9.1, 10.2, 12.7,
// 20.7, 27.9, 36.8.
static int launch_tiles(GemvTileArgs& a, hipStream_t st) {
    struct Tile {
        int rows, inputs;
        float alone, round;
    };
    static constexpr Tile tiles[] = {{32, 16, 0.63f, 0.72f}, {64, 16, 0.75f, 0.87f}, {64, 16, 1.2f, 0.8f},
                                     {128, 32, 2.1f, 2.5f},  {256, 32, 3.0f, 3.45f}, {384, 32, 4.0f, 4.75f}};
    const int cus = device_cu_count();
    int best = 0;
    float best_time = 0.f;
    for (int i = 0; i < 6; i++) {
        const long long wgs = (long long)ceil_div(a.rows, tiles[i].rows) * ceil_div(a.n_inputs, tiles[i].inputs);
        const float time = std::max(tiles[i].alone, tiles[i].round * (float)ceil_div(wgs, cus));
        if (i == 0 || time < best_time) {
            best = i;
            best_time = time;
        }
    }
    switch (best) {
        case 0: return launch_tile<2, 4, 1, 1, 2>(a, st);
        case 1: return launch_tile<4, 4, 1, 1, 4>(a, st);
        case 2: return launch_tile<4, 1, 1, 1, 4>(a, st);
        case 3: return launch_tile<8, 1, 1, 2, 4>(a, st);
        case 4: return launch_tile<16, 1, 1, 2, 4>(a, st);
        default: return launch_tile<12, 1, 2, 2, 3>(a, st);
    }
}

int gemv_q4k_launch(const uint8_t* const* ws, const float* x, long long x_stride, float* const* outs,
                    long long out_stride, const int32_t* row_counts, int n_mats, int nb, int batch,
                    hipStream_t st) {
    if (split_fits(nb, batch)) {
        GemvSplitArgs a{};
        long long rows = 0;
        for (int m = 0; m < n_mats; m++) {
            a.mat[m] = GemvMat{ws[m], outs[m], row_counts[m], 0};
            rows += row_counts[m];
        }
        a.nb = nb;
        a.x = x;
        a.x_stride = x_stride;
        a.out_stride = out_stride;
        a.n_inputs = batch;
        return launch_split(a, (int)rows, st);
    }
    GemvTileArgs t{};
    t.x = x;
    t.x_stride = x_stride;
    t.out_stride = out_stride;
    t.nb = nb;
    t.n_inputs = batch;
    for (int m = 0; m < n_mats; m++) {
        t.w = ws[m];
        t.out = outs[m];
        t.rows = row_counts[m];
        const int rc = launch_tiles(t, st);
        if (rc != NYION_OK) return rc;
    }
    return NYION_OK;
}

}  // namespace nyion
