// prefill_attention.hip — causal prefill attention on MFMA (gfx950).
//
// The reference prefills by calling ops::attention once per token with
// seq_len = abs_pos + 1 (swamp-engine/src/executor.rs:132-137, ops.rs:170-278):
// row i of a chunk that starts at position p attends to keys [0, p + i], the
// p cached ones first.  Here one kernel computes all rows of a chunk as a
// flash-attention style pass: bf16 q, k, v (and the p history tokens' k, v)
// in, fp32 accumulate, f32 out.
//
// Work decomposition.  A workgroup owns one kv head and eight (four at
// head_dim 64) (q head, 32-row block) pairs that read the same K/V: for GQA
// 4:1 these are the four q heads of the group on 64 rows, so every K/V tile
// staged in LDS feeds eight wavefronts.  Workgroups are numbered so that each XCD
// (workgroup id mod 8) takes a contiguous run of the (kv head, row block)
// list: with 8 kv heads every XCD's L2 holds the K/V of one head.  Within a
// head, row blocks are issued longest-first.  A launch too small for that to
// fill the chip splits the keys of its pairs as well (prefill_split_kernel).
//
// Per 64-key tile:
//   K tile  [64][D] bf16 -> LDS, rows padded by 16 bytes
//   V tile  [64][D] bf16 -> LDS as fp16, transposed to V^T [D][64] (key
//           pairs packed into 32-bit words, rows padded by 16 bytes)
//   S^T[64 keys][32 rows] = K . Q^T      v_mfma_f32_32x32x16_bf16, Q^T from
//                                        registers (loaded once)
//   online softmax per row (rows are lanes; 32 keys per lane per half), the
//   running max moved only when a half's weights against it grow too large
//   O[32 rows][D] += P . V               v_mfma_f32_32x32x16_f16, A = P in
//                                        fp16 converted in registers from the
//                                        S^T accumulators, B = V^T from LDS
// LDS holds two tiles: the next tile is written from registers (its global
// loads were issued a whole tile earlier) while the current one is consumed,
// with one barrier per tile.
//
// fp16 for P and V keeps 11 significant bits (p <= 2^14 after the lazy max),
// so the P.V product stays within the f32 reference's tolerance; V must lie
// within the fp16 range (|v| <= 65504).
#include <limits.h>
#include <math.h>

#include <algorithm>

#include "common.hpp"
#include "kv_write.hpp"

namespace nyion {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct PrefillArgs {
    const uint16_t* q;  // [N][Hq][D]
    const uint16_t* k;  // [N][Hkv][D]
    const uint16_t* v;
    const uint16_t* kh;  // [n_hist][Hkv][D]: the sequence's tokens before the chunk
    const uint16_t* vh;
    float* out;  // [N][Hq][D]
    int n;
    int n_hist;
    int n_heads;
    int n_kv_heads;
    int group;     // q heads per kv head
    int hw;        // q heads per workgroup (4, 2 or 1: the largest dividing the group)
    int rb_per_wg; // 32-row blocks per workgroup (wavefronts / hw)
    int n_rbg;     // row-block groups
    int n_items;   // kv heads x head subsets x row-block groups
    int causal;
    float scale_log2;
    // the chunk's paged K/V write, done by the kernel (kv_write == 0, no
    // pools: only the range check of its V): by the workgroups from attn_wgs
    // on, or (own_write) each workgroup of head subset 0 its own tokens' rows
    // for its kv head after its attention work
    WriteArgs kvw;
    int kv_write;
    int kv_dtype;
    int own_write;
    int attn_wgs;
};

constexpr int BN = 64;  // keys per tile

// Threads per workgroup: eight wavefronts at head_dim 128 (two per SIMD, one
// workgroup per CU), so each K/V tile staged in LDS feeds eight
// (q head, 32-row) pairs; four at head_dim 64.
template <int D>
constexpr int prefill_threads() {
    return D == 128 ? 512 : 256;
}
// Largest sum of one lane's 16 softmax weights of a half that is used as
// computed; above it the half's row max is taken and the weights redone.
// Every weight enters the P.V product as binary16, so the limit stays well
// below 65504.
constexpr float kPrefillSumLimit = 16384.0f;

// LDS tiles, padded by 16 bytes per row so that every lane's reads are one
// base address plus compile-time offsets (no per-read address registers):
//   K   [BN][D] bf16, row stride D*2+16 bytes;
//   V^T [D][BN] fp16, row stride BN*2+16 bytes.  Within each 16-key group the
//       keys sit in the order 0-3, 8-11, 4-7, 12-15, which is the order of
//       the PV k-step's B operand (lane half h holds keys 4h..4h+3 and
//       8+4h..8+4h+3), so one 16-byte read fetches it.
template <int D>
struct PrefillLds {
    static constexpr int KROW = D * 2 + 16;   // bytes
    static constexpr int VROW = BN * 2 + 16;  // bytes
    static constexpr int KBYTES = BN * KROW;
    static constexpr int VBYTES = D * VROW;
    static constexpr int BUF = KBYTES + VBYTES;
};

// Position of key w (0..15) of a 16-key group in V^T row order.
__device__ __forceinline__ int vt_pos(int w) {
    return (w & 3) | (((w >> 3) & 1) << 2) | (((w >> 2) & 1) << 3);
}

typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));

// max(v, v of lane ^ 32): v_permlane32_swap exchanges the two 32-lane halves
// without going through LDS (the result pair holds v and its partner in
// either order, depending on the half).
__device__ __forceinline__ float max_xor32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                    false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Two f32 -> one word of two fp16 (lo in the low half), round to nearest
// even; one v_cvt_pk_f16_f32.
__device__ __forceinline__ uint32_t pack_f16x2(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, halfx2{(_Float16)lo, (_Float16)hi});
}

// One tile's K (or V) in registers between its global loads and its LDS
// stores (K chunk u: key (tid+NT*u) / (D/8); V unit u: key pair and 8 dims).
// K is staged one tile ahead of V.
template <int D, int THREADS = prefill_threads<D>()>
struct KStage {
    static constexpr int NT = THREADS;
    static constexpr int LOADS = BN * (D / 8) / NT;
    u32x4 k[LOADS];
};
template <int D, int THREADS = prefill_threads<D>()>
struct VStage {
    static constexpr int NT = THREADS;
    static constexpr int UNITS = (BN / 2) * (D / 8) / NT;
    u32x4 v0[UNITS];
    u32x4 v1[UNITS];
};

// Buffer descriptor of a K or V source: n tokens of tok_stride elements
// from `base` (the bytes of one kv head's rows; the host keeps n *
// n_kv_heads * head_dim below 2^30, so every byte offset fits 31 bits).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t source_rsrc(const uint16_t* base, int n,
                                                               int tok_stride) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, n * tok_stride * 2, 0x00020000);
}

// Loads of the tile whose first key is token kt of a source of n tokens
// (kt may be negative for the first history tile).  A tile inside [0, n)
// is read with buffer loads (one per-thread offset, the tile offset in a
// scalar register); only a tile that reaches outside clamps K rows and
// zeroes V rows.
template <int D, int NT>
__device__ __forceinline__ void stage_load_k(KStage<D, NT>& st, const uint16_t* kbase, int tok_stride,
                                             int n, int kt, int tid) {
    constexpr int CPR = D / 8;
    constexpr int STEP = NT / CPR;  // keys between a thread's chunks
    if (kt >= 0 && kt + BN <= n) {
        // buffer loads: the source's descriptor and the tile offset in scalar
        // registers, one per-thread 32-bit offset (no per-lane address math)
        const __amdgpu_buffer_rsrc_t r = source_rsrc(kbase, n, tok_stride);
        const int off = ((tid / CPR) * tok_stride + 8 * (tid % CPR)) * 2;
        const int t0 = kt * tok_stride * 2, step = STEP * tok_stride * 2;
#pragma unroll
        for (int u = 0; u < KStage<D, NT>::LOADS; u++)
            st.k[u] = __builtin_amdgcn_raw_buffer_load_b128(r, off, t0 + u * step, 0);
        return;
    }
#pragma unroll
    for (int u = 0; u < KStage<D, NT>::LOADS; u++) {
        const int t = min(max(kt + tid / CPR + u * STEP, 0), n - 1);  // outside: finite, masked
        st.k[u] = *(const u32x4*)(kbase + (long long)t * tok_stride + 8 * (tid % CPR));
    }
}

template <int D, int NT>
__device__ __forceinline__ void stage_load_v(VStage<D, NT>& st, const uint16_t* vbase, int tok_stride,
                                             int n, int kt, int tid) {
    constexpr int STEP = 8 * (NT / (BN / 2));  // dims between a thread's units
    const int t = kt + 2 * (tid % (BN / 2));
    const int d0 = 8 * (tid / (BN / 2));
    if (kt >= 0 && kt + BN <= n) {
        const __amdgpu_buffer_rsrc_t r = source_rsrc(vbase, n, tok_stride);
        const int off = ((t - kt) * tok_stride + d0) * 2;
        const int t0 = kt * tok_stride * 2, row = tok_stride * 2;
#pragma unroll
        for (int u = 0; u < VStage<D, NT>::UNITS; u++) {
            st.v0[u] = __builtin_amdgcn_raw_buffer_load_b128(r, off + 2 * STEP * u, t0, 0);
            st.v1[u] = __builtin_amdgcn_raw_buffer_load_b128(r, off + 2 * STEP * u, t0 + row, 0);
        }
        return;
    }
#pragma unroll
    for (int u = 0; u < VStage<D, NT>::UNITS; u++) {
        st.v0[u] = t >= 0 && t < n ? *(const u32x4*)(vbase + (long long)t * tok_stride + d0 + STEP * u)
                                   : u32x4{0, 0, 0, 0};
        st.v1[u] = t + 1 >= 0 && t + 1 < n
                       ? *(const u32x4*)(vbase + (long long)(t + 1) * tok_stride + d0 + STEP * u)
                       : u32x4{0, 0, 0, 0};
    }
}

// The tile at key kt (relative to the chunk): keys below 0 come from the
// history, the rest from the chunk.  kt is uniform, so the selects are
// scalar and one copy of the loads serves both sources.
template <int D, int NT>
__device__ __forceinline__ void load_k_tile(KStage<D, NT>& st, const PrefillArgs& a,
                                            const uint16_t* kbase, const uint16_t* khbase,
                                            int tok_stride, int kt, int tid) {
    const bool hist = kt < 0;
    stage_load_k<D, NT>(st, hist ? khbase : kbase, tok_stride, hist ? a.n_hist : a.n,
                        hist ? kt + a.n_hist : kt, tid);
}
template <int D, int NT>
__device__ __forceinline__ void load_v_tile(VStage<D, NT>& st, const PrefillArgs& a,
                                            const uint16_t* vbase, const uint16_t* vhbase,
                                            int tok_stride, int kt, int tid) {
    const bool hist = kt < 0;
    stage_load_v<D, NT>(st, hist ? vhbase : vbase, tok_stride, hist ? a.n_hist : a.n,
                        hist ? kt + a.n_hist : kt, tid);
}

template <int D, int NT>
__device__ __forceinline__ void stage_store_k(const KStage<D, NT>& st, unsigned char* kslot, int tid) {
    using L = PrefillLds<D>;
    constexpr int CPR = D / 8;
#pragma unroll
    for (int u = 0; u < KStage<D, NT>::LOADS; u++) {
        const int id = tid + NT * u;
        *(u32x4*)(kslot + (id / CPR) * L::KROW + 16 * (id % CPR)) = st.k[u];
    }
}

template <int D, int NT>
__device__ __forceinline__ void stage_store_v(const VStage<D, NT>& st, unsigned char* vslot, int tid) {
    using L = PrefillLds<D>;
#pragma unroll
    for (int u = 0; u < VStage<D, NT>::UNITS; u++) {
        const int id = tid + NT * u;
        const int key = 2 * (id % (BN / 2));
        const int dc = id / (BN / 2);
        const int col = (key & ~15) + vt_pos(key & 15);  // even: keys key, key+1
#pragma unroll
        for (int e = 0; e < 8; e++) {
            // dim 8dc+e: low half from key, high half from key+1
            // bf16 -> f32 is a 16-bit shift (or mask for the high half); bf16
            // values in the fp16 range convert to fp16 exactly
            const uint32_t x0 = st.v0[u][e >> 1], x1 = st.v1[u][e >> 1];
            const float lo = __uint_as_float((e & 1) ? (x0 & 0xffff0000u) : (x0 << 16));
            const float hi = __uint_as_float((e & 1) ? (x1 & 0xffff0000u) : (x1 << 16));
            *(uint32_t*)(vslot + (8 * dc + e) * L::VROW + 2 * col) = pack_f16x2(lo, hi);
        }
    }
}

// Items first, first + step, ... < end of the chunk's K/V rows (`at` gives an
// item's row, kv head and four values) into the paged pools, with the V range
// check the binary16 P.V product needs; without pools, the check alone.
template <int D, class At>
__device__ __forceinline__ void write_items(const PrefillArgs& a, int first, int end, int step, At at) {
    float vmax = 0.f;
    auto each = [&](auto write) __attribute__((always_inline)) {
        for (int i = first; i < end; i += step) {
            int r, g, x;
            at(i, r, g, x);
            vmax = fmaxf(vmax, write(r, g, x));
        }
    };
    if (!a.kv_write)
        each([&](int r, int g, int x) {
            return v_absmax(*(const uint2*)(a.v + ((long long)r * a.n_kv_heads + g) * D + 4 * x));
        });
    else if (a.kv_dtype == NYION_KV_Q4_20B)  // 8 lanes per group: D / 4 is a multiple
        each([&](int r, int g, int x) { return write_kv_q4_vec(a.kvw, r, g, x); });
    else if (a.kv_dtype == NYION_KV_F16)
        each([&](int r, int g, int x) { return write_kv_vec<true>(a.kvw, r, g, x); });
    else
        each([&](int r, int g, int x) { return write_kv_vec<false>(a.kvw, r, g, x); });
    report_range(a.kvw.status, vmax >= 65520.f, kRangePrefillV);
}

// A workgroup's share of the write: the tokens of its row blocks for its kv
// head g (every (token, kv head) by exactly one workgroup).
template <int D>
__device__ __forceinline__ void write_chunk_rows(const PrefillArgs& a, int g, int hs, int rbg, int tid,
                                                 int threads) {
    if (!a.own_write || hs != 0) return;
    constexpr int VEC = D / 4;
    const int r0 = rbg * a.rb_per_wg * 32;
    const int r1 = min(a.n, r0 + a.rb_per_wg * 32);
    write_items<D>(a, tid, (r1 - r0) * VEC, threads, [&](int i, int& r, int& gi, int& x) {
        r = r0 + i / VEC;
        gi = g;
        x = i % VEC;
    });
}

// The whole write (of launches small enough for 32-bit item numbers), by the
// workgroups behind the first a.attn_wgs.
template <int D>
__device__ __forceinline__ void write_chunk_apart(const PrefillArgs& a, int wg, int wgs, int tid, int threads) {
    constexpr int VEC = D / 4;
    write_items<D>(a, wg * threads + tid, a.n * a.n_kv_heads * VEC, wgs * threads,
                   [&](int i, int& r, int& g, int& x) {
                       const int row = i / VEC;
                       r = row / a.n_kv_heads;
                       g = row - r * a.n_kv_heads;
                       x = i % VEC;
                   });
}

template <int D>
__global__ __launch_bounds__(prefill_threads<D>(), 512 / prefill_threads<D>()) void prefill_kernel(
    PrefillArgs a) {
    using L = PrefillLds<D>;
    constexpr int DT = D / 32;  // output dim tiles
    constexpr int KS = D / 16;  // k-steps of the S product

    // three K slots, then two V^T slots
    __shared__ __attribute__((aligned(16))) unsigned char lds[3 * L::KBYTES + 2 * L::VBYTES];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31;   // row (S^T col) / dim within tile (O col)
    const int h = lane >> 5;   // half

    if ((int)blockIdx.x >= a.attn_wgs) {
        write_chunk_apart<D>(a, (int)blockIdx.x - a.attn_wgs, (int)gridDim.x - a.attn_wgs, tid, prefill_threads<D>());
        return;
    }
    // workgroup -> work item: XCD x = id % 8 takes items [x*per, (x+1)*per)
    const int per = (a.n_items + 7) / 8;
    const int item = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (item >= a.n_items) return;
    const int p = item / a.n_rbg;                         // kv head * subsets + subset
    const int rbg = a.n_rbg - 1 - (item - p * a.n_rbg);  // longest first
    const int subsets = a.group / a.hw;
    const int g = p / subsets;
    const int hs = p - g * subsets;
    const int head = g * a.group + hs * a.hw + (wave % a.hw);
    const int row0 = (rbg * a.rb_per_wg + wave / a.hw) * 32;
    const int wg_row_end = min(a.n, (rbg + 1) * a.rb_per_wg * 32);
    // Keys are numbered relative to the chunk: history token t is key
    // t - n_hist (negative), chunk token t is key t.  History tiles end at
    // key -1, so the chunk's tiles start at key 0 whatever n_hist is, and
    // only the first history tile can be partial.
    const int key_end = a.causal ? wg_row_end : a.n;
    const int n_htiles = (a.n_hist + BN - 1) / BN;
    const int n_tiles = n_htiles + (key_end + BN - 1) / BN;
    const int kt0 = -n_htiles * BN;
    const int key_lo = -a.n_hist;                                  // first key of every row
    const int lim = a.causal ? min(row0 + j, a.n - 1) : a.n - 1;  // last key of this lane's row

    // Q^T operand (B of S^T = K.Q^T): row row0+j, dims 16s + 8h .. +7
    bf16x8 qreg[KS];
    {
        const int r = row0 + j;
        const bool ok = r < a.n;
        const uint16_t* qrow = a.q + ((long long)min(r, a.n - 1) * a.n_heads + head) * D;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            uint4 t = ok ? *(const uint4*)(qrow + 16 * s + 8 * h) : uint4{0, 0, 0, 0};
            qreg[s] = __builtin_bit_cast(bf16x8, t);
        }
    }

    floatx16 o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++) o[t] = floatx16{};
    float mrun = -1e30f;  // finite: exp2(s - mrun) of a masked s is 0, never NaN
    float lrun = 0.f;

    const uint16_t* kbase = a.k + (long long)g * D;
    const uint16_t* vbase = a.v + (long long)g * D;
    const uint16_t* khbase = a.kh + (long long)g * D;
    const uint16_t* vhbase = a.vh + (long long)g * D;
    const int tok_stride = a.n_kv_heads * D;
    unsigned char* const kslot0 = lds;
    unsigned char* const vslot0 = lds + 3 * L::KBYTES;
    KStage<D> kst;
    VStage<D> vst;

    // S^T of 32-key half kb of the tile in K slot `ks` (K rows kb*32 + j,
    // chunk 2s + h)
    auto scores_half = [&](const unsigned char* ks, int kb) {
        const unsigned char* kp = ks + (kb * 32 + j) * L::KROW + 16 * h;
        floatx16 st = floatx16{};
#pragma unroll
        for (int s0_ = 0; s0_ < KS; s0_ += 4) {
            bf16x8 kf[4];
#pragma unroll
            for (int s = 0; s < 4; s++) kf[s] = __builtin_bit_cast(bf16x8, *(const uint4*)(kp + 32 * (s0_ + s)));
#pragma unroll
            for (int s = 0; s < 4; s++) st = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s], qreg[s0_ + s], st, 0, 0, 0);
        }
        return st;
    };

    // Online softmax of half kb of the tile at key kt and O += P.V over its
    // two 16-key k-steps (consume_half).  Lane holds row row0+j, keys
    // kt + 32kb + 8(r/4) + 4h + r%4 in st[r].  The exps come before any
    // branch, so they interleave with the MFMAs issued before them.
    // Causal / range mask of half kb of the tile at key kt: the key of
    // st[r] is kt + 32kb + 4h + c(r), c(r) = 8(r/4) + r%4, compared as the
    // constant c(r) against this lane's bounds.
    auto mask_half = [&](floatx16& st, int kt, int kb) {
        const int hi = lim - kt - 32 * kb - 4 * h;
        const int lo = key_lo - kt - 32 * kb - 4 * h;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int c = 8 * (r >> 2) + (r & 3);
            st[r] = c <= hi && c >= lo ? st[r] : -INFINITY;
        }
    };
    // B operands of the PV product of half kb: V^T row 32dt + j, the 8 keys
    // of k-step t = 2kb + t2.  They are read before the softmax that
    // produces P, so the PV MFMAs do not wait on LDS.
    auto load_vhalf = [&](const unsigned char* vs, int kb, halfx8 (&vb)[2][DT]) {
        const unsigned char* vp = vs + j * L::VROW + 16 * h + 64 * kb;
#pragma unroll
        for (int t2 = 0; t2 < 2; t2++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
                vb[t2][dt] = __builtin_bit_cast(halfx8, *(const uint4*)(vp + 32 * dt * L::VROW + 32 * t2));
    };
    auto consume_half = [&](floatx16 st, const halfx8 (&vb)[2][DT]) {
        // p = exp2(s*scale - m), one FMA + one exp per score, converted to
        // fp16 pairs; the row sum adds the f32 values in two chains of plain
        // adds (a v_dot2 sum of the fp16 pairs competes with the MFMAs for
        // issue and measured 1-2 % slower).  A operands of the PV product: k-step
        // t2 of this half holds keys 16t2 + 8(e/4) + 4h + e%4 (e = 0..7).
        halfx8 pa[2];
        float psum = 0.f;
        auto exps = [&]() {
            float sa = 0.f, sb = 0.f;
#pragma unroll
            for (int t2 = 0; t2 < 2; t2++)
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[8 * t2 + e], a.scale_log2, -mrun));
                    const float p1 =
                        __builtin_amdgcn_exp2f(__builtin_fmaf(st[8 * t2 + e + 1], a.scale_log2, -mrun));
                    sa += p0;
                    sb += p1;
                    pa[t2][e] = (_Float16)p0;
                    pa[t2][e + 1] = (_Float16)p1;
                }
            psum = sa + sb;
        };
        // The running max m (log2 units, scaled) is not recomputed per half:
        // the exps run against the current m, and only when some lane's sum
        // of p exceeds kPrefillSumLimit (so some p may be past it, up to an
        // fp16 overflow) is the half's row max taken, m raised to it, O and
        // the row sum rescaled and the exps redone.  Every kept p is then at
        // most kPrefillSumLimit.  The first half of every row takes this
        // path (m starts at -1e30, so its p are inf); a NaN sum (NaN inputs)
        // does not, and propagates as in the f32 reference.
        exps();
        if (__any(psum > kPrefillSumLimit)) {
            float mt = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; r++) mt = fmaxf(mt, st[r]);
            mt = max_xor32(mt) * a.scale_log2;  // scale > 0: max commutes
            const float mnew = fmaxf(mrun, mt);
            const float alpha = __builtin_amdgcn_exp2f(mrun - mnew);
            mrun = mnew;
            lrun *= alpha;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                // O reg r of this lane is row 8(r/4) + 4h + r%4
                const float ar = __shfl(alpha, 8 * (r >> 2) + 4 * h + (r & 3));
#pragma unroll
                for (int t = 0; t < DT; t++) o[t][r] *= ar;
            }
            exps();
        }
        lrun += psum;
#pragma unroll
        for (int t2 = 0; t2 < 2; t2++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(pa[t2], vb[t2][dt], o[dt], 0, 0, 0);
    };
    auto tile_masked = [&](int kt) {
        return (kt + BN > a.n) || (a.causal && kt + BN - 1 > row0) || kt < key_lo;
    };
    auto kslot = [&](int it) { return kslot0 + (it % 3) * L::KBYTES; };

    // Pipeline over 32-key halves: the S MFMAs of the next half are issued
    // before the softmax of the current one, so the matrix and vector pipes
    // have independent work.  At the top of iteration it: K slots hold
    // tiles it and it+1, V slot it&1 holds tile it, s0 = S of tile it's
    // first half, and the staging registers hold K of tile it+2 and V of
    // tile it+1.  The iteration writes the staged K into the slot of tile
    // it-1 and the staged V into the other V slot (both last read one
    // iteration ago), issues the next global loads and synchronises once.
    // Prologue: K and V of tile 0 and K of tile 1 in one round of loads,
    // then K of tile 2 and V of tile 1 requested as soon as the staging
    // registers are in LDS.
    {
        KStage<D> kst1;
        load_k_tile(kst, a, kbase, khbase, tok_stride, kt0, tid);
        load_v_tile(vst, a, vbase, vhbase, tok_stride, kt0, tid);
        if (n_tiles > 1) load_k_tile(kst1, a, kbase, khbase, tok_stride, kt0 + BN, tid);
        stage_store_k(kst, kslot0, tid);
        stage_store_v(vst, vslot0, tid);
        if (n_tiles > 1) stage_store_k(kst1, kslot0 + L::KBYTES, tid);
    }
    if (n_tiles > 2) load_k_tile(kst, a, kbase, khbase, tok_stride, kt0 + 2 * BN, tid);
    if (n_tiles > 1) load_v_tile(vst, a, vbase, vhbase, tok_stride, kt0 + BN, tid);
    __syncthreads();
    floatx16 s0 = scores_half(kslot0, 0);

    auto step = [&](int it, bool masked) {
        const int kt = kt0 + it * BN;
        const unsigned char* vs = vslot0 + (it & 1) * L::VBYTES;
        halfx8 vb[2][DT];
        // Waves w and w + 4 of the workgroup share a SIMD, and at equal
        // priority the older one wins every issue conflict: it reached the
        // barrier ~1100 cycles before its partner on every tile.  The younger
        // wave takes priority for the first half of the step, so the two
        // arrive together (waits ~270 / ~170 cycles; 1-2 % faster).
        if (wave >= 4) __builtin_amdgcn_s_setprio(1);
        load_vhalf(vs, 0, vb);
        if (masked) mask_half(s0, kt, 0);
        floatx16 s1 = scores_half(kslot(it), 1);
        consume_half(s0, vb);
        s0 = scores_half(kslot(it + 1), 0);
        load_vhalf(vs, 1, vb);
        if (wave >= 4) __builtin_amdgcn_s_setprio(0);
        if (masked) mask_half(s1, kt, 1);
        consume_half(s1, vb);
        // a slot past the last tile is written and never read
        stage_store_k(kst, kslot(it + 2), tid);
        stage_store_v(vst, vslot0 + ((it + 1) & 1) * L::VBYTES, tid);
        if (it + 3 < n_tiles) load_k_tile(kst, a, kbase, khbase, tok_stride, kt + 3 * BN, tid);
        if (it + 2 < n_tiles) load_v_tile(vst, a, vbase, vhbase, tok_stride, kt + 2 * BN, tid);
        __syncthreads();
    };
    int it = 0;
    if (n_tiles > 1 && tile_masked(kt0)) step(it++, true);  // partial first history tile
    for (; it + 1 < n_tiles && !tile_masked(kt0 + it * BN); it++) step(it, false);
    for (; it + 1 < n_tiles; it++) step(it, true);
    {
        const int it = n_tiles - 1;
        const int kt = kt0 + it * BN;
        const unsigned char* vs = vslot0 + (it & 1) * L::VBYTES;
        floatx16 s1 = scores_half(kslot(it), 1);
        if (tile_masked(kt)) {
            mask_half(s0, kt, 0);
            mask_half(s1, kt, 1);
        }
        halfx8 vb[2][DT];
        load_vhalf(vs, 0, vb);
        consume_half(s0, vb);
        load_vhalf(vs, 1, vb);
        consume_half(s1, vb);
    }

    // epilogue: divide by the row sums and store
    const float lt = lrun + __shfl_xor(lrun, 32);
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int rr = 8 * (r >> 2) + 4 * h + (r & 3);
        const float lr = __shfl(lt, rr);
        const int rowg = row0 + rr;
        if (rowg < a.n) {
            const float inv = 1.0f / lr;
            float* orow = a.out + ((long long)rowg * a.n_heads + head) * D;
#pragma unroll
            for (int dt = 0; dt < DT; dt++) orow[32 * dt + j] = o[dt][r] * inv;
        }
    }

    write_chunk_rows<D>(a, g, hs, rbg, tid, prefill_threads<D>());
}

// ---------------------------------------------------------------------------
// Few work items: the keys split among groups of wavefronts
// ---------------------------------------------------------------------------
//
// A short chunk gives few (kv head, row block) items, and each walks its keys
// in one chain of tiles at the latency of a wavefront that has its SIMD to
// itself (1.0 us per 64-key tile at head_dim 64, 1.7 at 128).  Here a workgroup is NG groups of GW
// wavefronts: the GW wavefronts of a group are (q head, 32-row block) pairs
// that share K/V tiles, as in prefill_kernel, and the groups take NG equal
// runs of the keys of the same pairs, each with tile buffers of its own.  Two
// K and two V^T slots per group fit 160 KB where the pipelined kernel's three
// and two would not.  At the end the groups' (max, sum, O) are merged through
// LDS.  The staged V is range-checked on the way (history and chunk), which
// spares the launch that prefill_kernel needs for a history.
//
// Bound: issue.  A step of the two wavefronts of a SIMD takes 1.6 us at
// head_dim 64, and about a third each with the staging, the exps or the
// products alone; the phases of the two barely overlap.  Groups of 4 or 1
// x 4 at 64 spill or leave SIMDs empty.  Taken: 2 x 4 at 64, 4 x 2 at 128.
template <int D, int GW, int NG>
struct SplitLds {
    using L = PrefillLds<D>;
    static constexpr int GROUP = 2 * (L::KBYTES + L::VBYTES);
    static constexpr int PART = 64 * (D / 2) * 4 + 2 * 64 * 4;  // one wavefront's O, max and sum
    static constexpr int BYTES = NG * GROUP > (NG - 1) * GW * PART ? NG * GROUP : (NG - 1) * GW * PART;
};

template <int D, int GW, int NG>
__global__ __launch_bounds__(64 * GW * NG) void prefill_split_kernel(PrefillArgs a) {
    using L = PrefillLds<D>;
    using S = SplitLds<D, GW, NG>;
    constexpr int DT = D / 32;  // output dim tiles
    constexpr int KS = D / 16;  // k-steps of the S product
    constexpr int NT = 64 * GW;
    extern __shared__ __attribute__((aligned(16))) unsigned char split_lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int grp = wave / GW, gw = wave % GW;
    const int tid = (int)threadIdx.x - grp * NT;  // within the group
    const int j = lane & 31;
    const int h = lane >> 5;

    const int per = (a.n_items + 7) / 8;
    const int item = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (item >= a.n_items) return;
    const int p = item / a.n_rbg;
    const int rbg = a.n_rbg - 1 - (item - p * a.n_rbg);
    const int subsets = a.group / a.hw;
    const int g = p / subsets;
    const int hs = p - g * subsets;
    const int head = g * a.group + hs * a.hw + (gw % a.hw);
    const int row0 = (rbg * a.rb_per_wg + gw / a.hw) * 32;
    const int wg_row_end = min(a.n, (rbg + 1) * a.rb_per_wg * 32);
    const int key_end = a.causal ? wg_row_end : a.n;
    const int n_htiles = (a.n_hist + BN - 1) / BN;
    const int n_tiles = n_htiles + (key_end + BN - 1) / BN;
    const int key_lo = -a.n_hist;
    const int lim = a.causal ? min(row0 + j, a.n - 1) : a.n - 1;
    // this group's tiles [it0, it1); every group makes `steps` steps
    const int steps = (n_tiles + NG - 1) / NG;
    const int it0 = min(grp * steps, n_tiles), it1 = min(it0 + steps, n_tiles);
    const int kt0 = (it0 - n_htiles) * BN;

    bf16x8 qreg[KS];
    {
        // rows past the end repeat the last one and are not stored
        const uint16_t* qrow = a.q + ((long long)min(row0 + j, a.n - 1) * a.n_heads + head) * D;
#pragma unroll
        for (int s = 0; s < KS; s++) qreg[s] = __builtin_bit_cast(bf16x8, *(const uint4*)(qrow + 16 * s + 8 * h));
    }
    floatx16 o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++) o[t] = floatx16{};
    float mrun = -1e30f, lrun = 0.f, vmax = 0.f;

    const uint16_t* kbase = a.k + (long long)g * D;
    const uint16_t* vbase = a.v + (long long)g * D;
    const uint16_t* khbase = a.kh + (long long)g * D;
    const uint16_t* vhbase = a.vh + (long long)g * D;
    const int tok_stride = a.n_kv_heads * D;
    unsigned char* const kslots = split_lds + grp * S::GROUP;
    unsigned char* const vslots = kslots + 2 * L::KBYTES;
    KStage<D, NT> kst;
    VStage<D, NT> vst;
    // tile it0 + i, clamped to the group's last (with none of its own, the last of all)
    auto load_tile = [&](int i) __attribute__((always_inline)) {
        const int kt = kt0 + min(i, it1 - it0 - 1) * BN;
        load_k_tile(kst, a, kbase, khbase, tok_stride, kt, tid);
        load_v_tile(vst, a, vbase, vhbase, tok_stride, kt, tid);
    };
    auto store_tile = [&](int i) __attribute__((always_inline)) {
        stage_store_k(kst, kslots + (i & 1) * L::KBYTES, tid);
        stage_store_v(vst, vslots + (i & 1) * L::VBYTES, tid);
#pragma unroll
        for (int u = 0; u < VStage<D, NT>::UNITS; u++)
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                vmax = fmaxf(vmax, v_absmax(uint2{vst.v0[u][e], vst.v0[u][e + 1]}));
                vmax = fmaxf(vmax, v_absmax(uint2{vst.v1[u][e], vst.v1[u][e + 1]}));
            }
    };
    load_tile(0);
    store_tile(0);
    // q is waited for here: a wait inside the loop would also drain the loads
    // of the next tile, every step
#pragma unroll
    for (int s = 0; s < KS; s++) asm volatile("" : "+v"(qreg[s]));
    load_tile(1);
    __syncthreads();

    // The next tile into the slots that were last read before the barrier
    // that ended the previous step.  Of the two wavefronts of a SIMD one does
    // it before its products and one after them, so that one's LDS writes and
    // conversions run beside the other's matrix work.
    auto stage = [&](int i) __attribute__((always_inline)) {
        if (it0 + i + 1 < it1) {
            store_tile(i + 1);
            load_tile(i + 2);
        }
    };
    const bool early = wave < GW * NG / 2;
    for (int i = 0; i < steps; i++) {
        if (early) stage(i);
        if (it0 + i < it1) {
            const int kt = kt0 + i * BN;
            const unsigned char* ks = kslots + (i & 1) * L::KBYTES;
            const unsigned char* vs = vslots + (i & 1) * L::VBYTES;
            const bool masked = (kt + BN > a.n) || (a.causal && kt + BN - 1 > row0) || kt < key_lo;
            // both halves' scores first: their products run while the first
            // half's weights are computed, and its P.V while the second's are
            floatx16 sc[2];
#pragma unroll
            for (int kb = 0; kb < 2; kb++) {
                const unsigned char* kp = ks + (kb * 32 + j) * L::KROW + 16 * h;
                sc[kb] = floatx16{};
#pragma unroll
                for (int s = 0; s < KS; s++)
                    sc[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        __builtin_bit_cast(bf16x8, *(const uint4*)(kp + 32 * s)), qreg[s], sc[kb], 0, 0, 0);
            }
            if (masked) {
#pragma unroll
                for (int kb = 0; kb < 2; kb++) {
                    const int hi = lim - kt - 32 * kb - 4 * h;
                    const int lo = key_lo - kt - 32 * kb - 4 * h;
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int c = 8 * (r >> 2) + (r & 3);
                        sc[kb][r] = c <= hi && c >= lo ? sc[kb][r] : -INFINITY;
                    }
                }
            }
#pragma unroll
            for (int kb = 0; kb < 2; kb++) {
                const floatx16& st = sc[kb];
                // weights against the running max, which is raised (and they
                // are redone) only where a lane's sum passes the limit, as in
                // prefill_kernel
                halfx8 pa[2];
                float psum = 0.f;
                auto exps = [&]() __attribute__((always_inline)) {
                    float sa = 0.f, sb = 0.f;
#pragma unroll
                    for (int t2 = 0; t2 < 2; t2++)
#pragma unroll
                        for (int e = 0; e < 8; e += 2) {
                            const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[8 * t2 + e], a.scale_log2, -mrun));
                            const float p1 =
                                __builtin_amdgcn_exp2f(__builtin_fmaf(st[8 * t2 + e + 1], a.scale_log2, -mrun));
                            sa += p0;
                            sb += p1;
                            pa[t2][e] = (_Float16)p0;
                            pa[t2][e + 1] = (_Float16)p1;
                        }
                    psum = sa + sb;
                };
                exps();
                if (__any(psum > kPrefillSumLimit)) {
                    float mt = -INFINITY;
#pragma unroll
                    for (int r = 0; r < 16; r++) mt = fmaxf(mt, st[r]);
                    mt = max_xor32(mt) * a.scale_log2;
                    const float mnew = fmaxf(mrun, mt);
                    const float alpha = __builtin_amdgcn_exp2f(mrun - mnew);
                    mrun = mnew;
                    lrun *= alpha;
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const float ar = __shfl(alpha, 8 * (r >> 2) + 4 * h + (r & 3));
#pragma unroll
                        for (int t = 0; t < DT; t++) o[t][r] *= ar;
                    }
                    exps();
                }
                lrun += psum;
                const unsigned char* vp = vs + j * L::VROW + 16 * h + 64 * kb;
#pragma unroll
                for (int t2 = 0; t2 < 2; t2++)
#pragma unroll
                    for (int dt = 0; dt < DT; dt++)
                        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            pa[t2], __builtin_bit_cast(halfx8, *(const uint4*)(vp + 32 * dt * L::VROW + 32 * t2)),
                            o[dt], 0, 0, 0);
            }
        }
        if (!early) stage(i);
        __syncthreads();
    }
    report_range(a.kvw.status, vmax >= 65520.f, kRangePrefillV);

    // merge: the other groups' parts in order through LDS
    const float lt = lrun + __shfl_xor(lrun, 32);
    float4* const part0 = (float4*)split_lds;
    constexpr int PART4 = S::PART / 16;
    if (grp > 0) {
        float4* pp = part0 + ((grp - 1) * GW + gw) * PART4;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r += 4)
                pp[(dt * 4 + r / 4) * 64 + lane] = float4{o[dt][r], o[dt][r + 1], o[dt][r + 2], o[dt][r + 3]};
        ((float*)(pp + D * 8))[lane] = mrun;
        ((float*)(pp + D * 8))[64 + lane] = lt;
    }
    __syncthreads();
    if (grp == 0) {
        float mall = mrun, lall = 0.f;
#pragma unroll
        for (int q = 1; q < NG; q++) mall = fmaxf(mall, ((const float*)(part0 + ((q - 1) * GW + gw) * PART4 + D * 8))[lane]);
        {
            const float alpha = __builtin_amdgcn_exp2f(mrun - mall);
            lall = lt * alpha;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const float ar = __shfl(alpha, 8 * (r >> 2) + 4 * h + (r & 3));
#pragma unroll
                for (int dt = 0; dt < DT; dt++) o[dt][r] *= ar;
            }
        }
#pragma unroll 1
        for (int q = 1; q < NG; q++) {
            const float4* pp = part0 + ((q - 1) * GW + gw) * PART4;
            const float alpha = __builtin_amdgcn_exp2f(((const float*)(pp + D * 8))[lane] - mall);
            lall += ((const float*)(pp + D * 8))[64 + lane] * alpha;
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                float ar[4];
#pragma unroll
                for (int e = 0; e < 4; e++) ar[e] = __shfl(alpha, 8 * (r >> 2) + 4 * h + e);
#pragma unroll
                for (int dt = 0; dt < DT; dt++) {
                    const float4 v = pp[(dt * 4 + r / 4) * 64 + lane];
                    o[dt][r] = __builtin_fmaf(v.x, ar[0], o[dt][r]);
                    o[dt][r + 1] = __builtin_fmaf(v.y, ar[1], o[dt][r + 1]);
                    o[dt][r + 2] = __builtin_fmaf(v.z, ar[2], o[dt][r + 2]);
                    o[dt][r + 3] = __builtin_fmaf(v.w, ar[3], o[dt][r + 3]);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int rr = 8 * (r >> 2) + 4 * h + (r & 3);
            const float lr = __shfl(lall, rr);
            const int rowg = row0 + rr;
            if (rowg < a.n) {
                const float inv = 1.0f / lr;
                float* orow = a.out + ((long long)rowg * a.n_heads + head) * D;
#pragma unroll
                for (int dt = 0; dt < DT; dt++) orow[32 * dt + j] = o[dt][r] * inv;
            }
        }
    }
    write_chunk_rows<D>(a, g, hs, rbg, (int)threadIdx.x, NT * NG);
}

}  // namespace nyion

using namespace nyion;

// Work items of a launch whose workgroups (or groups) have `waves` (q head,
// 32-row block) pairs: 4, 2 or 1 q heads, the largest that divides the group
// and the wavefront count, the remaining wavefronts more row blocks of them.
static long long prefill_items(PrefillArgs& a, int waves) {
    a.hw = std::min(4, waves);
    while (a.group % a.hw) a.hw /= 2;
    a.rb_per_wg = waves / a.hw;
    a.n_rbg = (a.n + 32 * a.rb_per_wg - 1) / (32 * a.rb_per_wg);
    return (long long)a.n_kv_heads * (a.group / a.hw) * a.n_rbg;
}

template <int D, int GW, int NG>
static int launch_prefill_split(PrefillArgs& a, hipStream_t st) {
    a.n_items = (int)prefill_items(a, GW);
    constexpr int lds = SplitLds<D, GW, NG>::BYTES;
    static_assert(lds <= 160 * 1024, "LDS of a CU");
    static std::atomic<int> allowed[kMaxDevices];
    per_device_value(
        allowed,
        [] {
            return hipFuncSetAttribute((const void*)prefill_split_kernel<D, GW, NG>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
        },
        0);
    hipLaunchKernelGGL((prefill_split_kernel<D, GW, NG>), dim3(8 * ((a.n_items + 7) / 8)), dim3(64 * GW * NG), lds,
                       st, a);
    return check_launch("prefill");
}

template <int D>
static int launch_prefill(PrefillArgs& a, hipStream_t st, bool& split) {
    constexpr int GW = D == 64 ? 2 : 4, NG = D == 64 ? 4 : 2;
    // Keys split over a workgroup's groups where one such workgroup per CU
    // holds the launch and there are tiles enough to pipeline.  Measured (us,
    // whole kernel / split): 32/4 heads of 64, 384 rows 11.1 / 11.7, 450 rows
    // 12.1 / 12.2, 512 rows 13.1 / 12.3, 640 rows (320 workgroups, two rounds)
    // 15.3 / 18.1; 12/12 heads, 450 rows 13.3 / 12.6, 768 rows 17.7 / 15.0;
    // 32/8 heads of 128, 256 rows 14.9 / 15.5, 320 rows 16.7 / 16.7, 384 rows
    // 18.4 / 17.9, 1024 rows 37.3 / 29.4, 2048 rows after 2048 123 / 129; 512
    // rows after 1536 37.0 / 21.7 (d 64) and 59.0 / 43.3 (d 128); into 4-bit
    // pools the lines cross about 60 rows later.  With a history the split
    // kernel also saves the launch that checks its V, which outweighs the merge
    // at any length: one row after 128 12.5 / 9.7 (d 64) and 13.4 / 10.2 (d 128).
    const int tiles = (a.n_hist + BN - 1) / BN + (a.n + BN - 1) / BN;
    split = prefill_items(a, GW) <= device_cu_count() && (tiles >= (D == 64 ? 8 : 6) || a.n_hist > 0);
    if (split) return launch_prefill_split<D, GW, NG>(a, st);
    const long long items = prefill_items(a, prefill_threads<D>() / 64);
    if (items > (1LL << 30)) return set_error(NYION_ERR_UNSUPPORTED, "prefill: %lld work items", items);
    a.n_items = (int)items;
    constexpr int threads = prefill_threads<D>();
    int wgs = 8 * ((a.n_items + 7) / 8);
    // The write of the chunk's rows by workgroups of its own where idle CUs
    // hold enough of them to take fewer turns than the attention's workgroups
    // would, one after the other: a turn of 4-bit rows is 0.5 us of arithmetic
    // for the four wavefronts of a CU, one of f32 rows 0.3.  Measured (us, the
    // attention's workgroups / apart / as a launch of its own): 4-bit pools,
    // 12/12 heads of 64, 256 rows 17.7 / 9.3 / 13.6 and 400 rows 19.6 / 11.2 /
    // 15.9; 32/8 heads of 128, 68 rows 14.5 / 9.1 / 13.3; 32/4 of 64, 33 rows
    // 8.0 / 5.9 / 10.1; f32 pools, the same in turn 13.4 / 9.4, 15.6 / 11.4,
    // 11.3 / 9.1 and 6.9 / 5.9.
    const long long turns = (a.rb_per_wg * 32 * (D / 4) + threads - 1) / threads;
    const long long needed = ((long long)a.n * a.n_kv_heads * (D / 4) + threads - 1) / threads;
    const int idle = device_cu_count() - wgs;
    if (idle > 0 && (needed + idle - 1) / idle < turns) {
        a.own_write = 0;
        a.attn_wgs = wgs;
        wgs += (int)std::min<long long>(needed, idle);
    }
    hipLaunchKernelGGL(prefill_kernel<D>, dim3(wgs), dim3(threads), 0, st, a);
    return check_launch("prefill");
}

static int prefill_impl(const uint16_t* q, const uint16_t* k, const uint16_t* v,
                        const uint16_t* k_hist, const uint16_t* v_hist, int n_hist, int n,
                        int n_heads, int n_kv_heads, int head_dim, int causal, float scale,
                        float* out, void* k_pool, void* v_pool, const int32_t* block_table,
                        int block_tokens, int num_blocks, int kv_dtype, int start_pos,
                        nyion_stream_t stream) {
    clear_error();
    int rc;
    if ((rc = require_device()) != NYION_OK) return rc;
    if (!q || !k || !v || !out) return set_error(NYION_ERR_INVALID, "prefill: null q/k/v/out");
    if (n <= 0 || n_heads <= 0 || n_kv_heads <= 0 || n_heads % n_kv_heads)
        return set_error(NYION_ERR_INVALID, "prefill: n=%d heads=%d/%d", n, n_heads, n_kv_heads);
    if (head_dim != 64 && head_dim != 128)
        return set_error(NYION_ERR_UNSUPPORTED, "prefill: head_dim %d (supported: 64, 128)", head_dim);
    if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || !aligned(out, 16))
        return set_error(NYION_ERR_INVALID, "prefill: q/k/v/out must be 16-byte aligned");
    if (n_hist < 0) return set_error(NYION_ERR_INVALID, "prefill: n_hist %d", n_hist);
    if (n_hist > 0 && (!k_hist || !v_hist || !aligned(k_hist, 16) || !aligned(v_hist, 16)))
        return set_error(NYION_ERR_INVALID, "prefill: history needs 16-byte aligned k_hist/v_hist");
    // K/V byte offsets are 32-bit (buffer loads): below 2^30 elements per source
    if ((long long)n * n_kv_heads * head_dim >= (1LL << 30) ||
        (long long)n * n_heads * head_dim >= (1LL << 40))
        return set_error(NYION_ERR_UNSUPPORTED, "prefill: chunk of %d tokens too large", n);
    if ((long long)n_hist * n_kv_heads * head_dim >= (1LL << 30) ||
        (long long)n_hist + n + 2 * BN >= (1LL << 31))
        return set_error(NYION_ERR_UNSUPPORTED, "prefill: history of %d tokens too large", n_hist);
    const int group = n_heads / n_kv_heads;
    PrefillArgs a{};
    a.q = q;
    a.k = k;
    a.v = v;
    // with no history the history pointers are never read; they alias k/v
    a.kh = n_hist > 0 ? k_hist : k;
    a.vh = n_hist > 0 ? v_hist : v;
    a.out = out;
    a.n = n;
    a.n_hist = n_hist;
    a.n_heads = n_heads;
    a.n_kv_heads = n_kv_heads;
    a.group = group;
    a.causal = causal ? 1 : 0;
    a.own_write = 1;
    a.attn_wgs = INT_MAX;
    const float sc = scale > 0.f ? scale : 1.0f / sqrtf((float)head_dim);
    a.scale_log2 = sc * 1.4426950408889634f;
    if (k_pool || v_pool) {
        if (!k_pool || !v_pool || !block_table)
            return set_error(NYION_ERR_INVALID, "prefill: KV write needs k_pool, v_pool and block_table");
        if ((rc = prefill_write_args(a.kvw, k_pool, v_pool, block_table, block_tokens, num_blocks,
                                     n_kv_heads, head_dim, kv_dtype, start_pos, n, k, v)) != NYION_OK)
            return rc;
        a.kv_write = 1;
        a.kv_dtype = kv_dtype;
    } else {
        a.kvw.status = device_status_word();
    }
    hipStream_t st = (hipStream_t)stream;
    bool split = false;
    if ((rc = head_dim == 128 ? launch_prefill<128>(a, st, split) : launch_prefill<64>(a, st, split)) != NYION_OK)
        return rc;
    // V enters the P.V product as binary16: values of magnitude >= 65520 are
    // reported through the status word (the chunk's V by the kernel's own
    // tail; the history's by the split kernel as it stages it, or here)
    if (n_hist > 0 && !split &&
        (rc = v_range_check(v_hist, (long long)n_hist * n_kv_heads * head_dim, st)) != NYION_OK)
        return rc;
    return NYION_OK;
}

extern "C" int nyion_prefill_attention_bf16(const uint16_t* q, const uint16_t* k, const uint16_t* v,
                                            int n, int n_heads, int n_kv_heads, int head_dim,
                                            int causal, float scale, float* out, void* k_pool,
                                            void* v_pool, const int32_t* block_table,
                                            int block_tokens, int num_blocks, int kv_dtype,
                                            int start_pos, nyion_stream_t stream) {
    return prefill_impl(q, k, v, nullptr, nullptr, 0, n, n_heads, n_kv_heads, head_dim, causal,
                        scale, out, k_pool, v_pool, block_table, block_tokens, num_blocks,
                        kv_dtype, start_pos, stream);
}

extern "C" int nyion_prefill_attention_bf16_ctx(const uint16_t* q, const uint16_t* k,
                                                const uint16_t* v, const uint16_t* k_hist,
                                                const uint16_t* v_hist, int n_hist, int n,
                                                int n_heads, int n_kv_heads, int head_dim,
                                                int causal, float scale, float* out, void* k_pool,
                                                void* v_pool, const int32_t* block_table,
                                                int block_tokens, int num_blocks, int kv_dtype,
                                                int start_pos, nyion_stream_t stream) {
    return prefill_impl(q, k, v, k_hist, v_hist, n_hist, n, n_heads, n_kv_heads, head_dim, causal,
                        scale, out, k_pool, v_pool, block_table, block_tokens, num_blocks,
                        kv_dtype, start_pos, stream);
}

