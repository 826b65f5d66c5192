// The SVTR tail on fp16 halves (weights that bound every operand inside fp16's range), as one
// launch per transformer block and one before the first:
//   neck_qkv_kernel    x rows (transposed from channels first when they come so), LN1, qkv;
//   neck_block_kernel  attention, proj + residual, LN2, fc1, swish, fc2 + residual, and then
//                      the next block's LN1 and qkv, or the final LayerNorm + shortcut.
// Everything after the attention is local to a token row, and the attention needs only the
// line's q, k, v rows, so a workgroup takes R token rows through a whole block: the
// intermediate rows stay in LDS and registers, and only x and qkv cross HBM.
//
// Operands are split into fp16 halves, x = x_hi + x_lo, and a product is a_hi w_hi +
// a_hi w_lo + a_lo w_hi (exact products, fp32 sums).  Each operand is scaled by a power of two
// from its bound before the split (exact, undone on the sums), so that the low halves stay
// above fp16's subnormals.
//
// 512 threads.  In the attention wave w is head w: K and V go from the qkv rows straight into
// its MFMA operands (v_mfma_f32_16x16x16_f16), a line's keys 64 at a time with an online
// softmax.  In the products (v_mfma_f32_16x16x32_f16, weights as the A operand, token rows as
// columns) the waves share out the output columns, so each weight is read by one wave of the
// workgroup only and goes from L2 into registers without LDS: the planes are stored in the
// order of the operand registers (NeckBlockDev), 1 KB per load instruction.  Lane (c, g),
// c = lane % 16, g = lane / 16, holds of each output tile token row c at columns 4 g .. + 3.
//
// What bounds it: the chain of phases in one workgroup (cycle stamps of one line's workgroup, 16
// rows: 29200 cycles, of them 2300 to the line table, 8400 attention, 2600 + 3500 + 3600 around
// the loads of fc1's, fc2's and qkv's weights, 4 x 1300 products) over loads at 55 bytes a cycle
// into the CU (512 KB of weights per workgroup and block).  Measured with tables, transposes and
// launches: one channels-first line 93 -> 33 us, a page's tail and head 134 -> 74.  Tried on top:
// two workgroups per CU (128 registers spill: 94 us for 16384 rows against 76), V turned through
// LDS instead of loaded by dim (one line 34 us), query blocks in pairs (tiles of 64 rows spill).
#include <cmath>

#include "kernels.hpp"
#include "neck.hpp"
#include "neck_device.hpp"

namespace ppocr {

namespace {

constexpr int D = kNeckDim, H = kNeckHidden;
constexpr int kThreads = 512;
// LDS row strides: an odd number of 16-byte chunks, so that 8 lanes reading 16 bytes of 8
// consecutive rows touch all 32 banks
constexpr int kAS = 136;   // halves per row of an operand of 128 values
constexpr int kHS = 264;   // of the hidden layer (256)
constexpr int kXS = 124;   // floats per row of x
static_assert(D <= 120 && H <= 256 && kNeckHeadDim == 15, "tile geometry");

// The halves of two values: hi their nearest halves (low and high 16 bits), lo the nearest halves
// of the exact remainders.  Four instructions: the remainders are fp32 fmas that read the halves
// where they are (x - hi by way of a conversion back took ten).
__device__ __forceinline__ void split2(float x0, float x1, unsigned& hi, unsigned& lo) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    hi = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{x0, x1}, h2));
    float r0, r1;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(hi), "v"(x0));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r1) : "v"(hi), "v"(x1));
    lo = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{r0, r1}, h2));
}
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split4(const f32x4& x, u32x2& hi, u32x2& lo) {
    unsigned h0, h1, l0, l1;
    split2(x[0], x[1], h0, l0);
    split2(x[2], x[3], h1, l1);
    hi = u32x2{h0, h1};
    lo = u32x2{l0, l1};
}

// (low halves of a and b), (high halves of a and b)
__device__ __forceinline__ unsigned pair_lo(unsigned a, unsigned b) { return __builtin_amdgcn_perm(b, a, 0x05040100); }
__device__ __forceinline__ unsigned pair_hi(unsigned a, unsigned b) { return __builtin_amdgcn_perm(b, a, 0x07060302); }

__device__ __forceinline__ f32x4 mfma32(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// The maximum over the lanes c, c + 16, c + 32, c + 48, in each of them: the swaps exchange
// odd with even rows of 16 lanes, then the halves, in the vector ALU (no trip through LDS).
__device__ __forceinline__ float max_over_groups(float x) {
    const unsigned u = __float_as_uint(x);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const unsigned y = __float_as_uint(max_f32(__uint_as_float(a[0]), __uint_as_float(a[1])));
    const auto b = __builtin_amdgcn_permlane32_swap(y, y, false, false);
    return max_f32(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

template <int R>
struct Lds {
    __align__(16) _Float16 as[2][R * kAS];  // operand rows of 128: attention output, LN2, LN1
    __align__(16) _Float16 hs[2][R * kHS];  // hidden rows; its start also the channels-first tile
    __align__(16) float xs[R * kXS];        // x rows
    // a block's vectors: LN2's weight and bias, fc1's bias, the weight and bias of the LayerNorm at
    // the end, the next qkv's bias
    __align__(16) float ln2_w[D], ln2_b[D], b1[H], end_w[D], end_b[D], bq[kNeckQkvPad];
    int t0[R], t1[R];                       // each row's line: rows t0 .. t1 - 1 (t1 = 0: none)
    int base;
    // hs and xs together also stage the rows of qkv
    __device__ __forceinline__ uint8_t* stage() { return reinterpret_cast<uint8_t*>(hs); }
};
// A token row of qkv, 1536 bytes: per head 64 bytes of q, of k and of v.  q (times the
// attention's scale) and k: 16 high halves, then 16 low halves; v: 16 pairs (high, low).  All
// split after their power-of-two scaling, once here instead of once per use.  The sixteenth value
// of a head is 0 in q and k and 1 in v (unscaled), which makes row 15 of the attention's O^T
// the sum of the probabilities.
constexpr int kRowBytes = 4 * kNeckQkvPad, kPart = kRowBytes / 3;
constexpr int kStageStride = kRowBytes + 16;  // an odd number of 16-byte chunks

// The KS steps of 32 of one 16-column tile's weights, both planes: wf points at the tile,
// [step][plane][lane][8].
template <int KS>
struct Weights {
    f16x8 hi[KS], lo[KS];
    __device__ __forceinline__ void load(const uint16_t* wf, int lane) {
        const f16x8* p = reinterpret_cast<const f16x8*>(wf) + lane;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            hi[s] = p[(2 * s) * 64];
            lo[s] = p[(2 * s + 1) * 64];
        }
    }
};
constexpr int kTileHalves = 2 * 64 * 8;  // halves of one step of a tile (both planes)

// acc[t][rt] = the NT tiles' weights x the operand rows (planes act0, act1; rows 16 rt + c).  A
// single tile sums its three products apart and adds them at the end: its chain of MFMAs would
// otherwise wait for each one's result.
template <int KS, int NT, int RT>
__device__ __forceinline__ void products(const Weights<KS> (&w)[NT], const _Float16* act0, const _Float16* act1, int stride,
                                         int c, int g, f32x4 (&acc)[NT][RT]) {
    constexpr int A = NT == 1 ? 3 : 1;
    f32x4 s3[A][NT][RT];
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) s3[a][t][rt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        f16x8 bh[RT], bl[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int o = (16 * rt + c) * stride + 32 * s + 8 * g;
            bh[rt] = *reinterpret_cast<const f16x8*>(act0 + o);
            bl[rt] = *reinterpret_cast<const f16x8*>(act1 + o);
        }
#pragma unroll
        for (int pr = 0; pr < 3; ++pr)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    f32x4& x = s3[A == 3 ? pr : 0][t][rt];
                    x = mfma32(pr == 1 ? w[t].lo[s] : w[t].hi[s], pr == 2 ? bl[rt] : bh[rt], x);
                }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[t][rt] = A == 3 ? s3[0][t][rt] + (s3[A == 3 ? 1 : 0][t][rt] + s3[A == 3 ? 2 : 0][t][rt]) : s3[0][t][rt];
}

// LayerNorm of this thread's share of a row: a row is 32 units of 4 columns (the last two past
// D), 512 / R threads per row, thread `part` units part + (512 / R) j in v[j].  The sums run
// within a unit and then in one tree over the bits of the unit index, so a row's bits do not
// depend on R.  v becomes (v - mean) * inv_std.
template <int R>
__device__ __forceinline__ int unit_col(int part, int j) {
    return 4 * (part + kThreads / R * j);
}
template <int R>
__device__ __forceinline__ void layer_norm(float (&v)[R / 16][4], int part, float eps) {
    constexpr int U = R / 16, P = kThreads / R;
    auto tree = [&](float (&u)[U]) {
#pragma unroll
        for (int o = 1; o < P; o <<= 1)
#pragma unroll
            for (int j = 0; j < U; ++j) u[j] += __shfl_xor(u[j], o, 64);
#pragma unroll
        for (int n = U; n > 1; n /= 2)
#pragma unroll
            for (int j = 0; j < n / 2; ++j) u[j] = u[2 * j] + u[2 * j + 1];
        return u[0];
    };
    float u[U];
#pragma unroll
    for (int j = 0; j < U; ++j) u[j] = (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
    const float mean = __fdiv_rn(tree(u), (float)D);
#pragma unroll
    for (int j = 0; j < U; ++j) {
        float t = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[j][e] -= mean;
            t = fmaf(v[j][e], v[j][e], t);
        }
        u[j] = unit_col<R>(part, j) < D ? t : 0.0f;
    }
    const float inv = __fdiv_rn(1.0f, __fsqrt_rn(__fdiv_rn(tree(u), (float)D) + eps));
#pragma unroll
    for (int j = 0; j < U; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] *= inv;
}

// xs -> LayerNorm (w, b) -> as, times sy, in halves (zeros past D)
template <int R>
__device__ __forceinline__ void ln_to_operand(Lds<R>& l, int tid, const float* w, const float* b, float eps, float sy) {
    constexpr int U = R / 16, P = kThreads / R;
    const int row = tid / P, part = tid % P;
    float v[U][4];
    f32x4 lw[U], lb[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const int col = unit_col<R>(part, j), cc = col < D ? col : 0;
        lw[j] = *reinterpret_cast<const f32x4*>(w + cc);
        lb[j] = *reinterpret_cast<const f32x4*>(b + cc);
        const f32x4 x = *reinterpret_cast<const f32x4*>(l.xs + row * kXS + cc);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] = col < D ? x[e] : 0.0f;
    }
    layer_norm<R>(v, part, eps);
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const int col = unit_col<R>(part, j);
        f32x4 y;
        u32x2 hi, lo;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = col < D ? fmaf(v[j][e], lw[j][e], lb[j][e]) * sy : 0.0f;
        split4(y, hi, lo);
        *reinterpret_cast<u32x2*>(&l.as[0][row * kAS + col]) = hi;
        *reinterpret_cast<u32x2*>(&l.as[1][row * kAS + col]) = lo;
    }
}

// qkv of the rows in `as` (LN1's output times 2^qkv_ey): wave w the column tiles 3 w .. 3 w +
// 2 (a tile: q, k or v of one head), staged in LDS and stored as one contiguous piece.
template <int R>
__device__ __forceinline__ void qkv_rows(Lds<R>& l, const Weights<4> (&w)[3], const NeckBlockDev& k, float scale, int tid,
                                         int wave, int c, int g, int64_t r0, int64_t m, uint8_t* __restrict__ qkv) {
    constexpr int RT = R / 16;
    f32x4 acc[3][RT];
    products(w, l.as[0], l.as[1], kAS, c, g, acc);
    const float s = ldexpf(1.0f, -(k.qkv_e + k.qkv_ey));
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        const int tile = 3 * wave + t, part = tile >> 3;  // uniform
        const f32x4 bc = *reinterpret_cast<const f32x4*>(l.bq + 16 * tile + 4 * g);
        const float mul = ldexpf(1.0f, part == 0 ? k.attn_eq : part == 1 ? k.attn_ek : k.attn_ev);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            uint8_t* o = l.stage() + (16 * rt + c) * kStageStride + 64 * tile;
            f32x4 x;
            u32x2 hi, lo;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[e] = acc[t][rt][e] * s + bc[e];
                if (part == 0) x[e] = x[e] * scale;  // the Mul(scale) node, rounded as it
                x[e] = x[e] * mul;
            }
            if (part == 2) x[3] = g == 3 ? 1.0f : x[3];
            split4(x, hi, lo);
            if (part < 2) {
                *reinterpret_cast<u32x2*>(o + 8 * g) = hi;
                *reinterpret_cast<u32x2*>(o + 32 + 8 * g) = lo;
            } else {
                *reinterpret_cast<u32x4*>(o + 16 * g) =
                    u32x4{pair_lo(hi[0], lo[0]), pair_hi(hi[0], lo[0]), pair_lo(hi[1], lo[1]), pair_hi(hi[1], lo[1])};
            }
        }
    }
    __syncthreads();
    constexpr int CH = kRowBytes / 16;  // 16-byte chunks of a row
    const int64_t rows = min((int64_t)R, m - r0);
#pragma unroll
    for (int e = 0; e < R * CH / kThreads; ++e) {
        const int x = kThreads * e + tid, row = x / CH, ch = x % CH;
        if (row < rows)
            *reinterpret_cast<u32x4*>(qkv + r0 * kRowBytes + (int64_t)x * 16) =
                *reinterpret_cast<const u32x4*>(l.stage() + row * kStageStride + 16 * ch);
    }
}

// A channels-first tile (line b: [D][T_b] at D * t0_b): element e of this thread is row
// (512 e + tid) % R, channel (512 e + tid) / R, so neighbouring lanes read neighbouring steps.
// Rows in no line: zeros.
template <int R>
struct CfTile {
    static constexpr int N = (D * R + kThreads - 1) / kThreads;
    float v[N];
    __device__ __forceinline__ void load(const Lds<R>& l, int tid, int64_t r0, const float* __restrict__ src) {
#pragma unroll
        for (int e = 0; e < N; ++e) {
            const int x = kThreads * e + tid, r = x % R, ch = x / R;
            const int64_t t0 = l.t0[r], t1 = l.t1[r];
            v[e] = ch < D && t1 > 0 ? src[D * t0 + ch * (t1 - t0) + (r0 + r - t0)] : 0.0f;
        }
    }
    __device__ __forceinline__ void store(float* dst, int tid) const {
#pragma unroll
        for (int e = 0; e < N; ++e) {
            const int x = kThreads * e + tid, r = x % R, ch = x / R;
            if (ch < D) dst[r * kXS + ch] = v[e];
        }
    }
};

// Lines of the rows r0 .. r0 + R - 1 into t0 and t1 (clamped to [0, m)).  Ragged lines: every
// thread takes a line of a window of 512 and writes the rows it covers; the window starts at
// the last of 512 evenly spaced lines that begins at or before r0.
template <int R>
__device__ void line_table(Lds<R>& l, int tid, const int64_t* __restrict__ line_off, int64_t lines, int64_t line_len,
                           int64_t m, int64_t r0) {
    if (!line_off) {
        if (tid < R) {
            const int64_t r = r0 + tid, line = r / line_len, t0 = min(line * line_len, m);
            const bool in = r < m && line < lines;
            l.t0[tid] = in ? (int)t0 : 0;
            l.t1[tid] = in ? (int)min(t0 + line_len, m) : 0;
        }
        __syncthreads();
        return;
    }
    auto start = [&](int64_t line) { return min(max(line_off[line], (int64_t)0), m); };
    if (tid < R) l.t0[tid] = l.t1[tid] = 0;
    if (tid == 0) l.base = 0;
    __syncthreads();
    int64_t base = 0;
    if (lines > kThreads) {
        const int64_t step = (lines + kThreads - 1) / kThreads, line = tid * step;
        if (line < lines && start(line) <= r0) atomicMax(&l.base, tid);
        __syncthreads();
        base = l.base * step;
    }
    for (;; base += kThreads) {
        const int64_t line = base + tid;
        if (line < lines) {
            const int64_t s = start(line), e = min(max(line_off[line + 1], s), m);
            for (int64_t r = max(s, r0); r < min(e, r0 + R); ++r) {
                l.t0[r - r0] = (int)s;
                l.t1[r - r0] = (int)e;
            }
        }
        if (base + kThreads >= lines || start(base + kThreads) >= r0 + R) break;  // uniform
    }
    __syncthreads();
}

// The vectors of `l` from global memory, 16 bytes per thread (in flight until put).
struct Vectors {
    f32x4 v;
    int at;  // float index from ln2_w, or -1
    template <int R>
    __device__ __forceinline__ void load(int tid, const float* ln2_w, const float* ln2_b, const float* b1, const float* end_w,
                                         const float* end_b, const float* bq) {
        constexpr int Q = D / 4, QH = H / 4;  // 16-byte chunks
        static_assert(4 * Q + QH + kNeckQkvPad / 4 <= kThreads, "one chunk per thread");
        const float* p = nullptr;
        int x = tid;
        if (x < Q) p = ln2_w;
        else if ((x -= Q) < Q) p = ln2_b;
        else if ((x -= Q) < QH) p = b1;
        else if ((x -= QH) < Q) p = end_w;
        else if ((x -= Q) < Q) p = end_b;
        else if ((x -= Q) < kNeckQkvPad / 4) p = bq;
        at = p ? 4 * tid : -1;
        if (p) v = *reinterpret_cast<const f32x4*>(p + 4 * x);
    }
    template <int R>
    __device__ __forceinline__ void put(Lds<R>& l) const {
        if (at >= 0) *reinterpret_cast<f32x4*>(l.ln2_w + at) = v;
    }
};

// Before the first block: the rows' line table to tab, x (CF: transposed) through LN1 and qkv,
// and its rows to xout where the first block cannot read them where they are (xout not null).
// Rows whose pointer is not 16-byte aligned are read value by value.
template <int R, bool CF>
__global__ __launch_bounds__(kThreads, 2) void neck_qkv_kernel(NeckBlockDev k, float scale, const float* __restrict__ x, int64_t m,
                                                               const int64_t* __restrict__ line_off, int64_t lines,
                                                               int64_t line_len, int2* __restrict__ tab,
                                                               float* __restrict__ xout, uint8_t* __restrict__ qkv) {
    extern __shared__ __align__(16) uint8_t raw[];
    Lds<R>& l = *reinterpret_cast<Lds<R>*>(raw);
    constexpr int U = R / 16, P = kThreads / R;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(((tid >> 6) + (blockIdx.x >> 3)) & 7), c = lane & 15,
              g = lane >> 4;
    const int64_t r0 = (int64_t)blockIdx.x * R;
    Weights<4> w[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) w[t].load(k.qkv_f + (size_t)(3 * wave + t) * 4 * kTileHalves, lane);
    const int row = tid / P, part = tid % P;
    const bool aligned = (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    Vectors vec;
    vec.load<R>(tid, k.ln1_w, k.ln1_b, nullptr, nullptr, nullptr, k.qkv_bp);
    if constexpr (!CF) {
        // the rows first: the line table's loads wait behind them
        const int64_t rr = min(r0 + row, m - 1);
        f32x4 v[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int col = unit_col<R>(part, j), cc = col < D ? col : 0;
            const float* p = x + rr * D + cc;
            if (aligned) v[j] = *reinterpret_cast<const f32x4*>(p);
            else v[j] = f32x4{p[0], p[1], p[2], p[3]};
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int col = unit_col<R>(part, j);
            if (col < D) *reinterpret_cast<f32x4*>(l.xs + row * kXS + col) = v[j];
        }
    }
    vec.put(l);
    line_table<R>(l, tid, line_off, lines, line_len, m, r0);
    if (tid < R && r0 + tid < m) tab[r0 + tid] = int2{l.t0[tid], l.t1[tid]};
    if constexpr (CF) {
        CfTile<R> t;
        t.load(l, tid, r0, x);
        t.store(l.xs, tid);
        __syncthreads();
    }
    if (xout) {
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int col = unit_col<R>(part, j);
            if (col < D && r0 + row < m)
                *reinterpret_cast<f32x4*>(xout + (r0 + row) * D + col) =
                    *reinterpret_cast<const f32x4*>(l.xs + row * kXS + col);
        }
    }
    ln_to_operand<R>(l, tid, l.ln2_w, l.ln2_b, k.ln1_eps, ldexpf(1.0f, k.qkv_ey));
    __syncthreads();
    qkv_rows<R>(l, w, k, scale, tid, wave, c, g, r0, m, qkv);
}

// The attention of head `wave` for the R rows from r0, into `as` times 2^attn_ev (the scaling
// of v).  The tile's lines one after another: each line's keys meet every 16-query block that
// holds one of its rows, and a query keeps the result of its own line (so a line's values never
// reach another line's rows).  Per 64 keys: S^T = K Q^T, the running maximum, p =
// 2^15 e^(s - max), O^T += V^T P^T.  The 32 contraction values of a score step are k's high and
// low halves, against (q_hi, q_hi) and then (q_lo, 0): three products in two MFMAs.  A step of
// P^T takes two 16-key tiles u, u + 1: lane (c, g) keys 4 g .. + 3 of each, which are its own
// scores, and v at the same keys.
template <int R>
__device__ __forceinline__ void attention(Lds<R>& l, const NeckBlockDev& k, const uint8_t* __restrict__ qkv, int64_t r0,
                                          int64_t m, int wave, int c, int g) {
    constexpr int RT = R / 16, KT = 4;  // 16-key tiles per step
    const float ec = ldexpf(1.4426950408889634f, -(k.attn_eq + k.attn_ek));
    f16x8 qa[RT], qb[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const uint8_t* q = qkv + min(r0 + 16 * rt + c, m - 1) * kRowBytes + 64 * wave + 16 * (g & 1);
        qa[rt] = *reinterpret_cast<const f16x8*>(q);
        const u32x4 lo = *reinterpret_cast<const u32x4*>(q + 32);
        qb[rt] = __builtin_bit_cast(f16x8, g < 2 ? lo : u32x4{0, 0, 0, 0});
    }
    for (int row = 0; row < R;) {
        const int t0 = __builtin_amdgcn_readfirstlane(l.t0[row]), t1 = __builtin_amdgcn_readfirstlane(l.t1[row]);
        if (t1 <= 0) {  // in no line (or past the batch)
            ++row;
            continue;
        }
        const int end = (int)min((int64_t)R, t1 - r0);  // rows row .. end - 1 of the tile are of this line
        const int T = t1 - t0;
        f32x4 oa[RT];
        float mx[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            oa[rt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            mx[rt] = -INFINITY;
        }
        const uint8_t* kbase = qkv + (int64_t)t0 * kRowBytes + kPart + 64 * wave;
        // keys kb .. kb + 63 (past the line's end: its last key again, masked below): lane
        // (c, g) key 16 u + c at halves 8 g .. + 7, and v's dim c at keys 16 u + 4 g .. + 3
        f16x8 kf[KT];
        u32x4 vf[KT];
        const unsigned koff = c * kRowBytes + 16 * g, voff = 4 * g * kRowBytes + 4 * c;
        auto fetch = [&](int kb) {
            const uint8_t* base = kbase + (int64_t)kb * kRowBytes;
            if (kb + 16 * KT <= T) {  // uniform: lane offsets that stay, from a row the same in every lane
#pragma unroll
                for (int u = 0; u < KT; ++u) {
                    const uint8_t* p = base + 16 * u * kRowBytes;
                    kf[u] = *reinterpret_cast<const f16x8*>(p + koff);
#pragma unroll
                    for (int j = 0; j < 4; ++j) vf[u][j] = *reinterpret_cast<const unsigned*>(p + kPart + j * kRowBytes + voff);
                }
            } else {
                const int last = T - 1 - kb;
#pragma unroll
                for (int u = 0; u < KT; ++u) {
                    kf[u] = *reinterpret_cast<const f16x8*>(base + (unsigned)min(16 * u + c, last) * kRowBytes + 16 * g);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        vf[u][j] = *reinterpret_cast<const unsigned*>(
                            base + kPart + (unsigned)min(16 * u + 4 * g + j, last) * kRowBytes + 4 * c);
                }
            }
        };
        fetch(0);
        for (int kb = 0; kb < T; kb += 16 * KT) {
            f16x8 ka[KT], vh[KT / 2], vl[KT / 2];
#pragma unroll
            for (int u = 0; u < KT; ++u) ka[u] = kf[u];
#pragma unroll
            for (int u = 0; u < KT; u += 2) {
                u32x4 hi, lo;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const unsigned a = vf[u + j / 2][2 * (j & 1)], b = vf[u + j / 2][2 * (j & 1) + 1];
                    hi[j] = pair_lo(a, b);
                    lo[j] = pair_hi(a, b);
                }
                vh[u / 2] = __builtin_bit_cast(f16x8, hi);
                vl[u / 2] = __builtin_bit_cast(f16x8, lo);
            }
            if (kb + 16 * KT < T) fetch(kb + 16 * KT);  // under this step's work
            const int rem = T - kb;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                if (16 * rt >= end || 16 * rt + 16 <= row) continue;  // uniform: no query of this line
                f32x4 sc[KT];
                float bm = -INFINITY;
#pragma unroll
                for (int u = 0; u < KT; ++u) {
                    sc[u] = mfma32(ka[u], qa[rt], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
                    sc[u] = mfma32(ka[u], qb[rt], sc[u]);
                }
#pragma unroll
                for (int u = 0; u < KT; ++u) {
                    if (16 * u + 16 > rem) {  // uniform; the asm keeps it a branch, not selects
                        asm volatile("");
#pragma unroll
                        for (int j = 0; j < 4; ++j) sc[u][j] = (16 * u + 4 * g + j < rem) ? sc[u][j] : -INFINITY;
                    }
                    bm = max3_f32(max3_f32(bm, sc[u][0], sc[u][1]), sc[u][2], sc[u][3]);
                }
                bm = max_over_groups(bm);
                const float nm = max_f32(mx[rt], bm);
                // every step has a key inside the line, so nm is finite
                if (kb > 0) oa[rt] = oa[rt] * __builtin_amdgcn_exp2f((mx[rt] - nm) * ec);
                mx[rt] = nm;
                const float eb = fmaf(-nm, ec, 15.0f);
                f32x4 ob = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int u = 0; u < KT; u += 2) {
                    u32x4 h, r;
#pragma unroll
                    for (int j = 0; j < 8; j += 2) {
                        const f32x4& t = sc[u + j / 4];
                        unsigned hh, rr;
                        split2(__builtin_amdgcn_exp2f(fmaf(t[j & 3], ec, eb)),
                               __builtin_amdgcn_exp2f(fmaf(t[(j & 3) + 1], ec, eb)), hh, rr);
                        h[j / 2] = hh;
                        r[j / 2] = rr;
                    }
                    const f16x8 ph = __builtin_bit_cast(f16x8, h), pl = __builtin_bit_cast(f16x8, r);
                    f32x4& acc = (u & 2) ? ob : oa[rt];
                    acc = mfma32(vh[u / 2], ph, acc);
                    acc = mfma32(vh[u / 2], pl, acc);
                    acc = mfma32(vl[u / 2], ph, acc);
                }
                oa[rt] += ob;
            }
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            if (16 * rt >= end || 16 * rt + 16 <= row) continue;
            const float sum = __shfl(oa[rt][3], 48 + c, 64);  // sum(p) of query c
            const int q = 16 * rt + c;
            f32x4 x;
            u32x2 hi, lo;
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = __fdiv_rn(oa[rt][j], sum);
            x[3] = g == 3 ? 0.0f : x[3];  // the padding dim
            split4(x, hi, lo);
            if (q >= row && q < end) {
                *reinterpret_cast<u32x2*>(&l.as[0][q * kAS + 16 * wave + 4 * g]) = hi;
                *reinterpret_cast<u32x2*>(&l.as[1][q * kAS + 16 * wave + 4 * g]) = lo;
            }
        }
        row = end;
    }
}

// One transformer block for R token rows.  LAST: then the final LayerNorm and the shortcut
// (CF: channels first) into out; otherwise x to xout and the next block's qkv to qkv_next
// (another buffer than qkv, which other workgroups still read).
template <int R, bool LAST, bool CF>
__global__ __launch_bounds__(kThreads, 2) void neck_block_kernel(
    NeckBlockDev k, NeckBlockDev nx, float scale, const float* x, int64_t m, const int2* __restrict__ tab,
    const uint8_t* __restrict__ qkv, float* xout, uint8_t* __restrict__ qkv_next, const float* __restrict__ lnf_w,
    const float* __restrict__ lnf_b, float lnf_eps, const float* __restrict__ shortcut, float* __restrict__ out) {
    extern __shared__ __align__(16) uint8_t raw[];
    Lds<R>& l = *reinterpret_cast<Lds<R>*>(raw);
    constexpr int RT = R / 16, U = R / 16, P = kThreads / R;
    constexpr bool EARLY_Q = R < 64;  // the next qkv weights in registers a phase ahead, where they fit
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(((tid >> 6) + (blockIdx.x >> 3)) & 7), c = lane & 15,
              g = lane >> 4;
    const int64_t r0 = (int64_t)blockIdx.x * R;
    if (tid < R) {
        const int2 t = r0 + tid < m ? tab[r0 + tid] : int2{0, 0};
        l.t0[tid] = t.x;
        l.t1[tid] = t.y;
    }
    // this wave's weights of proj and its residual values: in flight during the attention
    Weights<4> wp[1];
    wp[0].load(k.proj_f + (size_t)wave * 4 * kTileHalves, lane);
    const int col = 16 * wave + 4 * g, cc = col < D ? col : 0;  // this lane's output columns
    f32x4 xv[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) xv[rt] = *reinterpret_cast<const f32x4*>(x + min(r0 + 16 * rt + c, m - 1) * D + cc);
    const f32x4 bp = *reinterpret_cast<const f32x4*>(k.proj_b + cc);
    const f32x4 b2 = *reinterpret_cast<const f32x4*>(k.fc2_b + cc);
    Vectors vec;
    vec.load<R>(tid, k.ln2_w, k.ln2_b, k.fc1_b, LAST ? lnf_w : nx.ln1_w, LAST ? lnf_b : nx.ln1_b, LAST ? nullptr : nx.qkv_bp);
    vec.put(l);
    __syncthreads();
    attention<R>(l, k, qkv, r0, m, wave, c, g);
    Weights<4> w1[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) w1[t].load(k.fc1_f + (size_t)(2 * wave + t) * 4 * kTileHalves, lane);
    __syncthreads();
    {  // x += proj(attention)
        f32x4 acc[1][RT];
        products(wp, l.as[0], l.as[1], kAS, c, g, acc);
        const float s = ldexpf(1.0f, -(k.proj_e + k.attn_ev));
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int e = 0; e < 4; ++e) xv[rt][e] = xv[rt][e] + (acc[0][rt][e] * s + bp[e]);
            if (col < D) *reinterpret_cast<f32x4*>(l.xs + (16 * rt + c) * kXS + col) = xv[rt];
        }
    }
    __syncthreads();
    ln_to_operand<R>(l, tid, l.ln2_w, l.ln2_b, k.ln2_eps, ldexpf(1.0f, k.mlp_ey));
    Weights<8> w2[1];
    w2[0].load(k.fc2_f + (size_t)wave * 8 * kTileHalves, lane);
    __syncthreads();
    {  // the hidden layer
        f32x4 acc[2][RT];
        products(w1, l.as[0], l.as[1], kAS, c, g, acc);
        const float s = ldexpf(1.0f, -(k.mlp_e1 + k.mlp_ey)), sh = ldexpf(1.0f, k.mlp_eh);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int unit = 16 * (2 * wave + t) + 4 * g;
            const f32x4 b1 = *reinterpret_cast<const f32x4*>(l.b1 + (unit < H ? unit : 0));
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                f32x4 z;
                u32x2 hi, lo;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    z[e] = swish_fast(acc[t][rt][e] * s + b1[e]) * sh;
                    z[e] = unit < H ? z[e] : 0.0f;
                }
                split4(z, hi, lo);
                *reinterpret_cast<u32x2*>(&l.hs[0][(16 * rt + c) * kHS + unit]) = hi;
                *reinterpret_cast<u32x2*>(&l.hs[1][(16 * rt + c) * kHS + unit]) = lo;
            }
        }
    }
    // what the end needs: the next block's qkv weights, or the shortcut
    Weights<4> wq[3];
    CfTile<R> sc_cf;
    f32x4 sc_rows[U];
    const int row = tid / P, part = tid % P;
    auto load_q = [&] {
#pragma unroll
        for (int t = 0; t < 3; ++t) wq[t].load(nx.qkv_f + (size_t)(3 * wave + t) * 4 * kTileHalves, lane);
    };
    if constexpr (!LAST) {
        if (EARLY_Q) load_q();
    } else if constexpr (CF) {
        sc_cf.load(l, tid, r0, shortcut);
    } else {
        const float* p = shortcut + min(r0 + row, m - 1) * D;
        const bool aligned = (reinterpret_cast<uintptr_t>(shortcut) & 15) == 0;
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int sc = unit_col<R>(part, j) < D ? unit_col<R>(part, j) : 0;
            if (aligned) sc_rows[j] = *reinterpret_cast<const f32x4*>(p + sc);
            else sc_rows[j] = f32x4{p[sc], p[sc + 1], p[sc + 2], p[sc + 3]};
        }
    }
    __syncthreads();
    {  // x += fc2(hidden)
        f32x4 acc[1][RT];
        products(w2, l.hs[0], l.hs[1], kHS, c, g, acc);
        const float s = ldexpf(1.0f, -(k.mlp_eh + k.mlp_e2));
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int e = 0; e < 4; ++e) xv[rt][e] = xv[rt][e] + (acc[0][rt][e] * s + b2[e]);
            if (col < D) {
                *reinterpret_cast<f32x4*>(l.xs + (16 * rt + c) * kXS + col) = xv[rt];
                const int64_t r = r0 + 16 * rt + c;
                if (!LAST && r < m) *reinterpret_cast<f32x4*>(xout + r * D + col) = xv[rt];
            }
        }
    }
    __syncthreads();
    if constexpr (!LAST) {
        ln_to_operand<R>(l, tid, l.end_w, l.end_b, nx.ln1_eps, ldexpf(1.0f, nx.qkv_ey));
        if (!EARLY_Q) load_q();
        __syncthreads();
        qkv_rows<R>(l, wq, nx, scale, tid, wave, c, g, r0, m, qkv_next);
    } else {
        float* sct = reinterpret_cast<float*>(l.hs);  // the hidden rows are read
        static_assert(sizeof(l.hs) >= sizeof(l.xs), "the shortcut tile fits the hidden rows");
        if constexpr (CF) {
            sc_cf.store(sct, tid);
            __syncthreads();
        }
        float v[U][4];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int oc = unit_col<R>(part, j);
            const f32x4 t = *reinterpret_cast<const f32x4*>(l.xs + row * kXS + (oc < D ? oc : 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) v[j][e] = oc < D ? t[e] : 0.0f;
        }
        layer_norm<R>(v, part, lnf_eps);
        const bool aligned = (reinterpret_cast<uintptr_t>(out) & 15) == 0;
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int oc = unit_col<R>(part, j);
            if (oc >= D || r0 + row >= m) continue;
            const f32x4 lw = *reinterpret_cast<const f32x4*>(l.end_w + oc), lb = *reinterpret_cast<const f32x4*>(l.end_b + oc);
            const f32x4 s = CF ? *reinterpret_cast<const f32x4*>(sct + row * kXS + oc) : sc_rows[j];
            f32x4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = fmaf(v[j][e], lw[e], lb[e]) + s[e];
            float* p = out + (r0 + row) * D + oc;
            if (aligned) {
                *reinterpret_cast<f32x4*>(p) = o;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) p[e] = o[e];
            }
        }
    }
}

// ---------------------------------------------------------------- planes, at creation
// (On the host, without half conversions in hardware, these took 3 ms of a tail's creation.)
__device__ __forceinline__ void put_halves(float v, uint16_t* hi, uint16_t* lo) {
    const _Float16 h = (_Float16)v;
    *hi = __builtin_bit_cast(uint16_t, h);
    *lo = __builtin_bit_cast(uint16_t, (_Float16)(v - (float)h));
}
// The model's index of index c padded per head to 16 (qkv's columns, proj's contraction), or one
// past any.
__device__ __forceinline__ int unpad(int c) {
    const int d = c % 16;
    return d < kNeckHeadDim ? c / 128 * D + c % 128 / 16 * kNeckHeadDim + d : INT32_MAX;
}

// The planes in operand order: thread x the value (tile, step, lane, j) of W [K][N] times mul.
// PAD 1: W's columns padded per head (qkv); 2: its rows (proj).
template <int PAD>
__global__ __launch_bounds__(256) void neck_fragments_kernel(const float* __restrict__ w, int K, int N, int steps, float mul,
                                                             uint16_t* __restrict__ out) {
    const int x = blockIdx.x * 256 + threadIdx.x, j = x & 7, lane = (x >> 3) & 63, ts = x >> 9;
    int col = 16 * (ts / steps) + lane % 16, k = 32 * (ts % steps) + 8 * (lane / 16) + j;
    if (PAD == 1) col = unpad(col);
    if (PAD == 2) k = unpad(k);
    uint16_t* f = out + (size_t)ts * kTileHalves + lane * 8 + j;
    put_halves(col < N && k < K ? w[k * N + col] * mul : 0.0f, f, f + 512);
}

// The planes [2][columns][128] of the separate kernels' GEMMs, a thread per value; PAD as above.
template <int PAD>
__global__ __launch_bounds__(256) void neck_columns_kernel(const float* __restrict__ w, int K, int N, int columns,
                                                           uint16_t* __restrict__ out) {
    const int x = blockIdx.x * 256 + threadIdx.x;
    if (x >= columns * 128) return;
    const int col = PAD == 1 ? unpad(x / 128) : x / 128, k = PAD == 2 ? unpad(x % 128) : x % 128;
    put_halves(col < N && k < K ? w[k * N + col] : 0.0f, out + x, out + columns * 128 + x);
}

// The staging order of the separate kernels' MLP (NeckBlockDev::mlp_h): thread x entry x % 4096 of
// tile x / 4096, of fc1's part and of fc2's.  fc2's contraction position 32 T + 16 q + 8 h + e
// holds hidden unit 32 T + 16 q + 8 (e / 4) + 4 h + e % 4, the order in which fc1's transposed
// MFMA output leaves the hidden values in registers.
__global__ __launch_bounds__(256) void neck_mlp_tiles_kernel(const float* __restrict__ fc1, const float* __restrict__ fc2,
                                                             float mul1, float mul2, uint16_t* __restrict__ out) {
    const int x = blockIdx.x * 256 + threadIdx.x, T = x >> 12, n = x & 4095, e = n & 7;
    uint16_t* t = out + (size_t)T * 16384;
    {  // [plane][chunk (16)][unit (32)][8]
        const int unit = 32 * T + ((n >> 3) & 31), k = 8 * (n >> 8) + e;
        put_halves(unit < H && k < D ? fc1[k * H + unit] * mul1 : 0.0f, t + n, t + 4096 + n);
    }
    {  // [plane][chunk (4)][column (128)][8]
        const int col = (n >> 3) & 127, c = n >> 10;
        const int unit = 32 * T + 16 * (c >> 1) + 8 * (e >> 2) + 4 * (c & 1) + (e & 3);
        put_halves(unit < H && col < D ? fc2[unit * D + col] * mul2 : 0.0f, t + 8192 + n, t + 12288 + n);
    }
}

// Whether two buffers of m rows share memory.
bool overlap(const float* a, const float* b, int64_t m) {
    const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b), n = (uintptr_t)m * D * sizeof(float);
    return x < y + n && y < x + n;
}

template <int R>
int go(const NeckDev& nk, const float* x_in, const float* shortcut, int64_t m, const int64_t* line_off, int64_t lines,
       int64_t line_len, bool cf, float* out, float* ws, hipStream_t st, const NeckMark& mark) {
    const unsigned grid = (unsigned)((m + R - 1) / R);
    float* x = ws;
    uint8_t* qkv[2] = {reinterpret_cast<uint8_t*>(ws + m * D), reinterpret_cast<uint8_t*>(ws + m * (D + kNeckQkvPad))};
    int2* tab = reinterpret_cast<int2*>(ws + m * (D + 2 * kNeckQkvPad));
    static_assert(D + 2 * kNeckQkvPad + 2 <= kNeckWsFloatsPerRow, "x, two qkv buffers and the line table in the workspace");
    // the residual of the first block: the input rows when they can be read as they are (row by
    // row while out is written, if the first block is the last)
    const bool keep = cf || (reinterpret_cast<uintptr_t>(x_in) & 15) || (nk.blocks == 1 && x_in != out && overlap(x_in, out, m));
    (cf ? neck_qkv_kernel<R, true> : neck_qkv_kernel<R, false>)<<<grid, kThreads, sizeof(Lds<R>), st>>>(
        nk.block[0], nk.scale, x_in, m, line_off, lines, line_len, tab, keep ? x : nullptr, qkv[0]);
    PPOCR_HIP(hipGetLastError());
    if (int e = mark("ln1_qkv")) return e;
    const float* xr = keep ? x : x_in;
    for (int b = 0; b < nk.blocks; ++b, xr = x) {
        const bool last = b + 1 == nk.blocks;
        if (last && cf && overlap(shortcut, out, m)) {
            // a workgroup's rows of out lie over other workgroups' part of the shortcut: its rows
            // first, into the qkv buffer that no kernel reads any more
            float* rows = reinterpret_cast<float*>(qkv[(b + 1) & 1]);
            if (int e = launch_cf_rows(shortcut, m, line_off, lines, line_len, rows, st)) return e;
            if (int e = mark("channels_first_to_rows")) return e;
            shortcut = rows;
            cf = false;
        }
        auto* kern = !last ? neck_block_kernel<R, false, false>
                     : cf  ? neck_block_kernel<R, true, true>
                           : neck_block_kernel<R, true, false>;
        kern<<<grid, kThreads, sizeof(Lds<R>), st>>>(nk.block[b], nk.block[last ? b : b + 1], nk.scale, xr, m, tab,
                                                    qkv[b & 1], x, qkv[(b + 1) & 1], nk.lnf_w, nk.lnf_b, nk.lnf_eps,
                                                    shortcut, out);
        PPOCR_HIP(hipGetLastError());
        if (int e = mark(last ? "block_final_ln_shortcut" : "block_ln1_qkv")) return e;
    }
    return PPOCR_OK;
}

}  // namespace

int launch_neck_planes(const NeckBlockDev& k, hipStream_t st) {
    auto mut = [](const uint16_t* p) { return const_cast<uint16_t*>(p); };
    auto mul = [](int e) { return std::ldexp(1.0f, e); };
    neck_columns_kernel<1><<<kNeckQkvPad / 2, 256, 0, st>>>(k.qkv_w, D, 3 * D, kNeckQkvPad, mut(k.qkv_h));
    neck_columns_kernel<2><<<D / 2, 256, 0, st>>>(k.proj_w, D, D, D, mut(k.proj_h));
    neck_mlp_tiles_kernel<<<8 * 16, 256, 0, st>>>(k.fc1_w, k.fc2_w, mul(k.mlp_e1), mul(k.mlp_e2), mut(k.mlp_h));
    neck_fragments_kernel<1><<<24 * 4 * 2, 256, 0, st>>>(k.qkv_w, D, 3 * D, 4, mul(k.qkv_e), mut(k.qkv_f));
    neck_fragments_kernel<2><<<8 * 4 * 2, 256, 0, st>>>(k.proj_w, D, D, 4, mul(k.proj_e), mut(k.proj_f));
    neck_fragments_kernel<0><<<16 * 4 * 2, 256, 0, st>>>(k.fc1_w, D, H, 4, mul(k.mlp_e1), mut(k.fc1_f));
    neck_fragments_kernel<0><<<8 * 8 * 2, 256, 0, st>>>(k.fc2_w, H, D, 8, mul(k.mlp_e2), mut(k.fc2_f));
    PPOCR_HIP(hipGetLastError());
    return PPOCR_OK;
}

int launch_neck_fused(const NeckDev& nk, const float* x_in, const float* shortcut, int64_t m, const int64_t* line_off,
                      int64_t lines, int64_t line_len, bool cf, float* out, float* ws, hipStream_t st,
                      const NeckMark& mark) {
    if (m > kNeckFusedRows) return fail(PPOCR_ERR_INVALID_ARG, "RecNeckHip: too many rows");
    // the smallest tile whose grid is at most a workgroup per CU: fewer rows, a shorter chain.
    // Measured (lines of 128, rows first): 128 rows 30 / 39 / 60 us with tiles of 16 / 32 / 64
    // rows, 4096: 40 / 45 / 66, 8192: 69 / 51 / 68, 16384: 128 / 89 / 76.  A tile's lines are
    // taken one after another, so lines of a row or two make a chain of it: 64 lines of one row 70
    // us, 4096 of one row 77, 8194 of one row 283, 2049 of four 111; the separate kernels, a
    // workgroup per line and head, take 69, 231, 396 and 162.  One line of 1000 rows 66, of 16384
    // rows 1415; the separate kernels 461 and 105410
    auto f = m <= 16 * 256 ? go<16> : m <= 32 * 256 ? go<32> : go<64>;
    return f(nk, x_in, shortcut, m, line_off, lines, line_len, cf, out, ws, st, mark);
}

}  // namespace ppocr
