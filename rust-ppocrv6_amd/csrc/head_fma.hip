// fp32 kernels of MatMul.12 (PPOCR_MODE_FP32_FMA): the accuracy anchor for the split kernels.
// Same contraction as compute_quantized_b_cols_avx2 (src/ops/matmul.rs:1338-1443) and
// transposed_b_tile_fma (src/ops/matmul.rs:1025-1087): fp32 products of the activation
// and the (exactly dequantised) weight, fp32 accumulation, then (sum * scale) + bias.
//
// The products run on v_mfma_f32_32x32x2_f32, which multiplies and sums in fp32 (154 TFLOP/s
// from registers on this chip, against 78 for the vector ALU's v_fma_f32 without packing).  A
// workgroup's tile is 128 rows x 128 classes: wave w owns rows 32 w .. + 31 and all 128 classes
// (four 32x32 accumulators), so a softmax statistic never crosses waves.  k passes through LDS
// in chunks of 16, two buffers (41 KB, so three workgroups per CU for the logits and the
// probabilities: chunks of 32 and two per CU took 377 us where this takes 363; the statistics
// and the rescues, with more registers, run two per CU); within 8 values of k lane half h holds k = 4 h .. 4 h + 3,
// one 16-byte LDS read for four MFMA steps (step e multiplies k = e and k = 4 + e), so a wave
// reads 5 KB of LDS per 16 MFMAs.
// Measured, 7680 x 120 x 18710 (an FP32 head's logits, 34.5 GFLOP, 575 MB written): 802 us with
// the vector ALU, 363 us here (95 TFLOP/s; 317 with no logits stored; matrix cores busy 68% of
// the time at 2.2 GHz).  The largest error against 64 bits is the same for both.
#include <algorithm>

#include "kernels.hpp"

namespace ppocr {

namespace {
constexpr int BM = kFmaRowsPerBlock, BN = kFmaCols, KC = 16;
constexpr int64_t kFmaRescueSlots = 128;  // row-block slots of a gather-mode (rescue) launch
// LDS row stride in floats: whole 16-byte chunks, an odd number of them, so 8 lanes reading
// 16 bytes each of 8 consecutive rows touch all 32 banks
constexpr int LST = KC + 4;
constexpr size_t kFmaLdsFloats = 2 * (size_t)(BM + BN) * LST;
static_assert(BM == 128 && BN == 128 && KC == 16, "the thread mappings below");

// Where the operands may be read 4 values of k at a time: k a multiple of 4, the row starts
// aligned (16 bytes for floats, 4 for int8), and 128 rows within 32-bit offsets.
constexpr int64_t kOffsetK = 1 << 24;
bool vec_rows(const float* p, int64_t k) { return k % 4 == 0 && k <= kOffsetK && reinterpret_cast<uintptr_t>(p) % 16 == 0; }
bool vec_rows(const int8_t* p, int64_t k) { return k % 4 == 0 && k <= kOffsetK && reinterpret_cast<uintptr_t>(p) % 4 == 0; }
// Most classes whose output rows r and r + 4 are addressed by 32-bit offsets.
constexpr int kOffsetClasses = 1 << 29;

// Row of slot j: contiguous rows, or (GATHER) an entry of the precision guard's row list of
// another kernel's pass (checked, not trusted: an entry outside [0, m) is skipped); -1: none.
template <bool GATHER>
__device__ __forceinline__ int64_t row_of(int64_t j, int64_t m, const int* list, int count) {
    if constexpr (GATHER) {
        const int64_t r = j < count ? (int64_t)list[j] : -1;
        return r >= 0 && r < m ? r : -1;
    }
    return j < m ? j : -1;
}

// The writer's tiles (EPI_LOGITS, EPI_PROBS over contiguous rows): workgroup b takes slot
// b % slots (workgroups go to the XCDs in turn, so with 8 slots a slot is an XCD), whose
// classes are per_slot consecutive tiles, and in it the tiles of one row block after another.
struct TileOrder {
    unsigned slots, per_slot;
};

// cpc: classes per vocabulary chunk; chunk c covers classes [c * cpc, (c + 1) * cpc) (the
// writer: the whole vocabulary).  Q: int8 weights.  VEC: both operands by 4 values of k (rows
// layout only).  line_len > 0: channels-first activations [lines][k][line_len].
template <int EPI, bool GATHER, bool Q, bool VEC>
__global__ __launch_bounds__(256, EPI == EPI_STATS || GATHER ? 2 : 3) void head_fma_kernel(
    const int8_t* __restrict__ q, const float* __restrict__ w, const float* __restrict__ scale,
    const float* __restrict__ bias, const float* __restrict__ a, int64_t m, int n, int k, int cpc,
    float* __restrict__ out, const float* __restrict__ row_max, const float* __restrict__ row_inv,
    Partial* __restrict__ part, int64_t line_len,
    const unsigned long long* __restrict__ guard_header, const int* __restrict__ guard_rows, unsigned guard_epoch,
    int guard_cap, TileOrder order) {
    extern __shared__ __align__(16) float lf[];  // two buffers of [BM + BN][LST]: rows, then classes
    __shared__ int64_t s_row[BM];                // the block's rows (-1: none)
    __shared__ __align__(16) float s_max[BM], s_inv[BM];
    __shared__ __align__(16) float s_const[4][2][BN];  // by tile, four in turn: scale, bias
    constexpr bool WRITER = EPI != EPI_STATS && !GATHER;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 31,
              h = lane >> 5;
    const int nk = (k + KC - 1) / KC;

    // Rows m0 .. m0 + BM - 1 (slots of the list with GATHER) x the tiles of classes from c0 to
    // c1, c0 < c1.
    auto block = [&](int64_t m0, int c0, int c1, int chunk, int count) {
        __syncthreads();  // the previous block is done with the tables
        if (tid < BM) {
            const int64_t r = row_of<GATHER>(m0 + tid, m, guard_rows, count);
            s_row[tid] = r;
            if (EPI == EPI_PROBS) {
                s_max[tid] = r >= 0 ? row_max[r] : 0.0f;
                s_inv[tid] = r >= 0 ? row_inv[r] : 0.0f;
            }
        }
        __syncthreads();
        // VEC: chunk x of the tile of classes from n0 into registers, rows and classes tid / 4 +
        // 64 it at k = 4 (tid % 4), and from there into an LDS buffer.  The addresses are a row's
        // and a tile's start, the same in every lane, plus 32-bit lane offsets that stay over a
        // tile: fp32 MFMAs and vector instructions do not overlap on a SIMD here, so each vector
        // instruction of the loop costs its cycles.  A row or class that is not there reads
        // another one of the batch (its results are never stored, and each result depends on its
        // own row and class alone).
        const int kq = 4 * (tid & 3), kq_last = (nk - 1) * KC + kq < k ? kq : 0;
        // Otherwise value by value: k = tid % 16 of rows and classes tid / 16 + 16 it (channels
        // first: row tid % 128, k = tid / 128 + 2 it, so neighbouring threads take neighbouring
        // steps), into the same registers and a step later into the LDS buffer.  (Loaded and
        // stored in one step, so that every step waited for memory: the statistics of 512 rows
        // of an FP32 head of 18710 x 121 131 us, 82 so, 7680 rows 928 and 720; the vector ALU's
        // kernel, more waves at once, 106 and 1125.)
        const int64_t any = m0 < m ? m0 : 0;
        int64_t arow[2];
        int64_t cf_row = 0;  // channels first: where this thread's row starts, at k = 0
        unsigned woff[2] = {0, 0};
        if constexpr (VEC) {
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                const int64_t row = s_row[(tid >> 2) + 64 * it];
                arow[it] = (row >= 0 ? row : any) * k;
            }
        } else if (line_len > 0) {
            const int64_t row = s_row[tid & (BM - 1)], r = row >= 0 ? row : any;
            cf_row = r / line_len * k * line_len + r % line_len;
        }
        f32x4 ca[2], cw[2];
        auto load = [&](int n0, int x) {
            if constexpr (!VEC) {
                int t = tid;
                asm volatile("" : "+v"(t));  // addresses from here on: kept over the loop they would spill
                const int kl = k - 1, kk = min(x * KC + (t & 15), kl);
                if (line_len > 0) {
                    const float* p = a + cf_row;
#pragma unroll
                    for (int it = 0; it < 8; ++it) ca[it >> 2][it & 3] = p[min(x * KC + (t >> 7) + 2 * it, kl) * line_len];
                } else {
#pragma unroll
                    for (int it = 0; it < 8; ++it) {
                        const int64_t row = s_row[(t >> 4) + 16 * it];
                        ca[it >> 2][it & 3] = a[(row >= 0 ? row : any) * k + kk];
                    }
                }
#pragma unroll
                for (int it = 0; it < 8; ++it) {
                    const int64_t e = (int64_t)min(n0 + (t >> 4) + 16 * it, n - 1) * k + kk;
                    if constexpr (Q) cw[it >> 2][it & 3] = __int_as_float((int)q[e]);
                    else cw[it >> 2][it & 3] = w[e];
                }
                return;
            }
            if (x == 0) {
#pragma unroll
                for (int it = 0; it < 2; ++it) woff[it] = (unsigned)min((tid >> 2) + 64 * it, n - 1 - n0) * (unsigned)k;
            }
            const unsigned kk = x + 1 == nk ? kq_last : kq;
            const float* ab = a + x * KC;
            const int64_t wb = (int64_t)n0 * k + x * KC;
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                ca[it] = *reinterpret_cast<const f32x4*>(ab + arow[it] + kk);
                if constexpr (Q) cw[it][0] = __int_as_float(*reinterpret_cast<const int*>(q + wb + (woff[it] + kk)));
                else cw[it] = *reinterpret_cast<const f32x4*>(w + wb + (woff[it] + kk));
            }
        };
        auto put = [&](int buf, int x) {
            if constexpr (!VEC) {
                int t = tid;
                asm volatile("" : "+v"(t));
                float* as = lf + (size_t)buf * (BM + BN) * LST;
                const int o = (t >> 4) * LST + (t & 15), oc = (t & (BM - 1)) * LST + (t >> 7);
                const bool in = x * KC + (t & 15) < k;  // past k: zeros
#pragma unroll
                for (int it = 0; it < 8; ++it) {
                    const float v = ca[it >> 2][it & 3], u = cw[it >> 2][it & 3];
                    if (line_len > 0) as[oc + 2 * it] = x * KC + (t >> 7) + 2 * it < k ? v : 0.0f;
                    else as[o + 16 * it * LST] = in ? v : 0.0f;
                    as[BM * LST + o + 16 * it * LST] = in ? (Q ? (float)__float_as_int(u) : u) : 0.0f;
                }
                return;
            }
            float* as = lf + (size_t)buf * (BM + BN) * LST + (tid >> 2) * LST + kq;
            if constexpr (Q) {
#pragma unroll
                for (int it = 0; it < 2; ++it) {
                    const int v = __float_as_int(cw[it][0]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) cw[it][j] = (float)(int8_t)(v >> (8 * j));
                }
            }
            // past k only where 4 of 8 values are multiplied (the other groups are skipped): zeros
            if (k % 8 != 0 && x + 1 == nk && x * KC + kq >= k) ca[0] = ca[1] = cw[0] = cw[1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                *reinterpret_cast<f32x4*>(as + 64 * it * LST) = ca[it];
                *reinterpret_cast<f32x4*>(as + (BM + 64 * it) * LST) = cw[it];
            }
        };
        // the constants of the tile from n0 (zeros past the chunk): loaded by the first 128
        // threads, stored for the epilogue of that tile
        float kc_s = 0.0f, kc_b = 0.0f;
        auto load_const = [&](int n0) {
            if (tid < BN) {
                const int c = min(n0 + tid, n - 1);
                kc_s = scale[c];
                kc_b = bias[c];
            }
        };
        auto put_const = [&](int par) {
            if (tid < BN) {
                s_const[par][0][tid] = kc_s;
                s_const[par][1][tid] = kc_b;
            }
        };

        RowStat st{-INFINITY, 0.0f, 0.0f, 0};  // EPI_STATS: row 32 wave + i, this half's classes
        bool refzero = true;
        f32x16 acc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = f32x16{};
        // A step is a chunk of k of a tile, the tiles one after another.  Step s first puts step
        // s + 1's operands (loaded into registers a step ago) into the other buffer and reads its
        // own second 8 values of k; its first 8, read in step s - 1, are multiplied meanwhile.
        // After the barrier it loads step s + 2 and reads the first 8 values of step s + 1 under
        // its second products: no product waits for an LDS read issued just before it.
        struct Step {
            int n0, x;
        };
        auto next = [&](Step q_) {  // past the last tile n0 stays at or past c1
            return q_.x + 1 < nk ? Step{q_.n0, q_.x + 1} : Step{q_.n0 < c1 ? q_.n0 + BN : q_.n0, 0};
        };
        struct Frag {
            f32x4 a, w[4];
        };
        auto frag = [&](int buf, int g, Frag& f) {
            const float* as = lf + (size_t)buf * (BM + BN) * LST + (32 * wave + i) * LST + 4 * h + 8 * g;
            const float* ws = lf + ((size_t)buf * (BM + BN) + BM + i) * LST + 4 * h + 8 * g;
            f.a = *reinterpret_cast<const f32x4*>(as);
#pragma unroll
            for (int t = 0; t < 4; ++t) f.w[t] = *reinterpret_cast<const f32x4*>(ws + 32 * t * LST);
        };
        auto product = [&](const Frag& f, int e, int t, const f32x16& c) {
            return EPI == EPI_STATS ? __builtin_amdgcn_mfma_f32_32x32x2f32(f.w[t][e], f.a[e], c, 0, 0, 0)
                                    : __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[e], f.w[t][e], c, 0, 0, 0);
        };
        auto products = [&](const Frag& f, int e0) {
#pragma unroll
            for (int e = e0; e < 4; ++e)
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[t] = product(f, e, t, acc[t]);
        };
        Step s0{c0, 0}, s1 = next(s0);
        load(c0, 0);
        put(0, 0);
        if (s1.n0 < c1) load(s1.n0, s1.x);
        load_const(c0);
        put_const(0);
        if (nk == 1 && s1.n0 < c1) load_const(s1.n0);
        __syncthreads();
        Frag f0, f1;
        frag(0, 0, f0);
        int buf = 0, par = 0;
        for (int n0 = c0; n0 < c1; n0 += BN, par = (par + 1) & 3) {
            for (int x = 0; x < nk; ++x) {
                const bool more = s1.n0 < c1;
                if (more) {
                    put(buf ^ 1, s1.x);
                    // the constants of four tiles: a slower wave may still read the last tile's
                    if (s1.x == 0) put_const((par + 1) & 3);
                }
                frag(buf, 1, f1);
                __builtin_amdgcn_sched_barrier(0);
                if (x == 0) {  // a tile's first products start from zero
#pragma unroll
                    for (int t = 0; t < 4; ++t) acc[t] = product(f0, 0, t, f32x16{});
                } else {
#pragma unroll
                    for (int t = 0; t < 4; ++t) acc[t] = product(f0, 0, t, acc[t]);
                }
                products(f0, 1);
                __builtin_amdgcn_sched_barrier(0);
                __syncthreads();
                const Step s2 = next(s1);
                if (s2.n0 < c1) {
                    load(s2.n0, s2.x);
                    if (s2.x == 0) load_const(s2.n0);
                }
                buf ^= 1;
                if (more) frag(buf, 0, f0);
                __builtin_amdgcn_sched_barrier(0);
                if (k - x * KC > 8) products(f1, 0);  // otherwise the rest of the chunk is zeros
                s1 = s2;
            }
            const float* s_sc = s_const[par][0];
            const float* s_bi = s_const[par][1];

            if (EPI == EPI_STATS) {
                // MFMA rows are classes: this lane holds row 32 wave + i at classes
                // n0 + 32 t + 8 (r / 4) + 4 h + r % 4, in increasing order
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    float tv[16], tmax = -INFINITY;
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int c = 32 * t + 8 * (r >> 2) + 4 * h + (r & 3);
                        tv[r] = n0 + c < c1 ? fmaf(acc[t][r], s_sc[c] * kLog2e, s_bi[c] * kLog2e) : -INFINITY;
                        tmax = fmaxf(tmax, tv[r]);
                    }
                    if (tmax > st.best) {
                        // the first of this lane's classes holding the maximum
                        int rr = 15;
#pragma unroll
                        for (int r = 14; r >= 0; --r) rr = (tv[r] == tmax) ? r : rr;
                        st.best = tmax;
                        st.idx = n0 + 32 * t + 8 * (rr >> 2) + 4 * h + (rr & 3);
                    }
                    const bool shift = st.best != -INFINITY &&
                                       (st.best > st.ref + 64.0f || st.best < st.ref - 64.0f);
                    if (__any(shift)) {
                        if (shift) {
                            st.sum *= __builtin_amdgcn_exp2f(st.ref - st.best);
                            st.ref = st.best;
                        }
                        refzero = false;
                    }
                    float e = 0.0f;
#pragma unroll
                    for (int r = 0; r < 16; ++r) e += __builtin_amdgcn_exp2f(refzero ? tv[r] : tv[r] - st.ref);
                    st.sum += e;
                }
            } else {
                // MFMA columns are classes: this lane holds class n0 + 32 t + i of rows
                // 32 wave + 8 (r / 4) + 4 h + r % 4
                float csc[4], cbi[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    csc[t] = s_sc[32 * t + i];
                    cbi[t] = s_bi[32 * t + i];
                }
                auto value = [&](int r, int lr, int t) {
                    if (EPI == EPI_LOGITS) return __fadd_rn(__fmul_rn(acc[t][r], csc[t]), cbi[t]);
                    return __builtin_amdgcn_exp2f(fmaf(acc[t][r], csc[t] * kLog2e, cbi[t] * kLog2e) - s_max[lr]) *
                           s_inv[lr];
                };
                // a whole tile: one 32-bit lane offset (4 h rows and i classes) from a row address that is the same in every lane
                const bool all = !GATHER && n <= kOffsetClasses && n0 + BN <= c1 && m0 + BM <= m;
                unsigned lo = (unsigned)(4 * h) * (unsigned)n + (unsigned)i;
                asm volatile("" : "+v"(lo));  // not before the products, where it would hold registers
                float* obase = out + (m0 + 32 * wave) * n + n0;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int lr = 32 * wave + 8 * (r >> 2) + 4 * h + (r & 3);
                    if (all) {
                        // no branch per value: at a branch the compiler waits for every store
                        // in flight
                        float* o = obase + (int64_t)(8 * (r >> 2) + (r & 3)) * n;
#pragma unroll
                        for (int t = 0; t < 4; ++t) o[lo + 32 * t] = value(r, lr, t);
                    } else {
                        const int64_t row = s_row[lr];
                        if (row < 0) continue;
#pragma unroll
                        for (int t = 0; t < 4; ++t)
                            if (n0 + 32 * t + i < c1) out[row * n + n0 + 32 * t + i] = value(r, lr, t);
                    }
                }
            }
        }

        if (EPI == EPI_STATS) {
            // the two halves of a row's classes (ties keep the lower class)
            RowStat other;
            other.best = __shfl_xor(st.best, 32, 64);
            other.sum = __shfl_xor(st.sum, 32, 64);
            other.ref = __shfl_xor(st.ref, 32, 64);
            other.idx = __shfl_xor(st.idx, 32, 64);
            st = stat_merge(st, other);
            const int64_t row = s_row[32 * wave + i];
            if (h == 0 && row >= 0) part[(int64_t)chunk * m + row] = Partial{st.best, st.sum, st.idx};
        }
    };

    if constexpr (WRITER) {
        const unsigned slot = blockIdx.x % order.slots, p = blockIdx.x / order.slots;
        const int64_t c0 = ((int64_t)slot * order.per_slot + p % order.per_slot) * BN;
        if (c0 < n) block((int64_t)(p / order.per_slot) * BM, (int)c0, (int)min(c0 + BN, (int64_t)n), 0, 0);
    } else {
        int count = 0;
        if constexpr (GATHER) {
            const unsigned long long hv = *guard_header;
            const unsigned c = (unsigned)(hv >> 32) == guard_epoch ? (unsigned)hv : 0u;
            count = c < (unsigned)guard_cap ? (int)c : guard_cap;
        }
        const int64_t nrows = GATHER ? (int64_t)count : m;
        const int chunk = blockIdx.x, c0 = (int)min((int64_t)chunk * cpc, (int64_t)n), c1 = min(n, n - c0 < cpc ? n : c0 + cpc);
        for (int64_t m0 = (int64_t)blockIdx.y * BM; m0 < nrows; m0 += (int64_t)gridDim.y * BM) {
            if (c0 < c1) {
                block(m0, c0, c1, chunk, count);
            } else if (EPI == EPI_STATS && tid < BM) {  // a chunk without classes
                const int64_t r = row_of<GATHER>(m0 + tid, m, guard_rows, count);
                if (r >= 0) part[(int64_t)chunk * m + r] = Partial{-INFINITY, 0.0f, 0};
            }
        }
    }
}

int check_fma_args(int64_t m, int64_t n, int64_t k) {
    if (n > 0x7fffffff - BN || k > 0x7fffffff - KC) return fail(PPOCR_ERR_INVALID_ARG, "MatMulQuantizedB: shape too large");
    if ((m + BM - 1) / BM > 65535) return fail(PPOCR_ERR_INVALID_ARG, "MatMulQuantizedB: m too large for the fp32 path");
    return PPOCR_OK;
}

// Every launch: grid.x vocabulary chunks of cpc classes, grid.y row-block slots.
template <int EPI, bool GATHER>
int fma_go(dim3 grid, const FmaWeights& fw, const float* a, int64_t m, int64_t n, int64_t k, int cpc, float* out,
           const float* row_max, const float* row_inv, Partial* part, int64_t line_len, const Guard* guard,
           hipStream_t st, TileOrder order = {1, 1}) {
    const bool vec = line_len == 0 && vec_rows(a, k) && (fw.q ? vec_rows(fw.q, k) : vec_rows(fw.w, k));
    auto go = [&](auto kern) {
        kern<<<grid, 256, kFmaLdsFloats * sizeof(float), st>>>(
            fw.q, fw.w, fw.scale, fw.bias, a, m, (int)n, (int)k, cpc, out, row_max, row_inv, part, line_len,
            guard ? guard->header : nullptr, guard ? guard->rows : nullptr, guard ? guard->epoch : 0u,
            guard ? guard->capacity : 0, order);
    };
    if (fw.q) vec ? go(head_fma_kernel<EPI, GATHER, true, true>) : go(head_fma_kernel<EPI, GATHER, true, false>);
    else vec ? go(head_fma_kernel<EPI, GATHER, false, true>) : go(head_fma_kernel<EPI, GATHER, false, false>);
    PPOCR_HIP(hipGetLastError());
    return PPOCR_OK;
}
}  // namespace

// The writer over contiguous rows.  From 64 tiles of classes up every XCD takes an eighth of
// the vocabulary: its slice of the weights (1.2 MB of an FP32 head) stays in its own L2, and
// the tiles of one row are written through one L2, where the halves of the cache lines that
// the tiles share (rows start at any 4-byte boundary) meet.
template <int EPI>
int writer_go(const FmaWeights& fw, const float* a, int64_t m, int64_t n, int64_t k, const float* row_max,
              const float* row_inv, float* out, hipStream_t st) {
    if (int e = check_fma_args(m, n, k)) return e;
    if (m <= 0 || n <= 0) return PPOCR_OK;
    const int64_t tiles = (n + BN - 1) / BN, blocks = (m + BM - 1) / BM;
    TileOrder order{tiles >= 64 ? 8u : 1u, 0};
    order.per_slot = (unsigned)((tiles + order.slots - 1) / order.slots);
    const int64_t grid = (int64_t)order.slots * order.per_slot * blocks;
    if (grid > 0x7fffffff) return fail(PPOCR_ERR_INVALID_ARG, "MatMulQuantizedB: shape too large");
    return fma_go<EPI, false>(dim3((unsigned)grid), fw, a, m, n, k, BN, out, row_max, row_inv, nullptr, 0, nullptr, st,
                              order);
}

int launch_logits_fma(const int8_t* q, const float* w, const float* scale, const float* bias,
                      const float* a, int64_t m, int64_t n, int64_t k, float* out, hipStream_t st) {
    return writer_go<EPI_LOGITS>(FmaWeights{q, w, scale, bias}, a, m, n, k, nullptr, nullptr, out, st);
}

int launch_probs_fma(const int8_t* q, const float* w, const float* scale, const float* bias,
                     const float* a, int64_t m, int64_t n, int64_t k, const float* row_max,
                     const float* row_inv, float* probs, hipStream_t st) {
    return writer_go<EPI_PROBS>(FmaWeights{q, w, scale, bias}, a, m, n, k, row_max, row_inv, probs, st);
}

int launch_stats_fma(const int8_t* q, const float* w, const float* scale, const float* bias,
                     const float* a, int64_t m, int64_t n, int64_t k, int nsplit, Partial* part,
                     hipStream_t st, int64_t line_len) {
    if (int e = check_fma_args(m, n, k)) return e;
    if (line_len < 0) return fail(PPOCR_ERR_INVALID_ARG, "RecHeadHip: bad line length");
    if (nsplit < 1 || nsplit > 1024) return fail(PPOCR_ERR_INVALID_ARG, "RecHeadHip: bad nsplit");
    if (m <= 0) return PPOCR_OK;
    const int ntiles = (int)((n + BN - 1) / BN);
    const int tpc = (ntiles + nsplit - 1) / nsplit;
    return fma_go<EPI_STATS, false>(dim3((unsigned)nsplit, (unsigned)((m + BM - 1) / BM)), FmaWeights{q, w, scale, bias},
                                    a, m, n, k, tpc * BN, nullptr, nullptr, nullptr, part, line_len, nullptr, st);
}

int launch_rescue_fma(int epi, const FmaWeights& fw, const float* a, int64_t m, int64_t n, int64_t k, int nsplit,
                      int classes_per_chunk, float* out, const float* row_max, const float* row_inv, Partial* part,
                      int64_t line_len, const Guard& guard, hipStream_t st) {
    if (int e = check_fma_args(m, n, k)) return e;
    if (line_len < 0) return fail(PPOCR_ERR_INVALID_ARG, "RecHeadHip: bad line length");
    if (m <= 0 || n <= 0) return PPOCR_OK;
    if (!guard.header || !guard.rows) return fail(PPOCR_ERR_INVALID_ARG, "RecHeadHip: rescue without a guard list");
    // the row count is on the device: a fixed number of row-block slots walk the list
    const unsigned slots = (unsigned)std::min<int64_t>((m + BM - 1) / BM, kFmaRescueSlots);
    int cpc = BN, chunks = (int)((n + BN - 1) / BN);
    if (epi == EPI_STATS) {
        if (nsplit < 1 || nsplit > 1024 || classes_per_chunk <= 0 || (int64_t)classes_per_chunk * nsplit < n)
            return fail(PPOCR_ERR_INVALID_ARG, "RecHeadHip: bad vocabulary chunks");
        cpc = classes_per_chunk;
        chunks = nsplit;
    }
    const dim3 grid((unsigned)chunks, slots);
    if (epi == EPI_LOGITS)
        return fma_go<EPI_LOGITS, true>(grid, fw, a, m, n, k, cpc, out, row_max, row_inv, part, line_len, &guard, st);
    if (epi == EPI_PROBS)
        return fma_go<EPI_PROBS, true>(grid, fw, a, m, n, k, cpc, out, row_max, row_inv, part, line_len, &guard, st);
    return fma_go<EPI_STATS, true>(grid, fw, a, m, n, k, cpc, out, row_max, row_inv, part, line_len, &guard, st);
}

}  // namespace ppocr
