// LayerStack dense layers for gfx950.
//
// The batch is processed in the bucket-sorted order produced by the stable
// bin sort (every 16-row tile belongs to one bucket), as the reference's
// sorted L1 kernels do (crates/cuda-native-runtime/kernels/native_kernels.cu:
// 2394-2432, 2502-2589).  Per-row arithmetic follows the reference CPU
// functions in crates/gpu-kernels/src/layerstack/ (dense_mm.rs,
// dense_mm_bucket.rs, crelu.rs, abs_pow2_scale.rs, concat_l1sqr_main.rs,
// elementwise.rs, slice2d.rs, ft_post_perspective.rs) and the loss kernels in
// crates/gpu-kernels/src/pointwise/{loss_wdl,loss_wrm}.rs; the launch order is
// the one of GpuTrainer::forward/backward (bins/nnue_train/src/
// trainer_layerstack.rs:2038-3936).
//
// MFMA (v_mfma_f32_16x16x4_f32) is used for the FT->L1 contraction only: the
// L1 forward (bucket + shared weights, K = ft_out) and the L1 weight gradient
// (K = rows of the batch).  Everything reduced over the batch goes through
// per-workgroup partials that are summed in a fixed order, so a step is
// bit-reproducible run to run (no float atomics anywhere).
#include "dense_kernels.hpp"

#include <type_traits>

#include "common.hpp"
#include "ft_kernels.hpp"

namespace tatara {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

typedef _Float16 half8 __attribute__((ext_vector_type(8)));


// ---------------------------------------------------------------------------
// L1 forward.  One wave per 16-row sorted tile (two with one bucket, the
// f32 form).
//   bucket part: l1_b[g] + combined . l1_w[g]^T   (accumulator starts at the bias,
//                as dense_mm_fwd_bucket_tiled_l1_sorted does); 0 for an invalid bucket
//   shared part: combined . l1s_w + l1s_b         (bias after the sum, as the
//                reference's sgemm + bias_add_per_row)
// MFMA operand layout (16x16x4 f32): lane l supplies A[l%16][l/16] and
// B[l/16][l%16]; the result holds D[4*(l/16)+r][l%16] in element r.  Each lane
// loads float4 column runs and feeds their components to four successive
// MFMAs, which permutes the K order consistently for A and B.
// ---------------------------------------------------------------------------
// T (1 or 2) consecutive tiles of bucket `bin`: the weights of each K-block
// are loaded once for all T tiles.  NJ (1 or 2) blocks of 16 L1 outputs:
// lane i computes outputs i and 16 + i (l1 = 32) from the same row loads.
template <int T, int NJ>
__device__ __forceinline__ void ls_l1_fwd_tiles(const LsDenseArgs& a, uint32_t tile0, int32_t bin, uint32_t lane) {
    const uint32_t i = lane % 16, q = lane / 16;
    const uint32_t ft_out = a.ft_out, l1 = a.l1;
    const bool bvalid = (uint32_t)bin < a.nb;
    // Operands are loaded unconditionally from always-valid addresses (row 0,
    // bucket 0, column l1-1) and masked afterwards: a guarded load would be
    // split into predicated dword loads and lose the 16-byte accesses.
    bool jvalid[NJ], wbvalid[NJ];
    const float4* W1[NJ];
    const float* Ws[NJ];
    float binit[NJ];
#pragma unroll
    for (int jt = 0; jt < NJ; ++jt) {
        const uint32_t j = 16 * jt + i;
        jvalid[jt] = j < l1;
        wbvalid[jt] = bvalid && jvalid[jt];
        const uint32_t ic = jvalid[jt] ? j : l1 - 1;
        W1[jt] = reinterpret_cast<const float4*>(a.l1_w + ((uint64_t)(bvalid ? bin : 0) * l1 + ic) * ft_out);
        Ws[jt] = a.l1s_w + ic;
        binit[jt] = wbvalid[jt] ? a.l1_b[bin * l1 + j] : 0.0f;
    }
    const float4* X[T];
    bool xvalid[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int32_t orig = a.perm[(tile0 + t) * 16 + i];
        xvalid[t] = orig >= 0;
        X[t] = reinterpret_cast<const float4*>(a.combined + (uint64_t)(orig >= 0 ? orig : 0) * ft_out);
    }
    floatx4 accb[T][NJ], accs[T][NJ];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int jt = 0; jt < NJ; ++jt) {
            accb[t][jt] = floatx4{binit[jt], binit[jt], binit[jt], binit[jt]};
            accs[t][jt] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    // ft_out % 64 == 0: whole groups of kU K-blocks; a group's operands are
    // loaded before its MFMAs so each wave keeps several loads in flight
    const uint32_t nk = ft_out / 16;
    constexpr uint32_t kU = T * NJ == 1 ? 4 : 2;
    for (uint32_t kb0 = 0; kb0 < nk; kb0 += kU) {
        float4 x[kU][T], wb[kU][NJ];
        float ws[kU][NJ][4];
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) {
            const uint32_t kb = kb0 + u;
#pragma unroll
            for (int t = 0; t < T; ++t) x[u][t] = X[t][kb * 4 + q];
            const uint32_t k = kb * 16 + 4 * q;
#pragma unroll
            for (int jt = 0; jt < NJ; ++jt) {
                wb[u][jt] = W1[jt][kb * 4 + q];
#pragma unroll
                for (int c = 0; c < 4; ++c) ws[u][jt][c] = Ws[jt][(uint64_t)(k + c) * l1];
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u)
#pragma unroll
            for (int jt = 0; jt < NJ; ++jt) {
                const float4 wv = wbvalid[jt] ? wb[u][jt] : zero4;
                const bool jv = jvalid[jt];
                const float w0 = jv ? ws[u][jt][0] : 0.f, w1 = jv ? ws[u][jt][1] : 0.f;
                const float w2 = jv ? ws[u][jt][2] : 0.f, w3 = jv ? ws[u][jt][3] : 0.f;
#pragma unroll
                for (int t = 0; t < T; ++t) {
                    const float4 xv = xvalid[t] ? x[u][t] : zero4;
                    accb[t][jt] = mfma4(xv.x, wv.x, accb[t][jt]);
                    accs[t][jt] = mfma4(xv.x, w0, accs[t][jt]);
                    accb[t][jt] = mfma4(xv.y, wv.y, accb[t][jt]);
                    accs[t][jt] = mfma4(xv.y, w1, accs[t][jt]);
                    accb[t][jt] = mfma4(xv.z, wv.z, accb[t][jt]);
                    accs[t][jt] = mfma4(xv.z, w2, accs[t][jt]);
                    accb[t][jt] = mfma4(xv.w, wv.w, accb[t][jt]);
                    accs[t][jt] = mfma4(xv.w, w3, accs[t][jt]);
                }
            }
    }
#pragma unroll
    for (int jt = 0; jt < NJ; ++jt) {
        const uint32_t j = 16 * jt + lane % 16;
        if (j >= l1) continue;
        const float bs = a.l1s_b[j];
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint64_t row = (uint64_t)(tile0 + t) * 16 + 4 * q + r;
                float* o = a.l1_sorted + row * 2 * l1;
                o[j] = bvalid ? accb[t][jt][r] : 0.0f;
                o[l1 + j] = accs[t][jt][r] + bs;
            }
    }
}

// The TF32 L1 forward's weight operands, once per forward: f16 copies of
// l1_w and of l1s_w transposed ([l1][ft_out], a lane's K values
// consecutive).  Thread i: bucket weight i, and shared weight i when
// i < l1 * ft_out (nb >= 1).  (The f32 forward reads the weights as they
// are: the transposed copy cost more than the strided loads it saved.)
__global__ __launch_bounds__(256) void ls_l1_weights_f16_kernel(LsDenseArgs a) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const uint64_t n_w = (uint64_t)a.nb * a.l1 * a.ft_out, n_s = (uint64_t)a.l1 * a.ft_out;
    if (i >= n_w) return;
    reinterpret_cast<_Float16*>(a.l1_w16)[i] = (_Float16)a.l1_w[i];
    if (i < n_s) {
        const uint64_t j = i / a.ft_out, k = i % a.ft_out;  // transposed [j][k] <- [k][j]
        reinterpret_cast<_Float16*>(a.l1s_wt16)[i] = (_Float16)a.l1s_w[k * a.l1 + j];
    }
}

// One wave per pair of 16-row sorted tiles: both in one pass when they
// belong to one bucket, else (at a bucket boundary) one pass each; a tile
// of bin -1 (all padding) is skipped.
template <int NJ>
__global__ __launch_bounds__(256) void ls_l1_fwd_kernel(LsDenseArgs a) {
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t tile0 = (blockIdx.x * 4 + wave) * 2;
    const uint32_t n_tiles = (uint32_t)(a.padded_b / 16);
    if (tile0 >= n_tiles) return;
    const int32_t bin0 = scalar_load(a.sorted_bin + (uint64_t)tile0 * 16);
    const int32_t bin1 = tile0 + 1 < n_tiles ? scalar_load(a.sorted_bin + (uint64_t)(tile0 + 1) * 16) : -1;
    if (bin0 >= 0 && bin0 == bin1) {
        ls_l1_fwd_tiles<2, NJ>(a, tile0, bin0, lane);
    } else {
        if (bin0 >= 0) ls_l1_fwd_tiles<1, NJ>(a, tile0, bin0, lane);
        if (bin1 >= 0) ls_l1_fwd_tiles<1, NJ>(a, tile0 + 1, bin1, lane);
    }
}

// The f32 L1 forward for batches of few tiles: a workgroup takes one tile, each
// of its 2 * NJ waves one of the tile's sums (bucket or shared, 16 outputs) over
// the whole K in the same order, so the sums are the two-tile kernel's bit for
// bit (split over K they would not be).  With one wave per two tiles such a
// batch leaves most SIMDs without a wave, and a wave waits for the loads of two
// to four K blocks at a time; here eight K blocks are loaded while the eight before
// them are multiplied.
template <int NJ>
__global__ __launch_bounds__(2 * NJ * 64) void ls_l1_fwd_sums_kernel(LsDenseArgs a) {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const uint32_t i = lane % 16, q = lane / 16;
    const uint32_t ft_out = a.ft_out, l1 = a.l1, tile = blockIdx.x;
    const int32_t bin = scalar_load(a.sorted_bin + (uint64_t)tile * 16);
    if (bin < 0) return;  // a trailing all-padding tile
    const bool shared = wave & 1u;
    const bool bvalid = (uint32_t)bin < a.nb;
    // unconditional loads from always-valid addresses, masked afterwards
    const int32_t orig = a.perm[tile * 16 + i];
    const bool xvalid = orig >= 0;
    const float4* X = reinterpret_cast<const float4*>(a.combined + (uint64_t)(xvalid ? orig : 0) * ft_out);
    const uint32_t j = 16 * (wave / 2) + i;
    const bool jvalid = j < l1, wvalid = jvalid && (shared || bvalid);
    const uint32_t ic = jvalid ? j : l1 - 1;
    const float4* W1 = reinterpret_cast<const float4*>(a.l1_w + ((uint64_t)(bvalid ? bin : 0) * l1 + ic) * ft_out);
    const float* Ws = a.l1s_w + ic;
    const float b0 = !shared && wvalid ? a.l1_b[bin * l1 + j] : 0.0f;
    floatx4 acc = {b0, b0, b0, b0};
    const uint32_t nk = ft_out / 16;
    constexpr uint32_t kU = 8;
    struct Group {
        float4 x[kU], w[kU];
    };
    auto load = [&](uint32_t kb0, Group& g) {  // past the end: the last block again, unused
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) {
            const uint32_t kb = kb0 + u < nk ? kb0 + u : nk - 1;
            g.x[u] = X[kb * 4 + q];
            if (shared) {
                const float* w = Ws + (uint64_t)(kb * 16 + 4 * q) * l1;
                g.w[u] = make_float4(w[0], w[l1], w[2 * l1], w[3 * l1]);
            } else {
                g.w[u] = W1[kb * 4 + q];
            }
        }
    };
    auto multiply = [&](uint32_t kb0, const Group& g) {
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) {
            if (kb0 + u >= nk) break;
            const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
            const float4 x = xvalid ? g.x[u] : zero4, w = wvalid ? g.w[u] : zero4;
            acc = mfma4(x.x, w.x, acc);
            acc = mfma4(x.y, w.y, acc);
            acc = mfma4(x.z, w.z, acc);
            acc = mfma4(x.w, w.w, acc);
        }
    };
    Group g0, g1;
    load(0, g0);
    for (uint32_t kb0 = 0; kb0 < nk; kb0 += 2 * kU) {
        load(kb0 + kU, g1);
        multiply(kb0, g0);
        load(kb0 + 2 * kU, g0);
        multiply(kb0 + kU, g1);
    }
    if (!jvalid) return;
    const float bs = shared ? a.l1s_b[j] : 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint64_t row = (uint64_t)tile * 16 + 4 * q + r;
        a.l1_sorted[row * 2 * l1 + (shared ? l1 : 0) + j] = shared ? acc[r] + bs : (bvalid ? acc[r] : 0.0f);
    }
}

// ---------------------------------------------------------------------------
// L1 forward with TF32-class products: f16 operands on the matrix cores
// (v_mfma_f32_16x16x32_f16, f32 sums).  Lane l supplies A[l%16][8(l/16)+e]
// (row l%16 of the tile, 8 consecutive K from the f16 `combined`, one
// 16-byte load) and B[8(l/16)+e][l%16] (output l%16: 8 consecutive K of its
// bucket weight row, rounded to f16, and 8 strided shared weights).  As the
// reference's tf32 path (per-bucket sgemm, then the bias,
// trainer_layerstack.rs:2388-2480) the bucket bias is added after the sum.
// ---------------------------------------------------------------------------
template <int NJ>
__global__ __launch_bounds__(256) void ls_l1_fwd_tf32_kernel(LsDenseArgs a) {
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t tile = blockIdx.x * 4 + wave;
    if ((uint64_t)tile * 16 >= a.padded_b) return;
    const int32_t bin = a.sorted_bin[tile * 16];
    if (bin < 0) return;  // trailing all-padding tile
    const uint32_t i = lane % 16, q = lane / 16;
    const uint32_t ft_out = a.ft_out, l1 = a.l1;
    const int32_t orig = a.perm[tile * 16 + i];
    const bool bvalid = (uint32_t)bin < a.nb;
    // unconditional loads from always-valid addresses, masked afterwards
    const bool xvalid = orig >= 0;
    const half8* X = reinterpret_cast<const half8*>(
        reinterpret_cast<const _Float16*>(a.combined16) + (uint64_t)(orig >= 0 ? orig : 0) * ft_out);
    bool jvalid[NJ], wbvalid[NJ];
    const half8 *W1[NJ], *Ws[NJ];
#pragma unroll
    for (int jt = 0; jt < NJ; ++jt) {
        const uint32_t j = 16 * jt + i;
        jvalid[jt] = j < l1;
        wbvalid[jt] = bvalid && jvalid[jt];
        const uint32_t ic = jvalid[jt] ? j : l1 - 1;
        W1[jt] = reinterpret_cast<const half8*>(reinterpret_cast<const _Float16*>(a.l1_w16) +
                                                ((uint64_t)(bvalid ? bin : 0) * l1 + ic) * ft_out);
        Ws[jt] = reinterpret_cast<const half8*>(reinterpret_cast<const _Float16*>(a.l1s_wt16) + (uint64_t)ic * ft_out);
    }
    floatx4 accb[NJ], accs[NJ];
#pragma unroll
    for (int jt = 0; jt < NJ; ++jt) accb[jt] = accs[jt] = floatx4{0.f, 0.f, 0.f, 0.f};
    const half8 zero8 = {};
    // ft_out % 64 == 0: K blocks of 32, four loaded before their MFMAs
    const uint32_t nk = ft_out / 32;
    constexpr uint32_t kU = 4;
    for (uint32_t kb0 = 0; kb0 < nk; kb0 += kU) {
        half8 x[kU], wb[kU][NJ], wsh[kU][NJ];
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) {
            const uint32_t k8 = (kb0 + u) * 4 + q;
            x[u] = X[k8];
#pragma unroll
            for (int jt = 0; jt < NJ; ++jt) {
                wb[u][jt] = W1[jt][k8];
                wsh[u][jt] = Ws[jt][k8];
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kU; ++u) {
            const half8 xv = xvalid ? x[u] : zero8;
#pragma unroll
            for (int jt = 0; jt < NJ; ++jt) {
                accb[jt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, wbvalid[jt] ? wb[u][jt] : zero8, accb[jt], 0, 0, 0);
                accs[jt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, jvalid[jt] ? wsh[u][jt] : zero8, accs[jt], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int jt = 0; jt < NJ; ++jt) {
        const uint32_t j = 16 * jt + lane % 16;
        if (j >= l1) continue;
        const float bb = bvalid ? a.l1_b[bin * l1 + j] : 0.0f;
        const float bs = a.l1s_b[j];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint64_t row = (uint64_t)tile * 16 + 4 * q + r;
            float* o = a.l1_sorted + row * 2 * l1;
            o[j] = bvalid ? accb[jt][r] + bb : 0.0f;
            o[l1 + j] = accs[jt][r] + bs;
        }
    }
}

// ---------------------------------------------------------------------------
// Extended-WRM weight sum (wrm_weight_sum, native_kernels.cu:520-544), as a
// deterministic two-level f64 reduction in position order.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void wrm_weight_partial_kernel(const float* __restrict__ score,
                                                                 uint32_t n, LossParams lp,
                                                                 double* __restrict__ partial) {
    __shared__ double s[256];
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    s[threadIdx.x] = i < n ? (double)wrm_weight_dev(score[i], lp) : 0.0;
    __syncthreads();
    if (threadIdx.x == 0) {
        double acc = 0.0;
        for (int k = 0; k < 256; ++k) acc += s[k];
        partial[blockIdx.x] = acc;
    }
}

// out[0] = sum of partial[0..n): thread t adds t, t + 256, ... in order, then
// the 256 thread sums are combined by a fixed pairwise tree (deterministic).
__global__ __launch_bounds__(256) void sum_partials_f64_kernel(const double* __restrict__ partial,
                                                               uint32_t n, double* __restrict__ out) {
    __shared__ double s[256];
    const uint32_t t = threadIdx.x;
    double acc = 0.0;
    for (uint32_t k = t; k < n; k += 256) acc += partial[k];
    s[t] = acc;
    __syncthreads();
    for (uint32_t w = 128; w > 0; w >>= 1) {
        if (t < w) s[t] = s[t] + s[t + w];
        __syncthreads();
    }
    if (t == 0) *out = s[0];
}

// ---------------------------------------------------------------------------
// Tail: one 64-lane workgroup per sorted 16-row tile (one bucket, the tile's
// rows being bucket-sorted and 16-aligned).  Lane l serves row r = l % 16 with
// quarter q = l / 16: its L2/4 consecutive L2 outputs in the forward, the
// L2 inputs k = q, q+4, .. in the backward, the L1 outputs k = q, q+4, .. of
// the L1-tail gradient.  The tile's L1 outputs, activations and gradients and
// the bucket's L2/L3 weights are in LDS, the L2 weights transposed so that a
// lane reads four outputs' weights at once.  Every
// per-row sum keeps the reference order (k ascending for L2, o ascending for
// L3 and for the L2 input gradient); the gradient partials are per tile, rows
// in order, and are reduced per bucket over the bucket's tiles.
//
// Bound by its chain of LDS round trips.  The L1 outputs as per-lane arrays
// indexed by lane went to scratch memory at l1 = 32, and every cell of the L2
// weight gradient read 32 LDS words: l1 32, l2 64, b 2048 88 -> 34 us;
// l1 16, l2 32, b 65536 70 -> 39 us; l1 8, l2 32, b 16384 22 -> 16 us.
// ---------------------------------------------------------------------------
template <int L1, int L2>
__global__ __launch_bounds__(64) void ls_tail_kernel(LsDenseArgs a, int32_t train) {
    constexpr int LE = L1 - 1;
    constexpr int LIN = 2 * LE;
    constexpr int OQ = L2 / 4;             // L2 outputs per lane
    constexpr int KQ = (LIN + 3) / 4;      // L2 inputs per lane (backward)
    constexpr int JQ = L1 / 4;             // L1 outputs per lane (backward)
    constexpr int WS = L2 + 4;             // row stride of the transposed weights: 16-byte rows, spread banks
    constexpr int IS = 4 * KQ + 4;         // row stride of the L2 inputs (zero past LIN)
    static_assert(L2 % 16 == 0 && L1 % 4 == 0, "quarters of whole float4");
    __shared__ __align__(16) float sW2[LIN * WS];  // [k][o]
    __shared__ float sB2[L2], sW3[L2];
    __shared__ float s_l1t[16][L1 + 1];
    __shared__ __align__(16) float s_l2in[16][IS];
    __shared__ float s_l2a[16][L2 + 1];
    __shared__ __align__(16) float s_dl2o[16][WS];
    __shared__ float s_dl2pre[16][LIN + 1];
    __shared__ float s_dl1[16][L1 + 1];
    __shared__ float s_dy[16];
    __shared__ double s_loss[16];
    __shared__ int32_t s_real[16];

    const uint32_t lane = threadIdx.x;
    const uint32_t r = lane % 16, q = lane / 16;
    const uint64_t tile = blockIdx.x;
    const uint64_t row = tile * 16 + r;
    // the tile's bucket: its first row is real unless the tile is all padding
    const int32_t orig0 = a.perm[tile * 16];
    const int32_t bin = orig0 >= 0 ? a.sorted_bin[tile * 16] : -1;
    const bool bvalid = bin >= 0 && (uint32_t)bin < a.nb;
    const int g = bvalid ? bin : 0;
    const int32_t orig = a.perm[row];
    const bool real = orig >= 0;
    if (q == 0) s_real[r] = real ? 1 : 0;
    if (bvalid) {
        const float* W2 = a.l2_w + (uint64_t)g * L2 * LIN;
        // 16-byte loads (a bucket's weights are a multiple of 16 floats), four
        // in flight: one at a time this loop was most of the kernel
        constexpr uint32_t N4 = L2 * LIN / 4, U = 4;
        for (uint32_t i0 = lane; i0 < N4; i0 += 64 * U) {
            float4 v[U];
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                const uint32_t i = i0 + 64 * u;
                v[u] = reinterpret_cast<const float4*>(W2)[i < N4 ? i : N4 - 1];
            }
#pragma unroll
            for (uint32_t u = 0; u < U; ++u) {
                if (i0 + 64 * u >= N4) break;
                const uint32_t e = 4 * (i0 + 64 * u);
                const float c[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) sW2[(e + j) % LIN * WS + (e + j) / LIN] = c[j];
            }
        }
        if (lane < (uint32_t)L2) {
            sB2[lane] = a.l2_b[g * L2 + lane];
            sW3[lane] = a.l3_w[g * L2 + lane];
        }
    }
    const float b3 = bvalid ? a.l3_b[g] : 0.0f;
    __syncthreads();  // s_real
    // bucket + shared L1 outputs, and what L2 reads of them; zero for padding
    const float* l1v = a.l1_sorted + tile * 16 * 2 * L1;
#pragma unroll
    for (uint32_t i = lane; i < 16u * L1; i += 64) {
        const uint32_t rr = i / L1, o = i % L1;
        const bool ok = s_real[rr] != 0;
        const float x = l1v[rr * 2 * L1 + o], y = l1v[rr * 2 * L1 + L1 + o];
        const float t = ok ? x + y : 0.0f;  // elementwise_add
        s_l1t[rr][o] = t;
        if (o < (uint32_t)LE) {
            s_l2in[rr][o] = crelu01(t * t * a.l1_sqr_scale);  // abs_pow2_scale_fwd
            s_l2in[rr][LE + o] = crelu01(t);                  // concat_l1sqr_main_fwd
        }
    }
    if (lane < 16)
        for (int k = LIN; k < 4 * KQ; ++k) s_l2in[lane][k] = 0.0f;
    __syncthreads();
    // L2 (dense_mm_fwd_bucket: the sum starts at the bias, k ascending) + CReLU
    float l2o[OQ];
#pragma unroll
    for (int j = 0; j < OQ; ++j) l2o[j] = bvalid ? sB2[OQ * q + j] : 0.0f;
    if (bvalid) {
#pragma unroll 4
        for (int k = 0; k < LIN; ++k) {
            const float x = s_l2in[r][k];
            const float4* w = reinterpret_cast<const float4*>(sW2 + k * WS + OQ * q);
#pragma unroll
            for (int j = 0; j < OQ; j += 4) {
                const float4 w4 = w[j / 4];
                l2o[j + 0] += x * w4.x;
                l2o[j + 1] += x * w4.y;
                l2o[j + 2] += x * w4.z;
                l2o[j + 3] += x * w4.w;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < OQ; ++j) s_l2a[r][OQ * q + j] = real ? crelu01(l2o[j]) : 0.0f;
    __syncthreads();
    if (q == 0) {
        // L3 (o ascending from the bias), net = l3 + skip, loss
        double loss_c = 0.0;
        float dy = 0.0f;
        if (real) {
            float l3 = 0.0f;
            if (bvalid) {
                l3 = b3;
#pragma unroll
                for (int o = 0; o < L2; ++o) l3 += s_l2a[r][o] * sW3[o];
            }
            const float net = l3 + s_l1t[r][LE];  // slice_extract_2d: the skip output
            a.net_output[orig] = net;
            loss_c = position_loss(net, a.score[orig], a.wdl[orig], a.wdl_lambda, a.loss, a.per_pos_norm,
                                   a.weight_sum, a.batch, dy);
        }
        s_dy[r] = dy;
        s_loss[r] = loss_c;
    }
    __syncthreads();
    if (lane == 0) {
        double acc = 0.0;
        for (int k = 0; k < 16; ++k) acc += s_loss[k];
        a.loss_partial[tile] = acc;
    }
    if (!train) return;

    // backward: L3 input gradient and the L2 CReLU mask for this lane's outputs
    const float dy = s_dy[r];
#pragma unroll
    for (int j = 0; j < OQ; ++j) {
        const int o = OQ * q + j;
        float acc = 0.0f;  // dense_mm_bwd_input_bucket, out_dim 1
        if (bvalid) acc += dy * sW3[o];
        const float d = (l2o[j] > 0.0f && l2o[j] < 1.0f) ? acc : 0.0f;  // crelu_grad
        s_dl2o[r][o] = real ? d : 0.0f;
    }
    __syncthreads();
    // L2 input gradient for this lane's inputs (o ascending), masked by the L1-tail CReLU
    float g2[KQ];
#pragma unroll
    for (int i = 0; i < KQ; ++i) g2[i] = 0.0f;
    if (bvalid) {
#pragma unroll 2
        for (int o = 0; o < L2; o += 4) {
            const float4 d4 = *reinterpret_cast<const float4*>(&s_dl2o[r][o]);
#pragma unroll
            for (int i = 0; i < KQ; ++i) {
                const int k = (int)q + 4 * i;
                const float4 w4 = *reinterpret_cast<const float4*>(sW2 + (k < LIN ? k : LIN - 1) * WS + o);
                g2[i] += d4.x * w4.x;
                g2[i] += d4.y * w4.y;
                g2[i] += d4.z * w4.z;
                g2[i] += d4.w * w4.w;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < KQ; ++i) {
        const int k = (int)q + 4 * i;
        if (k >= LIN) break;
        const float t = s_l1t[r][k < LE ? k : k - LE];
        const float pre = k < LE ? t * t * a.l1_sqr_scale : t;
        s_dl2pre[r][k] = (pre > 0.0f && pre < 1.0f) ? g2[i] : 0.0f;
    }
    __syncthreads();
    // L1-tail gradient for this lane's L1 outputs
#pragma unroll
    for (int i = 0; i < JQ; ++i) {
        const int k = (int)q + 4 * i;
        float d = 0.0f;
        if (real) {
            if (k < LE) {
                const float from_sqr = 2.0f * s_l1t[r][k] * a.l1_sqr_scale * s_dl2pre[r][k];  // abs_pow2_scale_grad
                d = s_dl2pre[r][LE + k] + from_sqr;                                             // elementwise_add
            } else {
                d = dy;  // slice_scatter_2d of the skip gradient
            }
        }
        a.dl1_sorted[row * L1 + k] = d;
        s_dl1[r][k] = d;
    }
    __syncthreads();

    // per-tile gradient partials, rows in order (padding rows hold zeros)
    if (bvalid) {
        const TailDims td{(uint32_t)L1, (uint32_t)L2, a.nb};
        const uint32_t cells = td.cells();
        float* part = a.tail_partial + tile * cells;
        // L2 weights: a lane takes cells of 4 outputs x 4 inputs (two 16-byte
        // LDS reads a row for 16 products)
        constexpr uint32_t KB = (LIN + 3) / 4;
        for (uint32_t blk = lane; blk < L2 / 4 * KB; blk += 64) {
            const uint32_t o = blk / KB * 4, k = blk % KB * 4;
            floatx4 acc[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
            for (int rr = 0; rr < 16; ++rr) {
                const floatx4 d = *reinterpret_cast<const floatx4*>(&s_dl2o[rr][o]);
                const floatx4 x = *reinterpret_cast<const floatx4*>(&s_l2in[rr][k]);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] += x * d[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (k + j < (uint32_t)LIN) part[(o + e) * LIN + k + j] = acc[e][j];
        }
        for (uint32_t c = td.off_b2() + lane; c < cells; c += 64) {
            float acc = 0.0f;
            if (c < td.off_w3()) {
                const uint32_t o = c - td.off_b2();
                for (int rr = 0; rr < 16; ++rr)
                    if (s_real[rr]) acc += s_dl2o[rr][o];
            } else if (c < td.off_b3()) {
                const uint32_t o = c - td.off_w3();
                for (int rr = 0; rr < 16; ++rr)
                    if (s_real[rr]) acc += s_l2a[rr][o] * s_dy[rr];
            } else if (c < td.off_b1()) {
                for (int rr = 0; rr < 16; ++rr)
                    if (s_real[rr]) acc += s_dy[rr];
            } else {
                const uint32_t o = c - td.off_b1();
                for (int rr = 0; rr < 16; ++rr)
                    if (s_real[rr]) acc += s_dl1[rr][o];
            }
            part[c] = acc;
        }
    }
    // shared L1 bias: every real row, including rows of an invalid bucket
    if (lane < (uint32_t)L1) {
        float acc = 0.0f;
        for (int rr = 0; rr < 16; ++rr)
            if (s_real[rr]) acc += s_dl1[rr][lane];
        a.b1s_partial[tile * L1 + lane] = acc;
    }
    // the bucket segments of the tile partials (first tile of each bin)
    if (tile == 0 && lane <= a.nb) a.tail_seg[lane] = a.bin_start[lane] / 16;
}

// ---------------------------------------------------------------------------
// Chunk table for the L1 weight gradient: every bin (including the invalid
// bin nb, whose rows still feed the shared weight) is split into chunks of at
// most kChunkTiles 16-row tiles.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void ls_chunk_table_kernel(const uint32_t* __restrict__ bin_start,
                                                             const uint32_t* __restrict__ bin_count, uint32_t nb,
                                                             uint32_t max_chunks, uint32_t* __restrict__ info) {
    // the bins' tile ranges and first chunks (at most 17 bins: nb <= 16 plus
    // the invalid bin), then one thread per chunk entry
    __shared__ uint32_t s_t0[17], s_t1[17], s_first[18];
    const uint32_t t = threadIdx.x;
    if (t <= nb) {
        s_t0[t] = bin_start[t] / 16;
        s_t1[t] = (bin_start[t] + bin_count[t] + 15) / 16;
    }
    __syncthreads();
    if (t == 0) {
        uint32_t c = 0;
        for (uint32_t g = 0; g <= nb; ++g) {
            s_first[g] = c;
            const uint32_t n = s_t1[g] > s_t0[g] ? (s_t1[g] - s_t0[g] + kChunkTiles - 1) / kChunkTiles : 0u;
            c = c + n < max_chunks ? c + n : max_chunks;
        }
        s_first[nb + 1] = c;
    }
    __syncthreads();
    const uint32_t total = s_first[nb + 1];
    for (uint32_t ci = t; ci < total; ci += blockDim.x) {
        uint32_t g = 0;
        while (g < nb && s_first[g + 1] <= ci) ++g;  // the bin whose chunks hold ci
        const uint32_t tile = s_t0[g] + (ci - s_first[g]) * kChunkTiles;
        info[3 * ci + 0] = g;
        info[3 * ci + 1] = tile;
        info[3 * ci + 2] = min(kChunkTiles, s_t1[g] - tile);
    }
    uint32_t* seg = info + 3 * max_chunks + 1;  // seg[g] = first chunk of bin g, seg[nb+1] = end
    if (t <= nb + 1) seg[t] = s_first[t];
    if (t == 0) info[3 * max_chunks] = total;
}

// ---------------------------------------------------------------------------
// Deterministic column sums of a partial matrix P[rows][n_cols]:
// out[seg][c] = sum over the segment's rows of P[r][c].  Thread (c, phase)
// sums rows phase, phase + PH, ... sequentially; the PH phase sums are then
// combined by a fixed pairwise tree.  Segment s covers rows
// [seg_rows[s], seg_rows[s+1]) when seg_rows is given, else all rows.
// ---------------------------------------------------------------------------

// COLS columns per workgroup and 1024 / COLS phases: 64 columns (16 phases)
// for wide matrices, 16 columns (64 phases) for tall narrow ones.
template <uint32_t COLS>
__global__ __launch_bounds__(1024) void reduce_rows_kernel(const float* __restrict__ P, uint32_t n_rows,
                                                           uint32_t n_cols, const uint32_t* __restrict__ seg_rows,
                                                           float* __restrict__ out) {
    constexpr uint32_t PH = 1024 / COLS;
    __shared__ float part[PH][COLS];
    const uint32_t lane = threadIdx.x % COLS, phase = threadIdx.x / COLS;
    const uint32_t c = blockIdx.x * COLS + lane;
    const uint32_t seg = blockIdx.y;
    const uint32_t r0 = seg_rows ? seg_rows[seg] : 0;
    const uint32_t r1 = seg_rows ? seg_rows[seg + 1] : n_rows;
    float acc = 0.0f;
    if (c < n_cols) {
#pragma unroll 8
        for (uint32_t r = r0 + phase; r < r1; r += PH) acc += P[(uint64_t)r * n_cols + c];
    }
    part[phase][lane] = acc;
    __syncthreads();
    for (uint32_t w = PH / 2; w > 0; w >>= 1) {
        if (phase < w) part[phase][lane] = part[phase][lane] + part[phase + w][lane];
        __syncthreads();
    }
    if (phase == 0 && c < n_cols) out[(uint64_t)seg * n_cols + c] = part[0][lane];
}

// The reduce_rows_kernel shape for a matrix n_cols wide: 16-column
// workgroups for narrow matrices, and for tall ones whose 64-column
// workgroups would not fill the chip (fewer rows per thread).
void reduce_rows(const float* P, uint32_t n_rows, uint32_t n_cols, const uint32_t* seg_rows, uint32_t n_seg,
                 float* out, hipStream_t stream) {
    // (n_rows: all segments' rows; 0 when unknown on the host)
    const bool tall = n_rows >= 256ull * n_seg && (uint64_t)ceil_div(n_cols, 64) * n_seg < 256;
    if (n_cols <= 16 || tall)
        reduce_rows_kernel<16><<<dim3(ceil_div(n_cols, 16), n_seg), 1024, 0, stream>>>(P, n_rows, n_cols, seg_rows,
                                                                                      out);
    else
        reduce_rows_kernel<64><<<dim3(ceil_div(n_cols, 64), n_seg), 1024, 0, stream>>>(P, n_rows, n_cols, seg_rows,
                                                                                      out);
}

// ---------------------------------------------------------------------------
// L1 weight gradient partials: P[chunk][o][k] = sum over the chunk's rows of
// dl1[row][o] * combined[row][k].  One wave owns 64 columns; lane (k, q) loads
// a float4 of combined so block c of its four MFMAs holds columns k0+4k+c.
// TF32: `combined` read as f16 (as the forward stored it); dl1 and the
// products stay f32.
// ---------------------------------------------------------------------------
template <bool TF32, int NJ>
__global__ __launch_bounds__(256) void ls_l1_wgrad_kernel(LsDenseArgs a) {
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t n_chunks = a.chunk_info[3 * a.max_chunks];
    const uint32_t chunk = blockIdx.x;
    if (chunk >= n_chunks) return;
    const uint32_t k0 = (blockIdx.y * 4 + wave) * 64;
    if (k0 >= a.ft_out) return;
    const uint32_t t0 = a.chunk_info[3 * chunk + 1], nt = a.chunk_info[3 * chunk + 2];
    const uint32_t o = lane % 16, q = lane / 16, kk = lane % 16;
    const uint32_t l1 = a.l1, ft_out = a.ft_out;
    const bool kvalid = k0 + 4 * kk < ft_out;
    // NJ blocks of 16 L1 outputs (lane o: outputs o and 16 + o)
    bool ovalid[NJ];
    uint32_t oc[NJ];
#pragma unroll
    for (int jt = 0; jt < NJ; ++jt) {
        ovalid[jt] = 16 * jt + o < l1;
        oc[jt] = ovalid[jt] ? 16 * jt + o : 0;
    }
    floatx4 acc[NJ][4];
#pragma unroll
    for (int jt = 0; jt < NJ; ++jt)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[jt][c] = floatx4{0.f, 0.f, 0.f, 0.f};
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    const uint32_t kc = kvalid ? k0 + 4 * kk : 0;  // always-valid column, masked below
    for (uint32_t tt = 0; tt < nt; ++tt) {
        // the tile's 16 rows are loaded before its 16 MFMAs (unconditional
        // loads from valid addresses, masked after the load)
        float4 xs[4];
        float ds[4][NJ];
        bool rvs[4];
#pragma unroll
        for (uint32_t s = 0; s < 4; ++s) {
            const uint64_t row = (uint64_t)(t0 + tt) * 16 + 4 * s + q;
            const int32_t orig = a.perm[row];
            rvs[s] = orig >= 0;
            const uint64_t xo = (uint64_t)(orig >= 0 ? orig : 0) * ft_out + kc;
            if constexpr (TF32) {
                typedef _Float16 h4 __attribute__((ext_vector_type(4)));
                const h4 h = *reinterpret_cast<const h4*>(reinterpret_cast<const _Float16*>(a.combined16) + xo);
                xs[s] = make_float4((float)h.x, (float)h.y, (float)h.z, (float)h.w);
            } else {
                xs[s] = *reinterpret_cast<const float4*>(a.combined + xo);
            }
#pragma unroll
            for (int jt = 0; jt < NJ; ++jt) ds[s][jt] = a.dl1_sorted[row * l1 + oc[jt]];
        }
#pragma unroll
        for (uint32_t s = 0; s < 4; ++s) {
            const float4 x = (rvs[s] && kvalid) ? xs[s] : zero4;
#pragma unroll
            for (int jt = 0; jt < NJ; ++jt) {
                const float d = ovalid[jt] ? ds[s][jt] : 0.0f;
                acc[jt][0] = mfma4(d, x.x, acc[jt][0]);
                acc[jt][1] = mfma4(d, x.y, acc[jt][1]);
                acc[jt][2] = mfma4(d, x.z, acc[jt][2]);
                acc[jt][3] = mfma4(d, x.w, acc[jt][3]);
            }
        }
    }
    if (!kvalid) return;
    float* P = a.w1_partial + (uint64_t)chunk * l1 * ft_out;
#pragma unroll
    for (int jt = 0; jt < NJ; ++jt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t oo = 16 * jt + 4 * q + r;
            if (oo >= l1) continue;
            float* dst = P + (uint64_t)oo * ft_out + k0 + 4 * kk;
            dst[0] = acc[jt][0][r];
            dst[1] = acc[jt][1][r];
            dst[2] = acc[jt][2][r];
            dst[3] = acc[jt][3][r];
        }
}

// ---------------------------------------------------------------------------
// L1 input gradient fused with the FT-post gradient.
// dcombined[c] = sum_o dl1[o] * l1_w[g][o][c]  +  sum_o dl1[o] * l1s_w[c][o]
// (the reference's two input-gradient kernels, added as in
// ft_post_perspective_grad_fused), then the pairwise CReLU gradient into dft
// (native_kernels.cu:2260-2302).  Grid (column block, row block): a wave owns
// 64 columns of the combined output over post_tiles sorted tiles and writes
// their ft_b gradient partials per perspective: f32 one for every kPostTiles of
// them, rows in order; f16 one for the row block.  The f16
// variant reads f16 raw sums and writes the f16 dft, scaled by dft_scale and
// clamped to +-65504 with a count of every clamp
// (ft_post_perspective_grad_fused_fp16, native_kernels.cu:2304-2352); the
// ft_b gradient stays unscaled f32.
//
// The two input gradients are [16 rows][L1] x [L1][64 columns] products per
// tile on the matrix cores (f32 operands and sums, o ascending).  MFMA operand
// layout (16x16x4 f32): lane l supplies A[l%16][l/16] and B[l/16][l%16];
// element r of the result is D[4*(l/16)+r][l%16].  Column group g's column
// l%16 is the wave's column 4 * (l%16) + g, so a lane ends with four rows of
// four consecutive columns and moves raw sums and dft in 16-byte (f16:
// 8-byte) pieces.
// With the sums as per-column FMAs (32 an element, plus the dl1 broadcasts)
// the kernel was bound by vector issue in f16.  ft_out 1536, b 65536: f16 273
// -> 193 us (0.8 GB, 4.2 TB/s); ft_out 512, l1 32, b 2048: 25 -> 18 us.  In f32
// memory bounds it (1.6 GB), and the step reads the raw sums here for the last
// time: with plain loads they took the last-level cache from the dft rows being
// written, and the kernel was slower than the per-column form it replaces.  The
// dense backward of a step, per-column form / plain loads / non-temporal ones, in us:
//   b 65536  ft 1536 l1 16  419 / 426 / 402   768 l1 8  202 / 210 / 194
//            640 l1 16      179 / 187 / 172   512 l1 16 150 / 161 / 154
//   b 32768  1152 l1 8      153 / 159 / 149   1024 l1 32 190 / 201 / 195
//            768 l1 8       113 / 114 / 109   512 l1 32 119 / 124 / 124
//   b 16384  1536 l1 16     118 / 121 / 116   768 l1 8  73 / 72 / 73
//            512 l1 16      76 / 61 / 60;  b 2048  512 l1 32  54 / 48 / 48
// (a whole step is not slower in any of them; workgroups of four waves gave 395 at
// 1536 but cost the step 5% at 512 l1 16, b 65536.)  The weights wait in LDS (each lane
// reads back what it wrote, so nothing is synchronised): in registers they
// cost a wave per SIMD.  The next tile's raw sums loaded ahead measured
// slower (255 us f16): 32 more registers, one wave per SIMD less.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float clamp_f16_range(float v, uint32_t& clamps) {
    if (v > 65504.0f) {
        ++clamps;
        return 65504.0f;
    }
    if (v < -65504.0f) {
        ++clamps;
        return -65504.0f;
    }
    return v;
}

template <int L1, bool H16>
__global__ __launch_bounds__(128) void ls_l1_input_post_kernel(LsDenseArgs a, uint32_t post_tiles) {
    constexpr int KC = L1 / 4;  // MFMAs per column group and gradient
    static_assert(L1 % 4 == 0, "whole MFMAs");
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    using Raw = typename std::conditional<H16, h4, floatx4>::type;
    // a lane's own weights of the current bucket: [bucket, shared][k][lane]
    __shared__ floatx4 s_w[2][KC][128];
    // f32: a wave's gradients of a tile, [row][column]
    __shared__ __align__(16) float s_g[H16 ? 1 : 2][H16 ? 1 : 16][64];
    const uint32_t ft_out = a.ft_out, half = ft_out / 2;
    const uint64_t batch = a.batch;
    const uint32_t tid = threadIdx.x, lane = tid % 64, i = lane % 16, q = lane / 16;
    // ft_out % 128 == 0: the wave's 64 columns lie in one perspective's half
    const uint32_t c = (blockIdx.x * 2 + tid / 64) * 64 + 4 * i;
    const uint32_t persp = c < half ? 0 : 1;
    const uint32_t p = c - persp * half;
    const Raw* raw = reinterpret_cast<const Raw*>(
        H16 ? static_cast<const void*>(persp ? a.ft_nstm16 : a.ft_stm16)
            : static_cast<const void*>(persp ? a.ft_nstm : a.ft_stm));
    // chunk-major dft: p and p + half are multiples of four, so a lane's run
    // lies in one chunk
    const uint64_t cstride = 2 * batch * kDftChunk;
    const uint64_t off_a = (uint64_t)(p / kDftChunk) * cstride + persp * batch * kDftChunk + p % kDftChunk;
    const uint64_t off_b =
        (uint64_t)((p + half) / kDftChunk) * cstride + persp * batch * kDftChunk + (p + half) % kDftChunk;
    Raw* dft = reinterpret_cast<Raw*>(H16 ? static_cast<void*>(a.dft16) : static_cast<void*>(a.dft));
    const floatx4 ba = *reinterpret_cast<const floatx4*>(a.ft_b + p);
    const floatx4 bb = *reinterpret_cast<const floatx4*>(a.ft_b + p + half);
#pragma unroll
    for (int k = 0; k < KC; ++k) {
        floatx4 v;
#pragma unroll
        for (int g = 0; g < 4; ++g) v[g] = a.l1s_w[(uint64_t)(c + g) * L1 + 4 * k + q];
        s_w[1][k][tid] = v;
    }
    int32_t cur_bin = -2;
    // ft_b gradients: f32, of the wave's column `lane` and of its partner, rows
    // in order; f16, of the lane's rows and columns (added up at the end)
    using Bias = typename std::conditional<H16, floatx4, float>::type;
    Bias acc_a = {}, acc_b = {};
    float(*g_t)[64] = s_g[H16 ? 0 : tid / 64];
    float* pp = a.ftb_partial + persp * ft_out + (H16 ? p : p - 4 * i + lane);
    uint32_t clamps = 0;
    const uint32_t tile0 = blockIdx.y * post_tiles;
    const uint32_t tiles_total = (uint32_t)(a.padded_b / 16);
    const uint32_t n_tiles = tile0 < tiles_total ? min(post_tiles, tiles_total - tile0) : 0u;
    if (n_tiles == 0) return;  // the grid covers whole row blocks only
    struct Tile {
        int4 rows;    // original rows of 4q .. 4q+3
        float d[KC];  // dl1 of row i, k = 4c + q
        int32_t bin;
    };
    auto load_tile = [&](uint32_t tile) -> Tile {
        Tile t;
        t.rows = *reinterpret_cast<const int4*>(a.perm + (uint64_t)tile * 16 + 4 * q);
#pragma unroll
        for (int k = 0; k < KC; ++k) t.d[k] = a.dl1_sorted[((uint64_t)tile * 16 + i) * L1 + 4 * k + q];
        t.bin = scalar_load(a.sorted_bin + (uint64_t)tile * 16);
        return t;
    };
    Tile cur = load_tile(tile0);
    for (uint32_t t = 0; t < n_tiles; ++t) {
        // the next tile's ids and dl1 (the last tile re-reads itself, unused)
        const Tile next = load_tile(t + 1 < n_tiles ? tile0 + t + 1 : tile0 + t);
        if (cur.bin >= 0) {  // else a trailing all-padding tile
            const int32_t rows[4] = {cur.rows.x, cur.rows.y, cur.rows.z, cur.rows.w};
            Raw xr[4], yr[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {  // row 0 (always valid) where the row is padding
                const uint64_t base = (uint64_t)(rows[r] >= 0 ? rows[r] : 0) * ft_out + p;
                if constexpr (H16) {
                    xr[r] = raw[base / 4];
                    yr[r] = raw[(base + half) / 4];
                } else {
                    xr[r] = __builtin_nontemporal_load(raw + base / 4);
                    yr[r] = __builtin_nontemporal_load(raw + (base + half) / 4);
                }
            }
            if (cur.bin != cur_bin) {
                cur_bin = cur.bin;
                const bool bvalid = (uint32_t)cur_bin < a.nb;
#pragma unroll
                for (int k = 0; k < KC; ++k) {
                    const floatx4 wb = *reinterpret_cast<const floatx4*>(
                        a.l1_w + ((uint64_t)(bvalid ? cur_bin : 0) * L1 + 4 * k + q) * ft_out + c);
                    s_w[0][k][tid] = bvalid ? wb : floatx4{0.f, 0.f, 0.f, 0.f};
                }
            }
            floatx4 da[4], db[4];  // [column group][row]
#pragma unroll
            for (int g = 0; g < 4; ++g) da[g] = db[g] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < KC; ++k) {
                const floatx4 w1 = s_w[0][k][tid], ws = s_w[1][k][tid];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    da[g] = mfma4(cur.d[k], w1[g], da[g]);
                    db[g] = mfma4(cur.d[k], ws[g], db[g]);
                }
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) da[g] += db[g];
            [[maybe_unused]] floatx4 gbs[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (H16 && rows[r] < 0) continue;
                floatx4 ga, gb;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float xa = (float)xr[r][g] + ba[g], xb = (float)yr[r][g] + bb[g];
                    const float dy = da[g][r];
                    const bool real = H16 || rows[r] >= 0;  // a padding row adds +0.0 (f16: skipped)
                    ga[g] = (real && xa > 0.0f && xa < 1.0f) ? dy * crelu01(xb) * a.ft_post_scale : 0.0f;
                    gb[g] = (real && xb > 0.0f && xb < 1.0f) ? dy * crelu01(xa) * a.ft_post_scale : 0.0f;
                }
                if constexpr (H16) {
                    acc_a += ga;
                    acc_b += gb;
                } else {
                    *reinterpret_cast<floatx4*>(&g_t[4 * q + r][4 * i]) = ga;
                    gbs[r] = gb;
                }
                if (!H16 && rows[r] < 0) continue;
                const uint64_t row = (uint64_t)rows[r] * kDftChunk;
                if constexpr (H16) {
                    floatx4 va = ga * a.dft_scale, vb = gb * a.dft_scale;
                    // one test of the largest magnitude (a NaN is ignored and
                    // passes, uncounted) keeps the clamps off the usual path
                    float top = 0.0f;
#pragma unroll
                    for (int g = 0; g < 4; ++g) top = fmaxf(top, fmaxf(fabsf(va[g]), fabsf(vb[g])));
                    if (top > 65504.0f) {
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            va[g] = clamp_f16_range(va[g], clamps);
                            vb[g] = clamp_f16_range(vb[g], clamps);
                        }
                    }
                    dft[(off_a + row) / 4] = __builtin_convertvector(va, h4);
                    dft[(off_b + row) / 4] = __builtin_convertvector(vb, h4);
                } else {
                    dft[(off_a + row) / 4] = ga;
                    dft[(off_b + row) / 4] = gb;
                }
            }
            if constexpr (!H16) {
                // the rows' gradients added in row order, a column per lane,
                // through the wave's own LDS (a wave's LDS accesses complete
                // in order)
                auto in_order = [&](float& acc) {
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int rr = 0; rr < 16; ++rr) acc += g_t[rr][lane];
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                };
                in_order(acc_a);
#pragma unroll
                for (int r = 0; r < 4; ++r) *reinterpret_cast<floatx4*>(&g_t[4 * q + r][4 * i]) = gbs[r];
                in_order(acc_b);
            }
        }
        if constexpr (!H16) {
            if ((t + 1) % kPostTiles == 0 || t + 1 == n_tiles) {  // the partial of these kPostTiles tiles
                float* o = pp + (uint64_t)((tile0 + t) / kPostTiles) * 2 * ft_out;
                o[0] = acc_a;
                o[half] = acc_b;
                acc_a = acc_b = 0.0f;
            }
        }
        cur = next;
    }
    if constexpr (H16) {  // the row block's partial: the four lanes of a column run hold different rows' sums
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            acc_a[g] += __shfl_xor(acc_a[g], 16);
            acc_b[g] += __shfl_xor(acc_b[g], 16);
            acc_a[g] += __shfl_xor(acc_a[g], 32);
            acc_b[g] += __shfl_xor(acc_b[g], 32);
        }
        if (q == 0) {
            float* o = pp + (uint64_t)blockIdx.y * 2 * ft_out;
            *reinterpret_cast<floatx4*>(o) = acc_a;
            *reinterpret_cast<floatx4*>(o + half) = acc_b;
        }
    }
    if (H16 && clamps) atomicAdd(a.clamp_counter, (unsigned long long)clamps);
}

// ---------------------------------------------------------------------------
// Dense gradient finalize + optimizer: one thread per parameter element of
// the nine non-FT groups (uniform_optim_group_layout order,
// trainer_layerstack.rs:676-705).
// ---------------------------------------------------------------------------
struct GroupTable {
    LsDenseGroup g[9];
    uint64_t start[10];
};

__global__ __launch_bounds__(256) void ls_dense_finalize_kernel(LsDenseArgs a, GroupTable gt,
                                                                OptScalars dense, OptScalars bias,
                                                                int32_t apply_update,
                                                                int32_t keep_grads) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= gt.start[9]) return;
    int gi = 0;
    while (i >= gt.start[gi + 1]) ++gi;
    const uint64_t e = i - gt.start[gi];
    const uint32_t l1 = a.l1, l2 = a.l2, nb = a.nb, ft_out = a.ft_out;
    const TailDims td{l1, l2, nb};
    const uint32_t cells = td.cells();
    float grad = 0.0f;
    auto tail_sum = [&](uint32_t g, uint32_t cell) { return a.tail_sum[(uint64_t)g * cells + cell]; };
    switch (gi) {
        case 0:  // ft_b: stm sum then nstm sum
            grad = a.ftb_sum[e] + a.ftb_sum[ft_out + e];
            break;
        case 1:  // l1_w [nb][l1][ft_out]: bucket segments of the chunk partials
            grad = a.w1_seg[e];
            break;
        case 2: {  // l1_b [nb][l1]
            grad = tail_sum((uint32_t)(e / l1), td.off_b1() + (uint32_t)(e % l1));
            break;
        }
        case 3: {  // l1s_w [ft_out][l1]: every bin's segment, invalid bin included
            const uint32_t k = (uint32_t)(e / l1), o = (uint32_t)(e % l1);
            float s = 0.0f;
            for (uint32_t g = 0; g <= nb; ++g) s += a.w1_seg[((uint64_t)g * l1 + o) * ft_out + k];
            grad = s;
            break;
        }
        case 4:  // l1s_b [l1]
            grad = a.b1s_sum[e];
            break;
        case 5: {  // l2_w [nb][l2][l2_in]
            const uint32_t per = l2 * td.l2_in();
            grad = tail_sum((uint32_t)(e / per), td.off_w2() + (uint32_t)(e % per));
            break;
        }
        case 6:  // l2_b [nb][l2]
            grad = tail_sum((uint32_t)(e / l2), td.off_b2() + (uint32_t)(e % l2));
            break;
        case 7:  // l3_w [nb][l2]
            grad = tail_sum((uint32_t)(e / l2), td.off_w3() + (uint32_t)(e % l2));
            break;
        default:  // l3_b [nb]
            grad = tail_sum((uint32_t)e, td.off_b3());
            break;
    }
    const LsDenseGroup& G = gt.g[gi];
    if (!apply_update) {
        G.grad[e] = grad;
        return;
    }
    OptScalars s = G.kind == 2 ? bias : dense;
    s.min_w = G.min_w;
    s.max_w = G.max_w;
    float W = G.w[e], M = G.m[e], V = G.v[e];
    radam_elem(W, M, V, grad, s);
    if (s.lookahead) {
        float S = G.slow[e];
        lerp_elem(W, S, s.alpha);
        G.slow[e] = S;
    }
    G.w[e] = W;
    G.m[e] = M;
    G.v[e] = V;
    G.grad[e] = keep_grads ? grad : 0.0f;
}

}  // namespace

uint32_t ls_tail_workgroups(uint32_t padded_b) { return ceil_div(padded_b, 16); }
uint32_t ls_post_workgroups(uint32_t padded_b) { return ceil_div(padded_b / 16, kPostTiles); }  // f16: at most
// Tiles per row block of the input-gradient kernel: eight (a column's weights
// loaded half as often) where that leaves the chip four waves per SIMD, else
// four.  Eight against four and sixteen at ft_out 1536 f16, b 65536: 211 /
// 225 / 216 us; at ft_out 512, l1 32, b 2048: 27 / 17 / 49 us.
static uint32_t post_block_tiles(uint32_t padded_b, uint32_t ft_out) {
    return (uint64_t)(padded_b / 16) * (ft_out / 64) >= 8 * 4096 ? 2 * kPostTiles : kPostTiles;
}
uint32_t ls_max_chunks(uint32_t padded_b, uint32_t nb) {
    return ceil_div(padded_b / 16, kChunkTiles) + nb + 1;
}

// Tiles from which the f32 L1 forward gives a wave two whole tiles (weights
// loaded once for 32 rows) instead of a workgroup one tile.  Dense forward
// phase, two tiles a wave / a workgroup a tile, in us:
//   b        ft 1536 l1 16   ft 768 l1 8   ft 512 l1 32   ft 256 l1 16
//   1024       96 / 45         59 / 31       77 / 47        39 / 30
//   4096      102 / 72         63 / 46       80 / 65        43 / 39
//   8192      123 / 99         75 / 60       90 / 79        48 / 45
//   16384     131 / 147        80 / 81       99 / 114       50 / 58
// The sums of few columns are short, and the line lies lower there.  A whole
// training step (and the phase):
//   b        ft 128 l1 8         ft 128 l1 32        ft 256 l1 8         ft 256 l1 32
//   3072      221 / 215 (32/29)   240 / 236 (42/38)   298 / 289 (37/29)   326 / 311 (53/38)
//   4096      230 / 229 (33/31)   251 / 254 (46/48)   314 / 302 (39/31)   338 / 329 (55/48)
//   6144      254 / 251 (36/45)   273 / 276 (50/57)   343 / 335 (44/46)   369 / 362 (58/58)
//   8192      269 / 275 (35/38)   290 / 302 (50/59)   369 / 373 (45/38)   401 / 402 (62/59)
//   10000     286 / 298 (39/41)   312 / 318 (54/60)   400 / 404 (47/40)   426 / 433 (64/62)
static uint32_t l1_pair_tiles(uint32_t ft_out) { return ft_out < 320 ? 2 * ft_out : 640; }

int32_t launch_ls_l1_forward(const LsDenseArgs& a, hipStream_t stream) {
    TATARA_REQUIRE(a.l1 >= 2 && a.l1 <= 32, "l1 must be in [2, 32]");
    TATARA_REQUIRE(a.ft_out % 64 == 0, "ft_out must be a multiple of 64");
    const bool two = a.l1 > 16;  // two blocks of 16 outputs
    TATARA_REQUIRE(!a.combined16 || (a.l1_w16 && a.l1s_wt16), "the TF32 L1 forward needs its f16 weights");
    const uint32_t tiles = a.padded_b / 16;
    if (tiles == 0) return kOk;
    if (a.combined16) {
        const uint64_t n_w = (uint64_t)a.nb * a.l1 * a.ft_out;
        ls_l1_weights_f16_kernel<<<ceil_div(n_w, 256), 256, 0, stream>>>(a);
        TATARA_LAUNCHED("ls_l1_weights_f16");
        if (two)
            ls_l1_fwd_tf32_kernel<2><<<ceil_div(tiles, 4), 256, 0, stream>>>(a);
        else
            ls_l1_fwd_tf32_kernel<1><<<ceil_div(tiles, 4), 256, 0, stream>>>(a);
    } else if (tiles < l1_pair_tiles(a.ft_out)) {
        if (two)
            ls_l1_fwd_sums_kernel<2><<<tiles, 256, 0, stream>>>(a);
        else
            ls_l1_fwd_sums_kernel<1><<<tiles, 128, 0, stream>>>(a);
    } else if (two) {
        ls_l1_fwd_kernel<2><<<ceil_div(tiles, 8), 256, 0, stream>>>(a);
    } else {
        ls_l1_fwd_kernel<1><<<ceil_div(tiles, 8), 256, 0, stream>>>(a);
    }
    TATARA_LAUNCHED("ls_l1_forward");
    return kOk;
}

int32_t launch_wrm_weight_sum(const float* score, uint32_t n, const LossParams& lp, double* out,
                              double* scratch, hipStream_t stream) {
    const uint32_t blocks = ceil_div(n, 256);
    if (blocks) {
        wrm_weight_partial_kernel<<<blocks, 256, 0, stream>>>(score, n, lp, scratch);
        TATARA_LAUNCHED("wrm_weight_sum");
    }
    sum_partials_f64_kernel<<<1, 256, 0, stream>>>(scratch, blocks, out);
    TATARA_LAUNCHED("wrm_weight_sum_reduce");
    return kOk;
}

int32_t launch_ls_tail(const LsDenseArgs& a, int32_t train, hipStream_t stream) {
    TATARA_REQUIRE(a.nb <= 16, "num_buckets must be <= 16");
    TATARA_REQUIRE(a.padded_b % 16 == 0, "the sorted batch is whole 16-row tiles");
    const uint32_t blocks = ls_tail_workgroups(a.padded_b);
    if (blocks == 0) return kOk;
    // one instantiation per accepted (l1, l2)
#define TATARA_TAIL(L1_, L2_)                                            \
    if (a.l1 == L1_ && a.l2 == L2_) {                                    \
        ls_tail_kernel<L1_, L2_><<<blocks, 64, 0, stream>>>(a, train);   \
        TATARA_LAUNCHED("ls_tail");                                      \
        return kOk;                                                      \
    }
    TATARA_TAIL(8, 16)
    TATARA_TAIL(8, 32)
    TATARA_TAIL(8, 64)
    TATARA_TAIL(16, 16)
    TATARA_TAIL(16, 32)
    TATARA_TAIL(16, 64)
    TATARA_TAIL(32, 16)
    TATARA_TAIL(32, 32)
    TATARA_TAIL(32, 64)
#undef TATARA_TAIL
    TATARA_REQUIRE(false, kLsDenseShapes);
    return kOk;
}

int32_t launch_ls_l1_weight_grad(const LsDenseArgs& a, hipStream_t stream) {
    ls_chunk_table_kernel<<<1, 256, 0, stream>>>(a.bin_start, a.bin_count, a.nb, a.max_chunks,
                                               a.chunk_info);
    TATARA_LAUNCHED("ls_chunk_table");
    dim3 grid(a.max_chunks, ceil_div(a.ft_out, 256));
    TATARA_REQUIRE(a.l1 >= 2 && a.l1 <= 32, "l1 must be in [2, 32]");
    const bool two = a.l1 > 16;
    if (a.combined16)
        (two ? ls_l1_wgrad_kernel<true, 2> : ls_l1_wgrad_kernel<true, 1>)<<<grid, 256, 0, stream>>>(a);
    else
        (two ? ls_l1_wgrad_kernel<false, 2> : ls_l1_wgrad_kernel<false, 1>)<<<grid, 256, 0, stream>>>(a);
    TATARA_LAUNCHED("ls_l1_weight_grad");
    return kOk;
}

int32_t launch_ls_l1_input_post(const LsDenseArgs& a, hipStream_t stream) {
    TATARA_REQUIRE(!a.dft16 || (a.ft_stm16 && a.ft_nstm16 && a.clamp_counter),
                   "an f16 dft needs the f16 raw sums and a clamp counter");
    const uint32_t block_tiles = post_block_tiles(a.padded_b, a.ft_out);
    const uint32_t rows = ceil_div(a.padded_b / 16, block_tiles);
    if (rows == 0) return kOk;
    TATARA_REQUIRE(a.ft_out % 128 == 0, "ft_out must be a multiple of 128");
    TATARA_REQUIRE(a.l1 == 8 || a.l1 == 16 || a.l1 == 32, kLsDenseShapes);
    const dim3 grid(a.ft_out / 128, rows);
    auto kernel = a.dft16 ? (a.l1 == 32   ? ls_l1_input_post_kernel<32, true>
                             : a.l1 == 16 ? ls_l1_input_post_kernel<16, true>
                                          : ls_l1_input_post_kernel<8, true>)
                          : (a.l1 == 32   ? ls_l1_input_post_kernel<32, false>
                             : a.l1 == 16 ? ls_l1_input_post_kernel<16, false>
                                          : ls_l1_input_post_kernel<8, false>);
    kernel<<<grid, 128, 0, stream>>>(a, block_tiles);
    TATARA_LAUNCHED("ls_l1_input_post");
    return kOk;
}

int32_t launch_ls_dense_finalize(const LsDenseArgs& a, LsDenseGroup* groups,
                                 const OptScalars& dense, const OptScalars& bias,
                                 int32_t apply_update, int32_t keep_grads, hipStream_t stream) {
    GroupTable gt;
    gt.start[0] = 0;
    for (int k = 0; k < 9; ++k) {
        gt.g[k] = groups[k];
        gt.start[k + 1] = gt.start[k] + groups[k].n;
    }
    const uint64_t n = gt.start[9];
    const TailDims td{a.l1, a.l2, a.nb};
    const uint32_t n_tail = ls_tail_workgroups(a.padded_b);
    const uint32_t n_post =
        a.dft16 ? ceil_div(a.padded_b / 16, post_block_tiles(a.padded_b, a.ft_out)) : ls_post_workgroups(a.padded_b);
    // bucket g's tile partials are the rows [tail_seg[g], tail_seg[g + 1])
    reduce_rows(a.tail_partial, n_tail, td.cells(), a.tail_seg, a.nb, a.tail_sum, stream);
    reduce_rows(a.b1s_partial, n_tail, a.l1, nullptr, 1, a.b1s_sum, stream);
    reduce_rows(a.ftb_partial, n_post, 2 * a.ft_out, nullptr, 1, a.ftb_sum, stream);
    reduce_rows(a.w1_partial, 0, a.l1 * a.ft_out, a.chunk_info + 3 * a.max_chunks + 1, a.nb + 1, a.w1_seg, stream);
    TATARA_LAUNCHED("reduce_rows");
    ls_dense_finalize_kernel<<<ceil_div(n, 256), 256, 0, stream>>>(a, gt, dense, bias, apply_update,
                                                                    keep_grads);
    TATARA_LAUNCHED("ls_dense_finalize");
    return kOk;
}

int32_t launch_ls_loss_reduce(const LsDenseArgs& a, hipStream_t stream) {
    return launch_sum_f64(a.loss_partial, ls_tail_workgroups(a.padded_b), a.loss_out, stream);
}

int32_t launch_reduce_rows(const float* P, uint32_t n_rows, uint32_t n_cols,
                           const uint32_t* seg_rows, uint32_t n_seg, float* out, hipStream_t stream) {
    TATARA_REQUIRE(seg_rows || n_seg == 1, "reduce_rows: n_seg must be 1 without segments");
    if (n_cols == 0 || n_seg == 0) return kOk;
    reduce_rows(P, n_rows, n_cols, seg_rows, n_seg, out, stream);
    TATARA_LAUNCHED("reduce_rows");
    return kOk;
}

int32_t launch_sum_f64(const double* partial, uint32_t n, double* out, hipStream_t stream) {
    sum_partials_f64_kernel<<<1, 256, 0, stream>>>(partial, n, out);
    TATARA_LAUNCHED("sum_f64");
    return kOk;
}

}  // namespace tatara
