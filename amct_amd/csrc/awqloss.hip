// Loss of one AWQ grid point: mean((y - yhat)^4) over all elements of two tensors of one dtype.
// Replaces the expression of amct_pytorch/algorithm/awq.py:96 `(ori_out - quant_out).float().pow(4).mean()`,
// which runs as four kernels and seven passes over the data, by one pass that reads both tensors once.
// The difference is rounded to the tensors' dtype before it is widened, as the reference's subtraction does;
// d^4 is (d*d)*(d*d) in fp32.  The sum is deterministic: a fixed number of blocks, each a fixed partition of the
// elements, per-block partials folded in a fixed order by one block (pass 2), which also divides by n.
// The order of summation differs from torch's, so results agree to fp32 rounding of the sum, not bit for bit.
#include <algorithm>

#include "amct_common.h"

namespace amct {

constexpr int kLossBlocks = 1024;      // partials (fixed, so the summation order does not depend on the device)
constexpr int kLossUnroll = 4;         // 16-byte vectors of each tensor in flight per lane

template <int DT> AMCT_DEV float loss_elem(const void* p, int64_t i) {
    if constexpr (DT == AMCT_F32) return reinterpret_cast<const float*>(p)[i];
    else if constexpr (DT == AMCT_BF16) return bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p)[i]);
    else return f16_bits_to_f32(reinterpret_cast<const uint16_t*>(p)[i]);
}

template <int DT>
__global__ __launch_bounds__(kBlock) void awq_loss_partial_k(const void* y, const void* yhat, int64_t n, float* partial) {
    constexpr int VEC = Tr<DT>::VEC;
    __shared__ float red[kBlock / 64];
    const int tid = threadIdx.x;
    const int64_t nvec = n / VEC;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    float s[kLossUnroll];
#pragma unroll
    for (int u = 0; u < kLossUnroll; ++u) s[u] = 0.f;
    const char* py = reinterpret_cast<const char*>(y);
    const char* ph = reinterpret_cast<const char*>(yhat);
    // vector v of the tensors belongs to lane v % stride; a lane keeps kLossUnroll running sums (vector u of its
    // iteration goes to sum u), so the partition and the order are fixed by n alone
    for (int64_t v0 = (int64_t)blockIdx.x * kBlock + tid; v0 < nvec; v0 += stride * kLossUnroll) {
        uint4 ra[kLossUnroll], rb[kLossUnroll];
#pragma unroll
        for (int u = 0; u < kLossUnroll; ++u) {
            const int64_t v = v0 + u * stride;
            const int64_t vc = v < nvec ? v : nvec - 1;              // unconditional loads, clamped
            ra[u] = ldg16_nt(py + vc * 16);
            rb[u] = ldg16_nt(ph + vc * 16);
        }
#pragma unroll
        for (int u = 0; u < kLossUnroll; ++u) {
            if (v0 + u * stride < nvec) {
                float a[VEC], b[VEC];
                unpack16<DT>(ra[u], a);
                unpack16<DT>(rb[u], b);
#pragma unroll
                for (int j = 0; j < VEC; ++j) {
                    const float d = round_to<DT>(a[j] - b[j]);
                    const float d2 = d * d;
                    s[u] = s[u] + d2 * d2;
                }
            }
        }
    }
    // the n % VEC elements behind the last whole vector: lane 0 of block 0
    if (blockIdx.x == 0 && tid == 0) {
        for (int64_t i = nvec * VEC; i < n; ++i) {
            const float d = round_to<DT>(loss_elem<DT>(y, i) - loss_elem<DT>(yhat, i));
            const float d2 = d * d;
            s[0] = s[0] + d2 * d2;
        }
    }
    float t = (s[0] + s[1]) + (s[2] + s[3]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) t = t + __shfl_xor(t, off, 64);
    if ((tid & 63) == 0) red[tid >> 6] = t;
    __syncthreads();
    if (tid == 0) {
        float b = red[0];
#pragma unroll
        for (int w = 1; w < kBlock / 64; ++w) b = b + red[w];
        partial[blockIdx.x] = b;
    }
}

// one block: lane l folds partials l, l + 256, ... in order, then the lanes meet; result / n
__global__ __launch_bounds__(kBlock) void awq_loss_final_k(const float* partial, int nparts, int64_t n, float* loss) {
    __shared__ float red[kBlock / 64];
    const int tid = threadIdx.x;
    float t = 0.f;
    for (int i = tid; i < nparts; i += kBlock) t = t + partial[i];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) t = t + __shfl_xor(t, off, 64);
    if ((tid & 63) == 0) red[tid >> 6] = t;
    __syncthreads();
    if (tid == 0) {
        float b = red[0];
#pragma unroll
        for (int w = 1; w < kBlock / 64; ++w) b = b + red[w];
        loss[0] = b / (float)n;
    }
}

// All candidate scales of a search in one launch, a thread block per grid point (amct_pytorch/algorithm/awq.py:85-88):
// mean ** ratio rounded to the activations' dtype and clamped at 1e-4, divided in fp64 by the geometric mean of its extremes,
// rounded to the dtype and clamped into [1e-4, largest finite].  As thirteen library launches per grid point these took
// longer than the fake-quantised weight they are for.  The powers are kept in the output between the two passes.
// 16 waves a block: a grid point is one block's work, and powers and fp64 quotients are long chains (20 points of 4096
// columns: 15.5 us with 4 waves, now 8.9).
constexpr int kCandThreads = 1024;
template <int DT> AMCT_DEV float dtype_max() { return DT == AMCT_F16 ? 65504.f : DT == AMCT_BF16 ? 3.38953138925153547590e38f : 3.40282346638528859812e38f; }
// torch.clamp of a value of the dtype: NaN stays NaN, the bound is rounded to the dtype
template <int DT> AMCT_DEV float clamp_low(float v) {
    const float lo = round_to<DT>(1e-4f);
    return v < lo ? lo : v;
}

template <int DT>
__global__ __launch_bounds__(kCandThreads) void awq_candidates_k(const void* mean, const float* ratios, void* out, int64_t cols) {
    __shared__ float smx[kCandThreads / 64], smn[kCandThreads / 64];
    const int tid = threadIdx.x;
    const float ratio = ratios[blockIdx.x];
    const int64_t base = (int64_t)blockIdx.x * cols;
    float mx = -__builtin_inff(), mn = __builtin_inff();
    for (int64_t c = tid; c < cols; c += kCandThreads) {
        const float x = load_scalar<DT>(mean, c);
        // the square root and the zeroth power as such, as the library's power does
        const float p = ratio == 0.5f ? sqrtf(x) : ratio == 0.f ? 1.f : powf(x, ratio);
        const float v = clamp_low<DT>(round_to<DT>(p));
        store_scalar<DT>(out, base + c, v);
        mx = fmax_nan(mx, v);
        mn = fmin_nan(mn, v);
    }
    team_minmax<64>(mn, mx);
    if ((tid & 63) == 0) {
        smx[tid >> 6] = mx;
        smn[tid >> 6] = mn;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kCandThreads / 64; ++w) {
        mx = fmax_nan(mx, smx[w]);
        mn = fmin_nan(mn, smn[w]);
    }
    const double norm = sqrt((double)mx * (double)mn);
    for (int64_t c = tid; c < cols; c += kCandThreads) {                 // a thread reads back what it wrote
        const double q = (double)load_scalar<DT>(out, base + c) / norm;
        const float v = clamp_low<DT>(round_to<DT>((float)q));
        store_scalar<DT>(out, base + c, v > dtype_max<DT>() ? dtype_max<DT>() : v);
    }
}

// The losses of a search from the partials of its grid points (kLossBlocks apart), folded as awq_loss_final_k folds them,
// and the first grid point whose loss is below infinity and below every earlier one: -1 if there is none.
// One block; a wave folds a quarter of a grid point's partials (lane l of quarter w those of l + 64 w, + 256, ...) with the
// loads of four quarters in flight, kPickGrids grid points between two barriers.  Bound by the latency of its loads: one grid
// point after the other, each behind the barriers of the one before, took 19 us for 20 of them, now 4.5 us.
constexpr int kPickThreads = 1024;
constexpr int kPickGrids = 64;                      // a lane of the first wave each, for the choice
constexpr int kPickLoads = kLossBlocks / kBlock;   // partials of a lane at most

__global__ __launch_bounds__(kPickThreads) void awq_pick_k(const float* partials, int nparts, int64_t n, int grids, float* losses, int32_t* winner) {
    constexpr int W = kBlock / 64, kWaves = kPickThreads / 64, kTasks = 4;
    __shared__ float red[kPickGrids * W];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float best = __builtin_inff();
    int at = -1;
    for (int g0 = 0; g0 < grids; g0 += kPickGrids) {
        const int count = grids - g0 < kPickGrids ? grids - g0 : kPickGrids;
        if (g0) __syncthreads();
        for (int t0 = wave; t0 < count * W; t0 += kWaves * kTasks) {
            float p[kTasks][kPickLoads];
#pragma unroll
            for (int k = 0; k < kTasks; ++k) {
                const int t = t0 + k * kWaves < count * W ? t0 + k * kWaves : t0;
                const float* src = partials + (int64_t)(g0 + t / W) * kLossBlocks;
#pragma unroll
                for (int l = 0; l < kPickLoads; ++l) {
                    const int i = (t % W) * 64 + lane + l * kBlock;
                    p[k][l] = src[i < nparts ? i : nparts - 1];
                }
            }
#pragma unroll
            for (int k = 0; k < kTasks; ++k) {
                const int t = t0 + k * kWaves;
                if (t >= count * W) break;
                float sum = 0.f;
#pragma unroll
                for (int l = 0; l < kPickLoads; ++l) {
                    if ((t % W) * 64 + lane + l * kBlock < nparts) sum = sum + p[k][l];
                }
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) sum = sum + __shfl_xor(sum, off, 64);
                if (lane == 0) red[t] = sum;
            }
        }
        __syncthreads();
        if (wave == 0) {
            float b = __builtin_inff();
            int mine = 0x7FFFFFFF;
            if (lane < count) {
                float v = red[lane * W];
#pragma unroll
                for (int w = 1; w < W; ++w) v = v + red[lane * W + w];
                v = v / (float)n;
                losses[g0 + lane] = v;
                if (v < b) {                         // false for NaN
                    b = v;
                    mine = g0 + lane;
                }
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                const float ob = __shfl_xor(b, off, 64);
                const int om = __shfl_xor(mine, off, 64);
                if (ob < b || (ob == b && om < mine)) {
                    b = ob;
                    mine = om;
                }
            }
            if (b < best) {
                best = b;
                at = mine;
            }
        }
    }
    if (tid == 0) *winner = at;
}

// *flag = 1 where x holds an infinity or a NaN: the check in front of a search, one pass where isfinite().all() makes five
template <int DT>
__global__ __launch_bounds__(kBlock) void nonfinite_k(const void* x, int64_t n, int vec_ok, int32_t* flag) {
    constexpr int VEC = Tr<DT>::VEC;
    bool bad = false;
    const int64_t nvec = vec_ok ? n / VEC : 0, stride = (int64_t)gridDim.x * kBlock;
    for (int64_t v0 = (int64_t)blockIdx.x * kBlock + threadIdx.x; v0 < nvec; v0 += stride * kLossUnroll) {
        uint4 raw[kLossUnroll];
#pragma unroll
        for (int u = 0; u < kLossUnroll; ++u) {
            const int64_t v = v0 + u * stride;
            raw[u] = ldg16(reinterpret_cast<const char*>(x) + (v < nvec ? v : nvec - 1) * 16);
        }
#pragma unroll
        for (int u = 0; u < kLossUnroll; ++u) {
            float f[VEC];
            unpack16<DT>(raw[u], f);
#pragma unroll
            for (int j = 0; j < VEC; ++j) bad = bad || !finite_f(f[j]);
        }
    }
    for (int64_t i = nvec * VEC + (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) bad = bad || !finite_f(load_scalar<DT>(x, i));
    if (bad) *flag = 1;
}

}  // namespace amct

using namespace amct;

static int loss_blocks(int64_t n, int dtype) {
    const int vec = dtype == AMCT_F32 ? 4 : 8;
    const int64_t blocks = (n / vec + (int64_t)kBlock * kLossUnroll - 1) / ((int64_t)kBlock * kLossUnroll);
    return (int)std::min<int64_t>(std::max<int64_t>(blocks, 1), kLossBlocks);
}

// n == 0: the mean of nothing is 0 / 0 = NaN, as torch's; this pass then writes zeros
static void loss_partials(const void* y, const void* yhat, int64_t n, int dtype, int blocks, float* partial, hipStream_t st) {
    const dim3 grid((unsigned)blocks);
    if (dtype == AMCT_F32) hipLaunchKernelGGL((awq_loss_partial_k<AMCT_F32>), grid, dim3(kBlock), 0, st, y, yhat, n, partial);
    else if (dtype == AMCT_F16) hipLaunchKernelGGL((awq_loss_partial_k<AMCT_F16>), grid, dim3(kBlock), 0, st, y, yhat, n, partial);
    else hipLaunchKernelGGL((awq_loss_partial_k<AMCT_BF16>), grid, dim3(kBlock), 0, st, y, yhat, n, partial);
}

extern "C" size_t amct_awq_loss_workspace_bytes(void) { return (size_t)kLossBlocks * sizeof(float); }

extern "C" int amct_awq_loss(const void* y, const void* yhat, int64_t n, int dtype, float* loss, void* workspace,
                             size_t workspace_bytes, amct_stream_t stream) {
    if (n < 0 || !loss) return AMCT_E_BADARG;
    if (dtype != AMCT_F32 && dtype != AMCT_F16 && dtype != AMCT_BF16) return AMCT_E_BADARG;
    if (n != 0 && (!y || !yhat)) return AMCT_E_BADARG;
    if (!workspace || workspace_bytes < amct_awq_loss_workspace_bytes() || ((uintptr_t)workspace & 3)) return AMCT_E_BADARG;
    if (n != 0 && (!aligned16(y) || !aligned16(yhat))) return AMCT_E_ALIGN;
    float* partial = reinterpret_cast<float*>(workspace);
    const int blocks = loss_blocks(n, dtype);
    loss_partials(y, yhat, n, dtype, blocks, partial, (hipStream_t)stream);
    hipLaunchKernelGGL(awq_loss_final_k, dim3(1), dim3(kBlock), 0, (hipStream_t)stream, partial, blocks, n, loss);
    return hip_status();
}

static bool loss_args_ok(int64_t n, int dtype) { return n >= 0 && (dtype == AMCT_F32 || dtype == AMCT_F16 || dtype == AMCT_BF16); }

extern "C" int amct_awq_loss_partials(const void* y, const void* yhat, int64_t n, int dtype, float* partials, amct_stream_t stream) {
    if (!loss_args_ok(n, dtype) || !partials || (n != 0 && (!y || !yhat))) return AMCT_E_BADARG;
    if (n != 0 && (!aligned16(y) || !aligned16(yhat))) return AMCT_E_ALIGN;
    loss_partials(y, yhat, n, dtype, loss_blocks(n, dtype), partials, (hipStream_t)stream);
    return hip_status();
}

extern "C" int amct_awq_pick(const float* partials, int64_t n, int dtype, int grids, float* losses, int32_t* winner, amct_stream_t stream) {
    if (!loss_args_ok(n, dtype) || grids <= 0 || !partials || !losses || !winner) return AMCT_E_BADARG;
    hipLaunchKernelGGL(awq_pick_k, dim3(1), dim3(kPickThreads), 0, (hipStream_t)stream, partials, loss_blocks(n, dtype), n, grids, losses, winner);
    return hip_status();
}

extern "C" int amct_awq_candidates(const void* mean, const float* ratios, void* out, int grids, int64_t cols, int dtype,
                                   amct_stream_t stream) {
    if (grids < 0 || cols < 0) return AMCT_E_BADARG;
    if (grids == 0 || cols == 0) return AMCT_OK;
    if (!mean || !ratios || !out) return AMCT_E_BADARG;
    const dim3 grid((unsigned)grids);
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case AMCT_F32: hipLaunchKernelGGL((awq_candidates_k<AMCT_F32>), grid, dim3(kCandThreads), 0, st, mean, ratios, out, cols); break;
        case AMCT_F16: hipLaunchKernelGGL((awq_candidates_k<AMCT_F16>), grid, dim3(kCandThreads), 0, st, mean, ratios, out, cols); break;
        case AMCT_BF16: hipLaunchKernelGGL((awq_candidates_k<AMCT_BF16>), grid, dim3(kCandThreads), 0, st, mean, ratios, out, cols); break;
        default: return AMCT_E_BADARG;
    }
    return hip_status();
}

extern "C" int amct_flag_nonfinite(const void* x, int64_t n, int dtype, int32_t* flag, amct_stream_t stream) {
    if (n < 0 || !flag) return AMCT_E_BADARG;
    if (n == 0) return AMCT_OK;
    if (!x) return AMCT_E_BADARG;
    const int vec = dtype == AMCT_F32 ? 4 : 8;
    const int64_t per = (int64_t)kBlock * kLossUnroll * vec;
    const dim3 grid((unsigned)std::min<int64_t>((n + per - 1) / per, 2048));
    const int vec_ok = aligned16(x);
    hipStream_t st = (hipStream_t)stream;
    switch (dtype) {
        case AMCT_F32: hipLaunchKernelGGL((nonfinite_k<AMCT_F32>), grid, dim3(kBlock), 0, st, x, n, vec_ok, flag); break;
        case AMCT_F16: hipLaunchKernelGGL((nonfinite_k<AMCT_F16>), grid, dim3(kBlock), 0, st, x, n, vec_ok, flag); break;
        case AMCT_BF16: hipLaunchKernelGGL((nonfinite_k<AMCT_BF16>), grid, dim3(kBlock), 0, st, x, n, vec_ok, flag); break;
        default: return AMCT_E_BADARG;
    }
    return hip_status();
}
