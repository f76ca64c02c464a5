// What surrounds the column loop of a GPTQ block: the update of the columns behind the block, and the two column orders.
// amct_pytorch/quantize_op/gptq_module.py:152-153 `weight[:, i2:] -= err_block @ hinv[i1:i2, i2:]`, :122 `weight[:, perm]` and
// :155 `weight[:, invperm]`.
//
// (Layers of more than 1024 columns are updated from bf16 parts instead: gptq_parts.hip.)
// gptq_trail_k: one 128 x 64 tile of W per thread block, W <- W - E U with fp32 MFMA: the product is summed first and
// subtracted once, as in the reference, but W is read and written once instead of three times more for a product that is
// written, read and subtracted.  E and U come 32 steps of the contraction at a time through LDS, the next 32 wait in
// registers, the tile of W is asked for at the start.  Bound by the fp32 matrix pipe and, with three blocks per CU, by what
// the loads of a block leave uncovered at its start.  Behind 128 columns of W[4096,4096]: 58.6 us for 3968 trailing columns
// (71 TFLOP/s; the register-only loop reaches 150), 32.0 for 2048, 9.4 for 256; the library's product and subtraction
// 87, 42, 28.  128 x 64 because the trailing part shrinks to nothing over the blocks of a layer: 64-row tiles read half as
// much again from L2, 128-column tiles leave CUs idle earlier.
// gptq_order_k: W[4096,4096] bf16, 21 us there and 22 back (indexing with the conversions around it 150 and 130).
#include "amct_common.h"

namespace amct {

typedef float t16f __attribute__((ext_vector_type(16)));
typedef float t4f __attribute__((ext_vector_type(4)));

constexpr int kTrRows = 128, kTrCols = 64, kTrK = 32;
constexpr int kTrLda = kTrK + 4, kTrLdb = kTrCols + 4;      // LDS strides in floats: 16-byte rows, 4 banks apart

struct TrailArgs {
    float* w;                                       // [rows][ld_w], at the first trailing column
    const float* err;                               // [rows][ld_e]
    const float* u;                                 // [count][ld_u], at the first trailing column
    int64_t ld_w, ld_e, ld_u, rows, cols;
    int count;
    int col_tiles;
};

// VEC: every row of the three matrices starts 16-byte aligned and count and cols are multiples of 4
template <bool VEC>
__global__ __launch_bounds__(kBlock) void gptq_trail_k(TrailArgs a) {
    __shared__ __align__(16) float ta[kTrRows * kTrLda], tb[kTrK * kTrLdb];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int64_t r0 = (int64_t)(blockIdx.x / (unsigned)a.col_tiles) * kTrRows;
    const int64_t c0 = (int64_t)(blockIdx.x % (unsigned)a.col_tiles) * kTrCols;
    // global -> registers -> LDS: a thread holds 4 consecutive floats of rows ar + 32 i of E and rows br + 16 i of U
    const int ar = tid >> 3, ak = (tid & 7) * 4;
    const int br = tid >> 4, bc = (tid & 15) * 4;
    const int64_t cb = c0 + bc;
    t4f va[4], vb[2];
    const float* pe[4];
    const float* pu[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) pe[i] = a.err + min(r0 + ar + 32 * i, a.rows - 1) * a.ld_e + ak;   // rows beyond: not stored
#pragma unroll
    for (int i = 0; i < 2; ++i) pu[i] = a.u + (int64_t)(br + 16 * i) * a.ld_u + cb;
    // whole block: every column is there; a stage of 32 steps is whole too, but for the last one of a short block
    const bool wide = c0 + kTrCols <= a.cols;
    auto load = [&](int k0) {
        if (VEC && wide && k0 + kTrK <= a.count) {
#pragma unroll
            for (int i = 0; i < 4; ++i) va[i] = *reinterpret_cast<const t4f*>(pe[i] + k0);
#pragma unroll
            for (int i = 0; i < 2; ++i) vb[i] = *reinterpret_cast<const t4f*>(pu[i] + (int64_t)k0 * a.ld_u);
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) va[i][e] = k0 + ak + e < a.count ? pe[i][k0 + e] : 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                vb[i][e] = k0 + br + 16 * i < a.count && cb + e < a.cols ? pu[i][(int64_t)k0 * a.ld_u + e] : 0.f;
    };
    auto store = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<t4f*>(ta + (ar + 32 * i) * kTrLda + ak) = va[i];
#pragma unroll
        for (int i = 0; i < 2; ++i) *reinterpret_cast<t4f*>(tb + (br + 16 * i) * kTrLdb + bc) = vb[i];
    };
    // wave: rows 32 wave .. + 31, all 64 columns in two MFMA tiles; lane: row / column lane % 32, four steps 4 (lane / 32) ..
    const int fr = lane & 31, fh = lane >> 5;
    const float* pa = ta + (32 * wave + fr) * kTrLda + 4 * fh;
    const float* pb = tb + 4 * fh * kTrLdb + fr;
    t16f acc[2];
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int x = 0; x < 16; ++x) acc[n][x] = 0.f;
    load(0);
    // acc[n][x]: row 8 (x / 4) + x % 4 behind rw, column 32 n + fr of the tile.  The tile of W is asked for behind the first
    // stage and needed behind the last.
    const int64_t rw = r0 + 32 * wave + 4 * fh;
    const bool inside = wide && r0 + kTrRows <= a.rows;      // whole block: no edge
    float* wp = a.w + rw * a.ld_w + c0 + fr;
    float old[2][16];
    if (inside) {
#pragma unroll
        for (int x = 0; x < 16; ++x) {
            const float* p = wp + (8 * (x / 4) + x % 4) * a.ld_w;
            old[0][x] = p[0];
            old[1][x] = p[32];
        }
    } else {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int x = 0; x < 16; ++x) {
                const int r = 8 * (x / 4) + x % 4;
                old[n][x] = rw + r < a.rows && c0 + 32 * n + fr < a.cols ? wp[r * a.ld_w + 32 * n] : 0.f;
            }
    }
    t4f fa[2];
    float fb[2][2][4];
    auto frag = [&](int s, int k) {
        fa[s] = *reinterpret_cast<const t4f*>(pa + k);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int n = 0; n < 2; ++n) fb[s][n][e] = pb[(k + e) * kTrLdb + 32 * n];
    };
    for (int k0 = 0; k0 < a.count; k0 += kTrK) {
        if (k0) __syncthreads();                    // everyone has read the stage before
        store();
        __syncthreads();
        if (k0 + kTrK < a.count) load(k0 + kTrK);
        frag(0, 0);
#pragma unroll
        for (int k = 0; k < kTrK; k += 8) {
            const int s = (k / 8) & 1;
            __builtin_amdgcn_sched_barrier(0);      // the next fragments are read under this one's products
            if (k + 8 < kTrK) frag(s ^ 1, k + 8);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int n = 0; n < 2; ++n) acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[s][e], fb[s][n][e], acc[n], 0, 0, 0);
        }
    }
    if (inside) {
#pragma unroll
        for (int x = 0; x < 16; ++x) {
            float* p = wp + (8 * (x / 4) + x % 4) * a.ld_w;
            p[0] = old[0][x] - acc[0][x];
            p[32] = old[1][x] - acc[1][x];
        }
    } else {
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int x = 0; x < 16; ++x) {
                const int r = 8 * (x / 4) + x % 4;
                if (rw + r < a.rows && c0 + 32 * n + fr < a.cols) wp[r * a.ld_w + 32 * n] = old[n][x] - acc[n][x];
            }
    }
}

// Column order of the weight, four rows per thread block through LDS so that memory sees whole lines both ways (picked
// column by column from memory a row costs a 64-byte sector per element).  Columns come in pieces of kPmCols.
//   GATHER: out[r][c] = dead[perm[c]] ? 0 : in[r][perm[c]], out fp32      (into the order of the Hessian's diagonal)
//   else:   out[r][perm[c]] = in[r][c], in fp32                            (and back)
constexpr int kPmRows = 4, kPmCols = 4096, kPmBlock = 512;

template <int DT, bool GATHER>
__global__ __launch_bounds__(kPmBlock) void gptq_order_k(const void* in, void* out, const int64_t* perm, const uint8_t* dead, int64_t rows,
                                                         int64_t cols) {
    __shared__ __align__(16) float piece[kPmCols][kPmRows];   // the four rows of a column side by side: one 16-byte access per column
    const int tid = threadIdx.x;
    const int64_t r0 = (int64_t)blockIdx.x * kPmRows;
    int64_t row[kPmRows];
#pragma unroll
    for (int r = 0; r < kPmRows; ++r) row[r] = min(r0 + r, rows - 1) * cols;       // rows beyond the matrix repeat its last one
    for (int64_t q0 = 0; q0 < cols; q0 += kPmCols) {
        const int np = (int)min((int64_t)kPmCols, cols - q0);
        if (q0) __syncthreads();
        if constexpr (GATHER) {
            for (int q = tid; q < np; q += kPmBlock) {
                const bool zero = dead[q0 + q] != 0;
                float v[kPmRows];
#pragma unroll
                for (int r = 0; r < kPmRows; ++r) v[r] = load_scalar<DT>(in, row[r] + q0 + q);
                *reinterpret_cast<float4*>(piece[q]) = zero ? make_float4(0.f, 0.f, 0.f, 0.f) : make_float4(v[0], v[1], v[2], v[3]);
            }
            __syncthreads();
            for (int64_t c = tid; c < cols; c += kPmBlock) {
                const int64_t q = perm[c] - q0;
                if (q < 0 || q >= np) continue;
                const float4 v = *reinterpret_cast<const float4*>(piece[q]);
                const float f[kPmRows] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int r = 0; r < kPmRows; ++r) reinterpret_cast<float*>(out)[row[r] + c] = f[r];
            }
        } else {
            for (int64_t c = tid; c < cols; c += kPmBlock) {
                const int64_t q = perm[c] - q0;
                if (q < 0 || q >= np) continue;
                float f[kPmRows];
#pragma unroll
                for (int r = 0; r < kPmRows; ++r) f[r] = reinterpret_cast<const float*>(in)[row[r] + c];
                *reinterpret_cast<float4*>(piece[q]) = make_float4(f[0], f[1], f[2], f[3]);
            }
            __syncthreads();
            for (int q = tid; q < np; q += kPmBlock) {
                const float4 v = *reinterpret_cast<const float4*>(piece[q]);
                const float f[kPmRows] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int r = 0; r < kPmRows; ++r) store_scalar<DT>(out, row[r] + q0 + q, f[r]);
            }
        }
    }
}

}  // namespace amct

using namespace amct;

extern "C" int amct_gptq_trail(float* w, int64_t ld_w, const float* err, int64_t ld_e, const float* u, int64_t ld_u, int64_t rows,
                               int64_t cols, int count, amct_stream_t stream) {
    if (rows < 0 || cols < 0 || count < 0 || ld_w < cols || ld_e < count || ld_u < cols) return AMCT_E_BADARG;
    if (rows == 0 || cols == 0 || count == 0) return AMCT_OK;
    if (!w || !err || !u) return AMCT_E_BADARG;
    const int64_t rt = (rows + kTrRows - 1) / kTrRows, ct = (cols + kTrCols - 1) / kTrCols;
    if (rt > 0x7FFFFFFF / ct) return AMCT_E_TOO_LARGE;
    const TrailArgs a{w, err, u, ld_w, ld_e, ld_u, rows, cols, count, (int)ct};
    const bool vec = count % 4 == 0 && cols % 4 == 0 && ld_e % 4 == 0 && ld_u % 4 == 0 && aligned16(err) && aligned16(u);
    const dim3 grid((unsigned)(rt * ct));
    if (vec) hipLaunchKernelGGL(gptq_trail_k<true>, grid, dim3(kBlock), 0, (hipStream_t)stream, a);
    else hipLaunchKernelGGL(gptq_trail_k<false>, grid, dim3(kBlock), 0, (hipStream_t)stream, a);
    return hip_status();
}

extern "C" int amct_gptq_order(const void* in, void* out, const int64_t* perm, const uint8_t* dead, int64_t rows, int64_t cols,
                               int back, int dtype, amct_stream_t stream) {
    if (rows < 0 || cols < 0) return AMCT_E_BADARG;
    if (dtype != AMCT_F32 && dtype != AMCT_F16 && dtype != AMCT_BF16) return AMCT_E_BADARG;
    if (rows == 0 || cols == 0) return AMCT_OK;
    if (!in || !out || !perm || (!back && !dead)) return AMCT_E_BADARG;
    const int64_t nb = (rows + kPmRows - 1) / kPmRows;
    if (nb > 0x7FFFFFFF) return AMCT_E_TOO_LARGE;
    const dim3 grid((unsigned)nb);
    hipStream_t st = (hipStream_t)stream;
#define AMCT_ORDER(DT)                                                                                                       \
    if (back) hipLaunchKernelGGL((gptq_order_k<DT, false>), grid, dim3(kPmBlock), 0, st, in, out, perm, dead, rows, cols);     \
    else hipLaunchKernelGGL((gptq_order_k<DT, true>), grid, dim3(kPmBlock), 0, st, in, out, perm, dead, rows, cols);
    switch (dtype) {
        case AMCT_F32: AMCT_ORDER(AMCT_F32) break;
        case AMCT_F16: AMCT_ORDER(AMCT_F16) break;
        default: AMCT_ORDER(AMCT_BF16) break;
    }
#undef AMCT_ORDER
    return hip_status();
}
