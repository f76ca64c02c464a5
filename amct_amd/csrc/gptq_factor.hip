// GPTQ: from the calibration Hessian to the factor that the column loop divides by and multiplies with.
// amct_pytorch/quantize_op/gptq_module.py:108-121 takes three library factorisations: chol(H), its inverse, and the upper
// Cholesky factor U of that inverse (H^-1 = U^T U).  With J the reversal of the index order, J H J = L L^T gives
// U = J L^-1 J: ONE Cholesky factorisation and ONE triangular inverse, k^3 / 3 multiply-adds each way, and no second
// factorisation of an already rounded inverse.
//
// Both run in place in one sweep over blocks of 64 columns of a [Cp, Cp] fp32 matrix W (Cp: columns up to a multiple of
// 64, padded with the identity).  Below the block being eliminated W holds what is left of J H J (lower triangle); in the
// rows at and above it, transposed, what is left of the inverse.  Eliminating block column j:
//     (Linv, T) = inverse Cholesky factor of W[j][j] and its transpose                   one thread block
//     W[r][j]   = W[r][j] Linv^T                      for every block row r != j          gqf_panel_k
//     W[r][s]   = W[r][s] - W[r][j] W[s][j]^T         s > j;  r < j or r >= s             gqf_update_k
//     W[j][s]   =         - T W[s][j]^T               s > j
// after which W's upper triangle holds L^-T.  The tile (j + 1, j + 1) is updated by thread block 0 of gqf_update_k, which
// goes on to factor it while the other blocks update the rest.  What bounds it is the chain of dependent pivots: 64 columns
// take 6.8 us at 2.4 GHz, with the launch, the tile's update and the way to memory and back 12.5 us, which hide the
// matrix products (fp32 MFMA) of the same launch once fewer than about 1000 tiles are left (20 us at 2000 tiles).
// 4096 columns: 1.5 ms, where the library's three factorisations take 28.6 ms.  From about 8000 columns on the matrix leaves the
// last-level cache and the sweeps over it bound the call instead (one per 64 columns, 535 MB read and written on average at
// 14336): 8192 columns 6.9 ms, 11008 16.3, 14336 35.3 (3.4 TB/s, 56 TFLOP/s), 65600 3.1 s; the library 81, 154 and 262 ms.
#include <algorithm>

#include "amct_common.h"

namespace amct {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int kFb = 64;                              // columns eliminated per step
constexpr int kFld = kFb + 4;                        // row stride of a tile in LDS, in floats: 16 rows apart meet no bank

// W = J (H with zero diagonal entries set to 1, rows and columns in the order perm, + damp I) J, identity beyond C (of each
// pair H[a][b] = H[b][a] the row of the one that comes later in the reversed order is read); one row
// per thread block, up to the end of its diagonal tile.  The row of H comes in whole, in pieces of kFgRow floats through
// LDS, and is picked apart there: picked straight from memory every element costs a 64-byte sector.
constexpr int kFgRow = 16384;
// Threads of a launch over half of (kFgMax / 64)^2 tiles stay below 2^32.  (A Hessian of that many columns is 256 GiB, the
// factor and the workspace as much again each.)
constexpr int64_t kFgMax = 262144;

__global__ __launch_bounds__(kBlock) void gqf_gather_k(const float* h, const int64_t* perm, const float* damp, float* w, int64_t C,
                                                       int64_t Cp) {
    extern __shared__ float hrow[];
    const int tid = threadIdx.x;
    const int64_t i = blockIdx.x;
    float* wr = w + i * Cp;
    const int64_t cols = (i / kFb + 1) * kFb;        // of this row
    if (i >= C) {
        for (int64_t c = tid; c < cols; c += kBlock) wr[c] = c == i ? 1.f : 0.f;
        return;
    }
    const float* hr = h + perm[C - 1 - i] * C;
    for (int64_t q0 = 0; q0 < C; q0 += kFgRow) {
        const int64_t q1 = min(C, q0 + kFgRow);
        if (q0) __syncthreads();
        for (int64_t q = q0 + tid; q < q1; q += kBlock) hrow[q - q0] = hr[q];
        __syncthreads();
        for (int64_t c = tid; c < cols; c += kBlock) {
            const int64_t q = c < C ? perm[C - 1 - c] : -1;
            if (q < 0) {
                if (q0 == 0) wr[c] = 0.f;
            } else if (q >= q0 && q < q1) {
                float v = hrow[q - q0];
                if (c == i) v = (v == 0.f ? 1.f : v) + *damp;
                wr[c] = v;
            }
        }
    }
}

AMCT_DEV float lane_value(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }

// 1 / sqrt(d): the hardware estimate and one Newton step (within two units in the last place)
AMCT_DEV float rsqrt_nr(float d) {
    const float y = __builtin_amdgcn_rsqf(d);
    const float e = __builtin_fmaf(-d * y, y, 1.0f);
    return __builtin_fmaf(0.5f * y, e, y);
}

// One panel of 16 columns of the tile, one row per lane, eliminated in registers: a pivot by lane read, one product per
// later column of the panel.  The rows above the pivot (the inverse so far) take the same operations as the rows below it;
// the pivot's own row starts the inverse's next row from zero.  The next pivot's column comes first and its 1 / sqrt runs
// under the updates of the others; every lane read of a step is issued before the first product that uses one (a read and
// its product back to back wait for one another: 275 cycles a column instead of 220).  The barriers keep that order.
AMCT_DEV void factor_panel(float* t, int p, int lane, int32_t* bad) {
    float a[16];
    float* row = t + lane * kFld + 16 * p;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const f4v v = *reinterpret_cast<const f4v*>(row + 4 * i);
        a[4 * i] = v[0]; a[4 * i + 1] = v[1]; a[4 * i + 2] = v[2]; a[4 * i + 3] = v[3];
    }
    float d = lane_value(a[0], 16 * p);
    float rs = rsqrt_nr(d);
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        ok = ok && d > 0.f;
        const bool mine = lane == 16 * p + k;
        const float q = mine ? rs : a[k] * rs;
        a[k] = q;
        if (k == 15) break;
        float ls[16];
#pragma unroll
        for (int s = k + 1; s < 16; ++s) ls[s] = lane_value(q, 16 * p + s);
#pragma unroll
        for (int s = k + 1; s < 16; ++s) a[s] = mine ? 0.f : a[s];
        __builtin_amdgcn_sched_barrier(0);
        a[k + 1] = __builtin_fmaf(-q, ls[k + 1], a[k + 1]);
        d = lane_value(a[k + 1], 16 * p + k + 1);
        rs = rsqrt_nr(d);
#pragma unroll
        for (int s = k + 2; s < 16; ++s) a[s] = __builtin_fmaf(-q, ls[s], a[s]);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (!ok && lane == 0) *bad = 1;
    // inside the panel's own 16 rows only the inverse goes on (on and above the diagonal)
#pragma unroll
    for (int k = 0; k < 15; ++k) a[k] = lane > 16 * p + k && lane < 16 * p + 16 ? 0.f : a[k];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const f4v v = {a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3]};
        *reinterpret_cast<f4v*>(row + 4 * i) = v;
    }
}

// rows 16 rt .. + 15 of columns 16 s .. + 15 behind panel p: C - Q_r Q_s^T, from zero in the panel's own rows
AMCT_DEV void factor_behind(float* t, int p, int rt, int s, int lane) {
    const int fr = lane & 15, fq = lane >> 4;
    const f4v fa = *reinterpret_cast<const f4v*>(t + (16 * rt + fr) * kFld + 16 * p + 4 * fq);
    const f4v fb = *reinterpret_cast<const f4v*>(t + (16 * s + fr) * kFld + 16 * p + 4 * fq);
    float* at = t + (16 * rt + 4 * fq) * kFld + 16 * s + fr;
    float c[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) c[r] = at[r * kFld];
    f4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) at[r * kFld] = (rt == p ? 0.f : c[r]) - acc[r];
}

// The 64 x 64 tile in LDS (lower triangle meaningful) -> its inverse Cholesky factor, transposed: t[r][c] = Linv[c][r]
// on and above the diagonal.  Four column panels of 16 by wave 0; behind panel p every wave first brings 16 rows of the
// next panel up to date, then wave 0 goes on with that panel while the others do the rest.  Whole block; ends with a
// barrier.
AMCT_DEV void factor_tile(float* t, int tid, int32_t* bad) {
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (wave == 0) factor_panel(t, 0, lane, bad);
    __syncthreads();
#pragma unroll 1
    for (int p = 0; p < 3; ++p) {
        factor_behind(t, p, wave, p + 1, lane);
        __syncthreads();
        if (wave == 0) factor_panel(t, p + 1, lane, bad);
        else
            for (int x = wave - 1; x < 4 * (2 - p); x += 3) factor_behind(t, p, x & 3, p + 2 + (x >> 2), lane);
        __syncthreads();
    }
}

// Step j: every tile of W that the elimination of block column j changes (see the top).  j = -1: only the first factor.
__global__ __launch_bounds__(kBlock) void gqf_update_k(float* w, float* linv, int32_t* bad, int64_t Cp, int n, int j) {
    __shared__ __align__(16) float ta[kFb * kFld], tb[kFb * kFld];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int m = n - 1 - j;                         // block columns behind j
    int r, s;
    if (blockIdx.x == 0) {
        r = s = j + 1;
    } else {
        const int above = (j + 1) * m;
        int b = (int)blockIdx.x - 1;
        if (b < above) {
            r = b / m;
            s = j + 1 + b % m;
        } else {                                     // the lower triangle behind j without its first tile, row by row
            b = b - above + 1;
            int i = (int)((__builtin_sqrtf(8.0f * (float)b + 1.0f) - 1.0f) * 0.5f);
            while ((i + 1) * (i + 2) / 2 <= b) ++i;
            while (i * (i + 1) / 2 > b) --i;
            r = j + 1 + i;
            s = j + 1 + b - i * (i + 1) / 2;
        }
    }
    const int fr = lane & 31, fh = lane >> 5;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    float* ct = w + ((int64_t)r * kFb + wr + 4 * fh) * Cp + (int64_t)s * kFb + wc + fr;   // row 8 (x / 4) + x % 4 of it: register x
    const bool fresh = r == j;                       // the rows of the inverse that start at this step
    float c[16];
#pragma unroll
    for (int x = 0; x < 16; ++x) c[x] = fresh ? 0.f : ct[(int64_t)(8 * (x / 4) + x % 4) * Cp];
    f16v acc;
#pragma unroll
    for (int x = 0; x < 16; ++x) acc[x] = 0.f;
    if (j >= 0) {
        const float* ga = w + (int64_t)r * kFb * Cp + (int64_t)j * kFb;
        const float* gb = w + (int64_t)s * kFb * Cp + (int64_t)j * kFb;
        const int row = tid >> 4, col = (tid & 15) * 4;
        f4v va[4], vb[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            va[i] = *reinterpret_cast<const f4v*>(ga + (int64_t)(row + 16 * i) * Cp + col);
            vb[i] = *reinterpret_cast<const f4v*>(gb + (int64_t)(row + 16 * i) * Cp + col);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            *reinterpret_cast<f4v*>(ta + (row + 16 * i) * kFld + col) = va[i];
            *reinterpret_cast<f4v*>(tb + (row + 16 * i) * kFld + col) = vb[i];
        }
        __syncthreads();
        const float* pa = ta + (wr + fr) * kFld + 4 * fh;
        const float* pb = tb + (wc + fr) * kFld + 4 * fh;
#pragma unroll
        for (int k = 0; k < kFb; k += 8) {
            const f4v fa = *reinterpret_cast<const f4v*>(pa + k), fb = *reinterpret_cast<const f4v*>(pb + k);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[e], acc, 0, 0, 0);
        }
    }
    if (blockIdx.x != 0) {
#pragma unroll
        for (int x = 0; x < 16; ++x) ct[(int64_t)(8 * (x / 4) + x % 4) * Cp] = c[x] - acc[x];
        return;
    }
    // block 0: the next diagonal tile -> LDS -> its inverse factor
    __syncthreads();                                 // every wave has read its fragments of ta
#pragma unroll
    for (int x = 0; x < 16; ++x) ta[(wr + 8 * (x / 4) + 4 * fh + x % 4) * kFld + wc + fr] = c[x] - acc[x];
    __syncthreads();
    factor_tile(ta, tid, bad);
    float* wd = w + (int64_t)(j + 1) * kFb * Cp + (int64_t)(j + 1) * kFb;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int e = tid + kBlock * i, y = e >> 6, x = e & 63;
        wd[(int64_t)y * Cp + x] = x >= y ? ta[y * kFld + x] : 0.f;
        linv[e] = y >= x ? ta[x * kFld + y] : 0.f;   // row-major Linv
    }
}

// W[r][j] <- W[r][j] Linv^T for 16 rows of one block row r != j per thread block; a wave owns 16 of the 64 columns.
__global__ __launch_bounds__(kBlock) void gqf_panel_k(float* w, const float* linv, int64_t Cp, int j) {
    __shared__ __align__(16) float ta[16 * kFld], tb[kFb * kFld];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    int g = blockIdx.x;                              // group of 16 rows, those of block row j left out
    if (g >= 4 * j) g += 4;
    float* wt = w + (int64_t)g * 16 * Cp + (int64_t)j * kFb;
    {
        const int row = tid >> 4, col = (tid & 15) * 4;
        *reinterpret_cast<f4v*>(ta + row * kFld + col) = *reinterpret_cast<const f4v*>(wt + (int64_t)row * Cp + col);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<f4v*>(tb + (row + 16 * i) * kFld + col) = *reinterpret_cast<const f4v*>(linv + (row + 16 * i) * kFb + col);
    }
    __syncthreads();
    const int fr = lane & 15, fq = lane >> 4;
    f4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kFb; k += 16) {
        const f4v fa = *reinterpret_cast<const f4v*>(ta + fr * kFld + k + 4 * fq);
        const f4v fb = *reinterpret_cast<const f4v*>(tb + (16 * wave + fr) * kFld + k + 4 * fq);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], acc, 0, 0, 0);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) wt[(int64_t)(4 * fq + x) * Cp + 16 * wave + fr] = acc[x];
}

// U[a][b] = W[C - 1 - b][C - 1 - a] (b >= a), zeros below: W's upper triangle holds L^-T
__global__ __launch_bounds__(kBlock) void gqf_store_k(const float* w, float* u, int64_t C, int64_t Cp) {
    __shared__ float tile[64][65];
    const int tid = threadIdx.x;
    const int64_t a0 = (int64_t)blockIdx.y * 64, b0 = (int64_t)blockIdx.x * 64;
    const int x = tid & 63;
    if (b0 + 63 >= a0) {
        // tile[i][x] = W[C - 1 - b0 - i][C - 1 - a0 - x]: rows of W, read backwards
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int y = (tid >> 6) + 4 * i;
            const int64_t wr = C - 1 - b0 - y, wc = C - 1 - a0 - x;
            tile[y][x] = (wr >= 0 && wc >= wr) ? w[wr * Cp + wc] : 0.f;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) tile[(tid >> 6) + 4 * i][x] = 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int y = (tid >> 6) + 4 * i;
        if (a0 + y < C && b0 + x < C) u[(a0 + y) * C + b0 + x] = tile[x][y];
    }
}

}  // namespace amct

using namespace amct;

extern "C" size_t amct_gptq_factor_workspace_bytes(int64_t cols) {
    if (cols <= 0) return 0;
    const size_t cp = (size_t)((cols + kFb - 1) / kFb * kFb);
    return (cp * cp + (size_t)kFb * kFb) * sizeof(float);
}

extern "C" int amct_gptq_factor(const float* hessian, const int64_t* perm, const float* damp, float* u, int32_t* bad, int64_t cols,
                                void* workspace, size_t workspace_bytes, amct_stream_t stream) {
    if (cols <= 0 || !hessian || !perm || !damp || !u || !bad || !workspace) return AMCT_E_BADARG;
    if (cols > kFgMax) return AMCT_E_TOO_LARGE;
    if (workspace_bytes < amct_gptq_factor_workspace_bytes(cols)) return AMCT_E_BADARG;
    if (!aligned16(workspace)) return AMCT_E_ALIGN;
    hipStream_t st = (hipStream_t)stream;
    const int64_t Cp = (cols + kFb - 1) / kFb * kFb;
    const int n = (int)(Cp / kFb);
    float* linv = (float*)workspace;
    float* w = linv + kFb * kFb;
    hipLaunchKernelGGL(gqf_gather_k, dim3((unsigned)Cp), dim3(kBlock), (size_t)std::min<int64_t>(cols, kFgRow) * sizeof(float), st,
                       hessian, perm, damp, w, cols, Cp);
    hipLaunchKernelGGL(gqf_update_k, dim3(1), dim3(kBlock), 0, st, w, linv, bad, Cp, n, -1);
    for (int j = 0; j < n; ++j) {
        if (n > 1) hipLaunchKernelGGL(gqf_panel_k, dim3((unsigned)(4 * (n - 1))), dim3(kBlock), 0, st, w, linv, Cp, j);
        const int m = n - 1 - j;
        if (m == 0) break;
        hipLaunchKernelGGL(gqf_update_k, dim3((unsigned)((j + 1) * m + m * (m + 1) / 2)), dim3(kBlock), 0, st, w, linv, bad, Cp, n, j);
    }
    hipLaunchKernelGGL(gqf_store_k, dim3((unsigned)n, (unsigned)n), dim3(kBlock), 0, st, w, u, cols, Cp);
    return hip_status();
}
