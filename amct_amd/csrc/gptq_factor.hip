// GPTQ: from the calibration Hessian to the factor that the column loop divides by and multiplies with.
// amct_pytorch/quantize_op/gptq_module.py:108-121 takes three library factorisations: chol(H), its inverse, and the upper
// Cholesky factor U of that inverse (H^-1 = U^T U).  With J the reversal of the index order, J H J = L L^T gives
// U = J L^-1 J: ONE Cholesky factorisation and ONE triangular inverse, k^3 / 3 multiply-adds each way, and no second
// factorisation of an already rounded inverse.
//
// Both run in place in one sweep over blocks of 64 columns of a [Cp, Cp] fp32 matrix W (Cp: columns up to a multiple of
// 64, padded with the identity).  Below the block being eliminated W holds what is left of J H J (lower triangle); in the
// rows at and above it, transposed, what is left of the inverse.  Eliminating block column j:
//     (Linv, T) = inverse Cholesky factor of W[j][j] and its transpose
//     P[r]      = W[r][j] Linv^T for every block row r != j;  P[j] = T
//     W[r][s]   = W[r][s] - P[r] P[s]^T         s > j;  r < j or r >= s
//     W[j][s]   =         - T P[s]^T            s > j
// after which W's upper triangle holds L^-T (W[r][j] = P[r] for r < j, W[j][j] = T).
// One launch per block column.  What bounds a step is a chain: the last update of tile (j + 1, j + 1), its 64 dependent
// pivots, then the panel that needs its inverse.  Launch j takes the chain on: its first n blocks, one per block row r, form
// P[r] (and, each for itself, P[j + 1]), bring tile (r, j + 1) up to date with steps j - 1 and j, and the one with r = j + 1 goes
// on to factor its tile.  The other blocks meanwhile do what is left of earlier steps, two steps at a time so that W is read and
// written half as often: launch j = 2 t the first half of the columns from j + 2 on with steps j - 2 and j - 1, launch 2 t + 1 the
// rest of them, and column j + 2 (which its chain does not reach, but the next one's needs) with step j - 1.  The panels of
// four steps are kept in the workspace; nothing is read that the same launch writes.  Every tile takes its steps in their order,
// one sum each.
// What a step takes: about 3 us of launch, 2 for the loads, 4 for the products (fp32 MFMA, each a chain of its own), 7 for the
// pivots, 16 in all while the other tiles fit beside it.  1024 columns 0.24 ms, 2816 0.69, 4096 1.17, where a launch for the panel
// and one for everything else took 0.25, 0.82 and 1.37 and the library's three factorisations take 28.6 (4096).  From about
// 8000 columns on the matrix leaves the last-level cache and the sweeps over it, one per two steps, bound the call: 8192 columns
// 5.6 ms, 11008 12.4, 14336 27 (one sweep per step 6.6, 16.2, 35; the library 81, 154 and 262 ms).
#include <algorithm>

#include "amct_common.h"

namespace amct {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int kFb = 64;                              // columns eliminated per step
constexpr int kFld = kFb + 4;                        // row stride of a tile in LDS, in floats: 16 rows apart meet no bank
constexpr int kFbThreads = 512;                      // of a step: two halves of four waves
// LDS of a step's blocks: four tiles.  While the blocks of a launch fit the chip twice over they are given more than half of a
// CU's 160 KB, so that the block of the chain has its CU to itself (4096 columns 1206 us, with three smaller blocks a CU 1279);
// beyond, the tiles are what a launch waits for, and two blocks wait for one another's loads (8192 columns 5.57 and 5.97 ms).
constexpr int kFbLds = 4 * kFb * kFld * 4, kFbLdsAlone = 84 * 1024;
static_assert(2 * kFbLds <= 160 * 1024 && 2 * kFbLdsAlone > 160 * 1024, "two blocks a CU, or one");

// W = J (H with zero diagonal entries set to 1, rows and columns in the order perm, + damp I) J, identity beyond C (of each
// pair H[a][b] = H[b][a] the row of the one that comes later in the reversed order is read); one row
// per thread block, up to the end of its diagonal tile.  The row of H comes in whole, in pieces of kFgRow floats through
// LDS, and is picked apart there: picked straight from memory every element costs a 64-byte sector.  Four loads in flight a lane, of 16 bytes where the
// rows lie on 16: 4096 columns 27.6 us, one word after the other 37.
constexpr int kFgRow = 16384;
// Threads of a launch over half of (kFgMax / 64)^2 tiles stay below 2^32.  (A Hessian of that many columns is 256 GiB, the
// factor and the workspace as much again each.)
constexpr int64_t kFgMax = 262144;

constexpr int kGatherLoads = 4;

__global__ __launch_bounds__(kBlock) void gqf_gather_k(const float* h, const int64_t* perm, const float* damp, float* w, int64_t C,
                                                       int64_t Cp, bool vec) {
    extern __shared__ __align__(16) float hrow[];
    const int tid = threadIdx.x;
    const int64_t i = blockIdx.x;
    float* wr = w + (i / kFb) * Cp * kFb + (i % kFb) * kFb;           // of tile (i / 64, 0)
    auto at = [](int64_t c) { return c / kFb * (kFb * kFb) + c % kFb; };
    const int64_t cols = (i / kFb + 1) * kFb;        // of this row
    if (i >= C) {
        for (int64_t c = tid; c < cols; c += kBlock) wr[at(c)] = c == i ? 1.f : 0.f;
        return;
    }
    const float* hr = h + perm[C - 1 - i] * C;
    for (int64_t q0 = 0; q0 < C; q0 += kFgRow) {
        const int64_t q1 = min(C, q0 + kFgRow);
        const int count = (int)(q1 - q0);
        if (q0) __syncthreads();
        if (vec) {
            for (int v0 = tid; v0 < count / 4; v0 += kGatherLoads * kBlock) {
                f4v v[kGatherLoads];
#pragma unroll
                for (int k = 0; k < kGatherLoads; ++k) v[k] = reinterpret_cast<const f4v*>(hr + q0)[min(v0 + k * kBlock, count / 4 - 1)];
#pragma unroll
                for (int k = 0; k < kGatherLoads; ++k)
                    if (v0 + k * kBlock < count / 4) reinterpret_cast<f4v*>(hrow)[v0 + k * kBlock] = v[k];
            }
        } else {
            for (int q = tid; q < count; q += kBlock) hrow[q] = hr[q0 + q];
        }
        __syncthreads();
        for (int64_t c0 = tid; c0 < cols; c0 += kGatherLoads * kBlock) {
            int64_t q[kGatherLoads];
#pragma unroll
            for (int k = 0; k < kGatherLoads; ++k) q[k] = perm[max(C - 1 - c0 - k * kBlock, (int64_t)0)];
#pragma unroll
            for (int k = 0; k < kGatherLoads; ++k) {
                const int64_t c = c0 + k * kBlock;
                if (c >= cols) break;
                if (c >= C) {
                    if (q0 == 0) wr[at(c)] = 0.f;
                } else if (q[k] >= q0 && q[k] < q1) {
                    float v = hrow[q[k] - q0];
                    if (c == i) v = (v == 0.f ? 1.f : v) + *damp;
                    wr[at(c)] = v;
                }
            }
        }
    }
}

AMCT_DEV float lane_value(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }

// One panel of 16 columns of the tile, one row per lane, eliminated in registers, four columns at a time.  The rows above a
// pivot (the inverse so far) take the same operations as the rows below it; the pivot's own row starts the inverse's next row
// from zero.  What a column waits for is the pivot before it: 1 / sqrt, a product, a difference.  The four pivots of a group
// depend on ten numbers only, those of its rows and columns: every lane reads them (at once) and goes through their chain by
// itself, the same operations as on the columns themselves without a lane read in between; the columns follow.  1 / sqrt is
// the hardware estimate and one Newton step (within two units in the last place).
AMCT_DEV void factor_panel(float* t, int p, int lane, int32_t* bad) {
    float a[16];
    float* row = t + lane * kFld + 16 * p;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const f4v v = *reinterpret_cast<const f4v*>(row + 4 * i);
        a[4 * i] = v[0]; a[4 * i + 1] = v[1]; a[4 * i + 2] = v[2]; a[4 * i + 3] = v[3];
    }
    const int own = lane - 16 * p;                   // this lane's pivot, if it is one of the panel's
    bool ok = true;
    float d[4][4];                                   // rows and columns k .. k + 3, lower triangle
    auto read_group = [&](int k) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int i = c; i < 4; ++i) d[i][c] = lane_value(a[k + c], 16 * p + k + i);
    };
    read_group(0);
    float q[4], far[8][4];                           // of the group before: its columns, and their rows k + 4 .. k + 11 as read
#pragma unroll
    for (int k = 0; k < 16; k += 4) {
        // the chain; between its operations the group before is taken from the columns that are not in this one
        const int columns = k == 0 ? 0 : 12 - k, all = 4 * columns;
        int slot = 0;
        auto fill = [&]() {
            const int f0 = all * slot / 24, f1 = all * (slot + 1) / 24;
            ++slot;
#pragma unroll
            for (int f = f0; f < f1; ++f) {
                const int c = f / columns, x = f % columns;
                a[k + 4 + x] = __builtin_fmaf(-q[c], far[x][c], a[k + 4 + x]);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        float rs[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            ok = ok && d[c][c] > 0.f;
            // rsqrt_nr, one operation of its chain at a time
            const float y = __builtin_amdgcn_rsqf(d[c][c]);
            fill();
            const float ny = -d[c][c] * y, hy = 0.5f * y;
            fill();
            const float e = __builtin_fmaf(ny, y, 1.0f);
            fill();
            rs[c] = __builtin_fmaf(hy, e, y);
            fill();
#pragma unroll
            for (int i = c + 1; i < 4; ++i) d[i][c] = d[i][c] * rs[c];
            fill();
#pragma unroll
            for (int x = c + 1; x < 4; ++x)
#pragma unroll
                for (int i = x; i < 4; ++i) d[i][x] = __builtin_fmaf(-d[i][c], d[x][c], d[i][x]);
            fill();
        }
        // the group's columns
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const bool mine = own == k + c;
            a[k + c] = mine ? rs[c] : a[k + c] * rs[c];
#pragma unroll
            for (int x = c + 1; x < 4; ++x) a[k + x] = __builtin_fmaf(-a[k + c], d[x][c], mine ? 0.f : a[k + x]);
        }
        if (k == 12) break;
        // the four columns behind, which the next chain needs: every lane is read before the first product (a read and its product
        // back to back wait for one another).  The group's own rows start from zero, each at its pivot.
        float l[4][4];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int x = 0; x < 4; ++x) l[x][c] = lane_value(a[k + c], 16 * p + k + 4 + x);
        const bool group = (unsigned)(own - k) < 4u;
#pragma unroll
        for (int c = 0; c < 4; ++c) q[c] = group && own > k + c ? 0.f : a[k + c];
#pragma unroll
        for (int x = k + 4; x < 16; ++x) a[x] = group ? 0.f : a[x];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int x = 0; x < 4; ++x) a[k + 4 + x] = __builtin_fmaf(-q[c], l[x][c], a[k + 4 + x]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int x = 0; x < 8 - k; ++x) far[x][c] = lane_value(a[k + c], 16 * p + k + 8 + x);
        read_group(k + 4);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (!ok && lane == 0) *bad = 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const f4v v = {a[4 * i], a[4 * i + 1], a[4 * i + 2], a[4 * i + 3]};
        *reinterpret_cast<f4v*>(row + 4 * i) = v;
    }
}

// rows 16 rt .. + 15 of columns 16 s .. + 15 behind panel p: C - Q_r Q_s^T, from zero in the panel's own rows
AMCT_DEV void factor_behind(float* t, int p, int rt, int s, int lane) {
    const int fr = lane & 15, fq = lane >> 4;
    f4v fa = *reinterpret_cast<const f4v*>(t + (16 * rt + fr) * kFld + 16 * p + 4 * fq);
    const f4v fb = *reinterpret_cast<const f4v*>(t + (16 * s + fr) * kFld + 16 * p + 4 * fq);
    if (rt == p) {                                   // of the panel's own rows only the inverse goes on (on and above the diagonal)
#pragma unroll
        for (int e = 0; e < 4; ++e) fa[e] = fr > 4 * fq + e ? 0.f : fa[e];
    }
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
        if (wave < 4) factor_behind(t, p, wave, p + 1, lane);
        __syncthreads();
        if (wave == 0) factor_panel(t, p + 1, lane, bad);
        else
            for (int x = wave - 1; x < 4 * (2 - p); x += kFbThreads / 64 - 1) factor_behind(t, p, x & 3, p + 2 + (x >> 2), lane);
        __syncthreads();
    }
}

// a 64 x 64 tile of memory: 4 x 4 floats a thread, row tid / 16 + 16 i, columns 4 (tid % 16) ..
struct FactorTile { f4v v[4]; };
AMCT_DEV FactorTile tile_load(const float* g, int tid) {
    FactorTile t;
#pragma unroll
    for (int i = 0; i < 4; ++i) t.v[i] = *reinterpret_cast<const f4v*>(g + (tid + kBlock * i) * 4);
    return t;
}
AMCT_DEV void tile_to_lds(float* lds, const FactorTile& t, int tid) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<f4v*>(lds + ((tid >> 4) + 16 * i) * kFld + (tid & 15) * 4) = t.v[i];
}
// ta tb^T of two tiles in LDS: a wave's 32 x 32, register x: row 8 (x / 4) + 4 (lane / 32) + x % 4, column lane % 32 of it
AMCT_DEV f16v tile_product(const float* ta, const float* tb, int wr, int wc, int lane) {
    const int fr = lane & 31, fh = lane >> 5;
    f16v acc;
#pragma unroll
    for (int x = 0; x < 16; ++x) acc[x] = 0.f;
    const float* pa = ta + (wr + fr) * kFld + 4 * fh;
    const float* pb = tb + (wc + fr) * kFld + 4 * fh;
#pragma unroll
    for (int k = 0; k < kFb; k += 8) {
        const f4v fa = *reinterpret_cast<const f4v*>(pa + k), fb = *reinterpret_cast<const f4v*>(pb + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[e], acc, 0, 0, 0);
    }
    return acc;
}
// t Linv^T of a tile and the inverse factor (rows of Linv) in LDS: a wave's 16 columns of the 64 rows, p[g][x]: row
// 16 g + 4 (lane / 16) + x, column 16 wave + lane % 16
struct FactorPanel { f4v p[4]; };
AMCT_DEV FactorPanel tile_panel(const float* t, const float* linv, int wave, int lane) {
    const int fr = lane & 15, fq = lane >> 4;
    FactorPanel r;
#pragma unroll
    for (int g = 0; g < 4; ++g) r.p[g] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kFb; k += 16) {
        const f4v fb = *reinterpret_cast<const f4v*>(linv + (16 * wave + fr) * kFld + k + 4 * fq);
        f4v fa[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) fa[g] = *reinterpret_cast<const f4v*>(t + (16 * g + fr) * kFld + k + 4 * fq);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int g = 0; g < 4; ++g) r.p[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[g][e], fb[e], r.p[g], 0, 0, 0);
    }
    return r;
}
AMCT_DEV void panel_store(float* to, int ld, const FactorPanel& r, int wave, int lane) {
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int x = 0; x < 4; ++x) to[(16 * g + 4 * (lane >> 4) + x) * ld + 16 * wave + (lane & 15)] = r.p[g][x];
}

struct FactorArgs {
    float* w;                                        // [n][n][64][64]
    float* panels;                                   // [4][n][64][64]: P of step j at j % 4, but for row j (T, in W)
    float* linv;                                     // [2][64][64], of the even and of the odd steps
    int32_t* bad;
    int n;
};

// the tiles of columns s0 .. s1 - 1 that steps a .. a + steps - 1 change
struct FactorRest {
    int a, steps, s0, s1;
    int tiles;                                       // (a + steps) (s1 - s0) of rows 0 .. a + steps - 1, then those on and below the diagonal
};

// Launch j (see the top); j = -1: only the first factor, j = n - 1: only the last panel.
__global__ __launch_bounds__(kFbThreads, 2) void gqf_step_k(FactorArgs a, int j, int chain, FactorRest near, FactorRest far) {
    extern __shared__ __align__(16) float tiles[];   // four of kFb * kFld
    constexpr int kT = kFb * kFld;
    const int n = a.n;
    const int half = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 8), tid = threadIdx.x & 255;
    const int lane = tid & 63, wave = tid >> 6;      // of the half
    float *ta = tiles + 2 * half * kT, *tb = ta + kT;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    const int mine = (wr + 4 * (lane >> 5)) * kFb + wc + (lane & 31);     // of a tile: register x in row 8 (x / 4) + x % 4 behind it
    auto tile = [&](int r, int s) { return a.w + ((int64_t)r * n + s) * (kFb * kFb); };
    auto panel = [&](int step) { return a.panels + (int64_t)(step & 3) * n * (kFb * kFb); };
    auto panel_tile = [&](int step, int r) {
        return tile_load(r == step ? tile(r, r) : panel(step) + (int64_t)r * (kFb * kFb), tid);
    };
    if ((int)blockIdx.x >= chain) {
        // two tiles a block, one for each half
        int b = (int)blockIdx.x - chain;
        const int near_blocks = (near.tiles + 1) / 2;
        const bool is_near = b < near_blocks;
        const FactorRest rest = is_near ? near : far;
        b = 2 * (is_near ? b : b - near_blocks) + half;
        const bool there = b < rest.tiles;           // the last block may have one tile only: its second half repeats it
        if (!there) b = rest.tiles - 1;
        const int m = rest.s1 - rest.s0, above = rest.a + rest.steps;
        int r, s;
        if (b < above * m) {
            r = b / m;
            s = rest.s0 + b % m;
        } else {                                     // column n - 1 - i holds i + 1 tiles from the diagonal down
            const int right = n - rest.s1;           // columns behind s1: the first ones of that order
            b += right * (right + 1) / 2 - above * m;
            int i = (int)((__builtin_sqrtf(8.0f * (float)b + 1.0f) - 1.0f) * 0.5f);
            while ((i + 1) * (i + 2) / 2 <= b) ++i;
            while (i * (i + 1) / 2 > b) --i;
            s = n - 1 - i;
            r = s + b - i * (i + 1) / 2;
        }
        float* ct = tile(r, s) + mine;
        // the rows of the inverse start at their own step, from zero
        const bool fresh = r >= rest.a && r < above;
        const int first = fresh ? r : rest.a;
        FactorTile pr = panel_tile(first, r), ps = panel_tile(first, s);
        float c[16];
#pragma unroll
        for (int x = 0; x < 16; ++x) c[x] = fresh ? 0.f : ct[(8 * (x / 4) + x % 4) * kFb];
        for (int step = rest.a; step < above; ++step) {
            if (step > rest.a) __syncthreads();      // everyone has read the tiles before
            if (step >= first) {
                tile_to_lds(ta, pr, tid);
                tile_to_lds(tb, ps, tid);
            }
            __syncthreads();
            if (step < first) continue;
            if (step + 1 < above) {
                pr = panel_tile(step + 1, r);
                ps = panel_tile(step + 1, s);
            }
            const f16v acc = tile_product(ta, tb, wr, wc, lane);
#pragma unroll
            for (int x = 0; x < 16; ++x) c[x] = c[x] - acc[x];
        }
        if (!there) return;
#pragma unroll
        for (int x = 0; x < 16; ++x) ct[(8 * (x / 4) + x % 4) * kFb] = c[x];
        return;
    }
    // the chain: block 0 has block row j + 1, the others the rows without it.  The first half keeps the tile (r, j + 1) and takes
    // step j - 1 from it while the second one forms the panels of step j.
    const bool more = j + 1 < n;                     // there is a column j + 1
    const int r = !more ? (int)blockIdx.x : blockIdx.x == 0 ? j + 1 : (int)blockIdx.x <= j + 1 ? (int)blockIdx.x - 1 : (int)blockIdx.x;
    const bool first = r == j + 1, self = r == j;
    float* ct = tile(r, more ? j + 1 : j) + mine;
    float *t0 = tiles, *t1 = tiles + kT;             // of the first half
    float c[16];
    if (j >= 0) {
        const bool old = more && j >= 1 && !self;    // step j - 1 changes this tile
        FactorPanel p, q;                            // P[r], P[j + 1]
        FactorTile raw;
        if (half == 0) {
            if (old) {
                const FactorTile pr = panel_tile(j - 1, r), ps = panel_tile(j - 1, j + 1);
                tile_to_lds(ta, pr, tid);
                tile_to_lds(tb, ps, tid);
            }
#pragma unroll
            for (int x = 0; x < 16; ++x) c[x] = more && r != j && r != j - 1 ? ct[(8 * (x / 4) + x % 4) * kFb] : 0.f;
            __syncthreads();
            if (old) {
                const f16v acc = tile_product(ta, tb, wr, wc, lane);
#pragma unroll
                for (int x = 0; x < 16; ++x) c[x] = c[x] - acc[x];
            }
            __syncthreads();                         // t0 and t1 are free
        } else {
            raw = tile_load(tile(r, j), tid);                                         // (T where r == j)
            const FactorTile inv = tile_load(a.linv + (j & 1) * kFb * kFb, tid);
            FactorTile top;
            if (more && !first) top = tile_load(tile(j + 1, j), tid);
            else top = raw;
            tile_to_lds(ta, top, tid);
            tile_to_lds(tb, inv, tid);
            __syncthreads();
            q = tile_panel(ta, tb, wave, lane);
            __syncthreads();
            if (more) panel_store(t1, kFld, q, wave, lane);
            if (self) tile_to_lds(t0, raw, tid);
        }
        if (!more) {                                 // the last column: raw was taken for P[j + 1]
            if (half == 1) panel_store(tile(r, j), kFb, q, wave, lane);
            return;
        }
        if (half == 1 && first) panel_store(panel(j) + (int64_t)r * (kFb * kFb), kFb, q, wave, lane);
        if (!first && !self) {
            if (half == 1) tile_to_lds(ta, raw, tid);
            __syncthreads();
            if (half == 1) {
                p = tile_panel(ta, tb, wave, lane);
                panel_store(t0, kFld, p, wave, lane);
                panel_store(panel(j) + (int64_t)r * (kFb * kFb), kFb, p, wave, lane);
                if (r < j) panel_store(tile(r, j), kFb, p, wave, lane);
            }
        }
        __syncthreads();
        if (half == 0) {
            const f16v acc = tile_product(first ? t1 : t0, t1, wr, wc, lane);
#pragma unroll
            for (int x = 0; x < 16; ++x) c[x] = c[x] - acc[x];
            if (!first) {
#pragma unroll
                for (int x = 0; x < 16; ++x) ct[(8 * (x / 4) + x % 4) * kFb] = c[x];
            }
        }
        if (!first) return;
    } else if (half == 0) {
#pragma unroll
        for (int x = 0; x < 16; ++x) c[x] = ct[(8 * (x / 4) + x % 4) * kFb];
    }
    // block row j + 1: its diagonal tile -> LDS -> its inverse factor
    float* td = tiles + 2 * kT;
    if (half == 0) {
#pragma unroll
        for (int x = 0; x < 16; ++x) td[(wr + 8 * (x / 4) + 4 * (lane >> 5) + x % 4) * kFld + wc + (lane & 31)] = c[x];
    }
    __syncthreads();
    factor_tile(td, threadIdx.x, a.bad);
    float* wd = tile(j + 1, j + 1);
    float* ld = a.linv + ((j + 1) & 1) * kFb * kFb;
#pragma unroll
    for (int i = 0; i < kFb * kFb / kFbThreads; ++i) {
        const int e = threadIdx.x + kFbThreads * i, y = e >> 6, x = e & 63;
        wd[e] = x >= y ? td[y * kFld + x] : 0.f;
        ld[e] = y >= x ? td[x * kFld + y] : 0.f;     // row-major Linv
    }
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
            tile[y][x] = (wr >= 0 && wc >= wr) ? w[(wr / kFb * (Cp / kFb) + wc / kFb) * (kFb * kFb) + wr % kFb * kFb + wc % kFb] : 0.f;
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
    return (cp * cp + 4 * cp * kFb + 2 * (size_t)kFb * kFb) * sizeof(float);     // W, the panels of four steps, the inverses of two
}

extern "C" int amct_gptq_factor(const float* hessian, const int64_t* perm, const float* damp, float* u, int32_t* bad, int64_t cols,
                                void* workspace, size_t workspace_bytes, amct_stream_t stream) {
    if (cols <= 0 || !hessian || !perm || !damp || !u || !bad || !workspace) return AMCT_E_BADARG;
    if (cols > kFgMax) return AMCT_E_TOO_LARGE;
    if (workspace_bytes < amct_gptq_factor_workspace_bytes(cols)) return AMCT_E_BADARG;
    if (!aligned16(workspace)) return AMCT_E_ALIGN;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(gqf_step_k), hipFuncAttributeMaxDynamicSharedMemorySize, kFbLdsAlone) != hipSuccess) {
        (void)hipGetLastError();
        return AMCT_E_HIP;
    }
    hipStream_t st = (hipStream_t)stream;
    const int64_t Cp = (cols + kFb - 1) / kFb * kFb;
    const int n = (int)(Cp / kFb);
    float* linv = (float*)workspace;
    float* panels = linv + 2 * kFb * kFb;
    float* w = panels + 4 * Cp * kFb;
    hipLaunchKernelGGL(gqf_gather_k, dim3((unsigned)Cp), dim3(kBlock), (size_t)std::min<int64_t>(cols, kFgRow) * sizeof(float), st,
                       hessian, perm, damp, w, cols, Cp, cols % 4 == 0 && aligned16(hessian));
    const FactorArgs a{w, panels, linv, bad, n};
    auto rest = [n](int a, int steps, int s0, int s1) {
        FactorRest r{a, steps, s0, s1 < n ? s1 : n, 0};
        if (a >= 0 && s0 < r.s1) {
            const int64_t left = n - s0, right = n - r.s1;
            r.tiles = (int)((int64_t)(a + steps) * (r.s1 - s0) + left * (left + 1) / 2 - right * (right + 1) / 2);
        }
        return r;
    };
    int split = 0;                                   // the columns of an even launch end here
    for (int j = -1; j < n; ++j) {
        const int chain = j < 0 ? 1 : j == n - 1 ? n - 1 : n;
        FactorRest near = rest(-1, 1, 0, 0), far = near;
        if (j >= 2 && j % 2 == 0) {
            // half of the tiles, at least the two columns that the next launch needs
            const int all = rest(j - 2, 2, j + 2, n).tiles;
            split = j + 4;
            while (split < n && 2 * rest(j - 2, 2, j + 2, split).tiles < all) ++split;
            far = rest(j - 2, 2, j + 2, split);
        } else if (j >= 1) {
            near = rest(j - 1, 1, j + 2, j + 3);
            far = rest(j - 3, 2, split, n);          // (none for j = 1)
        }
        const int blocks = chain + (near.tiles + 1) / 2 + (far.tiles + 1) / 2;
        if (blocks > 0) hipLaunchKernelGGL(gqf_step_k, dim3((unsigned)blocks), dim3(kFbThreads), blocks <= 2 * 256 ? kFbLdsAlone : kFbLds, st, a, j, chain, near, far);
    }
    hipLaunchKernelGGL(gqf_store_k, dim3((unsigned)n, (unsigned)n), dim3(kBlock), 0, st, w, u, cols, Cp);
    return hip_status();
}
