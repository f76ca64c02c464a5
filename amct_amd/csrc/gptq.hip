// GPTQ inner block: the column-by-column quantise / propagate-error loop of
// amct_pytorch/quantize_op/gptq_module.py:128-151 for one block of at most 128 columns, fused into one launch
// (the reference issues, per column, a fake-quant of an [N,1] slice, a division and a rank-1 update).
//
// Every row of the weight is independent inside the block:
//   for i in 0 .. count-1:
//       w    = W[n][i]
//       wq   = ((clamp(rne(w / s + z), qmin, qmax)) - z) * s                    (quant_dequant_weight)
//       err  = (w - wq) / Hinv[i][i]
//       W[n][j] -= err * Hinv[i][j]      for j = i .. count-1                   (one product, one subtraction)
//       E[n][i]  = err
// Two kernels.  Blocks of fewer than 128 columns (gptq_block_k):
// a wave owns four rows at a time with the columns across its lanes (2 per lane), so W[n][i] is a lane
// broadcast, the update is two multiplies and two subtractions per step, and the row's errors stay in
// registers until the row is done.  Full blocks of 128 columns (gptq_block_row_k, described there): 16 or 4
// lanes share a row.  The block of the inverse Hessian is read once per thread block into LDS.
// All arithmetic is fp32 with one rounding per operation, as in the eager reference: true divisions,
// round-half-even, product and subtraction rounded separately.
#include <utility>

#include "amct_common.h"
#include "gptq_parts.h"

namespace amct {

constexpr int kGqMax = 128;                         // columns per block at most
constexpr int kGqGaps = 16;
constexpr int64_t kGqWideRows = 8192;               // up to here sixteen lanes share a row, beyond it four
constexpr int kGqRows = 4;                          // rows a wave works on at the same time

struct GptqArgs {
    float* w;                                       // [rows][ld_w], the block starts at column 0 of this pointer
    float* err;                                     // [rows][ld_e]
    const float* hinv;                              // [count][ld_h]
    const float* scale;                             // [rows or 1][scale_stride or 0 ...]
    const int32_t* offset;                          // same layout, or null (symmetric)
    const int32_t* gidx;                            // [count] index of the scale column for each block column
    int64_t rows, ld_w, ld_e, ld_h, scale_stride;
    int count;
    int rows_per_wave;
    float qmin, qmax;
    uint16_t* parts;                                // [rows][3][ld_p]: the errors as three bf16 parts too, or null
    int64_t ld_p;
    int32_t* wide;                                  // set where the parts do not hold an error
};

__global__ __launch_bounds__(kBlock) void gptq_block_k(GptqArgs a) {
    extern __shared__ float hs[];                   // [count][count]
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int count = a.count;
    for (int i = tid; i < count * count; i += kBlock) {
        const int r = i / count, c = i - r * count;
        hs[i] = a.hinv[(int64_t)r * a.ld_h + c];
    }
    __syncthreads();
    const int c0 = lane, c1 = lane + 64;
    const bool v0 = c0 < count, v1 = c1 < count;
    const int64_t row_begin = ((int64_t)blockIdx.x * (kBlock / 64) + wave) * a.rows_per_wave;
    // kGqRows rows at a time: their chains of dependent operations (two divisions and ten more per step) are
    // independent of one another, so the wave issues one row's step while the others' results are on their way, and
    // the Hessian entries of a step are read from LDS once for all of them.  One row at a time ran at a fifth of the
    // vector-ALU issue rate.
    for (int rr = 0; rr < a.rows_per_wave; rr += kGqRows) {
        if (row_begin + rr >= a.rows) break;        // uniform for the wave
        float w0[kGqRows], w1[kGqRows], e0[kGqRows], e1[kGqRows], s0[kGqRows], s1[kGqRows], z0[kGqRows], z1[kGqRows];
        const int32_t g0 = v0 ? a.gidx[c0] : 0, g1 = v1 ? a.gidx[c1] : 0;
#pragma unroll
        for (int r = 0; r < kGqRows; ++r) {
            // rows beyond the matrix repeat its last row (loads stay unconditional; nothing is stored for them)
            const int64_t n = row_begin + rr + r < a.rows ? row_begin + rr + r : a.rows - 1;
            const float* wr = a.w + n * a.ld_w;
            w0[r] = v0 ? wr[c0] : 0.f;
            w1[r] = v1 ? wr[c1] : 0.f;
            e0[r] = 0.f;
            e1[r] = 0.f;
            // the factors of this row for every column of the block, one gather before the loop: lane j keeps
            // those of columns j and j + 64, and step i fetches them by lane broadcast like the weight itself
            const float* srow = a.scale + n * a.scale_stride;
            const int32_t* zrow = a.offset ? a.offset + n * a.scale_stride : nullptr;
            s0[r] = v0 ? srow[g0] : 1.f;
            s1[r] = v1 ? srow[g1] : 1.f;
            z0[r] = (zrow && v0) ? (float)zrow[g0] : 0.f;
            z1[r] = (zrow && v1) ? (float)zrow[g1] : 0.f;
        }
        const bool asym = a.offset != nullptr;
        for (int i = 0; i < count; ++i) {
            const int src = i & 63;                                // i is wave-uniform
            const float d = hs[i * count + i];
            const float h0 = v0 ? hs[i * count + c0] : 0.f;
            const float h1 = v1 ? hs[i * count + c1] : 0.f;
#pragma unroll
            for (int r = 0; r < kGqRows; ++r) {
                const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(i < 64 ? w0[r] : w1[r]), src));
                const float s = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(i < 64 ? s0[r] : s1[r]), src));
                const float z = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(i < 64 ? z0[r] : z1[r]), src));
                float t = w / s;
                if (asym) t = t + z;
                t = __builtin_rintf(t);
                t = __builtin_amdgcn_fmed3f(t, a.qmin, a.qmax);
                const float wq = (t - z) * s;
                const float err = (w - wq) / d;
                const float p0 = err * h0, p1 = err * h1;
                if (c0 >= i) w0[r] = w0[r] - p0;
                if (c1 >= i) w1[r] = w1[r] - p1;
                if (c0 == i) e0[r] = err;
                if (c1 == i) e1[r] = err;
            }
        }
#pragma unroll
        for (int r = 0; r < kGqRows; ++r) {
            const int64_t n = row_begin + rr + r;
            if (n < a.rows) {
                float* wr = a.w + n * a.ld_w;
                float* er = a.err + n * a.ld_e;
                if (v0) { wr[c0] = w0[r]; er[c0] = e0[r]; }
                if (v1) { wr[c1] = w1[r]; er[c1] = e1[r]; }
                if (a.parts) {
                    uint16_t* pr = a.parts + n * 3 * a.ld_p;
                    uint32_t h, m, l;
                    split_parts(e0[r], e1[r], h, m, l);
                    if (v0) { pr[c0] = (uint16_t)h; pr[a.ld_p + c0] = (uint16_t)m; pr[2 * a.ld_p + c0] = (uint16_t)l; }
                    if (v1) { pr[c1] = (uint16_t)(h >> 16); pr[a.ld_p + c1] = (uint16_t)(m >> 16); pr[2 * a.ld_p + c1] = (uint16_t)(l >> 16); }
                    if ((v0 && !parts_hold(e0[r])) || (v1 && !parts_hold(e1[r]))) *a.wide = 1;
                }
            }
        }
    }
}

// Full blocks of 128 columns: NL lanes share a row (64 / NL rows per wave) and each keeps 128 / NL of the row's columns in
// registers, column 4 NL m + 4 q + e in slot [m][e] of lane q of the row, so that loads and stores are 16 bytes per lane
// and the columns still to be updated stay spread over the lanes as the step advances.  The 128 steps are unrolled (the
// slots are registers).  Same operations per element as the kernel above, in the same order.
//
// What bounds it is the chain of a step (weight of column i by lane broadcast, quotient, rounding, error, the one slot that
// holds column i + 1): a thread block takes 128 chains whether the matrix has 16 rows or 14336.  So nothing else sits on it:
//   * both quotients are the fma sequence of div_fast with the reciprocals formed before the loop (10 dependent
//     instructions instead of the ~26 of two IEEE divisions, and the same bits); a wave in which a factor, a weight or an
//     error leaves the range in which that holds throws its result away and runs gptq_row_exact from the weights in memory;
//   * scale, offset and reciprocal of every slot are in registers before step 0 (fetched per step they put an index load
//     and a dependent gather in front of each chain);
//   * row i + 1 of the block of Hinv comes out of LDS during step i, and the slots of step i - 1 that step i does not read
//     are updated inside the chain of step i.
// A block of 128 columns of 4096 rows: 15.4 us, where one division after the other with the factors fetched step by step
// took 32.8 (49.7 with the factors of 32 groups gathered in column order); 14336 rows: 31.4, was 40.6.
// 4 or 16 lanes a row: with 16 the chip is full from 4096 rows on (1024 waves) and a step's updates are a fourth, but each
// wave computes the chain for 4 rows instead of 16.  Two thread blocks fit a CU (64 KB of LDS each), so 16 lanes hold all
// rows at once up to 8192 (4 / 16 lanes: 28.5 / 14.4 us at 512 rows, 30.3 / 21.3 at 8192, 30.5 / 30.2 at 11008, 31.4 / 36.7
// at 14336).
// Where the fma sequences hold: every scale and diagonal in [2^-60, 2^30), |offsets| and the clamp below 2^24, and, seen as
// the steps go by, |error| < 2^30 (with the others that bounds the weights below 2^61) and no difference other than 0
// under 2^-60 (its quotient's last correction would underflow).  NaN and infinity fail the test on the error.
struct GptqRange {
    float emax;                                     // largest |error|, NaN if there was one
    uint32_t dmin;                                  // 2 * bits(difference) - 1, smallest: a zero counts as large
};
constexpr float kGqLimit = 1073741824.0f;           // 2^30
constexpr uint32_t kGqTiny = 2u * (67u << 23) - 1u; // of 2^-60
AMCT_DEV bool range_ok(const GptqRange& r) { return r.emax < kGqLimit && r.dmin >= kGqTiny; }
AMCT_DEV bool range_divisor(const Divisor& d) { return d.fast && d.s < kGqLimit; }

// value held by lane Q of the row's NL lanes
template <int NL, int Q> AMCT_DEV float row_bcast(float v) {
    if constexpr (NL == 4) return quad_bcast<Q>(v);
    else return dpp_f<0x150 + Q>(v);                // row_newbcast: lane Q of every 16
}
// The same block with IEEE divisions, for the waves that leave the range of the fma sequence: a rolled loop, the slot of
// column i picked by comparison.
template <int NL, bool ASYM>
AMCT_DEV void gptq_row_exact(const float* hs, float (&w)[32 / NL][4], float (&eo)[32 / NL][4], const float (&s)[32 / NL][4],
                                            const float (&z)[32 / NL][4], float qmin, float qmax, int lane) {
    constexpr int M = 32 / NL;
    const int q = lane & (NL - 1);
#pragma clang loop unroll(disable)
    for (int i = 0; i < kGqMax; ++i) {
        const int mi = i / (4 * NL), ei = i & 3, src = (lane & ~(NL - 1)) + ((i >> 2) & (NL - 1));
        float wi = 0.f, sc = 1.f, zc = 0.f;
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool at = m == mi && e == ei;
                wi = at ? w[m][e] : wi;
                sc = at ? s[m][e] : sc;
                zc = at ? z[m][e] : zc;
            }
        wi = __shfl(wi, src, 64);
        sc = __shfl(sc, src, 64);
        zc = __shfl(zc, src, 64);
        float t = wi / sc;
        if (ASYM) t = t + zc;
        t = __builtin_rintf(t);
        t = __builtin_amdgcn_fmed3f(t, qmin, qmax);
        const float wq = (t - zc) * sc;
        const float err = (wi - wq) / hs[i * kGqMax + i];
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int c = 4 * NL * m + 4 * q + e;
                const float p = err * hs[i * kGqMax + c];
                if (c >= i) w[m][e] = w[m][e] - p;
                if (c == i) eo[m][e] = err;
            }
    }
}

// slot (m, e) of row lane q takes the update of step C: its column lies at or behind column C
template <int NL, int C> AMCT_DEV bool gptq_behind(int m, int e, int q) {
    constexpr int mc = C / (4 * NL), qc = (C >> 2) & (NL - 1), ec = C & 3;
    if (m != mc) return m > mc;
    return e >= ec ? q >= qc : q > qc;
}

// What a lane carries from step to step (a struct of constants-indexed arrays: the step number is a template argument)
template <int NL, bool ASYM> struct GptqRow {
    static constexpr int M = 32 / NL;               // 16-byte pieces of a row per lane
    float w[M][4], s[M][4], z[M][4], y[M][4], eo[M][4];
    float hprev[M][4], hcur[M][4];                  // rows i - 1 and i of the block of Hinv, this lane's columns
    float dd, ddy;                                  // diagonal of row i, its reciprocal
    float err_prev;
    float next;                                     // the slot of column i, up to date, before the choice of lanes
    GptqRange range;

    float prod[M][4];

    // the updates of step I - 1 that step I does not wait for (all slots but that of column I), product and subtraction
    // apart, dealt out over the kGqGaps places of the chain: they run where the chain waits for its own last result
    template <int I, int GAP> AMCT_DEV void fill(int q) {
        if constexpr (I > 0) {
            constexpr int mi = I / (4 * NL), ei = I & 3, mp = (I - 1) / (4 * NL);
            constexpr int n = 8 * (M - mp), f0 = n * GAP / kGqGaps, f1 = n * (GAP + 1) / kGqGaps;
#pragma unroll
            for (int f = f0; f < f1; ++f) {
                const int m = mp + f / 8, e = (f / 2) & 3;
                if (m == mi && e == ei) continue;
                if (f % 2 == 0) {
                    prod[m][e] = err_prev * hprev[m][e];
                } else {
                    const float u = w[m][e] - prod[m][e];
                    w[m][e] = gptq_behind<NL, I - 1>(m, e, q) ? u : w[m][e];
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }

    template <int I> AMCT_DEV void step(const float* hs, const float (*dg)[2], float qmin, float qmax, int q) {
        constexpr int mi = I / (4 * NL), qi = (I >> 2) & (NL - 1), ei = I & 3;
        constexpr int in = I + 1 < kGqMax ? I + 1 : I, mn = in / (4 * NL), en = in & 3;
        const float wi = row_bcast<NL, qi>(next);
        const float sc = row_bcast<NL, qi>(s[mi][ei]), yc = row_bcast<NL, qi>(y[mi][ei]);
        const float zi = ASYM ? row_bcast<NL, qi>(z[mi][ei]) : 0.f;
        float hnext[M][4];
#pragma unroll
        for (int m = mn; m < M; ++m) {
            const float4 h = *reinterpret_cast<const float4*>(&hs[in * kGqMax + 4 * NL * m + 4 * q]);
            hnext[m][0] = h.x; hnext[m][1] = h.y; hnext[m][2] = h.z; hnext[m][3] = h.w;
        }
        const float dn = dg[in][0], dny = dg[in][1];
        __builtin_amdgcn_sched_barrier(0);
        // t = wi / sc, err = dlt / dd: the sequence of div_fast, one operation to a gap.  A quotient that is a zero loses its
        // sign there: put back where a later result shows it (without an offset: in t; then dlt is never -0.0.  With one
        // the addition takes the sign of t, and dlt is -0.0 for a weight of -0.0)
        float q0 = wi * yc;
        fill<I, 0>(q);
        float r0 = __builtin_fmaf(-q0, sc, wi);
        fill<I, 1>(q);
        q0 = __builtin_fmaf(r0, yc, q0);
        fill<I, 2>(q);
        r0 = __builtin_fmaf(-q0, sc, wi);
        fill<I, 3>(q);
        float t = __builtin_fmaf(r0, yc, q0);
        fill<I, 4>(q);
        if constexpr (ASYM) t = t + zi;
        else t = __uint_as_float(__float_as_uint(t) | (__float_as_uint(wi) & 0x80000000u));
        fill<I, 5>(q);
        t = __builtin_rintf(t);
        fill<I, 6>(q);
        t = __builtin_amdgcn_fmed3f(t, qmin, qmax);
        fill<I, 7>(q);
        if constexpr (ASYM) t = t - zi;
        fill<I, 8>(q);
        t = t * sc;
        fill<I, 9>(q);
        const float dlt = wi - t;
        fill<I, 10>(q);
        float e0 = dlt * ddy;
        fill<I, 11>(q);
        float e1 = __builtin_fmaf(-e0, dd, dlt);
        fill<I, 12>(q);
        e0 = __builtin_fmaf(e1, ddy, e0);
        fill<I, 13>(q);
        e1 = __builtin_fmaf(-e0, dd, dlt);
        fill<I, 14>(q);
        float err = __builtin_fmaf(e1, ddy, e0);
        fill<I, 15>(q);
        if constexpr (ASYM) err = __uint_as_float(__float_as_uint(err) | (__float_as_uint(dlt) & 0x80000000u));
        range.dmin = min(range.dmin, 2u * __float_as_uint(dlt) - 1u);
        __builtin_amdgcn_sched_barrier(0);
        // the slot that holds column I + 1 (column I itself -- the reference's update runs from j = i,
        // W[n][i] -= err * Hinv[i][i]: not read again, but what the caller gets back -- shares its slot with columns of
        // the other lanes and is updated with them, among the pending slots of the next step)
        if constexpr (I + 1 < kGqMax) {
            const float p = err * hcur[mn][en];
            range.emax = fmax_nan(range.emax, __builtin_fabsf(err));
            eo[mi][ei] = q == qi ? err : eo[mi][ei];
            __builtin_amdgcn_sched_barrier(0);
            next = w[mn][en] - p;                   // (the lane of column I + 1 is behind column I: its value is taken as it is)
            w[mn][en] = gptq_behind<NL, I>(mn, en, q) ? next : w[mn][en];
        } else {
            range.emax = fmax_nan(range.emax, __builtin_fabsf(err));
            eo[mi][ei] = q == qi ? err : eo[mi][ei];
        }
        // (taken now: left to itself the compiler keeps every step's values alive for one long reduction at the end)
        asm volatile("" : "+v"(range.emax), "+v"(range.dmin), "+v"(eo[mi][ei]));
        __builtin_amdgcn_sched_barrier(0);
        err_prev = err;
        dd = dn;
        ddy = dny;
#pragma unroll
        for (int m = mi; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) hprev[m][e] = hcur[m][e];
#pragma unroll
        for (int m = mn; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 4; ++e) hcur[m][e] = hnext[m][e];
    }
    template <int... I>
    AMCT_DEV void steps(std::integer_sequence<int, I...>, const float* hs, const float (*dg)[2], float qmin, float qmax, int q) {
        (step<I>(hs, dg, qmin, qmax, q), ...);
    }
};

template <int NL, bool ASYM>
__global__ __launch_bounds__(kBlock) void gptq_block_row_k(GptqArgs a) {
    constexpr int M = 32 / NL;                                                   // 16-byte pieces of a row per lane
    struct Shared {
        float dg[kGqMax][2];                                                     // diagonal, its reciprocal
        float hs[kGqMax * kGqMax];                                               // [128][128]
        int dbad;
    };
    __shared__ __attribute__((aligned(16))) Shared sh;
    float* hs = sh.hs;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int q = lane & (NL - 1);
    const int64_t n = ((int64_t)blockIdx.x * (kBlock / 64) + wave) * (64 / NL) + lane / NL;
    const int64_t nc = n < a.rows ? n : a.rows - 1;              // rows beyond the matrix repeat its last row; not stored
    const float* wr = a.w + nc * a.ld_w + 4 * q;
    const float* srow = a.scale + nc * a.scale_stride;
    const int32_t* zrow = ASYM ? a.offset + nc * a.scale_stride : nullptr;
    if (tid == 0) sh.dbad = 0;
    GptqRow<NL, ASYM> r;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const float4 v = *reinterpret_cast<const float4*>(wr + 4 * NL * m);
        r.w[m][0] = v.x; r.w[m][1] = v.y; r.w[m][2] = v.z; r.w[m][3] = v.w;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int g = a.gidx[4 * NL * m + 4 * q + e];
            r.s[m][e] = srow[g];
            r.z[m][e] = ASYM ? (float)zrow[g] : 0.f;
        }
    }
    if (a.ld_h % 4 == 0 && (reinterpret_cast<uintptr_t>(a.hinv) & 15u) == 0) {
#pragma unroll
        for (int i = 0; i < kGqMax * kGqMax / (4 * kBlock); ++i) {
            const int v = tid + i * kBlock;
            *reinterpret_cast<float4*>(&hs[4 * v]) = *reinterpret_cast<const float4*>(a.hinv + (int64_t)(v >> 5) * a.ld_h + 4 * (v & 31));
        }
    } else {
        for (int i = tid; i < kGqMax * kGqMax; i += kBlock) hs[i] = a.hinv[(int64_t)(i >> 7) * a.ld_h + (i & 127)];
    }
    bool ok = true;
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const Divisor d = make_divisor(r.s[m][e]);
            r.y[m][e] = d.y;
            ok = ok && range_divisor(d) && __builtin_fabsf(r.z[m][e]) < 16777216.f;
            r.eo[m][e] = 0.f;
        }
    __syncthreads();
    if (tid < kGqMax) {
        const Divisor d = make_divisor(hs[tid * kGqMax + tid]);
        sh.dg[tid][0] = d.s;
        sh.dg[tid][1] = d.y;
        if (!range_divisor(d)) sh.dbad = 1;
    }
    __syncthreads();
    ok = ok && sh.dbad == 0 && __builtin_fabsf(a.qmin) < 16777216.f && __builtin_fabsf(a.qmax) < 16777216.f;

    r.range = GptqRange{0.f, 0xFFFFFFFFu};
    r.err_prev = 0.f;
    r.dd = sh.dg[0][0];
    r.ddy = sh.dg[0][1];
    r.next = r.w[0][0];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const float4 h = *reinterpret_cast<const float4*>(&hs[4 * NL * m + 4 * q]);
        r.hcur[m][0] = h.x; r.hcur[m][1] = h.y; r.hcur[m][2] = h.z; r.hcur[m][3] = h.w;
#pragma unroll
        for (int e = 0; e < 4; ++e) r.hprev[m][e] = 0.f;
    }
    r.steps(std::make_integer_sequence<int, kGqMax>(), hs, sh.dg, a.qmin, a.qmax, q);
    // what step 127 leaves pending: column 127 itself
    if (q == NL - 1) r.w[M - 1][3] = r.w[M - 1][3] - r.err_prev * r.hprev[M - 1][3];
    if (!wave_all(ok && range_ok(r.range))) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float4 v = *reinterpret_cast<const float4*>(wr + 4 * NL * m);
            r.w[m][0] = v.x; r.w[m][1] = v.y; r.w[m][2] = v.z; r.w[m][3] = v.w;
        }
        gptq_row_exact<NL, ASYM>(hs, r.w, r.eo, r.s, r.z, a.qmin, a.qmax, lane);
    }
    if (n < a.rows) {
        float* wo = a.w + n * a.ld_w + 4 * q;
        float* er = a.err + n * a.ld_e + 4 * q;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            *reinterpret_cast<float4*>(wo + 4 * NL * m) = make_float4(r.w[m][0], r.w[m][1], r.w[m][2], r.w[m][3]);
            *reinterpret_cast<float4*>(er + 4 * NL * m) = make_float4(r.eo[m][0], r.eo[m][1], r.eo[m][2], r.eo[m][3]);
        }
        if (a.parts) {
            uint16_t* pr = a.parts + n * 3 * a.ld_p + 4 * q;
            bool hold = true;
#pragma unroll
            for (int m = 0; m < M; ++m) {
                uint2 hi, mid, lo;
                split_parts(r.eo[m][0], r.eo[m][1], hi.x, mid.x, lo.x);
                split_parts(r.eo[m][2], r.eo[m][3], hi.y, mid.y, lo.y);
                *reinterpret_cast<uint2*>(pr + 4 * NL * m) = hi;
                *reinterpret_cast<uint2*>(pr + a.ld_p + 4 * NL * m) = mid;
                *reinterpret_cast<uint2*>(pr + 2 * a.ld_p + 4 * NL * m) = lo;
#pragma unroll
                for (int e = 0; e < 4; ++e) hold = hold && parts_hold(r.eo[m][e]);
            }
            if (!hold) *a.wide = 1;
        }
    }
}

}  // namespace amct

using namespace amct;

extern "C" int amct_gptq_block(float* w, int64_t ld_w, float* err, int64_t ld_e, const float* hinv, int64_t ld_h,
                               const float* scale, const int32_t* offset, int64_t scale_stride, const int32_t* gidx,
                               int64_t rows, int count, int qmin, int qmax, amct_stream_t stream) {
    return amct_gptq_block_parts(w, ld_w, err, ld_e, hinv, ld_h, scale, offset, scale_stride, gidx, rows, count, qmin, qmax, nullptr, 0,
                                 nullptr, stream);
}

extern "C" int amct_gptq_block_parts(float* w, int64_t ld_w, float* err, int64_t ld_e, const float* hinv, int64_t ld_h,
                                     const float* scale, const int32_t* offset, int64_t scale_stride, const int32_t* gidx,
                                     int64_t rows, int count, int qmin, int qmax, uint16_t* parts, int64_t ld_p, int32_t* wide,
                                     amct_stream_t stream) {
    if (parts && (ld_p < count || ld_p % 4 != 0 || !wide)) return AMCT_E_BADARG;
    if (reinterpret_cast<uintptr_t>(parts) & 7u) return AMCT_E_ALIGN;
    if (rows < 0 || count < 0 || count > kGqMax || qmin > qmax) return AMCT_E_BADARG;
    if (ld_w < count || ld_e < count || ld_h < count || scale_stride < 0) return AMCT_E_BADARG;
    if (rows == 0 || count == 0) return AMCT_OK;
    if (!w || !err || !hinv || !scale || !gidx) return AMCT_E_BADARG;
    GptqArgs a{};
    a.w = w; a.err = err; a.hinv = hinv; a.scale = scale; a.offset = offset; a.gidx = gidx;
    a.rows = rows; a.ld_w = ld_w; a.ld_e = ld_e; a.ld_h = ld_h; a.scale_stride = scale_stride;
    a.count = count; a.qmin = (float)qmin; a.qmax = (float)qmax;
    a.parts = parts; a.ld_p = ld_p; a.wide = wide;
    if (count == kGqMax && ld_w % 4 == 0 && ld_e % 4 == 0 && aligned16(w) && aligned16(err) && (rows + 15) / 16 <= 0x7FFFFFFF) {
        const bool wide = rows <= kGqWideRows;
        const int64_t per = (kBlock / 64) * (wide ? 4 : 16);
        const dim3 grid((unsigned)((rows + per - 1) / per));
        hipStream_t st = (hipStream_t)stream;
        if (wide && offset) hipLaunchKernelGGL((gptq_block_row_k<16, true>), grid, dim3(kBlock), 0, st, a);
        else if (wide) hipLaunchKernelGGL((gptq_block_row_k<16, false>), grid, dim3(kBlock), 0, st, a);
        else if (offset) hipLaunchKernelGGL((gptq_block_row_k<4, true>), grid, dim3(kBlock), 0, st, a);
        else hipLaunchKernelGGL((gptq_block_row_k<4, false>), grid, dim3(kBlock), 0, st, a);
        return hip_status();
    }
    // about 1024 thread blocks of 4 waves, each wave walking a few groups of kGqRows rows
    int64_t rpw = (rows + 4095) / 4096;
    rpw = (rpw + kGqRows - 1) / kGqRows * kGqRows;
    if (rpw < kGqRows) rpw = kGqRows;
    a.rows_per_wave = (int)rpw;
    const int64_t rows_per_block = rpw * (kBlock / 64);
    const int64_t nb = (rows + rows_per_block - 1) / rows_per_block;
    if (nb > 0x7FFFFFFF) return AMCT_E_UNSUPPORTED;
    const size_t lds = (size_t)count * count * sizeof(float);
    if (lds > 64 * 1024) return AMCT_E_UNSUPPORTED;
    hipLaunchKernelGGL(gptq_block_k, dim3((unsigned)nb), dim3(kBlock), lds, (hipStream_t)stream, a);
    return hip_status();
}
