// The update of the columns behind a GPTQ block, W <- W - E U (amct_pytorch/quantize_op/gptq_module.py:152-153), on the bf16 matrix
// pipe: fp32 numbers as exact sums of three bf16 parts, x = h + m + l (8 + 8 + 8 bits), and of the nine products of two such
// sums the six that matter (the other three are below 2^-25 of the product).  Six bf16 MFMAs take less than half the time of
// the fp32 ones, and err less: 32 products enter a sum with one rounding (of 128 steps, against fp64: 1.5e-7, the fp32 pipe
// 2.0e-7; sums are subtracted from W every 128 steps as in the reference: 512 steps 1.6e-7, in one fp32 sum 4.1e-7).
// The parts are made once: of U by gptq_split_k, of E by the column loop that computes it.  Parts of a value that is neither
// 0 nor in [2^-100, 2^60), NaN and infinities among them, may underflow or overflow: whoever makes them raises a flag, and
// the update goes back to the fp32 values.
#include "amct_common.h"
#include "gptq_parts.h"

namespace amct {

typedef float p4f __attribute__((ext_vector_type(4)));
typedef float p16f __attribute__((ext_vector_type(16)));
typedef __bf16 p8b __attribute__((ext_vector_type(8)));
typedef short p4s __attribute__((ext_vector_type(4)));
typedef short p8s __attribute__((ext_vector_type(8)));

// Rows of U (fp32 [cols][cols], upper triangle) -> [cols][3][ld] bf16, from the diagonal's multiple of 8 on.
// U[4096,4096]: 20 us, once a layer.
__global__ __launch_bounds__(kBlock) void gptq_split_k(const float* u, uint16_t* parts, int64_t cols, int64_t ld, int32_t* wide) {
    const int64_t row = blockIdx.x;
    const float* ur = u + row * cols;
    uint16_t* pr = parts + row * 3 * ld;
    bool ok = true;
    for (int64_t c = (row & ~(int64_t)7) + 8 * threadIdx.x; c < cols; c += 8 * kBlock) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = c + j < cols ? ur[c + j] : 0.f;
        uint4 h, m, l;
        split_parts(x[0], x[1], h.x, m.x, l.x);
        split_parts(x[2], x[3], h.y, m.y, l.y);
        split_parts(x[4], x[5], h.z, m.z, l.z);
        split_parts(x[6], x[7], h.w, m.w, l.w);
#pragma unroll
        for (int j = 0; j < 8; ++j) ok = ok && parts_hold(x[j]);
        stg16(pr + c, h);
        stg16(pr + ld + c, m);
        stg16(pr + 2 * ld + c, l);
    }
    if (!ok) *wide = 1;
}

struct PartsArgs {
    float* w;                                       // [rows][ld_w], at the first column to update
    const float* err;                               // [rows][ld_e]
    const float* u;                                 // [count][ld_u], at the first column to update
    const uint16_t* err_parts;                      // [rows][3][ld_ep]
    const uint16_t* u_parts;                        // [count][3][ld_up], at the first column to update
    const int32_t* wide;                            // set: the parts do not hold E or U
    int64_t ld_w, ld_e, ld_u, ld_ep, ld_up, rows, cols;
    int count;                                      // a multiple of 32
    int col_tiles, tiles;
    int vec_w;                                      // rows of w are 16-byte aligned, cols is a multiple of 4
};

// A direct-to-LDS load: wave-uniform 64-bit base, a byte offset per lane, lane l's 16 bytes land at lds + 16 l.  (Inline, with
// hand-counted waits: the compiler would wait for all of them before every LDS read.)
AMCT_DEV void parts_dma(uint32_t lds, const void* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(off), "s"(base) : "memory");
}
template <int N> AMCT_DEV void parts_wait() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory"); }

// 32 x 32 of W by one wave with fp32 MFMA, straight from memory: where the parts do not hold the values
AMCT_DEV void trail_exact(const PartsArgs& a, const int64_t r0, const int64_t c0, const int lane) {
    const int fr = lane & 31, fh = lane >> 5;
    const int64_t row = min(r0 + fr, a.rows - 1), col = min(c0 + fr, a.cols - 1);      // beyond: not stored
    for (int k0 = 0; k0 < a.count; k0 += kPartsSum) {
        p16f acc;
#pragma unroll
        for (int x = 0; x < 16; ++x) acc[x] = 0.f;
        for (int k = k0; k < min(k0 + kPartsSum, a.count); k += 2)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.err[row * a.ld_e + k + fh], a.u[(int64_t)(k + fh) * a.ld_u + col], acc, 0, 0, 0);
#pragma unroll
        for (int x = 0; x < 16; ++x) {
            const int64_t r = r0 + 8 * (x / 4) + 4 * fh + x % 4;
            if (r < a.rows && c0 + fr < a.cols) {
                float* p = a.w + r * a.ld_w + c0 + fr;
                *p = *p - acc[x];
            }
        }
    }
}

// A 64 x 64 tile of W per block: 2 x 2 waves of 32 x 32.  Stages of 32 steps, two in LDS, filled by direct-to-LDS loads, one
// barrier each; the fragments of the next stage are read under the products of this one.  Three blocks fit a CU and wait
// for one another's loads of parts and of W.  W[4096,.] behind 512 columns: 3584 / 1024 / 128 columns 101 / 34 / 9.8 us (the fp32
// kernel 134 / 43 / 22; bf16 products at 0.9 PFLOP/s, half of what a register-only loop reaches: the loads, the fragment reads
// and the products take about as long as one another); behind 128 columns, where W's own bytes count as much, 40 / 14 / 7.5
// (47 / 16 / 8.0).  128 x 128 tiles, one block of three stages a CU: 115 / 33 / 10.2 and 57 / 16 / 8.0.
constexpr int kPartsTile = 64;
__global__ __launch_bounds__(kBlock, 3) void gptq_trail_parts_k(PartsArgs a) {
    constexpr int T = 2, kTile = kPartsTile, kPlane = 64 * kTile, kStage = 6 * kPlane, kStages = 2, kPieces = 3;   // T: 16 x 16 tiles of a wave
    __shared__ __align__(1024) uint8_t lds[kStages * kStage];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // block -> tile: consecutive blocks go to the eight dies in turn, each with an L2 of its own.  A die takes a run of an order
    // that goes down 8 rows of tiles and on to the next column: the blocks it runs at a time share 8 rows' E (1.6 MB of 512
    // steps) and a few columns' U (512 columns behind 512: 16.2 us, row after row 22.0).
    const unsigned per = gridDim.x / 8, logical = blockIdx.x % 8 * per + blockIdx.x / 8;
    if (logical >= (unsigned)a.tiles) return;       // whole block (before any barrier)
    const unsigned ct = (unsigned)a.col_tiles, rt = (unsigned)a.tiles / ct;
    const unsigned band = logical / (8 * ct), place = logical % (8 * ct), tall = min(8u, rt - 8 * band);
    const int64_t r0 = (int64_t)(8 * band + place % tall) * kTile;
    const int64_t c0 = (int64_t)(place / tall) * kTile;
    const int wi = wave >> 1, wj = wave & 1, fr = lane & 15, fg = lane >> 4;
    // a lane's four values of tile (m, n): row 16 m + lane % 16, columns 16 n + 4 (lane / 16) .. + 3 of the wave's tile
    const int64_t rw = r0 + 16 * T * wi + fr, cw = c0 + 16 * T * wj + 4 * fg;
    float* wp = a.w + rw * a.ld_w + cw;
    const bool inside = a.vec_w && r0 + kTile <= a.rows && c0 + kTile <= a.cols;
    p4f old[T][T], acc[T][T];
    if (inside) {
#pragma unroll
        for (int m = 0; m < T; ++m)
#pragma unroll
            for (int n = 0; n < T; ++n) old[m][n] = *reinterpret_cast<const p4f*>(wp + 16 * m * a.ld_w + 16 * n);
    } else {
#pragma unroll
        for (int m = 0; m < T; ++m)
#pragma unroll
            for (int n = 0; n < T; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) old[m][n][r] = a.w[min(rw + 16 * m, a.rows - 1) * a.ld_w + min(cw + 16 * n + r, a.cols - 1)];
    }
#pragma unroll
    for (int m = 0; m < T; ++m)
#pragma unroll
        for (int n = 0; n < T; ++n) acc[m][n] = p4f{0.f, 0.f, 0.f, 0.f};

    // Memory -> LDS, per part.  E: a row is 32 steps in four 16-byte chunks, swapped by the row; U: a step is kTile columns in
    // 32-byte units, swapped by the step: a fragment read (16 rows' chunk; 4 columns of 4 steps out of each 8) meets in no bank.
    // Rows and columns beyond the matrix repeat its last ones (not stored).
    auto swap_e = [](int row) { return (row >> 2) & 3; };
    auto swap_u = [](int k) { return ((k >> 1) & 1) | ((k >> 3) & 1) << 1; };
    uint32_t off_e[kPieces], off_u[kPieces];
#pragma unroll
    for (int j = 0; j < kPieces; ++j) {
        const int q = wave * kPieces + j;
        {
            const int part = q / (2 * T), row = 16 * (q % (2 * T)) + (lane >> 2);
            const int64_t r = min(r0 + row, a.rows - 1) - r0;
            off_e[j] = (uint32_t)(2 * ((r * 3 + part) * a.ld_ep + 8 * ((lane & 3) ^ swap_e(row))));
        }
        {
            const int part = q / (2 * T), k = 16 / T * (q % (2 * T)) + lane / (4 * T), at = lane % (4 * T);
            const int64_t c = min(c0 + 8 * ((((at >> 1) ^ swap_u(k)) << 1) | (at & 1)), (a.cols - 1) & ~(int64_t)7) - c0;
            off_u[j] = (uint32_t)(2 * ((3 * k + part) * a.ld_up + c));
        }
    }
    const uint16_t *eb = a.err_parts + r0 * 3 * a.ld_ep, *ub = a.u_parts + c0;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds);
    const int stages = a.count / 32, last = stages - 1;
    auto fetch = [&](int buf, int s) {
        const uint32_t to = lds0 + buf * kStage + wave * kPieces * 1024;
        const uint16_t *es = eb + 32 * s, *us = ub + (int64_t)(96 * s) * a.ld_up;
#pragma unroll
        for (int j = 0; j < kPieces; ++j) {
            parts_dma(to + j * 1024, es, off_e[j]);
            parts_dma(to + 3 * kPlane + j * 1024, us, off_u[j]);
        }
    };
    const int kl = 8 * fg + (fr >> 2);              // the step whose 4 columns this lane reads for the transposition (and + 4)
    const int at_e = (16 * T * wi + fr) * 64 + ((fg ^ swap_e(fr)) * 16);
    int at_u[T];
#pragma unroll
    for (int n = 0; n < T; ++n) at_u[n] = 3 * kPlane + kl * (2 * kTile) + ((wj * T + n) ^ swap_u(kl)) * 32 + (lane & 3) * 8;
    p8s fe[2][T][3], fu[2][T][3];
    // fragment q of a stage: rows first, the smallest parts first
    auto read_one = [&](int buf, int set, int q) {
        const int part = 2 - q / (2 * T), x = q % (2 * T);
        const uint8_t* st = lds + buf * kStage + part * kPlane;
        if (x < T) {
            fe[set][x][part] = *reinterpret_cast<const p8s*>(st + at_e + x * 1024);
        } else {
            typedef __attribute__((address_space(3))) p4s lds_p4s;
            const p4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_p4s*)(st + at_u[x - T]));
            const p4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_p4s*)(st + at_u[x - T] + 4 * 2 * kTile));
            fu[set][x - T][part] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    };
    // products of the parts whose places add up to at most 2, the smallest first; U is the first operand (see wp).  Behind each
    // of the first ones a fragment of the next stage is read.
    auto products = [&](int set, int buf) {
        int x = 0;
#pragma unroll
        for (int t = 2; t >= 0; --t)
#pragma unroll
            for (int p = 0; p <= t; ++p)
#pragma unroll
                for (int m = 0; m < T; ++m)
#pragma unroll
                    for (int n = 0; n < T; ++n, ++x) {
                        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(p8b, fu[set][n][t - p]),
                                                                           __builtin_bit_cast(p8b, fe[set][m][p]), acc[m][n], 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        if (x < 6 * T) {
                            read_one(buf, set ^ 1, x);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
    };
    auto subtract = [&]() {
#pragma unroll
        for (int m = 0; m < T; ++m)
#pragma unroll
            for (int n = 0; n < T; ++n) {
                old[m][n] = old[m][n] - acc[m][n];
                acc[m][n] = p4f{0.f, 0.f, 0.f, 0.f};
            }
    };
    constexpr int kPer = 2 * kPieces;               // loads of a wave and stage
#pragma unroll
    for (int s = 0; s < kStages; ++s) fetch(s, min(s, last));                 // (beyond the last: repeats it, nobody reads it)
    parts_wait<(kStages - 1) * kPer>();
    // (the tile of W, asked for before those loads, is there too; used here, the compiler waits for it now and not among the
    // loads of a later stage, which it does not count)
#pragma unroll
    for (int m = 0; m < T; ++m)
#pragma unroll
        for (int n = 0; n < T; ++n) asm volatile("" : "+v"(old[m][n]));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int q = 0; q < 6 * T; ++q) read_one(0, 0, q);
    int buf = 0;
    auto step = [&](int set, int s) {
        const int next = buf + 1 == kStages ? 0 : buf + 1;
        parts_wait<(kStages - 2) * kPer>();         // the next stage is there, this one is in registers
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        fetch(buf, min(s + kStages, last));
        products(set, next);                  // (behind the last stage: its repetition)
        if ((s + 1) % (kPartsSum / 32) == 0) subtract();
        buf = next;
    };
    for (int s = 0; s < stages; s += 2) {
        step(0, s);
        if (s + 1 < stages) step(1, s + 1);
    }
    if (stages % (kPartsSum / 32) != 0) subtract();
    parts_wait<0>();                                // no load may land after the block has given its LDS back
    if (*a.wide) {                                  // whole block
        trail_exact(a, r0 + 32 * wi, c0 + 32 * wj, lane);
        return;
    }
    if (inside) {
#pragma unroll
        for (int m = 0; m < T; ++m)
#pragma unroll
            for (int n = 0; n < T; ++n) *reinterpret_cast<p4f*>(wp + 16 * m * a.ld_w + 16 * n) = old[m][n];
    } else {
#pragma unroll
        for (int m = 0; m < T; ++m)
#pragma unroll
            for (int n = 0; n < T; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (rw + 16 * m < a.rows && cw + 16 * n + r < a.cols) wp[16 * m * a.ld_w + 16 * n + r] = old[m][n][r];
    }
}

}  // namespace amct

using namespace amct;

extern "C" int amct_gptq_split(const float* u, uint16_t* parts, int64_t cols, int64_t ld, int32_t* wide, amct_stream_t stream) {
    if (cols < 0 || ld < cols || ld % 8 != 0) return AMCT_E_BADARG;
    if (cols == 0) return AMCT_OK;
    if (!u || !parts || !wide) return AMCT_E_BADARG;
    if (cols > 0x7FFFFFFF) return AMCT_E_TOO_LARGE;
    if (!aligned16(parts)) return AMCT_E_ALIGN;
    hipLaunchKernelGGL(gptq_split_k, dim3((unsigned)cols), dim3(kBlock), 0, (hipStream_t)stream, u, parts, cols, ld, wide);
    return hip_status();
}

extern "C" int amct_gptq_trail_parts(float* w, int64_t ld_w, const float* err, int64_t ld_e, const float* u, int64_t ld_u,
                                     const uint16_t* err_parts, int64_t ld_ep, const uint16_t* u_parts, int64_t ld_up, const int32_t* wide,
                                     int64_t rows, int64_t cols, int count, amct_stream_t stream) {
    if (rows < 0 || cols < 0 || count < 0 || ld_w < cols || ld_e < count || ld_u < cols || ld_ep < count || ld_up < cols) return AMCT_E_BADARG;
    if (count % 32 != 0 || ld_ep % 8 != 0 || ld_up % 8 != 0) return AMCT_E_BADARG;
    if (rows == 0 || cols == 0 || count == 0) return AMCT_OK;
    if (!w || !err || !u || !err_parts || !u_parts || !wide) return AMCT_E_BADARG;
    if (!aligned16(err_parts) || !aligned16(u_parts)) return AMCT_E_ALIGN;
    if (ld_ep >= (int64_t(1) << 22) || ld_up >= (int64_t(1) << 22)) return AMCT_E_TOO_LARGE;      // 32-bit offsets inside a stage
    const int64_t rt = (rows + kPartsTile - 1) / kPartsTile, ct = (cols + kPartsTile - 1) / kPartsTile;
    if (rt > 0x7FFFFFF0 / ct) return AMCT_E_TOO_LARGE;
    const PartsArgs a{w, err, u, err_parts, u_parts, wide, ld_w, ld_e, ld_u, ld_ep, ld_up, rows, cols, count, (int)ct, (int)(rt * ct),
                      cols % 4 == 0 && ld_w % 4 == 0 && aligned16(w)};
    hipLaunchKernelGGL(gptq_trail_parts_k, dim3((unsigned)((rt * ct + 7) / 8 * 8)), dim3(kBlock), 0, (hipStream_t)stream, a);
    return hip_status();
}
