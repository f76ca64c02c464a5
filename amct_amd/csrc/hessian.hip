// GPTQ Hessian accumulation on the matrix pipe: H <- beta * H + alpha * X^T X, the update of
// amct_pytorch/quantize_op/gptq_module.py:176-181 (hessian *= n / (n + b); x = sqrt(2 / n) * x.float();
// hessian += x @ x.t()) for 16-bit calibration activations X [tokens, columns].
//
// The products of two bf16 (or fp16) values are exact in fp32 and the MFMA accumulates in fp32, so the matrix
// product of the 16-bit inputs is the reference's fp32 product up to the order of the sum; the factor 2 / n is
// applied once to the sum instead of sqrt(2 / n) to every element.
//
// hess_syrk_k owns one square tile of the lower triangle and reads X as it lies in memory, tokens by columns: a step of 64
// tokens of the tile's two column ranges goes to LDS by direct-to-LDS loads, and the transposing LDS read
// (ds_read_b64_tr_b16: of a block of 4 tokens x 16 columns, lane i gets the 4 tokens of column i) makes MFMA operands of it.
// Two or three stages of LDS, one barrier per step; the fragments of the second half of a step are read under the products of
// the first half, those of the next step under the products of the second.
// A tile is 64, 128 or 192 columns wide, 2 x 2 waves of half that: see hs_width.  The epilogue
// applies beta and alpha, writes the tile and its mirror image, so H stays exactly symmetric, and notes whether everything
// it wrote is finite: as library passes over H that check took as long as the update itself (75 us at 4096 columns).
// X[2048,4096] bf16 into an empty / a running H[4096,4096]: 48 / 52 us, where 128-column tiles fed by a kernel that transposed X
// first took 75 / 82; 512 columns 12 / 12 (39 / 40), 2816 30 / 31 (49 / 53), 11008 295 / 351 (335 / 403).  At 4096 columns the
// products take about 31 us (21 at the rate of a register-only loop, 8 more are the loads' and LDS's), the rest is the launch
// and H itself, 64 MB written and half of it read, all tiles at the same time.
// Every sum runs over the tokens in order, 16 to an instruction, whatever the tile: GPTQ's codes follow the last bits of H
// (sums of 32 tokens an instruction, as far from the exact ones, moved codes in 7 rows of 100 of a [4096,4096] layer).
#include <type_traits>

#include "amct_common.h"

namespace amct {

typedef float h4f __attribute__((ext_vector_type(4)));
typedef float h16f __attribute__((ext_vector_type(16)));
typedef __bf16 h8bf __attribute__((ext_vector_type(8)));
typedef _Float16 h8h __attribute__((ext_vector_type(8)));
typedef short h4s __attribute__((ext_vector_type(4)));
typedef short h8s __attribute__((ext_vector_type(8)));

constexpr int kHsK = 64;                             // tokens per step

// X [T, C] -> [T, ld], columns beyond C zero: rows that start 16-byte aligned, where those of X do not.
__global__ __launch_bounds__(kBlock) void hess_align_k(const uint16_t* x, uint16_t* xa, int64_t T, int64_t C, int64_t ld) {
    const int64_t c = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * 8;
    if (c >= ld) return;
    for (int64_t t = blockIdx.y; t < T; t += gridDim.y) {
        uint16_t v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = c + j < C ? x[t * C + c + j] : (uint16_t)0;
        uint4 q;
        q.x = v[0] | (uint32_t)v[1] << 16;
        q.y = v[2] | (uint32_t)v[3] << 16;
        q.z = v[4] | (uint32_t)v[5] << 16;
        q.w = v[6] | (uint32_t)v[7] << 16;
        stg16(xa + t * ld + c, q);
    }
}

__global__ void hess_clear_k(int32_t* bad) { *bad = 0; }

struct SyrkArgs {
    const uint16_t* x;                               // [T, ld], rows 16-byte aligned
    float* h;                                        // [C, C]
    int64_t T, C, ld;
    int nb;                                          // tiles per side
    int per_die;                                     // tiles of the lower triangle per die (rounded up)
    int64_t ntiles;                                  // nb (nb + 1) / 2
    float beta, alpha;
    int vec;                                         // rows of H are 16-byte aligned
    int32_t* bad;                                    // set where an element of the new H is not finite, or null
};

template <bool F16>
AMCT_DEV h16f hs_mfma(const h8s& a, const h8s& b, const h16f& c) {
    if constexpr (F16) return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8h, a), __builtin_bit_cast(h8h, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(h8bf, a), __builtin_bit_cast(h8bf, b), c, 0, 0, 0);
}

// A direct-to-LDS load: wave-uniform 64-bit base, a byte offset per lane, lane l's 16 bytes land at lds + 16 l.  (Inline, with
// hand-counted waits: the compiler would wait for all of them before every LDS read.)
AMCT_DEV void hs_dma(uint32_t lds, const void* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(off), "s"(base) : "memory");
}
template <int N> AMCT_DEV void hs_wait() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory"); }
AMCT_DEV void hs_meet() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// W: half the 32-column MFMA tiles per side of a block (2, 4 or 6): W / 2 of them per side of a wave.  128-column tiles take two stages so
// that two blocks fit a CU, and one's epilogue runs under the other's products: X[2048,11008] 295 us, with three stages and
// one block 381.
template <int W> struct SyrkShape {
    static constexpr int kTile = 32 * W;
    static constexpr int kRow = 2 * kTile;           // bytes of a token in LDS
    static constexpr int kOperand = kHsK * kRow;
    static constexpr int kStage = 2 * kOperand;
    static constexpr int kStages = W == 4 ? 2 : 3;
    static constexpr int kLds = kStages * kStage;
    static constexpr int kPerCu = 160 * 1024 / kLds;
    static_assert(W == 2 || W == 4 || W == 6, "the swaps of LDS units below are for these");
    static_assert(kLds >= 4 * (16 * W) * (16 * W) * 4, "the epilogue's patches");
};

template <bool F16, int W>
__global__ __launch_bounds__(kBlock, SyrkShape<W>::kPerCu) void hess_syrk_k(SyrkArgs a) {
    using S = SyrkShape<W>;
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // block -> tile (bi, bj) of the lower triangle, bi >= bj.  The chip hands consecutive blocks to its eight dies in
    // turn, and each die has an L2 of its own: block id works on tile (id % 8) * per + id / 8 of an order in which
    // consecutive tiles form compact patches (bands of 8 rows of tiles, inside a band column after column), so the blocks
    // that a die runs at a time share their operand tiles.
    const int per = a.per_die;
    const int64_t logical = (int64_t)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || logical >= a.ntiles) return;         // whole block (before any barrier)
    int bi, bj;
    {
        // band b holds the rows 8 b .. min(8 b + 7, nb - 1); rows before it hold 8 b (8 b + 1) / 2 tiles
        int b = (int)((__builtin_sqrtf(8.0f * (float)logical + 1.0f) - 1.0f) * 0.5f) >> 3;
        while ((int64_t)(8 * (b + 1)) * (8 * (b + 1) + 1) / 2 <= logical) ++b;
        while ((int64_t)(8 * b) * (8 * b + 1) / 2 > logical) --b;
        const int r0 = 8 * b, r1 = min(8 * b + 7, a.nb - 1), H = r1 - r0 + 1;
        int o = (int)(logical - (int64_t)r0 * (r0 + 1) / 2);
        if (o < (r0 + 1) * H) {                      // the columns that every row of the band has
            bj = o / H;
            bi = r0 + o % H;
        } else {                                     // the triangle at the band's end: column r0 + 1 + c has H - 1 - c rows
            o -= (r0 + 1) * H;
            int c = 0;
            while (o >= H - 1 - c) { o -= H - 1 - c; ++c; }
            bj = r0 + 1 + c;
            bi = bj + o;
        }
    }
    bi = __builtin_amdgcn_readfirstlane(bi);         // (a square root is not scalar arithmetic)
    bj = __builtin_amdgcn_readfirstlane(bj);
    const bool diag = bi == bj;
    const int64_t i0 = (int64_t)bi * S::kTile, j0 = (int64_t)bj * S::kTile;
    const int wi = wave >> 1, wj = wave & 1;         // 2 x 2 waves of 16 W x 16 W

    // Memory -> LDS: per operand and step 64 tokens x 4 W chunks of 16 bytes, token after token; a wave moves W pieces of 1 KB.
    // A fragment read takes 4 tokens x 64 bytes from each half of 8 tokens: the 32-byte units of a token are swapped by the
    // token, so that four consecutive tokens' pairs of units lie in different banks (a token is 128, 256 or 384 bytes).
    // Columns beyond C repeat the last ones of X (their sums are not stored), tokens beyond T the last one (cleared below).
    auto swap = [](int t) { return W == 4 ? 2 * (t & 3) : t & 2; };
    const uint32_t row_bytes = (uint32_t)(a.ld * 2);
    uint32_t off_a[W], off_b[W];                     // bytes from the tile's first column at the step's first token
#pragma unroll
    for (int p = 0; p < W; ++p) {
        const int q = (wave * W + p) * 64 + lane, t = q / (4 * W), at = q % (4 * W);
        const int c = 8 * ((((at >> 1) ^ swap(t)) << 1) | (at & 1));
        off_a[p] = (uint32_t)t * row_bytes + 2 * (uint32_t)(min(i0 + c, a.ld - 8) - i0);
        off_b[p] = (uint32_t)t * row_bytes + 2 * (uint32_t)(min(j0 + c, a.ld - 8) - j0);
    }
    const int steps = (int)((a.T + kHsK - 1) / kHsK), last = steps - 1;
    const int tail = (int)(a.T - (int64_t)last * kHsK);                       // tokens of the last step
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds);
    auto fetch = [&](int stage, int step) {
        const uint16_t* xs = a.x + (int64_t)step * kHsK * a.ld;
        const uint32_t to = lds0 + stage * S::kStage + wave * W * 1024;
        if (step == last && tail < kHsK) {
#pragma unroll
            for (int p = 0; p < W; ++p) {
                const int t = ((wave * W + p) * 64 + lane) / (4 * W);
                const uint32_t back = t < tail ? 0u : (uint32_t)(t - tail + 1) * row_bytes;
                hs_dma(to + p * 1024, xs + i0, off_a[p] - back);
                hs_dma(to + p * 1024 + S::kOperand, xs + j0, off_b[p] - back);
            }
            return;
        }
#pragma unroll
        for (int p = 0; p < W; ++p) {
            hs_dma(to + p * 1024, xs + i0, off_a[p]);
            hs_dma(to + p * 1024 + S::kOperand, xs + j0, off_b[p]);
        }
    };
    // the tokens beyond T in the last step's stage, before anyone reads it
    auto clear_tail = [&](int stage) {
        const int z0 = tail * S::kRow / 16, z1 = S::kOperand / 16;
        for (int z = z0 + tid; z < z1; z += kBlock) {
            *reinterpret_cast<uint4*>(lds + stage * S::kStage + z * 16) = make_uint4(0, 0, 0, 0);
            *reinterpret_cast<uint4*>(lds + stage * S::kStage + S::kOperand + z * 16) = make_uint4(0, 0, 0, 0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        hs_meet();
    };

    // Fragment of 32 columns and 16 tokens: lane l holds column l % 32 and the tokens 8 (l / 32) .. + 7, each sum in the order of
    // the tokens.  Group l / 16 of the lanes reads 4 tokens x 16 columns, a lane 4 columns of token (l % 16) / 4, and is given its
    // own column by the transposition; then the 4 tokens behind (swapped alike).
    constexpr int N = W / 2;                         // 32-column tiles per side of a wave
    const int tl = 8 * (lane >> 5) + ((lane & 15) >> 2), half = (lane >> 4) & 1;
    int at_a[N], at_b[N];
#pragma unroll
    for (int m = 0; m < N; ++m) {
        at_a[m] = tl * S::kRow + ((wi * W + 2 * m + half) ^ swap(tl)) * 32 + (lane & 3) * 8;
        at_b[m] = S::kOperand + tl * S::kRow + ((wj * W + 2 * m + half) ^ swap(tl)) * 32 + (lane & 3) * 8;
    }
    auto fragment = [&](int at) {
        typedef __attribute__((address_space(3))) h4s lds_h4s;
        const h4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_h4s*)(lds + at));
        const h4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_h4s*)(lds + at + 4 * S::kRow));
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    h8s fa[2][2][N], fb[2][2][N];                    // [half of a stage: 32 tokens][16 tokens][tile]
    constexpr int kReads = 4 * N, kProducts = 2 * N * N;
    auto read_one = [&](int stage, int u, int q) {   // q < 4 N: fragment of half u
        const int ks = q / (2 * N), x = q % (2 * N), base = stage * S::kStage + (2 * u + ks) * 16 * S::kRow;
        if (x < N) fa[u][ks][x] = fragment(base + at_a[x]);
        else fb[u][ks][x - N] = fragment(base + at_b[x - N]);
    };
    h16f acc[N][N];
#pragma unroll
    for (int m = 0; m < N; ++m)
#pragma unroll
        for (int n = 0; n < N; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.f;
    // the products of half u, the fragments of the next half dealt out behind them; the column fragment is the first
    // operand: sums 4 q .. + 3 of tile (m, n) are H[32 m + lane % 32][32 n + 8 q + 4 (lane / 32) + 0 .. 3] of the wave's tile
    auto products = [&](int u, bool more, int stage, int v) {
#pragma unroll
        for (int x = 0; x < kProducts; ++x) {
            const int ks = x / (N * N), m = x / N % N, n = x % N;
            acc[m][n] = hs_mfma<F16>(fb[u][ks][n], fa[u][ks][m], acc[m][n]);
            __builtin_amdgcn_sched_barrier(0);
            if (more) {
#pragma unroll
                for (int q = x * kReads / kProducts; q < (x + 1) * kReads / kProducts; ++q) read_one(stage, v, q);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    if (steps > 0) {
        constexpr int kPer = 2 * W;                  // loads of a wave and stage
        // (steps beyond the last repeat it: the counts of the waits stay the same, and nobody reads those stages)
#pragma unroll
        for (int s = 0; s < S::kStages; ++s) fetch(s, min(s, last));
        hs_wait<(S::kStages - 1) * kPer>();
        hs_meet();
        if (last == 0 && tail < kHsK) clear_tail(0);
#pragma unroll
        for (int q = 0; q < kReads; ++q) read_one(0, 0, q);
        int stage = 0;
        for (int s = 0; s < last; ++s) {
            const int next = stage + 1 == S::kStages ? 0 : stage + 1;
            products(0, true, stage, 1);
            hs_wait<(S::kStages - 2) * kPer>();       // the next stage is there, this one is in registers
            hs_meet();
            if (s + 1 == last && tail < kHsK) clear_tail(next);
            fetch(stage, min(s + S::kStages, last));
            products(1, true, next, 0);
            stage = next;
        }
        products(0, true, stage, 1);
        products(1, false, 0, 0);
        hs_wait<0>();                                // no load may land after the block has given its LDS back
    }

    // ---- epilogue -------------------------------------------------------------------------------------------
    // The sums go through LDS, a patch per wave, so that H is read and written in whole rows of the wave's tile both ways, and
    // by loops: unrolled over the registers it was 144 stores with their checks that every wave fetched from memory as
    // instructions and ran once.  16-byte units of a row are swapped by the row (unit_of): 16 rows' same unit, which
    // 16 lanes write at a time, lie in different banks.
    hs_meet();                                       // every wave is done with the stages
    constexpr int kRows = 16 * W, kUnits = 4 * W;    // of the patch; a unit is 4 columns
    auto unit_of = [](int row, int u) {
        return u ^ (W == 4 ? (row ^ (row >> 4)) & 15 : ((row >> 1) ^ (row >> 4)) & 7);
    };
    h4f* patch = reinterpret_cast<h4f*>(lds + wave * (S::kLds / 4));
#pragma unroll
    for (int m = 0; m < N; ++m)
#pragma unroll
        for (int n = 0; n < N; ++n)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                h4f v;
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = a.alpha * acc[m][n][4 * q + r];
                const int row = 32 * m + (lane & 31);
                patch[row * kUnits + unit_of(row, 8 * n + 2 * q + (lane >> 5))] = v;
            }
    // Addresses: one block-uniform base per wave plus 32-bit lane offsets (cols < 2^22 is checked by the host).
    const bool have = a.beta != 0.f;
    const uint32_t C32 = (uint32_t)a.C;
    const int64_t wi0 = i0 + wi * kRows, wj0 = j0 + wj * kRows;               // the wave's first row and column
    float* hw = a.h + wi0 * a.C + wj0;                                        // H[wi0][wj0]
    float* hm = a.h + wj0 * a.C + wi0;                                        // its mirror image H[wj0][wi0]
    const int rows_left = (int)min((int64_t)kRows, a.C - wi0), cols_left = (int)min((int64_t)kRows, a.C - wj0);   // may be <= 0
    bool finite = true;                              // of everything this lane writes (the mirror image repeats it)
    // VEC: rows of H are 16-byte aligned and a lane takes four columns, which are inside H or outside together; else one.  Lanes
    // outside read what the first lane does and write nothing: no branches between the loads, of which a lane has kBatch in
    // flight.  (Element by element, with a branch each, the tiles at the edge of H took 25 us, and a launch waits for its
    // slowest block.)
    auto finish = [&](auto vec_tag) {
        constexpr bool VEC = decltype(vec_tag)::value;
        constexpr int V = VEC ? 4 : 1, kPieces = kRows / V, kTurns = kRows * kPieces / 64, kBatch = VEC ? 2 * W : 8;
        static_assert(kTurns % kBatch == 0, "batches");
        const float* pf = reinterpret_cast<const float*>(patch);
        auto in_patch = [&](int row, int col) { return (row * kUnits + unit_of(row, col >> 2)) * 4 + (col & 3); };
#pragma unroll 1
        for (int b = 0; b < kTurns; b += kBatch) {
            float old[kBatch][V];
            if (have) {
#pragma unroll
                for (int x = 0; x < kBatch; ++x) {
                    const int e = (b + x) * 64 + lane, row = e / kPieces, col = V * (e % kPieces);
                    const float* from = hw + (row < rows_left && col < cols_left ? (uint32_t)row * C32 + (uint32_t)col : 0u);
                    if constexpr (VEC) *reinterpret_cast<h4f*>(old[x]) = *reinterpret_cast<const h4f*>(from);
                    else old[x][0] = *from;
                }
            }
#pragma unroll
            for (int x = 0; x < kBatch; ++x) {
                const int e = (b + x) * 64 + lane, row = e / kPieces, col = V * (e % kPieces), at = in_patch(row, col);
                float v[V];
                if constexpr (VEC) *reinterpret_cast<h4f*>(v) = patch[at >> 2];
                else v[0] = pf[at];
                if (have) {
#pragma unroll
                    for (int r = 0; r < V; ++r) v[r] = old[x][r] * a.beta + v[r];
                    if constexpr (VEC) patch[at >> 2] = *reinterpret_cast<const h4f*>(v);
                    else reinterpret_cast<float*>(patch)[at] = v[0];
                }
                if (row < rows_left && col < cols_left) {
                    float* to = hw + ((uint32_t)row * C32 + (uint32_t)col);
                    if constexpr (VEC) *reinterpret_cast<h4f*>(to) = *reinterpret_cast<const h4f*>(v);
                    else *to = v[0];
#pragma unroll
                    for (int r = 0; r < V; ++r) finite = finite && finite_f(v[r]);
                }
            }
        }
        if (diag) return;                            // the tile on the diagonal is its own mirror image
        // mirror image: a lane takes V rows of one column of the patch (the patch is the wave's own: no barrier)
#pragma unroll 1
        for (int b = 0; b < kTurns; b += 4) {
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const int e = (b + x) * 64 + lane, col = e / kPieces, row = V * (e % kPieces);
                float v[V];
#pragma unroll
                for (int r = 0; r < V; ++r) v[r] = pf[in_patch(row + r, col)];
                if (col < cols_left && row < rows_left) {
                    float* to = hm + ((uint32_t)col * C32 + (uint32_t)row);
                    if constexpr (VEC) *reinterpret_cast<h4f*>(to) = *reinterpret_cast<const h4f*>(v);
                    else *to = v[0];
                }
            }
        }
    };
    if (rows_left > 0 && cols_left > 0) {
        if (a.vec) finish(std::true_type{});
        else finish(std::false_type{});
    }
    if (a.bad && !finite) *a.bad = 1;
}

}  // namespace amct

using namespace amct;

static int64_t hs_round_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

// The width of the tiles by their number, for 256 CUs.  64 columns while three tiles a CU hold them all (to 2432 columns): short
// tiles, many of them (2048 tokens of 512 / 2048 columns: 11.9 / 23.4 us, with 128 columns 24.2 / 29.1; at 2560 columns 31.4 and 30.4).
// Else 128, two a CU.  Where these need a second round for a few more (3969 columns and on) but tiles of 192 columns do with one
// a CU (to 4224), 192: 4096 columns 47.8 us, with 128 62.6; 3968 columns 46.8 and 40.2; 4608 90.1 and 66.8.  Not where rows of H
// are not 16-byte aligned: a column a lane, four waves a CU take 25 us longer over their H (512 tokens of 4098 columns: 49.0 / 58.8
// into an empty / a running H, with 128 44.2 / 52.8, from the transposed copy 41.9 / 59.1).
static int hs_width(int64_t cols, bool vec) {
    auto tiles = [cols](int64_t side) { const int64_t nb = (cols + side - 1) / side; return nb * (nb + 1) / 2; };
    if (tiles(64) <= 3 * 256) return 2;
    return vec && tiles(128) > 2 * 256 && tiles(192) <= 256 ? 6 : 4;
}


template <bool F16, int W> static void hs_launch(SyrkArgs a, hipStream_t st) {
    a.nb = (int)((a.C + 32 * W - 1) / (32 * W));
    a.ntiles = (int64_t)a.nb * (a.nb + 1) / 2;
    a.per_die = (int)((a.ntiles + 7) / 8);
    hipLaunchKernelGGL((hess_syrk_k<F16, W>), dim3((unsigned)(8 * (int64_t)a.per_die)), dim3(kBlock), SyrkShape<W>::kLds, st, a);
}

extern "C" size_t amct_hessian_update_workspace_bytes(int64_t tokens, int64_t cols) {
    if (tokens <= 0 || cols <= 0) return 0;
    return (size_t)hs_round_up(cols, 128) * (size_t)hs_round_up(tokens, kHsK) * 2;
}

static int hessian_launch(float* hessian, const void* x, int64_t tokens, int64_t cols, float beta, float alpha, int dtype, int32_t* bad,
                          bool clear, void* workspace, size_t workspace_bytes, amct_stream_t stream);

extern "C" int amct_hessian_update(float* hessian, const void* x, int64_t tokens, int64_t cols, float beta, float alpha,
                                   int dtype, void* workspace, size_t workspace_bytes, amct_stream_t stream) {
    return hessian_launch(hessian, x, tokens, cols, beta, alpha, dtype, nullptr, false, workspace, workspace_bytes, stream);
}

extern "C" int amct_hessian_update_checked(float* hessian, const void* x, int64_t tokens, int64_t cols, float beta, float alpha,
                                           int dtype, int32_t* bad, void* workspace, size_t workspace_bytes, amct_stream_t stream) {
    return hessian_launch(hessian, x, tokens, cols, beta, alpha, dtype, bad, true, workspace, workspace_bytes, stream);
}

extern "C" int amct_hessian_update_flag(float* hessian, const void* x, int64_t tokens, int64_t cols, float beta, float alpha, int dtype,
                                        int32_t* flag, void* workspace, size_t workspace_bytes, amct_stream_t stream) {
    return hessian_launch(hessian, x, tokens, cols, beta, alpha, dtype, flag, false, workspace, workspace_bytes, stream);
}

static int hessian_launch(float* hessian, const void* x, int64_t tokens, int64_t cols, float beta, float alpha, int dtype, int32_t* bad,
                          bool clear, void* workspace, size_t workspace_bytes, amct_stream_t stream) {
    if (tokens < 0 || cols <= 0 || !hessian) return AMCT_E_BADARG;
    if (dtype != AMCT_BF16 && dtype != AMCT_F16) return AMCT_E_UNSUPPORTED;
    if (tokens != 0 && !x) return AMCT_E_BADARG;
    if (cols >= (int64_t(1) << 22)) return AMCT_E_TOO_LARGE;                  // 32-bit offsets inside a tile, block ids
    const size_t need = (size_t)hs_round_up(cols, 128) * (size_t)hs_round_up(tokens > 0 ? tokens : 1, kHsK) * 2;
    if (!workspace || workspace_bytes < need) return AMCT_E_BADARG;
    if (!aligned16(workspace) || (reinterpret_cast<uintptr_t>(hessian) & 3u) != 0 || (reinterpret_cast<uintptr_t>(x) & 1u) != 0)
        return AMCT_E_ALIGN;
    hipStream_t st = (hipStream_t)stream;
    SyrkArgs a{reinterpret_cast<const uint16_t*>(x), hessian, tokens, cols, cols, 0, 0, 0, beta, alpha,
               cols % 4 == 0 && aligned16(hessian), bad};
    if (bad && clear) hipLaunchKernelGGL(hess_clear_k, dim3(1), dim3(1), 0, st, bad);
    if (cols % 8 != 0 || !aligned16(x)) {
        a.ld = hs_round_up(cols, 8);
        if (tokens > 0)
            hipLaunchKernelGGL(hess_align_k, dim3((unsigned)((a.ld / 8 + kBlock - 1) / kBlock), (unsigned)(tokens < 65535 ? tokens : 65535)),
                               dim3(kBlock), 0, st, reinterpret_cast<const uint16_t*>(x), reinterpret_cast<uint16_t*>(workspace), tokens, cols,
                               a.ld);
        a.x = reinterpret_cast<const uint16_t*>(workspace);
    }
#define AMCT_HS(W)                                              \
    case W:                                                     \
        if (dtype == AMCT_F16) hs_launch<true, W>(a, st);       \
        else hs_launch<false, W>(a, st);                        \
        break;
    switch (hs_width(cols, a.vec != 0)) {
        AMCT_HS(2) AMCT_HS(4) AMCT_HS(6)
    }
#undef AMCT_HS
    return hip_status();
}
