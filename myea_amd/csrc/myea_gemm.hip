// myea_gemm.hip — dense FP32 contraction for gfx950 (CDNA4) on the BF16 matrix cores, LDS-staged.
//
// One kernel template covers the three contractions of the fully-connected and LSTM path:
//   forward  Y  = X W^T          (A k-contiguous, B k-contiguous)   Forward_Pass__FC,
//            Neural_Network__Forward_Pass__OpenMP.cpp:4517-4557
//   backward dX = delta W        (A k-contiguous, B n-contiguous)   Backward_Pass__FC, Neural_Network__Backward_Pass__OpenMP.cpp:1044-1082
//   weights  dW += delta^T X     (A m-contiguous, B n-contiguous)   Update_Derivative_Weight__FC,
//            Neural_Network__Update_Derivative_Weight__OpenMP.cpp:178-216
//
// Arithmetic.  gfx950 multiplies FP32 at 157 TFLOP/s and BF16 at 2.5 PFLOP/s.  An FP32 number below 2^103 is the sum of three
// BF16 numbers, but for a power of two that keeps the smallest of them normal (myea_split.h): hi = x rounded to BF16, mid = (x
// - hi) rounded to BF16, lo = what is left (8 + 8 + 8 significant bits, signs included, cover the 24 of x; both differences
// are exact in FP32).  Of the nine products of two such sums the six with a weight above 2^-24 are formed - hi hi, hi mid, mid
// hi, mid mid, hi lo, lo hi - each exact in the matrix unit, all accumulated in FP32.  What is left out is below 2^-25 of a
// product.  The five smaller products have an accumulator of their own, added at the end: an accumulator as large as the
// result is rounded (to nearest, as measured) once per 16 k's, where v_mfma_f32_32x32x2_f32 rounds it at every second k, and
// from 16 k's on (fewer are another kernel's) the measured error against 64-bit sums is smaller than that instruction's
// (normal operands, 2-norm: 4e-7 against 1.15e-6 at k = 4096, 1.3e-7 against 4.1e-7 at k = 512; positive ones: 3.1e-7 against
// 8.4e-7 at k = 4096, 6.0e-7 against 1.7e-6 at k = 16384).  Six BF16 instructions for 16 k's take 6 x 32 cycles of a SIMD's
// matrix unit where the FP32 ones take 8 x 64: the ceiling moves from 157 to 419 TFLOP/s, and to 190 at the 1.14 PFLOP/s that
// a large BF16 product was measured to sustain on this card.  Measured, FP32 instruction -> this: 1024 x 4096 x 4096 forward
// 296 -> 197 us, its weight gradient 303 -> 196 us (176 TFLOP/s), 16384 x 2048 x 512 307 -> 199 us, 512 x 2048 x 2048 44.5 ->
// 37.4; 333 x 1201 x 1201, whose rows are no 16-byte multiples and which is a short product now, 50 -> 21 us.
// Infinities and NaN do not survive the split (inf - inf), nor do finite values whose scaled hi is a BF16 infinity: such a product
// always leaves a non-finite accumulator, and a wavefront that finds one computes its accumulators again with the FP32
// instruction (redo_in_f32), so the results are those of FP32 arithmetic there too.
//
// Tiling: a workgroup of 256 lanes (4 wavefronts, 2 x 2) owns a BM x BN tile of C; each wavefront owns (BM/2) x (BN/2) as
// TM x TN accumulators of v_mfma_f32_32x32x16_bf16 (16 VGPRs each).  A K step moves BK columns: global -> registers (asked for
// two steps ahead or four), split there once, three BF16 planes -> LDS (two stages, one barrier per step).  What bounds a step is
// issue: per 16 k's of a 128 x 128 tile a wavefront has 24 matrix instructions (768 cycles) and about 120 vector ones (480), so
// the splitting of the next step is spread between the matrix instructions of this one (2048 x 2048 x 2048: 114 us with the
// compiler's order, 98 us so).  An operand's place in LDS does not depend on its orientation in memory:
//   [plane][k / 8][row][8 k's]     a fragment (row l % 32, k's 8 (l / 32) .. + 7 of lane l) is one conflict-free ds_read_b128
// Counted (1024 x 4096 x 4096, two workgroups a tile): the matrix unit is busy 56 % of the clocks, 5 vector instructions a matrix
// instruction, no bank conflicts; 64 x 64 tiles (1024 x 1000 x 4096) 37 %, and a k-contiguous operand's stores, four chunks of a row at a
// time, lose a sixth of the clocks to conflicts there.
// A k-contiguous operand is read as two 16-byte loads per lane, the other kind as eight 4-byte loads that are coalesced over
// the rows; neither needs more than 4-byte alignment, so odd widths and leading dimensions take the same path.
//
// Accumulator layout of v_mfma_f32_32x32x16_bf16, as of v_mfma_f32_32x32x2_f32: register r of lane l holds
//   C[(r / 4) * 8 + (l / 32) * 4 + (r % 4)][l % 32].
#include <cstdlib>
#include <mutex>

#include "myea_device_af.h"
#include "myea_kernels.h"
#include "myea_split.h"

namespace myea {

namespace {

constexpr int kThreads = 256;
constexpr int kBK = 32;   // slabs and halves of a k range are multiples of this

// K columns per step: two stages of the 128 x 128 tile at 16 leave room for two workgroups a CU, the smaller tiles take a whole
// 128-byte line of a k-contiguous row at a time
constexpr int step_of(int bm, int bn) { return bm * bn >= 128 * 128 ? 16 : 32; }

// Where one operand tile (ROWS x BK, three planes) lies in an LDS stage: 16-byte chunks of 8 k's.
template <int ROWS, int BK>
struct PlaneShape {
    static constexpr int kChunkRow = ROWS * 16 + 64;            // bytes of one [k / 8] slice; the pad keeps the slices' equal rows on different banks
    static constexpr int kPlane = (BK / 8) * kChunkRow;
    static constexpr int kBytes = 3 * kPlane;
    static constexpr int kChunks = ROWS * BK / 8;
    static constexpr int kPerThread = kChunks / kThreads;
    static_assert(kChunks % kThreads == 0, "a tile's chunks go round the workgroup evenly");
    static __device__ __forceinline__ int at(int plane, int k8, int row) { return plane * kPlane + k8 * kChunkRow + row * 16; }
};

// Global -> registers -> three planes in LDS for one operand tile; `AHEAD` steps wait in registers.
template <int ROWS, int BK, bool KC, int AHEAD>
struct SplitMover {
    using S = PlaneShape<ROWS, BK>;
    float reg[AHEAD][S::kPerThread][8];
    const float *ptr[S::kPerThread];   // the chunk's first element in the step that is loaded next
    long ld, step;

    static __device__ __forceinline__ int row_of(int p) { const int q = threadIdx.x + p * kThreads; return KC ? q / (BK / 8) : q % ROWS; }
    static __device__ __forceinline__ int k8_of(int p) { const int q = threadIdx.x + p * kThreads; return KC ? q % (BK / 8) : q / ROWS; }

    // base: operand origin; row0: first row (m or n) of the tile; rows beyond the extent repeat the last one (never stored)
    __device__ __forceinline__ void init(const float *base, long ld_, int row0, int extent, int k0)
    {
        ld = ld_; step = KC ? (long)BK : (long)BK * ld;
#pragma unroll
        for (int p = 0; p < S::kPerThread; ++p) {
            const long row = min(row0 + row_of(p), extent - 1), k = k0 + k8_of(p) * 8;
            ptr[p] = base + (KC ? row * ld + k : k * ld + row);
        }
    }

    // asks for a whole step, and moves on to the next one if there is another whole one (`more`)
    __device__ __forceinline__ void load(int slot, bool more)
    {
        const long onward = more ? step : 0;
#pragma unroll
        for (int p = 0; p < S::kPerThread; ++p) {
            if (KC) {
                *reinterpret_cast<f32x4 *>(reg[slot][p]) = *reinterpret_cast<const f32x4_any *>(ptr[p]);
                *reinterpret_cast<f32x4 *>(reg[slot][p] + 4) = *reinterpret_cast<const f32x4_any *>(ptr[p] + 4);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) reg[slot][p][e] = ptr[p][e * ld];
            }
            ptr[p] += onward;
        }
    }

    // the last, partial step: `left` k's, zeros behind them (in both operands)
    __device__ __forceinline__ void load_tail(int left)
    {
#pragma unroll
        for (int p = 0; p < S::kPerThread; ++p)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                reg[0][p][e] = 0.f;
                if (k8_of(p) * 8 + e < left) reg[0][p][e] = ptr[p][KC ? (long)e : e * ld];
            }
    }

    __device__ __forceinline__ void store(int slot, char *tile) const
    {
#pragma unroll
        for (int p = 0; p < S::kPerThread; ++p) {
            unsigned hi[4], mid[4], lo[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) split_pair(reg[slot][p][2 * e], reg[slot][p][2 * e + 1], hi[e], mid[e], lo[e]);
            const int row = row_of(p), k8 = k8_of(p);
            *reinterpret_cast<u32x4 *>(tile + S::at(0, k8, row)) = (u32x4){hi[0], hi[1], hi[2], hi[3]};
            *reinterpret_cast<u32x4 *>(tile + S::at(1, k8, row)) = (u32x4){mid[0], mid[1], mid[2], mid[3]};
            *reinterpret_cast<u32x4 *>(tile + S::at(2, k8, row)) = (u32x4){lo[0], lo[1], lo[2], lo[3]};
        }
    }
};

struct GemmDev {
    const float *A, *B;
    float *C;
    int M, N, K;
    long lda, ldb, ldc;
    int accumulate, epilogue;
    const float *bias;
    float *aux_out;
    const float *colscale;
    const float *pre, *val;
    int act;
    float steep;
    const float *addend;
    long ld_addend;
    float *col_partials;
    const float *hats;
    int nbm, nbn;
    int ksplit, kchunk;   // split-K: number of slabs and k's per slab (multiple of BK); slab s writes C + s * slab
    long slab;
    float *pair_partials;    // not null: ksplit == 2 and the two workgroups of a tile combine their halves in the launch
    unsigned *pair_tickets;
    unsigned *pair_fault, *pair_host_flag;   // raised when the wait for the tile's other half runs out of polls
    unsigned pair_polls;
    int pair_local;          // the two workgroups of a tile run on one XCD (ids equal mod 8): its L2 is where they meet
};

__device__ __forceinline__ unsigned pair_xcc_id() { return __builtin_amdgcn_s_getreg(20 | (3 << 11)) & 15u; }   // HW_REG_XCC_ID[3:0]

struct TilePlace {
    int m0, n0, wave_m, wave_n, lane32, half;
    long slab_offset;
};

// The accumulators of one wavefront go out: a lane owns one column of each 32 x 32 accumulator (rows
// (r / 4) * 8 + half * 4 + r % 4), so per-column operands are read once.  The kind of epilogue, the class of the
// activation and the presence of an addend are the same for every element of a launch, and whether a tile lies wholly
// inside the matrix is the same for every element of the tile: all four are template parameters, decided once per tile,
// and the element loop carries no test of them (it carried a dozen branches per element before, 5 - 10 us per tile).
//   KIND 0 store | 3 add onto C (one hardware add per element, performed at the L2: every element is owned by exactly one
//        lane of one workgroup, so the result is the C + v a load / add / store gives, and nothing waits for C to come in)
//   KIND 1 forward: C = v + bias, aux_out = AF(C) * column multiplier; CLASS 0 no aux_out, 1 piecewise linear (linear, ReLU,
//        leaky: s < 0 ? slope * s : s, ReLU's zero kept exact), 2 through exp (sigmoid, tanh: a / (1 + exp(k s)) - b)
//   KIND 2 C = v * AF'(pre, steep, val); CLASS 1 piecewise (q < 0 ? steep * slope : steep), 2 smooth (tanh, sigmoid);
//        with col_partials, the sum of each 32-row accumulator's column goes out too: 16 values per lane, the two lanes
//        of a column combined, one store per (32-row block, column) - the bias gradient needs no pass of its own over C
// Edge tiles (WHOLE false) run the same arithmetic behind a bounds test per element, so an element's value does not
// depend on the tile shape it was computed in.
template <int KIND, int CLASS, bool ADDEND, bool WHOLE, int TM, int TN>
__device__ __forceinline__ void store_tile_as(const GemmDev &p, const f32x16 (&acc)[TM][TN], const TilePlace &at)
{
    const bool relu = p.act == MYEA_AF_RELU, tanh_like = p.act == MYEA_AF_TANH;
    const float slope = p.act == MYEA_AF_LINEAR ? 1.f : 0.01f;                       // piecewise classes (ReLU handled by `relu`)
    const float ek = tanh_like ? -2.f : -1.f, ea = tanh_like ? 2.f : 1.f, eb = tanh_like ? 1.f : 0.f;
    const float d_neg = relu ? 0.f : (p.act == MYEA_AF_LINEAR ? p.steep : p.steep * 0.01f);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = at.n0 + at.wave_n + j * 32 + at.lane32;
        if (!WHOLE && col >= p.N) continue;
        float bias = 0.f, cs = 1.f;
        if (KIND == 1) {
            if (p.bias) bias = p.bias[col];
            if (CLASS != 0 && p.colscale) cs = p.colscale[col];
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            int row0 = at.m0 + at.wave_m + i * 32 + at.half * 4;
            asm volatile("" : "+v"(row0));   // the addresses of this accumulator's rows are formed here: hoisted, those of all accumulators together spill
            float column_sum = 0.f, column_sum2 = 0.f;   // per kind: see col_partials
            // What an accumulator's elements read from other tensors - the addend, the pre-activation or the activation, x-hat -
            // is asked for four elements at a time, ahead of their arithmetic: read where it is used, every load would sit behind
            // the store of the element before it (the compiler may not move it across: the tensors could overlap) and cost its
            // own trip to memory.  (All sixteen at once need 48 more registers than the 128 x 128 tile leaves.)
#pragma unroll
            for (int rq = 0; rq < 4; ++rq) {
            float addend_v[4], operand_v[4], hats_v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = row0 + rq * 8 + e;
                addend_v[e] = 0.f; operand_v[e] = 0.f; hats_v[e] = 0.f;
                if (!WHOLE && row >= p.M) continue;
                const long o = (long)row * p.ldc + col + at.slab_offset;
                if (ADDEND) addend_v[e] = p.addend[(long)row * p.ld_addend + col];
                if (KIND == 2) {
                    operand_v[e] = CLASS == 1 ? p.pre[o] : p.val[o];
                    if (p.hats) hats_v[e] = p.hats[o];
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = rq * 4 + e;
                const int row = row0 + rq * 8 + e;
                if (!WHOLE && row >= p.M) continue;
                const long o = (long)row * p.ldc + col + at.slab_offset;
                float v = acc[i][j][r];
                if (ADDEND) v += addend_v[e];
                if (KIND == 1) {
                    v += bias;
                    p.C[o] = v;
                    {
#pragma clang fp contract(off)   // as for the derivative's sums below: the same bits from every tile shape
                        column_sum = column_sum + v;
                        column_sum2 = column_sum2 + v * v;
                    }
                    if (CLASS == 1) {
                        const float neg = slope * v;
                        p.aux_out[o] = (v < 0.f ? (relu ? 0.f : neg) : v) * cs;
                    } else if (CLASS == 2) {
                        const float e = expf(ek * v);
                        p.aux_out[o] = (ea / (1.f + e) - eb) * cs;
                    }
                } else if (KIND == 2) {
                    float dv;
                    if (CLASS == 1) {
                        dv = operand_v[e] < 0.f ? d_neg : p.steep;
                    } else {
                        const float y = operand_v[e];
                        dv = tanh_like ? p.steep * (1.f - y * y) : p.steep * y * (1.f - y);
                    }
                    {
#pragma clang fp contract(off)   // the sum takes the stored, rounded product - never a fused multiply-add - so every tile shape gives the same bits
                        const float out = v * dv;
                        p.C[o] = out;
                        column_sum = column_sum + out;
                        if (p.hats) column_sum2 = column_sum2 + out * hats_v[e];
                    }
                } else if (KIND == 3) {
                    unsafeAtomicAdd(&p.C[o], v);
                } else {
                    p.C[o] = v;
                }
            }
            }
            if ((KIND == 1 || KIND == 2) && p.col_partials) {
                const float both = column_sum + __shfl_xor(column_sum, 32);   // the column's other 16 rows of this accumulator
                const float both2 = column_sum2 + __shfl_xor(column_sum2, 32);
                const int block_row = at.m0 + at.wave_m + i * 32;
                if (at.half == 0 && (WHOLE || block_row < p.M)) {
                    if (KIND == 2 && !p.hats) {
                        p.col_partials[(long)(block_row >> 5) * p.N + col] = both;
                    } else {   // pairs: forward (sum, sum of squares); derivative with hats (sum of C * hats, sum of C)
                        float *pair = p.col_partials + (long)(block_row >> 5) * 2 * p.N + col;
                        pair[0] = KIND == 1 ? both : both2;
                        pair[p.N] = KIND == 1 ? both2 : both;
                    }
                }
            }
        }
    }
}

template <bool WHOLE, int TM, int TN>
__device__ __forceinline__ void store_tile_kind(const GemmDev &p, const f32x16 (&acc)[TM][TN], const TilePlace &at)
{
    const bool smooth = p.act == MYEA_AF_TANH || p.act == MYEA_AF_SIGMOID;
    if (p.epilogue == EPI_FC_FORWARD) {          // the launcher admits no addend on this kind nor on an accumulating launch
        if (!p.aux_out) store_tile_as<1, 0, false, WHOLE, TM, TN>(p, acc, at);
        else if (smooth) store_tile_as<1, 2, false, WHOLE, TM, TN>(p, acc, at);
        else store_tile_as<1, 1, false, WHOLE, TM, TN>(p, acc, at);
    } else if (p.epilogue == EPI_FC_DERIVE) {
        if (p.addend) { if (smooth) store_tile_as<2, 2, true, WHOLE, TM, TN>(p, acc, at); else store_tile_as<2, 1, true, WHOLE, TM, TN>(p, acc, at); }
        else { if (smooth) store_tile_as<2, 2, false, WHOLE, TM, TN>(p, acc, at); else store_tile_as<2, 1, false, WHOLE, TM, TN>(p, acc, at); }
    } else if (p.accumulate) {
        store_tile_as<3, 0, false, WHOLE, TM, TN>(p, acc, at);
    } else {
        if (p.addend) store_tile_as<0, 0, true, WHOLE, TM, TN>(p, acc, at);
        else store_tile_as<0, 0, false, WHOLE, TM, TN>(p, acc, at);
    }
}

// The accumulators of one wavefront again, with the FP32 matrix instruction and operands straight from memory: for products in
// which infinities, NaN or overflows took part.  Rows and columns beyond the matrix repeat the last one.
template <bool A_KC, bool B_KC, int TM, int TN>
__device__ __forceinline__ void redo_in_f32(const GemmDev &p, f32x16 (&acc)[TM][TN], int row, int col, int half, int k_begin, int k_end)
{
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    for (long k0 = k_begin; k0 < k_end; k0 += 2) {
        const long k = k0 + half;
        float a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const long m = min(row + i * 32, p.M - 1);
            a[i] = k < k_end ? p.A[A_KC ? m * p.lda + k : k * p.lda + m] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const long n = min(col + j * 32, p.N - 1);
            b[j] = k < k_end ? p.B[B_KC ? n * p.ldb + k : k * p.ldb + n] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
}

template <int BM, int BN>
constexpr int stage_bytes() { return PlaneShape<BM, step_of(BM, BN)>::kBytes + PlaneShape<BN, step_of(BM, BN)>::kBytes; }

// One workgroup's share of a contraction: tile number `block` of problem `p`, staged through `smem`.
template <int BM, int BN, bool A_KC, bool B_KC>
__device__ __forceinline__ void gemm_tile(const GemmDev &p, const int block, char *smem)
{
    constexpr int TM = BM / 64, TN = BN / 64;  // 32x32 accumulators per wavefront along m / n
    constexpr int BK = step_of(BM, BN);
    using SA = PlaneShape<BM, BK>;
    using SB = PlaneShape<BN, BK>;
    constexpr int kAhead = BM * BN > 64 * 64 ? 2 : 4;   // steps that wait in registers (even: a step's stage is known at compile time)
    using MA = SplitMover<BM, BK, A_KC, kAhead>;
    using MB = SplitMover<BN, BK, B_KC, kAhead>;
    constexpr int kStage = SA::kBytes + SB::kBytes;  // one LDS stage = A planes then B planes

    // Workgroup -> tile.  Consecutive workgroup ids land on different XCDs (8 of them, each with its own
    // L2), so give every XCD a contiguous run of tile ids, and walk tiles in bands of 8 m-tiles so that a
    // run shares its B columns and a small set of A rows.
    const int nblocks = p.nbm * p.nbn;
    const int split = block / nblocks;   // split-K slab of this workgroup
    int pid = block - split * nblocks;
    if ((nblocks & 7) == 0) pid = (pid & 7) * (nblocks >> 3) + (pid >> 3);
    const int k_begin = split * p.kchunk, k_end = (int)min((long)p.K, (long)k_begin + p.kchunk);
    constexpr int kBand = 8;
    const int band = pid / (kBand * p.nbn);
    const int band_first = band * kBand;
    const int band_rows = min(p.nbm - band_first, kBand);
    const int in_band = pid - band * kBand * p.nbn;
    const int m0 = (band_first + in_band % band_rows) * BM;
    const int n0 = (in_band / band_rows) * BN;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lane32 = lane & 31, half = lane >> 5;
    const int wave_m = (wave >> 1) * (BM / 2), wave_n = (wave & 1) * (BN / 2);

    f32x16 acc[TM][TN], small[TM][TN];   // the hi hi products; the others
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = small[i][j][r] = 0.f;

    bf16x8 fa[BK / 16][3][TM], fb[BK / 16][3][TN];
    auto read = [&](const char *la) {
        const char *lb = la + SA::kBytes;
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks)
#pragma unroll
            for (int pl = 2; pl >= 0; --pl) {
#pragma unroll
                for (int i = 0; i < TM; ++i) fa[ks][pl][i] = *reinterpret_cast<const bf16x8 *>(la + SA::at(pl, ks * 2 + half, wave_m + i * 32 + lane32));
#pragma unroll
                for (int j = 0; j < TN; ++j) fb[ks][pl][j] = *reinterpret_cast<const bf16x8 *>(lb + SB::at(pl, ks * 2 + half, wave_n + j * 32 + lane32));
            }
    };
    auto multiply = [&]() {
        constexpr int pa[6] = {0, 2, 1, 0, 1, 0}, pb[6] = {2, 0, 1, 1, 0, 0};   // hi hi last
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks)
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        (q < 5 ? small[i][j] : acc[i][j]) = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[ks][pa[q]][i], fb[ks][pb[q]][j], q < 5 ? small[i][j] : acc[i][j], 0, 0, 0);
    };
    // The order of a step's instructions: the fragments first, then some of the splitting's between every two matrix instructions,
    // which leave the wavefront idle otherwise (left alone the compiler splits everything before the first of them).  A pair of
    // elements takes 13 vector instructions; room for 32 is left, so that the splitting is done behind two fifths of the matrix
    // instructions and its stores have the others to land behind (us at room for 13 -> 32: 512 x 2048 x 2048 40.6 -> 36.6,
    // 1024 x 1000 x 4096 76 -> 68.7, 1024 x 4096 x 4096 194 -> 185).
    constexpr int kMatrix = 6 * TM * TN * (BK / 16), kWrites = 3 * (MA::S::kPerThread + MB::S::kPerThread), kRoom = 32 * 4 * (MA::S::kPerThread + MB::S::kPerThread);
    auto interleave = [&]() {
        __builtin_amdgcn_sched_group_barrier(0x100, 3 * (TM + TN) * (BK / 16), 0);   // LDS reads
#pragma unroll
        for (int q = 0; q < kMatrix; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);           // a matrix instruction
            __builtin_amdgcn_sched_group_barrier(0x002, (kRoom + kMatrix - 1) / kMatrix + 1, 0);   // vector arithmetic
            if (q % (kMatrix / kWrites) == kMatrix / kWrites - 1) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);   // an LDS write
        }
    };
    // The whole steps.  While step kt multiplies from its stage, step kt + 1 is split out of the registers into the other stage,
    // those registers ask for step kt + 1 + kAhead, and one barrier ends the step.  Loads and stores behind the last whole step
    // repeat it: no branch in the loop, so every wait counts exactly the loads it needs.
    MA moveA;
    MB moveB;
    moveA.init(p.A, p.lda, m0, p.M, k_begin);
    moveB.init(p.B, p.ldb, n0, p.N, k_begin);
    const int whole = (k_end - k_begin) / BK, left = (k_end - k_begin) - whole * BK;
    if (whole > 0) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            moveA.load(u, u + 1 < whole);
            moveB.load(u, u + 1 < whole);
        }
        moveA.store(0, smem);
        moveB.store(0, smem + SA::kBytes);
        moveA.load(0, kAhead + 1 < whole);
        moveB.load(0, kAhead + 1 < whole);
        __syncthreads();
        for (int kt = 0; kt < whole; kt += kAhead) {
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                if (u > 0 && kt + u >= whole) break;
                char *next = smem + ((u + 1) & 1) * kStage;
                read(smem + (u & 1) * kStage);   // in front of the stores: the compiler cannot tell the stages apart
                moveA.store((u + 1) % kAhead, next);
                moveB.store((u + 1) % kAhead, next + SA::kBytes);
                moveA.load((u + 1) % kAhead, kt + u + 2 + kAhead < whole);
                moveB.load((u + 1) % kAhead, kt + u + 2 + kAhead < whole);
                multiply();
                interleave();
                __syncthreads();
            }
        }
    }
    if (left > 0) {
        moveA.init(p.A, p.lda, m0, p.M, k_end - left);
        moveB.init(p.B, p.ldb, n0, p.N, k_end - left);
        moveA.load_tail(left);
        moveB.load_tail(left);
        moveA.store(0, smem);
        moveB.store(0, smem + SA::kBytes);
        __syncthreads();
        read(smem);
        multiply();
    }
    {   // an infinity, a NaN or a value that is a BF16 infinity took part (or the result itself is one): FP32 says what it is
        float finite = 0.f;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[i][j][r] = unscaled(acc[i][j][r] + small[i][j][r]);
                    finite = fmaf(acc[i][j][r], 0.f, finite);
                }
        if (__any(finite != 0.f)) redo_in_f32<A_KC, B_KC, TM, TN>(p, acc, m0 + wave_m + lane32, n0 + wave_n + lane32, half, k_begin, k_end);
    }

    if (BM == BN && p.pair_partials) {   // only launches of square tiles are split this way
        // Two workgroups share this tile, one per half of k (their ids are equal mod 8: the same XCD).  Whoever is done first
        // leaves its accumulators and goes; the other adds them and carries on to the epilogue.  The sum is half 0 + half 1
        // either way.  The wait below is for a workgroup that has nothing left to do but store its tile and raise its flag.
        __shared__ unsigned s_ticket;
        const int tile = block - split * nblocks;
        unsigned *ticket = p.pair_tickets + 2 * tile, *flag = ticket + 1;
        float *partial = p.pair_partials + (size_t)tile * (BM * BN);
        if (threadIdx.x == 0) s_ticket = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (s_ticket == 0u) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        __hip_atomic_store(partial + ((i * TN + j) * 16 + r) * kThreads + threadIdx.x, acc[i][j][r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this wavefront's stores are complete
            __syncthreads();
            // Publishes the tile stored above.  On one XCD the stores (performed at the L2, acknowledged) are visible to every load
            // that bypasses its compute unit's L1, and the flag carries this workgroup's XCC id for the other to check; a release
            // at device scope writes the whole L2's dirty lines back first and its acquire sends the partner's loads to memory:
            // measured 6 k + 5 k clocks against 2 k + 1.5 k.
            if (threadIdx.x == 0) {
                if (p.pair_local) __hip_atomic_store(flag, 0x100u | (pair_xcc_id() + 1u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else __hip_atomic_store(flag, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            }
            return;
        }
        // The wait is bounded.  When it runs out the other half is not there to add: this workgroup raises the network's fault
        // words (a device word the update kernels look at, a pinned host word the next call that looks reports) and leaves
        // without storing its tile.  Ticket and flag stay as they are - a late partner still raises its flag - and the host
        // clears both before these buffers serve another launch.
        __shared__ unsigned s_there;
        if (threadIdx.x == 0) {
            unsigned there = 0u;
            for (unsigned polls = 0; polls < p.pair_polls; ++polls) {   // plain looks; the acquire that makes the tile visible comes once, behind them
                there = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (there != 0u) break;
                __builtin_amdgcn_s_sleep(1);
            }
            // on one XCD nothing more is needed; a partner that ran elsewhere (never seen: the host probed the placement) is a fault
            if (p.pair_local && there != 0u && there != (0x100u | (pair_xcc_id() + 1u))) there = 0u;
            if (!p.pair_local && there != 0u) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            if (there != 0u) {
                __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // as the next launch expects them
                __hip_atomic_store(flag, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
                if (p.pair_fault) __hip_atomic_store(p.pair_fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (p.pair_host_flag) __hip_atomic_store(p.pair_host_flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
            s_there = there;
        }
        __syncthreads();
        if (s_there == 0u) return;
        // The other half, an accumulator at a time: its sixteen values are asked for together (device-scope loads one behind the
        // other, each used before the next was issued, cost a trip to the L2 apiece: 350 clocks x 16 x the tile's accumulators).
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                float other[16];
                if (p.pair_local) {   // served by the L2, never by this compute unit's L1
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        other[r] = __hip_atomic_load(partial + ((i * TN + j) * 16 + r) * kThreads + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } else {
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        other[r] = __builtin_nontemporal_load(partial + ((i * TN + j) * 16 + r) * kThreads + threadIdx.x);
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = split == 0 ? acc[i][j][r] + other[r] : other[r] + acc[i][j][r];
            }
    }
    // Epilogue.  What kind it is, whether an addend joins and whether the tile lies wholly inside the matrix are the same
    // for every element of the tile: they are decided once, and the element loops of whole tiles carry no such test.
    const TilePlace at{m0, n0, wave_m, wave_n, lane32, half, (long)split * p.slab};
    if (m0 + BM <= p.M && n0 + BN <= p.N) store_tile_kind<true, TM, TN>(p, acc, at);
    else store_tile_kind<false, TM, TN>(p, acc, at);
}

template <int BM, int BN, bool A_KC, bool B_KC>
__global__ __launch_bounds__(kThreads, 2) void gemm_f32_kernel(GemmDev p)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    gemm_tile<BM, BN, A_KC, B_KC>(p, (int)blockIdx.x, smem);
}

// Two independent contractions in one launch, 128 x 128 tiles each: workgroups [0, first_blocks) work on `a` (A k-contiguous,
// B n-contiguous: dX = delta W), the others on `b` (both operands k-strided: dW += delta^T X).  A batch of 1024 gives dX only
// 256 such tiles - one workgroup per CU, one wavefront per SIMD, too little to keep the matrix pipe busy - while dW has
// four times as many, quarter as long.  Launched together, a CU holds one long dX workgroup next to a succession of
// dW workgroups: two wavefronts per SIMD throughout, and the dW tiles' stores fall at different moments behind
// the dX workgroup's MFMAs instead of all at once.
// At a batch of 512 the same holds one size down: dX as 64 x 64 tiles (256 of them for 2048-wide layers) beside dW as
// 128 x 128 tiles over the short k = batch, equal work per workgroup, one of each per CU.
template <int BMA, int BNA>
__global__ __launch_bounds__(kThreads, 2) void gemm_pair_kernel(GemmDev a, GemmDev b, int first_blocks)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    if ((int)blockIdx.x < first_blocks) gemm_tile<BMA, BNA, true, false>(a, (int)blockIdx.x, smem);
    else gemm_tile<128, 128, false, false>(b, (int)blockIdx.x - first_blocks, smem);
}

template <int BM, int BN, bool A_KC, bool B_KC>
int launch_one(hipStream_t stream, GemmDev d)
{
    constexpr size_t lds_bytes = 2 * stage_bytes<BM, BN>();
    auto kern = gemm_f32_kernel<BM, BN, A_KC, B_KC>;
    static std::once_flag attr_once;  // per instantiation; launches may come from several host threads
    static hipError_t attr_status = hipSuccess;
    std::call_once(attr_once, [&] { attr_status = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes); });
    if (attr_status != hipSuccess) return hip_fail(attr_status, "hipFuncSetAttribute(gemm_f32_kernel)");
    d.nbm = (d.M + BM - 1) / BM;
    d.nbn = (d.N + BN - 1) / BN;
    const long nblocks = (long)d.nbm * d.nbn * d.ksplit;
    if (nblocks <= 0 || nblocks > 0x7fffffffL) { set_last_error("gemm: grid of %ld workgroups out of range", nblocks); return MYEA_E_INVALID; }
    hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(kThreads), lds_bytes, stream, d);
    MYEA_HIP_TRY(hipGetLastError());
    return MYEA_OK;
}

template <int BM, int BN>
int launch_layout(hipStream_t stream, const GemmDev &d, bool a_kc, bool b_kc)
{
    if (a_kc && b_kc) return launch_one<BM, BN, true, true>(stream, d);
    if (a_kc && !b_kc) return launch_one<BM, BN, true, false>(stream, d);
    if (!a_kc && !b_kc) return launch_one<BM, BN, false, false>(stream, d);
    return launch_one<BM, BN, false, true>(stream, d);
}

// ---- a short product ----------------------------------------------------------------------------------------------------
// A product with too few 64 x 64 tiles to occupy the chip - a batch of 128 in front of 256 units is 8 of them - spends the tiled
// kernel's time in its K steps, one behind the other on a few compute units.  Here a workgroup owns 32 rows x 32 columns and its
// WAVES wavefronts share k: each takes every WAVES-th run of 32 k's, a run ahead of the one it splits and multiplies; no barrier until the
// wavefronts' accumulators are added, in wavefront order, by the first, which runs the tiled kernel's epilogue.  What bounds it is
// the latency of the first operands and the splitting, which every workgroup of a row or column of tiles repeats.  Loading a k-contiguous
// operand in whole lines and turning it round in LDS, and addresses that are scalar but for a lane's constant, took (us) 256 x 1024, k =
// 1024 forward 11.8 -> 10.4, backward 11.0 -> 9.3; 512 x 100, k = 2048 18.2 -> 14.5; 64 x 512, k = 512 7.4 -> 6.0; 333 x 1201, k = 1201 20.9
// -> 20.7 and 21.4 -> 19.2 (three runs in registers instead of two: no better at long k, 0.3 - 0.9 worse at short).
// launch_gemm says up to where it pays.
constexpr int kShortMost = 256;   // workgroups: one of eight wavefronts per compute unit
constexpr int kShortRun = 32;   // k's: one 128-byte line of a k-contiguous row

// Operands are read through buffer instructions: the lane's part of an address is set up once, a run's part is scalar, and the range ends
// where this workgroup's k's do.  short_fits: offsets are 32 bits wide.
inline bool short_fits(const GemmDev &d, bool a_kc, bool b_kc)
{
    const long most = 0x1c000000L;   // floats
    auto fits = [&](bool kc, long ld, long rows) { return kc ? 32 * ld + d.K < most : ((long)d.K + 2 * kShortRun * 8) * ld + rows < most; };
    return fits(a_kc, d.lda, d.M) && fits(b_kc, d.ldb, d.N);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t short_range(const float *base, long floats)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, (int)(floats * (long)sizeof(float)), 0x00020000);
}

// An operand whose k's are not contiguous: a lane's eight k's are eight loads, 32 columns - a line - each; k's beyond the last lie beyond
// the range and read as zeros.
template <bool KC, int WAVES, bool TURN>
struct ShortOperand {
    float reg[2][2][8];   // [slot][group of 16 k's][k]
    __amdgpu_buffer_rsrc_t range;
    int lane_at, run_at, ld;   // bytes

    // rows (columns) from `first` on, k's from k_begin to k_end; the wavefront's first run is `run` k's further on
    __device__ __forceinline__ void init(const float *base, long ld_, int first, int extent, int k_begin, int k_end, int run, float *)
    {
        const int lane = threadIdx.x & 63;
        range = short_range(base + (long)k_begin * ld_ + first, (long)(k_end - k_begin - 1) * ld_ + (extent - first));
        ld = (int)ld_ * 4;
        lane_at = (lane >> 5) * 8 * ld + min(lane & 31, extent - 1 - first) * 4;
        run_at = run * ld;
    }
    __device__ __forceinline__ void load(int slot, int)
    {
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int e = 0; e < 8; ++e) reg[slot][g][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(range, lane_at, run_at + (g * 16 + e) * ld, 0));
        run_at += kShortRun * WAVES * ld;
    }
    __device__ __forceinline__ void place(int) {}
    __device__ __forceinline__ void fetch(int slot, int g, float (&x)[8]) const
    {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = reg[slot][g][e];
    }
};

// An operand whose k's are contiguous.  The matrix instruction wants a lane to hold eight k's of one row: loaded so, every load instruction
// touches 32 rows' lines for 16 bytes each, and the address path takes a line at a time.  So eight lanes bring a row's 128 bytes - any
// alignment - and the wavefront turns them round in 4 KiB of LDS of its own: 16-byte chunks, XOR-swizzled by row, no barrier.
template <int WAVES>
struct ShortOperand<true, WAVES, true> {
    u32x4 reg[2][4];   // [slot][rows 8 q + lane / 8]
    __amdgpu_buffer_rsrc_t range;
    int lane_at[4], run_at;   // bytes
    float *tile;          // [32 rows][32 k's]

    static __device__ __forceinline__ int chunk(int row, int c) { return row * 32 + ((c ^ ((row >> 1) & 7)) << 2); }
    __device__ __forceinline__ void init(const float *base, long ld, int first, int extent, int k_begin, int k_end, int run, float *tile_)
    {
        const int lane = threadIdx.x & 63, last = min(31, extent - 1 - first);
        tile = tile_;
        range = short_range(base + first * ld + k_begin, last * ld + (k_end - k_begin));
#pragma unroll
        for (int q = 0; q < 4; ++q) lane_at[q] = (min(q * 8 + (lane >> 3), last) * (int)ld + (lane & 7) * 4) * 4;
        run_at = run * 4;
    }
    __device__ __forceinline__ void load(int slot, int left)   // left: k's from the run's first on
    {
        if (left >= kShortRun) {
#pragma unroll
            for (int q = 0; q < 4; ++q) reg[slot][q] = __builtin_amdgcn_raw_buffer_load_b128(range, lane_at[q], run_at, 0);
        } else {   // the rest of a row: word by word, the row's last in the place of those beyond it, and zeros in their place
            const int mine = left - (int)(threadIdx.x & 7) * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int back = (e - min(e, mine - 1)) * 4;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const unsigned v = __builtin_amdgcn_raw_buffer_load_b32(range, lane_at[q] + e * 4 - back, run_at, 0);
                    reg[slot][q][e] = e < mine ? v : 0u;
                }
            }
        }
        run_at += kShortRun * WAVES * 4;
    }
    __device__ __forceinline__ void place(int slot)
    {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int q = 0; q < 4; ++q) *reinterpret_cast<u32x4 *>(tile + chunk(q * 8 + (lane >> 3), lane & 7)) = reg[slot][q];
    }
    __device__ __forceinline__ void fetch(int, int g, float (&x)[8]) const
    {
        const int lane = threadIdx.x & 63, row = lane & 31, c = g * 4 + (lane >> 5) * 2;
        *reinterpret_cast<f32x4 *>(x) = *reinterpret_cast<const f32x4 *>(tile + chunk(row, c));
        *reinterpret_cast<f32x4 *>(x + 4) = *reinterpret_cast<const f32x4 *>(tile + chunk(row, c + 1));
    }
};

// The same in the lanes that multiply it.  Where A has only a few rows, or a tile's rows of A and of B are few together, the instructions
// are few lines each, and the trip through LDS and the set-up of the ranges are what remains.  us, direct against turned round: 1 x 256, k = 784
// 7.3 | 7.6; 8 x 1000, k = 1000 9.0 | 9.9; 16 x 1000 9.3 | 9.1; 24 x 2048, k = 2048 17.3 | 14.5; k = 4096: 9 x 10 21.0 | 23.6, 16 x 16 22.4 |
// 23.7, 64 x 1 22.9 | 24.3, 14 x 20 22.5 | 23.4, 32 x 4 23.5 | 23.7, 16 x 20 23.1 | 23.3, 16 x 24 24.0 | 23.5.
inline bool short_direct(const GemmDev &d)
{
    constexpr int kRows = 8, kRowsTogether = 34;
    return d.M <= kRows || min(d.M, 32) + min(d.N, 32) <= kRowsTogether;
}
template <int WAVES>
struct ShortOperand<true, WAVES, false> {
    float reg[2][2][8];   // [slot][group of 16 k's][k]
    const float *at;      // of the run that is loaded next
    int mine;             // k's from this lane's first one in that run on

    __device__ __forceinline__ void init(const float *base, long ld, int first, int extent, int k_begin, int k_end, int run, float *)
    {
        const int lane = threadIdx.x & 63, k0 = k_begin + run + (lane >> 5) * 8;
        at = base + min(first + (lane & 31), extent - 1) * ld + k0;
        mine = k_end - k0;
    }
    __device__ __forceinline__ void load(int slot, int)
    {
        if (mine >= 24) {   // this lane's last k of the run is the 24th
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                *reinterpret_cast<f32x4 *>(reg[slot][g]) = *reinterpret_cast<const f32x4_any *>(at + g * 16);
                *reinterpret_cast<f32x4 *>(reg[slot][g] + 4) = *reinterpret_cast<const f32x4_any *>(at + g * 16 + 4);
            }
        } else {
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    reg[slot][g][e] = 0.f;
                    if (g * 16 + e < mine) reg[slot][g][e] = at[g * 16 + e];
                }
        }
        at += kShortRun * WAVES; mine -= kShortRun * WAVES;
    }
    __device__ __forceinline__ void place(int) {}
    __device__ __forceinline__ void fetch(int slot, int g, float (&x)[8]) const
    {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = reg[slot][g][e];
    }
};

template <bool A_KC, bool B_KC, int WAVES, bool TURN>
__global__ __launch_bounds__(64 * WAVES) void short_gemm_kernel(GemmDev p)
{
    // a wavefront's tiles of its operands, 4 KiB each; the accumulators of those behind the first take their place
    constexpr int kTiles = A_KC && B_KC ? 2 : 1;
    __shared__ __attribute__((aligned(16))) float tiles[WAVES][kTiles][1024];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane32 = lane & 31, half = lane >> 5;
    const int nblocks = p.nbm * p.nbn, split = (int)blockIdx.x / nblocks, pid = (int)blockIdx.x - split * nblocks;
    const int m0 = pid % p.nbm * 32, n0 = pid / p.nbm * 32;
    const int k_begin = split * p.kchunk, k_end = (int)min((long)p.K, (long)k_begin + p.kchunk);
    f32x16 acc[1][1], small;   // the hi hi products; the others
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][0][r] = small[r] = 0.f;
    ShortOperand<A_KC, WAVES, TURN> a;
    ShortOperand<B_KC, WAVES, TURN> b;
    const int first = k_begin + wave * kShortRun;
    a.init(p.A, p.lda, m0, p.M, k_begin, k_end, wave * kShortRun, tiles[wave][0]);
    b.init(p.B, p.ldb, n0, p.N, k_begin, k_end, wave * kShortRun, tiles[wave][kTiles - 1]);
    const int runs = first < k_end ? (k_end - first - 1) / (kShortRun * WAVES) + 1 : 0;
    int left = k_end - first;
    auto load = [&](int slot) {
        a.load(slot, left); b.load(slot, left);
        left -= kShortRun * WAVES;
    };
    auto multiply = [&](int slot) {
        a.place(slot); b.place(slot);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            bf16x8 pa[3], pb[3];
            float xa[8], xb[8];
            a.fetch(slot, g, xa); b.fetch(slot, g, xb);
            split_eight(xa, pa);
            split_eight(xb, pb);
#pragma unroll
            for (int q = 0; q < 5; ++q) small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pa[kSmallA[q]], pb[kSmallB[q]], small, 0, 0, 0);
            acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pa[0], pb[0], acc[0][0], 0, 0, 0);
        }
    };
    if (runs > 0) load(0);
    for (int r = 0; r < runs; r += 2) {
        if (r + 1 < runs) load(1);
        multiply(0);
        if (r + 1 >= runs) break;
        if (r + 2 < runs) load(0);
        multiply(1);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][0][r] += small[r];
    if (wave) {
#pragma unroll
        for (int r = 0; r < 4; ++r) *reinterpret_cast<f32x4 *>(&tiles[wave][0][(r * 64 + lane) * 4]) = (f32x4){acc[0][0][r * 4], acc[0][0][r * 4 + 1], acc[0][0][r * 4 + 2], acc[0][0][r * 4 + 3]};
    }
    __syncthreads();
    if (wave) return;
    float finite = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES - 1; ++w)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const f32x4 v = *reinterpret_cast<const f32x4 *>(&tiles[w + 1][0][(r * 64 + lane) * 4]);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[0][0][r * 4 + e] += v[e];
        }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        acc[0][0][r] = unscaled(acc[0][0][r]);
        finite = fmaf(acc[0][0][r], 0.f, finite);
    }
    if (__any(finite != 0.f)) redo_in_f32<A_KC, B_KC, 1, 1>(p, acc, m0 + lane32, n0 + lane32, half, k_begin, k_end);
    const TilePlace at{m0, n0, 0, 0, lane32, half, (long)split * p.slab};
    if (m0 + 32 <= p.M && n0 + 32 <= p.N) store_tile_kind<true, 1, 1>(p, acc, at);
    else store_tile_kind<false, 1, 1>(p, acc, at);
}

template <int WAVES>
void launch_short_waves(hipStream_t stream, const GemmDev &d, bool a_kc, bool b_kc, long nblocks)
{
    const dim3 grid((unsigned)nblocks), group(64 * WAVES);
    if (a_kc && b_kc) hipLaunchKernelGGL((short_gemm_kernel<true, true, WAVES, true>), grid, group, 0, stream, d);
    else if (a_kc) hipLaunchKernelGGL((short_gemm_kernel<true, false, WAVES, true>), grid, group, 0, stream, d);
    else if (b_kc) hipLaunchKernelGGL((short_gemm_kernel<false, true, WAVES, true>), grid, group, 0, stream, d);
    else hipLaunchKernelGGL((short_gemm_kernel<false, false, WAVES, true>), grid, group, 0, stream, d);
}

int launch_short(hipStream_t stream, GemmDev d, bool a_kc, bool b_kc)
{
    d.nbm = (d.M + 31) / 32;
    d.nbn = (d.N + 31) / 32;
    const long nblocks = (long)d.nbm * d.nbn * d.ksplit;
    if (nblocks <= 0 || nblocks > 0x7fffffffL) { set_last_error("gemm: grid of %ld workgroups out of range", nblocks); return MYEA_E_INVALID; }
    // The registers admit eight wavefronts a compute unit.  More workgroups than compute units: of four wavefronts each, so that two
    // share one instead of the second waiting for the first.  us, eight -> four, 333 x 1201 (418 workgroups): k = 64 7.5 -> 5.7, 256
    // 9.5 -> 7.8, 1000 20.9 -> 18.2; up to one per compute unit: 10 x 1000, k = 1000 9.4 against 10.8.
    if (nblocks > kShortMost) launch_short_waves<4>(stream, d, a_kc, b_kc, nblocks);
    else if (a_kc && b_kc && short_direct(d)) hipLaunchKernelGGL((short_gemm_kernel<true, true, 8, false>), dim3((unsigned)nblocks), dim3(64 * 8), 0, stream, d);
    else launch_short_waves<8>(stream, d, a_kc, b_kc, nblocks);
    MYEA_HIP_TRY(hipGetLastError());
    return MYEA_OK;
}

// ---- a shallow product --------------------------------------------------------------------------------------------------
// With few k's there is nothing to gain from the BF16 planes and something to lose: a single product or a pair of them is rounded once by
// the FP32 instruction and a little more than once by the six (k = 1: 2.6e-8 against 2.5e-8), and a sum that one large product
// dominates stays up to 1.7 times less exact until an instruction's 16 k's are full.  Such a product is bound by the latency of its
// operands and the stores of C, so it can as well be exact: a wavefront owns 32 rows x 32 columns, takes its operands straight
// from memory and multiplies with v_mfma_f64_16x16x4_f64 (as many cycles a k as the FP32 instruction's on 64-bit sums); what is
// rounded is the result.  Infinities, NaN and subnormals need no care.
//   operands: lane l takes k = l / 16 of every four and one row (A) or column (B) of each half of the tile
//   result:   register i of lane l holds row 4 i + l / 16, column l % 16.  Which row of C that is is chosen by the rows that A's lanes
//             take: with the rows below, lanes l and l ^ 16 hold each other's half of what the epilogue's layout gives them.
constexpr int kShallow = 16;   // k's of one v_mfma_f32_32x32x16_bf16
typedef double f64x4 __attribute__((ext_vector_type(4)));

template <bool A_KC, bool B_KC>
__global__ __launch_bounds__(kThreads) void shallow_gemm_kernel(GemmDev p)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lane16 = lane & 15, quad = lane >> 4;
    const int tile = (int)blockIdx.x * (kThreads / 64) + wave;   // columns first: a workgroup stores whole runs of C's rows
    if (tile >= p.nbm * p.nbn) return;
    const int m0 = tile / p.nbn * 32, n0 = tile % p.nbn * 32;
    long a_row[2], b_col[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int i = lane16 >> 2, g = lane16 & 3;   // of the result's row 4 i + g
        a_row[t] = min(m0 + ((g & 1) * 2 + t) * 8 + (g >> 1) * 4 + i, p.M - 1);
        b_col[t] = min(n0 + t * 16 + lane16, p.N - 1);
    }
    f64x4 sum[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) sum[t][u] = (f64x4){0., 0., 0., 0.};
    float a[kShallow / 4][2], b[kShallow / 4][2];
#pragma unroll
    for (int e = 0; e < kShallow / 4; ++e) {
        if (e * 4 >= p.K) break;
        const long k = e * 4 + quad;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            a[e][t] = b[e][t] = 0.f;
            if (k < p.K) {
                a[e][t] = p.A[A_KC ? a_row[t] * p.lda + k : k * p.lda + a_row[t]];
                b[e][t] = p.B[B_KC ? b_col[t] * p.ldb + k : k * p.ldb + b_col[t]];
            }
        }
    }
#pragma unroll
    for (int e = 0; e < kShallow / 4; ++e) {
        if (e * 4 >= p.K) break;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < 2; ++u) sum[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[e][t], (double)b[e][u], sum[t][u], 0, 0, 0);
    }
    f32x16 acc[1][1];
    const bool odd = quad & 1;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float first = (float)sum[t][0][i], second = (float)sum[t][1][i];
            const float kept = odd ? second : first, other = __shfl_xor(odd ? first : second, 16);
            acc[0][0][t * 4 + i] = odd ? other : kept;
            acc[0][0][8 + t * 4 + i] = odd ? kept : other;
        }
    const TilePlace at{m0, n0, 0, 0, lane & 31, lane >> 5, 0L};
    if (p.M - m0 >= 32 && p.N - n0 >= 32) store_tile_kind<true, 1, 1>(p, acc, at);
    else store_tile_kind<false, 1, 1>(p, acc, at);
}

int launch_shallow(hipStream_t stream, GemmDev d, bool a_kc, bool b_kc)
{
    d.nbm = (d.M + 31) / 32;
    d.nbn = (d.N + 31) / 32;
    const long tiles = (long)d.nbm * d.nbn;
    if (tiles > 0x7fffffffL) { set_last_error("gemm: %ld tiles of 32 x 32 out of range", tiles); return MYEA_E_INVALID; }
    const dim3 grid((unsigned)((tiles + kThreads / 64 - 1) / (kThreads / 64))), group(kThreads);
    if (a_kc && b_kc) hipLaunchKernelGGL((shallow_gemm_kernel<true, true>), grid, group, 0, stream, d);
    else if (a_kc) hipLaunchKernelGGL((shallow_gemm_kernel<true, false>), grid, group, 0, stream, d);
    else if (b_kc) hipLaunchKernelGGL((shallow_gemm_kernel<false, true>), grid, group, 0, stream, d);
    else hipLaunchKernelGGL((shallow_gemm_kernel<false, false>), grid, group, 0, stream, d);
    MYEA_HIP_TRY(hipGetLastError());
    return MYEA_OK;
}

// ---- a narrow product ---------------------------------------------------------------------------------------------------
// C [M][N] = A B with N <= 32 and K <= 64 - a layer of an independently recurrent stack over T x batch rows, forward or backward.
// The tiled kernel spends such a launch on its set-up and its stages: a few microseconds of instructions fetched to be run once.  Here a wavefront owns 32 rows of C: the
// lane's operands of v_mfma_f32_32x32x2f32 are asked for straight from memory, all of a round of 32 k's together (A: lane l
// takes row l % 32 at k + l / 32; B: column l % 32), then the round's 16 matrix instructions; no LDS, one round or two.  The
// accumulator has the layout of the tiled kernel's, so its epilogue (store_tile_kind) finishes the tile: every kind of
// epilogue, the same arithmetic per element.
template <bool A_KC, bool B_KC>
__global__ __launch_bounds__(kThreads) void narrow_gemm_kernel(GemmDev p)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lane32 = lane & 31, half = lane >> 5;
    const int m0 = (int)blockIdx.x * 128, row = m0 + wave * 32 + lane32;
    const bool in_m = row < p.M, in_n = lane32 < p.N;
    f32x16 acc[1][1];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][0][r] = 0.f;
    const float *a_at = A_KC ? p.A + (long)row * p.lda + half : p.A + (long)half * p.lda + row;
    const float *b_at = B_KC ? p.B + (long)lane32 * p.ldb + half : p.B + (long)half * p.ldb + lane32;
    const long a_step = A_KC ? 2 : 2 * p.lda, b_step = B_KC ? 2 : 2 * p.ldb;   // from one pair of k's to the next
    for (int k0 = 0; k0 < p.K; k0 += 32) {
        float a[16], b[16];
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const bool in_k = k0 + 2 * s + half < p.K;
            a[s] = (in_m && in_k) ? a_at[s * a_step] : 0.f;
            b[s] = (in_n && in_k) ? b_at[s * b_step] : 0.f;
        }
#pragma unroll
        for (int s = 0; s < 16; ++s) acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], b[s], acc[0][0], 0, 0, 0);
        a_at += 16 * a_step; b_at += 16 * b_step;
    }
    const TilePlace at{m0, 0, wave * 32, 0, lane32, half, 0L};
    if (m0 + 128 <= p.M && p.N == 32) store_tile_kind<true, 1, 1>(p, acc, at);
    else store_tile_kind<false, 1, 1>(p, acc, at);
}

// ---- the weight gradient of a narrow layer ------------------------------------------------------------------------------
// dW = delta^T X with at most 32 outputs (columns of delta) and at most 32 inputs (columns of X) over many rows - a layer of an
// independently recurrent stack over T x batch rows.  Two rows of delta and of X, as they lie in memory, ARE the operands of
// v_mfma_f32_32x32x2f32 (lane l: column l % 32 of row l / 32): a wavefront walks its share of the rows with two coalesced
// loads and one matrix instruction per pair of rows, no LDS, no tile edges to test; a loop of a few dozen instructions.
// The wavefronts of a workgroup add their 32 x 32 accumulators in wavefront order and store one slab [H][In]; the slabs
// are added by launch_slab_sum_add, as the slabs of a split-K launch are.  (The tiled kernel spends its time on such a
// shape in its set-up and its epilogue.)
constexpr int kNarrowAhead = 16;   // pairs of rows a wavefront asks for at once: its whole share when the launch is not capped
constexpr int kNarrowWaves = 8;    // wavefronts a workgroup: fewer slabs to add afterwards
__device__ __forceinline__ void narrow_dw(const float *__restrict__ delta, const float *__restrict__ x, float *__restrict__ slabs,
                                          int H, int In, long rows, long rows_per_wave)
{
    __shared__ float handed[kNarrowWaves - 1][16][64];   // the accumulators of the wavefronts behind the first
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 31, half = lane >> 5;
    const long first = ((long)blockIdx.x * kNarrowWaves + wave) * rows_per_wave;
    const long last = first + rows_per_wave < rows ? first + rows_per_wave : rows;
    const bool in_delta = col < H, in_x = col < In;
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    for (long r0 = first; r0 < last; r0 += 2 * kNarrowAhead) {
        float a[kNarrowAhead], b[kNarrowAhead];
#pragma unroll
        for (int u = 0; u < kNarrowAhead; ++u) {
            const long row = r0 + 2 * u + half;
            a[u] = (in_delta && row < last) ? delta[row * H + col] : 0.f;
            b[u] = (in_x && row < last) ? x[row * In + col] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < kNarrowAhead; ++u) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u], b[u], acc, 0, 0, 0);
    }
    if (wave) {
#pragma unroll
        for (int r = 0; r < 16; ++r) handed[wave - 1][r][lane] = acc[r];
    }
    __syncthreads();
    if (wave || !in_x) return;
    float *slab = slabs + (size_t)blockIdx.x * H * In;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = (r >> 2) * 8 + half * 4 + (r & 3);   // the accumulator's row of this lane's column
        float v = acc[r];
#pragma unroll
        for (int w = 0; w < kNarrowWaves - 1; ++w) v += handed[w][r][lane];
        if (m < H) slab[m * In + col] = v;
    }
}

__global__ __launch_bounds__(64 * kNarrowWaves) void narrow_dw_kernel(const float *__restrict__ delta, const float *__restrict__ x, float *__restrict__ slabs,
                                                             int H, int In, long rows, long rows_per_wave)
{
    narrow_dw(delta, x, slabs, H, In, rows, rows_per_wave);
}

// The same for a table of layers, grid (slabs, layers): as launches of their own they were 5.6 us each, a few dozen workgroups
// at a time (29 layers of at most 32 x 32 over 7168 rows: 161 us of launches in turns on two streams, 15 us here).
__global__ __launch_bounds__(64 * kNarrowWaves) void narrow_dw_jobs_kernel(const NarrowDwJob *__restrict__ jobs, long rows, long rows_per_wave)
{
    const NarrowDwJob job = jobs[blockIdx.y];
    narrow_dw(job.delta, job.x, job.slabs, (int)job.H, (int)job.In, rows, rows_per_wave);
}

}  // namespace

// Number of K slabs for a contraction whose M x N alone does not fill the chip; 1 when the plain launch already does.
// Short k: about one workgroup per CU with 64 x 64 tiles, each slab at least 128 k's deep.
static long split_k_wanted(int M, int N, int K)
{
    const long tiles_128 = (long)((M + 127) / 128) * ((N + 127) / 128);
    if (tiles_128 * 2 >= 256) return 1;
    long want, most = 16;
    if (K >= 4096) {
        // long k (weight gradients over T x batch rows): enough slabs for ~1000 workgroups of 128 x 64, each slab at least
        // 1024 k's deep - the larger tile's operand reuse is worth more than the pass over the slabs that sums them
        // (a product no larger than one 64 x 64 tile has no operand reuse to protect: slabs 256 k's deep, up to 32 of them)
        const bool one_tile = M <= 64 && N <= 64;
        want = (512 + tiles_128 - 1) / tiles_128;
        const long by_k = K / (one_tile ? 256 : 1024);
        if (want > by_k) want = by_k;
        if (one_tile) most = 32;
    } else {
        const long tiles_64 = (long)((M + 63) / 64) * ((N + 63) / 64);
        want = (256 + tiles_64 - 1) / tiles_64;
        const long max_by_k = K / 128 > 0 ? K / 128 : 1;
        if (want > max_by_k) want = max_by_k;
    }
    if (want > most) want = most;
    return want < 1 ? 1 : want;
}

int gemm_split_k(int M, int N, int K)
{
    const long want = split_k_wanted(M, N, K);
    if (want == 1) return 1;
    // the launcher rounds the chunk up to a multiple of 32: return the slab count that rounding produces
    const int chunk = (int)(((K + want - 1) / want + kBK - 1) / kBK * kBK);
    return (int)(((long)K + chunk - 1) / chunk);
}

// No k up to K takes more slabs than this: what a workspace for them is sized by.  (Fewer k's may take more of them: 16 at 4095,
// 4 at 4096.  On either side of that line the wanted number only grows with k, and the rounding of the chunk only lowers it.)
int gemm_split_k_most(int M, int N, int K)
{
    const long shallow = split_k_wanted(M, N, K < 4095 ? K : 4095), deep = split_k_wanted(M, N, K);
    return (int)(shallow > deep ? shallow : deep);
}

unsigned gemm_pair_polls()
{
    const char *e = std::getenv("MYEA_GEMM_PAIR_SPIN_POLLS");
    if (e && *e) { const unsigned long long v = std::strtoull(e, nullptr, 10); return v > 0xffffffffull ? 0xffffffffu : (unsigned)v; }
    return 1u << 24;
}

bool gemm_pair_k_128(int M, int N, int K)
{
    const long tiles_128 = (long)((M + 127) / 128) * ((N + 127) / 128);
    return tiles_128 <= kGemmPairTiles && tiles_128 % 8 == 0 && tiles_128 >= 128 && K >= 2048;
}

bool gemm_can_fuse_activation(int act)
{
    return act == MYEA_AF_LINEAR || act == MYEA_AF_RELU || act == MYEA_AF_LEAKY_RELU || act == MYEA_AF_PARAMETRIC_RELU ||
           act == MYEA_AF_TANH || act == MYEA_AF_SIGMOID;
}

// checks a problem and fills the kernel's argument block
static int prepare_gemm(const GemmParams &p, GemmDev &d)
{
    if (p.M <= 0 || p.N <= 0 || p.K < 0) { set_last_error("gemm: bad shape M=%d N=%d K=%d", p.M, p.N, p.K); return MYEA_E_INVALID; }
    if (!p.A || !p.B || !p.C) { set_last_error("gemm: null operand"); return MYEA_E_INVALID; }
    const long a_min = p.a_k_contiguous ? p.K : p.M, b_min = p.b_k_contiguous ? p.K : p.N;
    if (p.lda < a_min || p.ldb < b_min || p.ldc < p.N) { set_last_error("gemm: leading dimension smaller than the row length"); return MYEA_E_INVALID; }
    if (p.epilogue == EPI_FC_DERIVE && (!p.pre || !p.val)) { set_last_error("gemm: derive epilogue without pre/val"); return MYEA_E_INVALID; }
    if (p.addend && (p.epilogue == EPI_FC_FORWARD || p.accumulate)) { set_last_error("gemm: an addend goes with a plain or a derivative epilogue only"); return MYEA_E_INVALID; }
    if (p.epilogue == EPI_FC_DERIVE && !gemm_can_fuse_activation(p.act)) { set_last_error("gemm: activation %d cannot be fused", p.act); return MYEA_E_INVALID; }
    if (p.epilogue == EPI_FC_FORWARD && p.aux_out && !gemm_can_fuse_activation(p.act)) { set_last_error("gemm: activation %d cannot be fused", p.act); return MYEA_E_INVALID; }

    d.A = p.A; d.B = p.B; d.C = p.C;
    d.M = p.M; d.N = p.N; d.K = p.K;
    d.lda = p.lda; d.ldb = p.ldb; d.ldc = p.ldc;
    d.accumulate = (p.accumulate && !p.c_is_zero) ? 1 : 0; d.epilogue = p.epilogue;   // onto zeros a store gives the same values as an add
    d.bias = p.bias; d.aux_out = p.aux_out; d.colscale = p.colscale;
    d.pre = p.pre; d.val = p.val; d.act = p.act; d.steep = p.steep;
    d.addend = p.addend; d.ld_addend = p.ld_addend;
    d.col_partials = p.col_partials; d.hats = p.hats;
    if (p.col_partials && p.epilogue == EPI_NONE) { set_last_error("gemm: column partial sums go with the forward and the derivative epilogue only"); return MYEA_E_INVALID; }
    if (p.hats && (p.epilogue != EPI_FC_DERIVE || !p.col_partials)) { set_last_error("gemm: hats go with the derivative epilogue's column sums"); return MYEA_E_INVALID; }
    if (p.addend && (p.epilogue == EPI_FC_FORWARD || p.ld_addend < p.N)) { set_last_error("gemm: addend needs EPI_NONE / EPI_FC_DERIVE and ld_addend >= N"); return MYEA_E_INVALID; }
    d.nbm = d.nbn = 0;
    d.ksplit = 1; d.kchunk = p.K > 0 ? p.K : 1; d.slab = 0;
    d.pair_partials = nullptr; d.pair_tickets = nullptr;
    d.pair_fault = p.pair_fault; d.pair_host_flag = p.pair_host_flag; d.pair_polls = p.pair_polls;
    {   // MYEA_GEMM_PAIR_LOCAL=0: the two workgroups of a tile meet through device-scope release / acquire wherever they run
        static const bool local_off = [] { const char *e = std::getenv("MYEA_GEMM_PAIR_LOCAL"); return e && e[0] == '0'; }();
        d.pair_local = (!local_off && device_groups_share_xcd()) ? 1 : 0;
    }
    if (p.split_k > 1) {
        if (p.epilogue != EPI_NONE || p.accumulate || p.addend) { set_last_error("gemm: split-K writes plain partial slabs"); return MYEA_E_INVALID; }
        const int chunk = (int)(((long)p.K + p.split_k - 1) / p.split_k + kBK - 1) / kBK * kBK;
        d.kchunk = chunk;
        d.ksplit = (int)(((long)p.K + chunk - 1) / chunk);
        d.slab = p.split_k_slab;
        if (d.ksplit != p.split_k) { set_last_error("gemm: split-K count %d does not divide K=%d into %d-wide chunks; use gemm_split_k()", p.split_k, p.K, chunk); return MYEA_E_INVALID; }
    }
    return MYEA_OK;
}

// Slabs the narrow weight-gradient kernel writes for these shapes: 0 when the shape is not its own (the tiled kernel takes it).
// A wavefront gets at least 32 rows (one round of loads), a launch at most 128 workgroups.
constexpr int kNarrowSlabs = 128;
int narrow_dw_slabs(size_t H, size_t In, size_t rows)
{
    if (H == 0 || In == 0 || H > 32 || In > 32 || rows < 512 || rows > 0x7fffffffu) return 0;
    static const bool off = [] { const char *e = std::getenv("MYEA_NARROW_DW"); return e && e[0] == '0'; }();
    if (off) return 0;
    size_t per_wave = 2 * kNarrowAhead;
    while ((rows + kNarrowWaves * per_wave - 1) / (kNarrowWaves * per_wave) > kNarrowSlabs) per_wave *= 2;
    return (int)((rows + kNarrowWaves * per_wave - 1) / (kNarrowWaves * per_wave));
}

// No number of rows up to `rows` takes more: 128 at 32768 rows, 65 at 32769.
int narrow_dw_slabs_most(size_t H, size_t In, size_t rows)
{
    constexpr size_t full = (size_t)kNarrowSlabs * kNarrowWaves * 2 * kNarrowAhead;   // the most rows that every wavefront takes in one round
    return narrow_dw_slabs(H, In, rows < full ? rows : full);
}

// even: a matrix instruction takes a pair of rows
static long narrow_rows_per_wave(size_t rows, int S) { return (long)(((rows + (size_t)S * kNarrowWaves - 1) / ((size_t)S * kNarrowWaves) + 1) / 2 * 2); }

// delta [rows][H], x [rows][In], both dense; slabs: narrow_dw_slabs(H, In, rows) x [H][In]
int launch_narrow_dw(hipStream_t stream, const float *delta, const float *x, float *slabs, size_t H, size_t In, size_t rows)
{
    const int S = narrow_dw_slabs(H, In, rows);
    if (S <= 0 || !delta || !x || !slabs) { set_last_error("narrow weight gradient: %zu x %zu over %zu rows is not its shape", H, In, rows); return MYEA_E_INVALID; }
    hipLaunchKernelGGL(narrow_dw_kernel, dim3((unsigned)S), dim3(64 * kNarrowWaves), 0, stream, delta, x, slabs, (int)H, (int)In, (long)rows, narrow_rows_per_wave(rows, S));
    MYEA_HIP_TRY(hipGetLastError());
    return MYEA_OK;
}

int launch_narrow_dw_jobs(hipStream_t stream, const NarrowDwJob *jobs, size_t count, size_t rows)
{
    if (count == 0) return MYEA_OK;
    const int S = narrow_dw_slabs(1, 1, rows);   // the same for every layer that is narrow
    if (count > 65535 || S <= 0) { set_last_error("narrow weight gradients: %zu layers over %zu rows in one launch", count, rows); return MYEA_E_INVALID; }
    hipLaunchKernelGGL(narrow_dw_jobs_kernel, dim3((unsigned)S, (unsigned)count), dim3(64 * kNarrowWaves), 0, stream, jobs, (long)rows, narrow_rows_per_wave(rows, S));
    MYEA_HIP_TRY(hipGetLastError());
    return MYEA_OK;
}

int launch_gemm(hipStream_t stream, const GemmParams &p)
{
    GemmDev d;
    {
        const int rc = prepare_gemm(p, d);
        if (rc != MYEA_OK) return rc;
    }
    const bool a_kc = p.a_k_contiguous != 0, b_kc = p.b_k_contiguous != 0;

    // a narrow product over many rows: the kernel that feeds the matrix unit straight from memory (MYEA_NARROW_GEMM=0: the tiled one)
    static const bool narrow_off = [] { const char *e = std::getenv("MYEA_NARROW_GEMM"); return e && e[0] == '0'; }();
    if (!narrow_off && p.N <= 32 && p.K <= 64 && p.M >= 256 && d.ksplit == 1) {
        const dim3 grid((unsigned)((p.M + 127) / 128));
        if (a_kc && b_kc) hipLaunchKernelGGL((narrow_gemm_kernel<true, true>), grid, dim3(kThreads), 0, stream, d);
        else if (a_kc) hipLaunchKernelGGL((narrow_gemm_kernel<true, false>), grid, dim3(kThreads), 0, stream, d);
        else if (b_kc) hipLaunchKernelGGL((narrow_gemm_kernel<false, true>), grid, dim3(kThreads), 0, stream, d);
        else hipLaunchKernelGGL((narrow_gemm_kernel<false, false>), grid, dim3(kThreads), 0, stream, d);
        MYEA_HIP_TRY(hipGetLastError());
        return MYEA_OK;
    }
    // Fewer k's than one BF16 instruction takes: the sums in 64 bits.  Exactness decides the line, and the time is no worse than the FP32
    // instruction's was (us, FP32 tiles / BF16 planes / this: 333 x 1201 x 10 5.2 / 8.4 / 5.3, 2049 x 2050 x 10 10.0 / 8.6 / 9.1, 4096 x
    // 4096 x 3 20.7 / 15.1 / 15.3, 16384 x 512 x 10 13.4 / 9.7 / 12.3); at 16 k's and large outputs the planes win (16384 x 512: 9.9
    // against 16).
    if (p.K < kShallow && d.ksplit == 1) return launch_shallow(stream, d, a_kc, b_kc);
    // Tile choice: 128 x 128 from one workgroup per CU (256 CUs) on - its operand reuse is worth more than a second workgroup
    // (2048 x 2048 x 2048, 256 such tiles: 98 us, 512 tiles of 64 x 128: 110 us), unless half of it would lie outside the matrix
    // (49152 rows, 40 columns, k = 64: 11.2 us, as 128 x 64 8.7) - else 64-row tiles to keep the chip filled for short-M / short-N
    // problems.
    const long tiles_128 = (long)((p.M + 127) / 128) * ((p.N + 127) / 128);
    const bool pair_128 = p.pair_partials && p.pair_tickets && d.ksplit == 1 && gemm_pair_k_128(p.M, p.N, p.K);   // see below
    if (tiles_128 * d.ksplit >= 256 && !pair_128 && p.M > 64 && p.N > 64) return launch_layout<128, 128>(stream, d, a_kc, b_kc);   // slabs of a split k count: they fill the chip like tiles do
    // At most one 64 x 64 tile per compute unit but enough of them, and a k worth splitting: two workgroups per tile, half of k each, combined in
    // the launch - a second wavefront per SIMD to fill the first one's waits, which such a launch otherwise lacks.
    // MYEA_GEMM_PAIR_K=0 keeps one workgroup per tile.
    static const int pair_k = [] { const char *e = std::getenv("MYEA_GEMM_PAIR_K"); return e ? std::atoi(e) : 3; }();   // bit 0: 64 x 64 tiles, bit 1: 128 x 128
    const bool pair_k_off = !(pair_k & 1);
    // The same one size up: at most one 128 x 128 tile per compute unit (a batch of 1024 in front of 4096 units) would run as 64 x
    // 128 tiles to put two workgroups on every compute unit; two workgroups sharing a 128 x 128 tile's k do that with the larger
    // tile's operand reuse.
    if ((pair_k & 2) && pair_128) {
        d.ksplit = 2;
        d.kchunk = (int)(((long)p.K + 1) / 2 + kBK - 1) / kBK * kBK;
        d.pair_partials = p.pair_partials; d.pair_tickets = p.pair_tickets;
        return launch_layout<128, 128>(stream, d, a_kc, b_kc);
    }
    const long tiles_64 = (long)((p.M + 63) / 64) * ((p.N + 63) / 64);
    if (p.pair_partials && p.pair_tickets && !pair_k_off && d.ksplit == 1 && tiles_64 <= kGemmPairTiles && tiles_64 % 8 == 0 && tiles_64 >= 128 && p.K >= 512) {
        d.ksplit = 2;
        d.kchunk = (int)(((long)p.K + 1) / 2 + kBK - 1) / kBK * kBK;
        d.pair_partials = p.pair_partials; d.pair_tickets = p.pair_tickets;
        return launch_layout<64, 64>(stream, d, a_kc, b_kc);
    }
    // The short product below 128 tiles of 64 x 64, slabs counted, at any k: two of its workgroups a compute unit are enough there.  us, 64 x
    // 64 tiles -> short, k = 64, 256, 1024, 4096 (the layouts' mean): 512 x 512 (256 workgroups) 4.7 -> 4.5, 7.9 -> 5.4, 21.1 -> 10.5, 75 ->
    // 32; 640 x 768 (480) 5.6 -> 5.8, 8.3 -> 7.6, 21.6 -> 17.3, 75 -> 57; with a third workgroup a unit, 700 x 900 (638), 5.6 -> 7.5, 8.6 ->
    // 10.6, 22.4 -> 25.9, 76 -> 85.  (128 tiles exactly, 512 x 1024, would gain as well, 21.5 -> 17.7 at k = 1024, but are what a paired launch
    // takes as tiles, and a product has the same bits there and alone.)
    if (tiles_64 * d.ksplit < 128 && short_fits(d, a_kc, b_kc)) return launch_short(stream, d, a_kc, b_kc);
    if (tiles_128 * 2 * d.ksplit < 256) return launch_layout<64, 64>(stream, d, a_kc, b_kc);
    if (p.M <= p.N) return launch_layout<64, 128>(stream, d, a_kc, b_kc);
    return launch_layout<128, 64>(stream, d, a_kc, b_kc);
}

// `a` = (A k-contiguous, B n-contiguous), `b` = (both k-strided), neither split along k, any alignment, and `a` no
// more than about one 128 x 128 tile per CU: both in ONE launch (gemm_pair_kernel).  Returns MYEA_OK when launched, 1 when the pair form does not apply (the caller launches the two one after the other), a negative code on an error.
// Either product has the bits that launch_gemm gives it: what that sends to a kernel of other sums (fewer than 16 k's) does not pair.
int launch_gemm_pair(hipStream_t stream, const GemmParams &a, const GemmParams &b)
{
    if (!a.a_k_contiguous || a.b_k_contiguous || b.a_k_contiguous || b.b_k_contiguous || a.split_k > 1 || b.split_k > 1) return 1;
    if (a.K < kShallow || b.K < kShallow) return 1;
    GemmDev da, db;
    int rc = prepare_gemm(a, da);
    if (rc != MYEA_OK) return rc;
    rc = prepare_gemm(b, db);
    if (rc != MYEA_OK) return rc;
    db.nbm = (b.M + 127) / 128; db.nbn = (b.N + 127) / 128;
    const long nb = (long)db.nbm * db.nbn;
    // Worth it when `a` alone would leave the CUs with one workgroup each and `b` brings about as much work in at least as
    // many pieces: `a` as 128 x 128 tiles if that gives 128 .. 256 of them, else as 64 x 64 tiles under the same test.
    auto fits = [&](int tile) {
        const long na = (long)((a.M + tile - 1) / tile) * ((a.N + tile - 1) / tile);
        const double wa = (double)a.K * tile * tile * (double)na, wb = (double)b.K * 128.0 * 128.0 * (double)nb;
        return na >= 128 && na <= 256 && (na & 7) == 0 && nb >= na && wa <= 2.0 * wb && wb <= 2.0 * wa;
    };
    constexpr size_t lds_b = 2 * stage_bytes<128, 128>();
    if (fits(128)) {
        da.nbm = (a.M + 127) / 128; da.nbn = (a.N + 127) / 128;
        const long na = (long)da.nbm * da.nbn;
        constexpr size_t lds_bytes = lds_b;
        static std::once_flag attr_once;
        static hipError_t attr_status = hipSuccess;
        std::call_once(attr_once, [&] { attr_status = hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_pair_kernel<128, 128>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes); });
        if (attr_status != hipSuccess) return hip_fail(attr_status, "hipFuncSetAttribute(gemm_pair_kernel)");
        hipLaunchKernelGGL((gemm_pair_kernel<128, 128>), dim3((unsigned)(na + nb)), dim3(kThreads), lds_bytes, stream, da, db, (int)na);
    } else if (fits(64)) {
        da.nbm = (a.M + 63) / 64; da.nbn = (a.N + 63) / 64;
        const long na = (long)da.nbm * da.nbn;
        constexpr size_t lds_a = 2 * stage_bytes<64, 64>();
        constexpr size_t lds_bytes = lds_a > lds_b ? lds_a : lds_b;
        static std::once_flag attr_once;
        static hipError_t attr_status = hipSuccess;
        std::call_once(attr_once, [&] { attr_status = hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_pair_kernel<64, 64>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes); });
        if (attr_status != hipSuccess) return hip_fail(attr_status, "hipFuncSetAttribute(gemm_pair_kernel)");
        hipLaunchKernelGGL((gemm_pair_kernel<64, 64>), dim3((unsigned)(na + nb)), dim3(kThreads), lds_bytes, stream, da, db, (int)na);
    } else {
        return 1;
    }
    MYEA_HIP_TRY(hipGetLastError());
    return MYEA_OK;
}

}  // namespace myea

extern "C" int myea_hip_gemm_f32(void *stream, int a_k_contiguous, int b_k_contiguous, int accumulate, size_t M, size_t N, size_t K,
                                 const float *A, size_t lda, const float *B, size_t ldb, float *C, size_t ldc)
{
    if (M > 0x7fffffffu || N > 0x7fffffffu || K > 0x7fffffffu) { myea::set_last_error("gemm: dimension too large"); return MYEA_E_INVALID; }
    myea::GemmParams p{};
    p.A = A; p.B = B; p.C = C;
    p.M = (int)M; p.N = (int)N; p.K = (int)K;
    p.lda = (long)lda; p.ldb = (long)ldb; p.ldc = (long)ldc;
    p.a_k_contiguous = a_k_contiguous; p.b_k_contiguous = b_k_contiguous;
    p.accumulate = accumulate;
    p.epilogue = myea::EPI_NONE;
    return myea::launch_gemm(static_cast<hipStream_t>(stream), p);
}
