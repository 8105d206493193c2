// myea_lstm_planes.hip — the time loop of an LSTM layer of 16 .. 512 cells (one cell per block, any width) as ONE launch, its recurrent
// products on the BF16 matrix cores.
//
// Shape of the work.  A MEMBER is a workgroup that stays on its compute unit for all time steps and owns 16 cells; a GROUP is the members
// that cover all C cells for the same examples of one direction, all on one XCD, whose L2 is where they meet (workgroup ids that are equal
// mod 8 share an XCD: probed once per process, and compared again in every launch).  A group owns one or several ROW TILES of 16 examples;
// a UNIT is one time step of one row tile.  Eight wavefronts of a member contract - its slice of the recurrent weights stays in registers,
// split into the three planes of myea_split.h once per launch (96 of a lane's 168 registers at 512 cells) - and four more, one a SIMD and
// with priority there, do the gate math, a lane per (example, cell): so neither the tensors a step reads and writes nor the gate math stand
// in front of the next row tile's products, and a wait for data is never one for stores.
//
// Forward: every wavefront takes the k blocks wave, wave + 8, ... of h[t-1] from the exchange buffer straight into the operand registers of
// v_mfma_f32_16x16x32_bf16 (h travels as its three planes, in the operand's order); the transposed product puts the four gates of one
// (example, cell) into one accumulator; the eight partial tiles meet in LDS.  Backward: a member contracts over the 64 k's of its own gate
// deltas, which never leave its LDS, and hands every other member the 16 columns of dh that are that one's (FP32 shares, added in a fixed
// order): a quarter of the bytes that reading all members' deltas takes, which was built and measured too (200 cells x 60 examples x 50
// steps 162 us against 107, 512 x 16 x 64 361 against 200: a compute unit takes 50 bytes a clock from L2 at best).
//
// Waiting.  There is no barrier between the members: a word of the exchange buffer that is not written yet is absent (every bit set - no
// number any member stores, a NaN of that pattern becomes another), and whoever needs it looks at the data itself until all of it is there
// (512 cells, one row tile: 2.7 us a step, against 5.6 with stores, a counter and its poll one behind the other).  A wait is
// bounded by `spin_polls` looks; the wavefront that gives up raises the launch's give-up word and the host's flag, every wavefront that
// waits leaves when it sees the word, one that does not wait runs out of units.  Words are used again:
//   * h of step t lies in slot t mod 4.  At unit (t, r) the slot of step t + 1 holds h[t-3], which every member read before it stored
//     h[t-2], which this member has seen whole (before the barrier behind its products of step t-1): it may take its own words back, and
//     does so with vmcnt(0) in front of storing h[t]; whoever looks for h[t+1] has seen h[t];
//   * shares of step j lie in slot j mod 2 and have one reader, who takes them back as soon as it has them, acknowledged before its member
//     stores shares of step j + 1 (a barrier lies between); a producer writes shares of step j + 2 after it has seen those of step j + 1.
//     So the buffer is absent as a whole again when the loop ends, and needs no clearing between launches.
// The host only launches when every workgroup of the grid can be resident at once (one per compute unit).
//
// Several row tiles per group (more examples than the device holds groups for): forward, a wavefront asks for the next unit's h behind its
// barrier; backward, the unit before is contracted while the gates of this one are worked on.
//
// Measured (MI355X, microseconds a pass, one launch per time step or the FP32 loops -> here; forward, backward): 200 cells x 60 examples x 50
// steps 271 -> 107, 274 -> 107; 512 x 16 x 64 365 -> 178, 412 -> 200; 512 x 256 x 64 410 -> 255, stays (see backward_most_tiles); 300 x 128 x
// 30, two directions 290 -> 104, 293 -> 147; 64 x 512 x 30 130 -> 63, 107 -> 56; 480 x 512 x 30 568 -> 234, 649 -> 624; 128 x 256 x 32 127 -> 69,
// 102 -> 66; 256 x 256 x 32 173 -> 79, 153 -> 80; 256 x 1024 x 32 466 -> 209, 582 -> 449.  What bounds a step
// of one row tile at 512 cells: 0.6 us of gate math behind the partial tiles, 0.6 of products, 0.5 from a store to another
// member's look, the rest the looks themselves; of several: the exchange (48 KB a unit and member forward, 96 KB backward).
//
// Precision: h and the deltas are the exact sums of their planes; errors as in myea_gemm.hip.  A product that is not finite (an infinite
// weight, a sum beyond 2^79) is computed again from the FP32 numbers, in 64 bits.
//
// Gate math: Forward_Pass__LSTM__Gates_CIF_AF_State (NN/Neural_Network__Recurrent_Forward_Pass__OpenMP.cpp:1042-1191),
// __States_AF (:1547-1582), __Output (:1351-1418); backward: Backward_Pass__LSTM_Derivative__Output
// (NN/Neural_Network__Recurrent_Backward_Pass__OpenMP.cpp:1130-1273), __Cell_State_AF (:1275-1327),
// __Gates_CIF_AF_State (:1329-1604).  NN/ = Neural_Network_Library_Windows/Source_Files/Neural_Network/.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>
#include <vector>

#include "myea_kernels.h"
#include "myea_split.h"

namespace myea {
namespace {

constexpr int kCells = 16, kRows = 16;       // cells of a member, examples of a row tile
constexpr int kAuxSc1 = 16;                  // a buffer access beyond this compute unit's L1
constexpr unsigned kBufferWord3 = 0x00020000u;   // raw buffer of dwords
constexpr unsigned kAbsent = 0xffffffffu, kAlmost = 0xfffffffeu;   // "not written yet"; what a NaN of that pattern becomes
constexpr int kSlots = 4;                    // forward: steps of h the exchange buffer holds
constexpr int kCellPad = 68;                 // floats between two cells of a partial tile in LDS: 16 examples x 4 gates, and 4 that spread the banks
constexpr int kQuadPad = 80;                 // floats between two groups of four cells of a sum of shares: 16 examples x 4 cells, and 16 that spread the banks
constexpr int kMaxPlaneGroups = 256;
constexpr int kSyncWords = 2 + kMaxPlaneGroups;   // the give-up word, a word per group, a scrap word

struct PlaneGeometry {
    int T, B, Bmax, C;
    int dirs, row_groups, row_tiles, rs;     // groups = dirs * row_groups; a group owns rs row tiles of the row_tiles there are
    int members;                             // workgroups of a group
    int absent;                              // test switch: no wait ever ends
    unsigned spin_polls;
};
struct PlaneSync {
    unsigned *give_up;     // device word, polled; behind it one word per group: the XCC id its first member ran on (+ 1)
    unsigned *host_flag, *fault;
    char *exchange;
    unsigned group_bytes;  // of the exchange buffer per group
};

__device__ __forceinline__ void lds_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// 1 / (1 + exp2(scale s)), scale in two parts: exp2 of the rounded product times (1 + what the rounding left), a Newton step behind the
// reciprocal - as exact as expf and a division, at half their instructions
__device__ __forceinline__ float logistic(float s, float scale_hi, float scale_lo)
{
    const float t = s * scale_hi;
    const float left = __builtin_fmaf(s, scale_lo, __builtin_fmaf(s, scale_hi, -t));
    const float e = __builtin_amdgcn_exp2f(t);
    const float d = 1.f + __builtin_fmaf(e, left * 0.693147180559945309f, e);
    const float y = __builtin_amdgcn_rcpf(d);
    const float better = __builtin_fmaf(__builtin_fmaf(-d, y, 1.f), y, y);
    return t > 120.f ? 0.f : t < -120.f ? 1.f : better;   // beyond: infinities on the way; the value is within 2^-120 of this
}
__device__ __forceinline__ float sigmoid_f(float s) { return logistic(s, -1.44269502162933349609375f, -1.92596299112661746887e-8f); }
__device__ __forceinline__ float tanh_f(float s) { return 2.f * logistic(s, -2.8853900432586669921875f, -3.85192598225323493774e-8f) - 1.f; }   // AF_TANH_real

__device__ __forceinline__ unsigned xcc_id() { return __builtin_amdgcn_s_getreg(20 | (3 << 11)) & 15u; }   // HW_REG_XCC_ID[3:0]

// workgroup id -> (group, member): the XCD of ids = x (mod 8) hosts the groups x, x + 8, ...
__device__ __forceinline__ bool place(unsigned id, int members, int groups, int &group, int &member)
{
    const int xcd = (int)(id & 7), slot = (int)(id >> 3);
    group = (slot / members) * 8 + xcd;
    member = slot % members;
    return group < groups;
}

__device__ __forceinline__ void raise(const PlaneSync &w, unsigned code)
{
    __hip_atomic_store(w.give_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(w.host_flag, code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(w.fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the members of a group must share an XCD's L2: the first to get here writes its XCC id, the others compare
__device__ __forceinline__ void check_same_xcd(const PlaneSync &w, int group)
{
    if (threadIdx.x != 0) return;
    const unsigned mine = xcc_id() + 1u;
    unsigned seen = 0u;
    if (!__hip_atomic_compare_exchange_strong(w.give_up + 1 + group, &seen, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) && seen != mine) raise(w, 2u);
}

// One look at data that is not all there yet: may the wait go on?  The give-up word is looked at every 16th time.
__device__ __forceinline__ bool wait_on(const PlaneSync &w, unsigned &polls)
{
    if ((--polls & 15u) != 0u) return true;
    const unsigned stop = __hip_atomic_load(w.give_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(stop)) return false;
    if (polls == 0u) {
        if ((threadIdx.x & 63) == 0) raise(w, 1u);
        return false;
    }
    return true;
}

__device__ __forceinline__ unsigned umax4(u32x4 v, unsigned m) { return max(max(max(v[0], v[1]), max(v[2], v[3])), m); }

template <int W, int KB>
__global__ __launch_bounds__(64 * (W + 4)) void lstm_planes_forward_kernel(PlaneGeometry g, LstmResidentDir d0, LstmResidentDir d1, PlaneSync w)
{
    constexpr int NCT = 4, kPart = kCells * kCellPad;     // tiles of gate columns; floats of a wavefront's partial tile
    extern __shared__ __attribute__((aligned(16))) float smem[];
    __shared__ unsigned s_dead;
    float *const parts = smem;                            // [2][W][kPart]
    float *const state = smem + 2 * W * kPart;            // [rs][2][256]: cell state and output of the lane's (example, cell)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);

    int group, member;
    if (!place(blockIdx.x, g.members, g.dirs * g.row_groups, group, member)) return;
    const int dir = group % g.dirs, rg = group / g.dirs;
    const LstmResidentDir &d = dir ? d1 : d0;
    const int C = g.C, G = 4 * C, T = g.T, c0 = member * kCells, blocks = (C + 31) / 32;
    const int tiles = min(g.rs, g.row_tiles - rg * g.rs);
    check_same_xcd(w, group);
    const __amdgpu_buffer_rsrc_t exchange = __builtin_amdgcn_make_buffer_rsrc(w.exchange + (size_t)group * w.group_bytes, 0, (int)w.group_bytes, (int)kBufferWord3);
    const unsigned tile_bytes = (unsigned)blocks * 3072u, slot_bytes = (unsigned)g.rs * tile_bytes;
    auto slot_of = [&](int t, int r) { return ((unsigned)t & (kSlots - 1)) * slot_bytes + (unsigned)r * tile_bytes; };
    if (threadIdx.x == 0) s_dead = 0u;

    if (wave < W) {
        // ---- the contraction
        const int col16 = lane & 15, quad = lane >> 4;
        // the weights: gate column i of tile ct is gate i % 4 of cell 4 ct + i / 4
        bf16x8 wf[KB][NCT][3];
#pragma unroll
        for (int i = 0; i < KB; ++i)
#pragma unroll
            for (int ct = 0; ct < NCT; ++ct) {
                const int wc = c0 + ct * 4 + col16 / 4, k = (wave + W * i) * 32 + quad * 8;
                float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                if (wc < C && k < C) load_eight<true>(x, d.Wrec + ((size_t)(col16 & 3) * C + wc) * C + k, 0, k, C);
                split_eight(x, wf[i][ct]);
            }
        // a block's second half has no owner where the members are an odd number
        const bool tail_lane = quad >= 2 && (g.members & 1);
        u32x4 fr[KB][3];   // the wavefront's blocks of 32 k's of a unit
#pragma unroll
        for (int i = 0; i < KB; ++i)
#pragma unroll
            for (int p = 0; p < 3; ++p) fr[i][p] = (u32x4){0u, 0u, 0u, 0u};
        const unsigned in_lane = (unsigned)wave * 3072u + (unsigned)lane * 16u;
        auto load_block = [&](int i, int t, int r) {   // h of step t, row tile r
            const int kb = wave + W * i;
            if (kb >= blocks || (tail_lane && kb == blocks - 1)) return;
            const unsigned at = slot_of(t, r) + in_lane + (unsigned)i * (W * 3072u);
#pragma unroll
            for (int p = 0; p < 3; ++p) fr[i][p] = __builtin_amdgcn_raw_buffer_load_b128(exchange, (int)(at + (unsigned)p * 1024u), 0, kAuxSc1);
        };
        auto all_there = [&]() {
            unsigned m = 0u;
#pragma unroll
            for (int i = 0; i < KB; ++i)
#pragma unroll
                for (int p = 0; p < 3; ++p) m = umax4(fr[i][p], m);
            return __all(m != kAbsent && !g.absent);
        };
        lds_barrier();
        for (int r = 0; r < tiles; ++r) lds_barrier();   // the first step has no recurrent term
        int u = tiles;
#pragma unroll
        for (int i = 0; i < KB; ++i) load_block(i, 0, 0);
        for (int t = 1; t < T; ++t)
            for (int r = 0; r < tiles; ++r, ++u) {
                unsigned polls = g.spin_polls;
                while (!all_there()) {
                    if (!wait_on(w, polls)) { if (lane == 0) s_dead = 1u; return; }
                    asm volatile("" ::: "memory");
#pragma unroll
                    for (int i = 0; i < KB; ++i) load_block(i, t - 1, r);
                }
                f32x4 acc[NCT], small[NCT];
#pragma unroll
                for (int ct = 0; ct < NCT; ++ct) acc[ct] = small[ct] = (f32x4){0.f, 0.f, 0.f, 0.f};
                int tn = t, rn = r + 1;
                if (rn == tiles) { rn = 0; ++tn; }
#pragma unroll
                for (int i = 0; i < KB; ++i) {
                    bf16x8 h[3];
#pragma unroll
                    for (int p = 0; p < 3; ++p) {
                        asm volatile("" : "+v"(fr[i][p]));   // as the compiler sees it nothing is on its way into these registers from here on
                        h[p] = __builtin_bit_cast(bf16x8, fr[i][p]);
                    }
                    if (wave + W * i < blocks) {
#pragma unroll
                        for (int q = 0; q < 5; ++q)
#pragma unroll
                            for (int ct = 0; ct < NCT; ++ct) small[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i][ct][kSmallA[q]], h[kSmallB[q]], small[ct], 0, 0, 0);
#pragma unroll
                        for (int ct = 0; ct < NCT; ++ct) acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i][ct][0], h[0], acc[ct], 0, 0, 0);
                    }
                }
                float *to = parts + ((u & 1) * W + wave) * kPart + col16 * 4;
#pragma unroll
                for (int ct = 0; ct < NCT; ++ct) *reinterpret_cast<f32x4 *>(to + (ct * 4 + quad) * kCellPad) = acc[ct] + small[ct];
                lds_barrier();
                if (tn < T) {
#pragma unroll
                    for (int i = 0; i < KB; ++i) load_block(i, tn - 1, rn);
                }
            }
        return;
    }

    // ---- the gates: four wavefronts, a lane per (example, cell), ahead of the others where they share a SIMD
    __builtin_amdgcn_s_setprio(3);
    const int pair = threadIdx.x - 64 * W, row = pair >> 4, cell = pair & 15;
    const int k = c0 + cell, kc = min(k, C - 1);
    float e_bias[4], e_peep[3];
#pragma unroll
    for (int q = 0; q < 4; ++q) e_bias[q] = d.bias[q * C + kc];
#pragma unroll
    for (int q = 0; q < 3; ++q) e_peep[q] = d.peep[q * C + kc];
    asm volatile("" : "+v"(e_bias[0]), "+v"(e_bias[1]), "+v"(e_bias[2]), "+v"(e_bias[3]), "+v"(e_peep[0]), "+v"(e_peep[1]), "+v"(e_peep[2]));
    for (int i = pair; i < 512 * tiles; i += 256) state[i] = 0.f;
    // where this lane's words of h go: even cells the first and the third plane, odd cells the second
    const unsigned out_lane = (unsigned)(k >> 5) * 3072u + (unsigned)((k & 31) >> 3) * 256u + (unsigned)row * 16u + (unsigned)((k & 7) >> 1) * 4u;
    const bool even = !(cell & 1);
    const unsigned out_first = out_lane + (even ? 0u : 1024u), out_third = out_lane + 2048u;
    // a time step's part of a tensor is found by scalar arithmetic, the lane's place in it by 32-bit offsets
    const ptrdiff_t step = (d.reverse ? -1 : 1) * (ptrdiff_t)g.Bmax * C;   // floats of a [Bmax][C] tensor from one step to the next
    ptrdiff_t at_now = d.reverse ? (T - 1) * (ptrdiff_t)g.Bmax * C : 0;
    const int first_row = rg * g.rs * kRows;
    float e_in[4];
    unsigned keep_c = 1u, keep_h = 1u;
    auto load_inputs = [&](ptrdiff_t time, int t, int r) {
        const float *in = d.acts + 4 * time;
        const unsigned at = (unsigned)min(first_row + r * kRows + row, g.B - 1) * (unsigned)G + (unsigned)kc;
#pragma unroll
        for (int q = 0; q < 4; ++q) e_in[q] = in[at + (unsigned)(q * C)];
        if (d.zone_state) keep_c = (d.zone_state + (size_t)(d.reverse ? T - 1 - t : t) * d.zone_stride)[kc];
        if (d.zone_output) keep_h = (d.zone_output + (size_t)(d.reverse ? T - 1 - t : t) * d.zone_stride)[kc];
    };
    load_inputs(at_now, 0, 0);
    lds_barrier();
    int u = 0;
    for (int t = 0; t < T; ++t) {
        for (int r = 0; r < tiles; ++r, ++u) {
            lds_barrier();
            const unsigned dead = s_dead;
            if (t >= kSlots - 1) {   // the slot of the step after this one is free: everybody has read what it holds
                const unsigned at = slot_of(t + 1, r);
                __builtin_amdgcn_raw_buffer_store_b32(kAbsent, exchange, (int)(at + out_first), 0, 0);
                if (even) __builtin_amdgcn_raw_buffer_store_b32(kAbsent, exchange, (int)(at + out_third), 0, 0);
            }
            const int ex = first_row + r * kRows + row;
            const bool valid = ex < g.B && k < C;
            f32x4 sum = {0.f, 0.f, 0.f, 0.f};
            if (t > 0) {
                const float *from = parts + (u & 1) * W * kPart + cell * kCellPad + row * 4;
                f32x4 part[W];
#pragma unroll
                for (int wv = 0; wv < W; ++wv) part[wv] = *reinterpret_cast<const f32x4 *>(from + wv * kPart);
                __builtin_amdgcn_sched_barrier(0);   // all of them requested before the first is waited for
#pragma unroll
                for (int wv = 0; wv < W; ++wv) sum += part[wv];
            }
            const float cp = state[r * 512 + pair];
            float rec[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) rec[q] = unscaled(sum[q]);
            if (!(fabsf(rec[0]) < INFINITY && fabsf(rec[1]) < INFINITY && fabsf(rec[2]) < INFINITY && fabsf(rec[3]) < INFINITY)) {
                // a weight or a sum beyond the planes' range: again, in 64 bits
                const unsigned base = slot_of(t - 1, r) + (unsigned)row * 16u;
                double s[4] = {0., 0., 0., 0.};
                for (int j = 0; j < C && valid; ++j) {
                    const unsigned at = base + (unsigned)(j >> 5) * 3072u + (unsigned)((j & 31) >> 3) * 256u + (unsigned)((j & 7) >> 1) * 4u;
                    double h = 0.;
                    for (int p = 0; p < 3; ++p) {
                        const unsigned both = __builtin_amdgcn_raw_buffer_load_b32(exchange, (int)(at + (unsigned)p * 1024u), 0, kAuxSc1);
                        h += (double)__uint_as_float(j & 1 ? both & 0xffff0000u : both << 16);
                    }
                    for (int q = 0; q < 4; ++q) s[q] = fma(h * 0x1p-24, (double)d.Wrec[((size_t)q * C + k) * C + j], s[q]);
                }
                for (int q = 0; q < 4; ++q) rec[q] = (float)s[q];
            }
            float si = e_in[1] + rec[1] + e_bias[1], gf = 0.f;
            if (t > 0) {
                si += cp * e_peep[0];
                gf = sigmoid_f(e_in[2] + rec[2] + e_bias[2] + cp * e_peep[1]);
            }
            const float gi = sigmoid_f(si);
            const float z = tanh_f(e_in[0] + rec[0] + e_bias[0]);
            float cs = t > 0 ? z * gi + gf * cp : z * gi;
            cs = keep_c ? cs : cp;
            const float a = tanh_f(cs);
            const float go = sigmoid_f(e_in[3] + rec[3] + e_bias[3] + cs * e_peep[2]);
            float hv = a * go;
            if (d.zone_output) {
                hv = keep_h ? hv : state[r * 512 + 256 + pair];
                state[r * 512 + 256 + pair] = hv;
            }
            state[r * 512 + pair] = cs;
            if (t + 1 < T) {
                const float own = valid ? hv : 0.f;
                const float other = __uint_as_float((unsigned)__builtin_amdgcn_mov_dpp((int)__float_as_uint(own), 0xB1, 0xF, 0xF, true));
                unsigned hi, mid, lo;
                split_pair(even ? own : other, even ? other : own, hi, mid, lo);
                const unsigned at = slot_of(t, r);
                __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): the words taken back for the step after this one are absent for everybody
                __builtin_amdgcn_raw_buffer_store_b32(min(even ? hi : mid, kAlmost), exchange, (int)(at + out_first), 0, 0);
                if (even) __builtin_amdgcn_raw_buffer_store_b32(min(lo, kAlmost), exchange, (int)(at + out_third), 0, 0);
            }
            if (dead) return;
            const ptrdiff_t at_then = at_now;
            if (r + 1 < tiles) load_inputs(at_now, t, r + 1);
            else if (t + 1 < T) load_inputs(at_now + step, t + 1, 0);
            if (valid) {
                float *acts = d.acts + 4 * at_then, *pc = d.c + at_then, *pca = d.ca + at_then, *ph = d.h + at_then;
                const unsigned at_c = (unsigned)ex * (unsigned)C + (unsigned)k, at_g = at_c + (unsigned)ex * (unsigned)(3 * C);
                acts[at_g] = z; acts[at_g + (unsigned)C] = gi; acts[at_g + (unsigned)(2 * C)] = gf; acts[at_g + (unsigned)(3 * C)] = go;
                pc[at_c] = cs; pca[at_c] = a; ph[at_c] = hv;
            }
        }
        at_now += step;
    }
}

// dh[t] += dG[t'] Wrec (t' = the step processed before t in this pass), every member contracting over its own 64 k's - the gate deltas it
// has just computed and keeps in LDS - and handing each other member the share of its 16 columns.
template <int W, int TW>
__global__ __launch_bounds__(64 * (W + 4)) void lstm_planes_backward_kernel(PlaneGeometry g, LstmResidentDir d0, LstmResidentDir d1, PlaneSync w)
{
    constexpr unsigned kPlaneBytes = 2u * 3u * 1024u;     // the member's gate deltas of a unit: [2 blocks of 32 k's][3 planes][64 lanes][16 bytes]
    constexpr int kShare = 4 * kQuadPad;                  // floats of a wavefront's sum of shares
    extern __shared__ __attribute__((aligned(16))) float smem[];
    __shared__ unsigned s_dead;
    __shared__ double s_fold[4][7][16];
    char *const planes = reinterpret_cast<char *>(smem);                       // [2][kPlaneBytes]
    float *const own = smem + 2 * kPlaneBytes / sizeof(float);                 // [2][16 examples][64 k's], FP32
    float *const shares = own + 2 * kRows * 64;                                // [2][W][kShare]
    float *const state = shares + 2 * W * kShare;                              // [rs][4][256]: of the step before: delta i, delta f, f, delta c
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);

    int group, member;
    if (!place(blockIdx.x, g.members, g.dirs * g.row_groups, group, member)) return;
    const int dir = group % g.dirs, rg = group / g.dirs;
    const LstmResidentDir &d = dir ? d1 : d0;
    const int C = g.C, T = g.T, c0 = member * kCells, members = g.members;
    const int tiles = min(g.rs, g.row_tiles - rg * g.rs);
    check_same_xcd(w, group);
    if (threadIdx.x == 0) s_dead = 0u;

    if (wave < W) {
        // ---- the contraction, transposed: an accumulator holds four consecutive columns of one example
        // [2 steps][row tiles][consumer][producer][64 lanes][16 bytes]
        const __amdgpu_buffer_rsrc_t exchange = __builtin_amdgcn_make_buffer_rsrc(w.exchange + (size_t)group * w.group_bytes, 0, (int)w.group_bytes, (int)kBufferWord3);
        const unsigned tile_bytes = (unsigned)(members * members) * 1024u, slot_bytes = (unsigned)g.rs * tile_bytes;
        auto slot_of = [&](int j, int r) { return ((unsigned)j & 1u) * slot_bytes + (unsigned)r * tile_bytes + (unsigned)lane * 16u; };
        const int col16 = lane & 15, quad = lane >> 4;
        bf16x8 wf[TW][2][3];   // k = 4 cell + gate
#pragma unroll
        for (int i = 0; i < TW; ++i)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int n = (wave * TW + i) * 16 + col16;
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int c = c0 + b * 8 + quad * 2 + e / 4;
                    x[e] = 0.f;
                    if (n < C && c < C) x[e] = d.Wrec[((size_t)(e & 3) * C + c) * C + n];
                }
                split_eight(x, wf[i][b]);
            }
        // the shares of the step after (j, r), from the gate deltas the other four wavefronts left for unit u
        auto contract = [&](int u, int j, int r) {
            const char *from = planes + (unsigned)(u & 1) * kPlaneBytes + lane * 16;
            bf16x8 dg[2][3];
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int p = 0; p < 3; ++p) dg[b][p] = *reinterpret_cast<const bf16x8 *>(from + (b * 3 + p) * 1024);
            f32x4 acc[TW], small[TW];
#pragma unroll
            for (int i = 0; i < TW; ++i) acc[i] = small[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int q = 0; q < 5; ++q)
#pragma unroll
                    for (int i = 0; i < TW; ++i) small[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i][b][kSmallA[q]], dg[b][kSmallB[q]], small[i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < TW; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i][b][0], dg[b][0], acc[i], 0, 0, 0);
            }
            const unsigned to = slot_of(j + 1, r) + (unsigned)member * 1024u;
#pragma unroll
            for (int i = 0; i < TW; ++i) {
                const int consumer = wave * TW + i;
                if (consumer >= members) continue;
                f32x4 v = acc[i] + small[i];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = unscaled(v[e]);
                if (!(fabsf(v[0]) < INFINITY && fabsf(v[1]) < INFINITY && fabsf(v[2]) < INFINITY && fabsf(v[3]) < INFINITY)) {
                    // an operand or a sum beyond the planes' range: again, in 64 bits
                    for (int e = 0; e < 4; ++e) {
                        const int n = consumer * 16 + quad * 4 + e;
                        double sum = 0.;
                        for (int k = 0; k < 64 && n < C; ++k) {
                            const int c = c0 + (k >> 2);
                            if (c < C) sum = fma((double)own[(u & 1) * (kRows * 64) + col16 * 64 + k], (double)d.Wrec[((size_t)(k & 3) * C + c) * C + n], sum);
                        }
                        v[e] = (float)sum;
                    }
                }
                u32x4 bits;
#pragma unroll
                for (int e = 0; e < 4; ++e) bits[e] = min(__float_as_uint(v[e]), kAlmost);
                __builtin_amdgcn_raw_buffer_store_b128(bits, exchange, (int)(to + (unsigned)(consumer * members) * 1024u), 0, 0);
            }
        };
        lds_barrier();
        int u = 0, j_before = -1, r_before = 0;
        for (int j = 0; j < T; ++j)
            for (int r = 0; r < tiles; ++r, ++u) {
                if (j > 0) {   // the shares of this unit from the wavefront's producers: wave, wave + W, ...
                    const unsigned at = slot_of(j, r) + (unsigned)(member * members + wave) * 1024u;
                    u32x4 got[TW];
                    unsigned polls = g.spin_polls;
                    for (;;) {
#pragma unroll
                        for (int i = 0; i < TW; ++i) {
                            got[i] = (u32x4){0u, 0u, 0u, 0u};
                            if (wave + i * W < members) got[i] = __builtin_amdgcn_raw_buffer_load_b128(exchange, (int)(at + (unsigned)(i * W) * 1024u), 0, kAuxSc1);
                        }
                        unsigned m = 0u;
#pragma unroll
                        for (int i = 0; i < TW; ++i) m = umax4(got[i], m);
                        if (__all(m != kAbsent && !g.absent)) break;
                        if (!wait_on(w, polls)) { if (lane == 0) s_dead = 1u; return; }
                        asm volatile("" ::: "memory");
                    }
                    // taken: absent again before this member hands out the shares of the step after this one, two before these words' next
                    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int i = 0; i < TW; ++i) {
                        if (wave + i * W < members) __builtin_amdgcn_raw_buffer_store_b128((u32x4){kAbsent, kAbsent, kAbsent, kAbsent}, exchange, (int)(at + (unsigned)(i * W) * 1024u), 0, 0);
                        sum += __builtin_bit_cast(f32x4, got[i]);
                    }
                    *reinterpret_cast<f32x4 *>(shares + ((u & 1) * W + wave) * kShare + quad * kQuadPad + col16 * 4) = sum;
                }
                if (tiles > 1) {
                    // this unit's sums to the gates, and while they work on them the unit before is contracted; what that unit's look took is
                    // absent for everybody: only this unit's own stores may still be on their way
                    __builtin_amdgcn_s_waitcnt(0x0F70 | TW);
                    lds_barrier();
                    if (j_before >= 0 && j_before + 1 < T) contract(u - 1, j_before, r_before);
                    j_before = j; r_before = r;
                } else {
                    lds_barrier();
                    if (j + 1 < T) {
                        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
                        lds_barrier();
                        contract(u, j, r);
                    }
                }
                if (s_dead) return;
            }
        return;
    }

    // ---- the gates: four wavefronts, a lane per (example, cell), ahead of the others where they share a SIMD
    __builtin_amdgcn_s_setprio(3);
    const int pair = threadIdx.x - 64 * W, row = pair >> 4, cell = pair & 15;
    const int k = c0 + cell, kc = min(k, C - 1);
    float e_peep[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) e_peep[q] = d.peep[q * C + kc];
    asm volatile("" : "+v"(e_peep[0]), "+v"(e_peep[1]), "+v"(e_peep[2]));
    // this pass walks the direction's steps from its last to its first
    const ptrdiff_t step = (d.reverse ? 1 : -1) * (ptrdiff_t)g.Bmax * C;
    ptrdiff_t at_now = d.reverse ? 0 : (T - 1) * (ptrdiff_t)g.Bmax * C;
    const int first_row = rg * g.rs * kRows;
    float e_act[4], e_ca, e_dh, e_cp, e_cs;
    auto load_operands = [&](ptrdiff_t time, int s, int r) {   // s: the direction's step
        const unsigned ex = (unsigned)min(first_row + r * kRows + row, g.B - 1), at = ex * (unsigned)C + (unsigned)kc, at_g = at + ex * (unsigned)(3 * C);
        const float *acts = d.acts + 4 * time;
#pragma unroll
        for (int q = 0; q < 4; ++q) e_act[q] = acts[at_g + (unsigned)(q * C)];
        e_ca = (d.ca + time)[at]; e_dh = (d.dh + time)[at]; e_cs = (d.c + time)[at];
        e_cp = (d.c + time + (s > 0 ? step : 0))[at];   // (no step before the first: any value, it is not used)
    };
    double sums[7] = {0., 0., 0., 0., 0., 0., 0.};   // over the lane's examples and steps: dz, di, df, do, di c', df c', do c (c': the state of the step before)
    load_operands(at_now, T - 1, 0);
    lds_barrier();
    int u = 0;
    for (int j = 0; j < T; ++j) {
        const int s = T - 1 - j;
        for (int r = 0; r < tiles; ++r, ++u) {
            const int ex = first_row + r * kRows + row;
            const bool valid = ex < g.B && k < C;
            float rec = 0.f, n_di = 0.f, n_df = 0.f, n_f = 0.f, n_dc = 0.f;
            float *const before = state + r * 1024 + pair;
            lds_barrier();
            const unsigned dead = s_dead;
            if (j > 0) {
                const float *from = shares + (u & 1) * W * kShare + (cell >> 2) * kQuadPad + row * 4 + (cell & 3);
                float part[W];
#pragma unroll
                for (int wv = 0; wv < W; ++wv) part[wv] = from[wv * kShare];
                n_di = before[0]; n_df = before[256]; n_f = before[512]; n_dc = before[768];
                __builtin_amdgcn_sched_barrier(0);   // all of them requested before the first is waited for
#pragma unroll
                for (int wv = 0; wv < W; ++wv) rec += part[wv];
            }
            const float dh = e_dh + rec;
            const float z = e_act[0], gi = e_act[1], gf = e_act[2], go = e_act[3], a = e_ca;
            float ddo = go * (1.f - go) * (dh * a);
            float e = dh * go * (1.f - a * a);
            e += e_peep[2] * ddo;
            if (j > 0) {
                e += e_peep[0] * n_di;
                e += e_peep[1] * n_df;
                e += n_dc * n_f;
            }
            float dz = e * gi * (1.f - z * z);
            float di = (e * z) * (gi * (1.f - gi));
            float df = s > 0 ? (e * e_cp) * (gf * (1.f - gf)) : 0.f;
            if (!valid) dz = di = df = ddo = 0.f;
            const float cp = s > 0 ? e_cp : 0.f, cs = e_cs;
            if (j + 1 < T) {
                unsigned hi[2], mid[2], lo[2];
                split_pair(dz, di, hi[0], mid[0], lo[0]);
                split_pair(df, ddo, hi[1], mid[1], lo[1]);
                char *to = planes + (unsigned)(u & 1) * kPlaneBytes + (cell >> 3) * 3072 + (((cell & 7) >> 1) * 16 + row) * 16 + (cell & 1) * 8;
                *reinterpret_cast<u32x2 *>(to) = (u32x2){hi[0], hi[1]};
                *reinterpret_cast<u32x2 *>(to + 1024) = (u32x2){mid[0], mid[1]};
                *reinterpret_cast<u32x2 *>(to + 2048) = (u32x2){lo[0], lo[1]};
                *reinterpret_cast<f32x4 *>(own + (u & 1) * (kRows * 64) + row * 64 + cell * 4) = (f32x4){dz, di, df, ddo};
                if (tiles == 1) lds_barrier();
            }
            if (dead) return;
            before[0] = di; before[256] = df; before[512] = gf; before[768] = e;
            const ptrdiff_t at_then = at_now;
            const int rn = r + 1 < tiles ? r + 1 : 0, jn = r + 1 < tiles ? j : j + 1;
            if (jn < T) load_operands(jn > j ? at_now + step : at_now, T - 1 - jn, rn);
            if (valid) {
                float *pg = d.dG + 4 * at_then;
                const unsigned at_c = (unsigned)ex * (unsigned)C + (unsigned)k, at_g = at_c + (unsigned)ex * (unsigned)(3 * C);
                pg[at_g] = dz; pg[at_g + (unsigned)C] = di; pg[at_g + (unsigned)(2 * C)] = df; pg[at_g + (unsigned)(3 * C)] = ddo;
                (d.dh + at_then)[at_c] = dh; (d.dc + at_then)[at_c] = e;
                sums[0] += dz; sums[1] += di; sums[2] += df; sums[3] += ddo;
                sums[4] += di * cp; sums[5] += df * cp; sums[6] += ddo * cs;
            }
        }
        at_now += step;
    }
    if (!d.sums) return;
    // the sums over the group's examples, in a fixed order; the other wavefronts wait for nothing any more
#pragma unroll
    for (int v = 0; v < 7; ++v) {
        double x = sums[v];
        x += __shfl_xor(x, 16);
        x += __shfl_xor(x, 32);
        if (lane < 16) s_fold[wave - W][v][lane] = x;
    }
    lds_barrier();
    if (pair < 7 * 16) {
        const int v = pair >> 4, cl = pair & 15;
        if (c0 + cl < C) d.sums[((size_t)rg * 7 + v) * C + c0 + cl] = (float)(((s_fold[0][v][cl] + s_fold[1][v][cl]) + s_fold[2][v][cl]) + s_fold[3][v][cl]);
    }
}

__global__ void planes_clear_kernel(unsigned *words, int n, u32x4 *exchange, size_t chunks)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (size_t c = i; c < (size_t)n; c += (size_t)gridDim.x * blockDim.x) words[c] = 0u;
    for (size_t c = i; c < chunks; c += (size_t)gridDim.x * blockDim.x) exchange[c] = (u32x4){kAbsent, kAbsent, kAbsent, kAbsent};
}


// ---- host ----------------------------------------------------------------------------------------------------------------
using PlaneKernel = void (*)(PlaneGeometry, LstmResidentDir, LstmResidentDir, PlaneSync);
struct PlaneKernelInfo {
    PlaneKernel fn = nullptr;
    int waves = 0;
    bool ready = false;
    hipError_t status = hipSuccess;
};
std::mutex g_planes_mutex;

constexpr size_t kMaxLds = 156 * 1024;   // dynamic LDS a workgroup may ask for
size_t forward_lds(int waves, int rs) { return (size_t)2 * waves * kCells * kCellPad * sizeof(float) + (size_t)rs * 512 * sizeof(float); }

// by the number of blocks of 32 k's: up to 8, up to 16 (one or two a wavefront)
PlaneKernelInfo g_forward[2] = {{lstm_planes_forward_kernel<8, 1>, 8}, {lstm_planes_forward_kernel<8, 2>, 8}};

// by the number of members: up to 8, 16, 32 (consumers a wavefront serves: 1, 2, 4)
PlaneKernelInfo g_backward[3] = {{lstm_planes_backward_kernel<8, 1>, 8}, {lstm_planes_backward_kernel<8, 2>, 8}, {lstm_planes_backward_kernel<8, 4>, 8}};
size_t backward_lds(int rs) { return (size_t)2 * 6 * 1024 + ((size_t)2 * kRows * 64 + (size_t)2 * 8 * 4 * kQuadPad + (size_t)rs * 1024) * sizeof(float); }

PlaneKernelInfo *ready(PlaneKernelInfo &k)
{
    std::lock_guard<std::mutex> lock(g_planes_mutex);
    if (!k.ready) {
        k.status = hipFuncSetAttribute(reinterpret_cast<const void *>(k.fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMaxLds);
        k.ready = true;
    }
    return k.status == hipSuccess ? &k : nullptr;
}
PlaneKernelInfo *forward_kernel(size_t C)
{
    const size_t blocks = (C + 31) / 32;
    return C < 16 || blocks > 16 ? nullptr : ready(g_forward[(blocks - 1) / 8]);
}
PlaneKernelInfo *backward_kernel(int members) { return ready(g_backward[members <= 8 ? 0 : members <= 16 ? 1 : 2]); }
unsigned polls()
{
    const char *e = std::getenv("MYEA_LSTM_RESIDENT_SPIN_POLLS");
    if (e && *e) { const unsigned long long v = std::strtoull(e, nullptr, 10); return v < 16 ? 16u : (v > 0x7ffffff0ull ? 0x7ffffff0u : (unsigned)v & ~15u); }
    return 400000u;
}
bool flag_set(const char *name, char value)
{
    const char *e = std::getenv(name);
    return e && e[0] == value;
}

// Row tiles a group at which one launch a step is not the faster form yet, both sides measured over 16 time steps, us.  A loop's step costs
// the members' shares, tile by tile, and more than that once a XCD's shares of two steps (2 members^2 KiB a tile) outgrow its 4 MiB of L2; a launch a
// step costs its launch, and less the better its width fills tiles (multiples of 32 have a kernel of their own).
// Backward, loop against launches, up to the line and beyond it: 128 cells 8 tiles (4093 examples) 340 | 374, 100 cells 310 | 311, 12 tiles
// 462 | 424; 160 x 2301 (6) 283 | 298, 2309 (7) 310 | 297; 256 x 1277 (5) 285 | 298, 1533 (6) 343 | 318; 384 x 509 (4) 228 | 248, 637 (5) 289 |
// 263; 480 x 509 (4) 304 | 316, 517 (5) 349 | 322; 300 x 773 (7) 280 | 326, 1021 (8) 388 | 373; 200 x 1541 (7) 298 | 316, 2045 (8) 383 | 339; 500
// x 765 (6) 523 | 538, 1021 (8) 697 | 566.  Two directions' launches share the device: 100 x 2045 (8) 307 | 314; 128 x 1277 (5) 193 | 218, 1533
// (6) 259 | 247; 160 x 957 (5) 216 | 226, 1149 (6) 280 | 250; 256 x 509 (4) 208 | 210, 637 (5) 283 | 248; 448 x 189 (3) 167 | 208, 253 (4) 279 |
// 245; 300 x 381 (6) 249 | 313; 500 x 317 (5) 433 | 481, 381 (6) 524 | 506.  512 cells and more than one tile: the loop of
// myea_lstm_resident.hip is the faster one (figures there), or one launch a step where that does not hold the batch (512 examples, 30 steps:
// 642 us against 670).
size_t backward_most_tiles(size_t C, int dirs)
{
    if (C == 512) return 1;
    if (C % 32 != 0) return dirs == 1 ? (C <= 128 ? 8 : C <= 320 ? 7 : 6) : (C <= 128 ? 8 : C <= 320 ? 6 : 5);
    return dirs == 1 ? (C <= 128 ? 8 : C <= 224 ? 6 : C <= 320 ? 5 : 4) : (C <= 224 ? 5 : C <= 320 ? 4 : 3);
}
// Forward: 480 x 3712 (29 tiles) 894 | 1743, 300 x 3712 790 | 832, 200 x 7424 839 | 867; 100 x 8189 (16) 450 | 515, 14848 (29) 836 | 756.
size_t forward_most_tiles(size_t C) { return C <= 128 ? 16 : 29; }

constexpr int kMostCus = 256;   // the buffers are sized for
// groups of one direction that are resident at once
size_t groups_that_fit(int cus, size_t C, int dirs) { return (size_t)cus / 8 / ((C + kCells - 1) / kCells) * 8 / (size_t)dirs; }

}  // namespace

int lstm_planes_plan(size_t C, size_t cells_per_block, size_t B, size_t Bmax, int dirs, LstmPlanesPlan *plan)
{
    *plan = LstmPlanesPlan{};
    if (flag_set("MYEA_LSTM_RESIDENT", '0') || cells_per_block != 1 || B == 0 || dirs < 1 || dirs > 2 || C < 16 || C > 512) return MYEA_OK;
    if (!device_groups_share_xcd()) return MYEA_OK;
    int dev = -1, cus = 0;
    MYEA_HIP_TRY(hipGetDevice(&dev));
    MYEA_HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    cus = std::min(cus, kMostCus);
    const int members = (int)(C + kCells - 1) / kCells;
    const size_t most = groups_that_fit(cus, C, dirs);
    if (most == 0) return MYEA_OK;
    const size_t tiles = (B + kRows - 1) / kRows, rs = (tiles + most - 1) / most;
    // offsets into a time step's rows are 32 bits wide (a group's exchange: 29 tiles x 192 KiB forward, 8 x 2 MiB backward)
    if (rs > forward_most_tiles(C) || Bmax * 4 * C > 0x3fffffffu) return MYEA_OK;
    PlaneKernelInfo *k = forward_kernel(C);
    if (!k || !backward_kernel(members) || forward_lds(k->waves, (int)rs) > kMaxLds) return MYEA_OK;
    plan->ok = true; plan->members = members; plan->rs = (int)rs; plan->row_tiles = (int)tiles;
    plan->row_groups = (int)((tiles + rs - 1) / rs);
    const int groups = plan->row_groups * dirs;
    if (groups > kMaxPlaneGroups) { plan->ok = false; return MYEA_OK; }
    plan->grid = 8 * ((groups + 7) / 8) * members;
    plan->cus = cus;
    plan->backward = rs <= backward_most_tiles(C, dirs) && backward_lds((int)rs) <= kMaxLds;
    return MYEA_OK;
}

// row tiles of all groups of a direction, those of the last one rounded up, for up to B examples
static size_t planes_tiles(size_t C, size_t B, int dirs, size_t most_tiles)
{
    const size_t most = groups_that_fit(kMostCus, C, dirs);
    return std::min((B + kRows - 1) / kRows + most, most * most_tiles);
}

size_t lstm_planes_exchange_floats(size_t C, size_t B, int dirs)
{
    if (C < 16 || C > 512 || B == 0) return 0;
    return (size_t)dirs * planes_tiles(C, B, dirs, forward_most_tiles(C)) * ((C + 31) / 32) * 3072 * kSlots / sizeof(float);
}

size_t lstm_planes_shares_floats(size_t C, size_t B, int dirs)
{
    if (C < 16 || C > 512 || B == 0) return 0;
    const size_t members = (C + kCells - 1) / kCells;
    return (size_t)dirs * 2 * planes_tiles(C, B, dirs, backward_most_tiles(C, dirs)) * members * members * 256;
}

static int prepare(hipStream_t s, const LstmPlanesPlan &plan, size_t T, size_t B, size_t Bmax, size_t C, int dirs, unsigned *sync, unsigned *host_flag, unsigned *fault,
                   float *exchange, size_t exchange_floats, size_t group_bytes, bool clear, PlaneGeometry *g, PlaneSync *w)
{
    if (!plan.ok || T < 2 || T > 0x7fffffffu / 4u) { set_last_error("resident LSTM: no plan for this layer"); return MYEA_E_INVALID; }
    const int groups = plan.row_groups * dirs;
    const size_t bytes = group_bytes * (size_t)groups;
    if (!exchange || (reinterpret_cast<uintptr_t>(exchange) & 15u) || exchange_floats * sizeof(float) < bytes) {
        set_last_error("resident LSTM: the exchange buffer holds %zu floats, the layer needs %zu", exchange ? exchange_floats : (size_t)0, bytes / sizeof(float));
        return MYEA_E_INVALID;
    }
    g->T = (int)T; g->B = (int)B; g->Bmax = (int)Bmax; g->C = (int)C;
    g->dirs = dirs; g->row_groups = plan.row_groups; g->row_tiles = plan.row_tiles; g->rs = plan.rs; g->members = plan.members;
    g->absent = flag_set("MYEA_LSTM_RESIDENT_TEST_ABSENT_MEMBER", '1') ? 1 : 0;
    g->spin_polls = polls();
    w->give_up = sync; w->host_flag = host_flag; w->fault = fault ? fault : sync + 1 + kMaxPlaneGroups;
    w->exchange = reinterpret_cast<char *>(exchange); w->group_bytes = (unsigned)group_bytes;
    const size_t chunks = clear ? bytes / 16 : 0;
    const int words = 1 + groups;
    const size_t work = chunks / 1024 + (size_t)(words + 511) / 512, blocks = work > 1024 ? 1024 : work;
    hipLaunchKernelGGL(planes_clear_kernel, dim3((unsigned)blocks), dim3(512), 0, s, sync, words, reinterpret_cast<u32x4 *>(exchange), chunks);
    MYEA_HIP_TRY(hipGetLastError());
    return MYEA_OK;
}

int launch_lstm_planes_forward(hipStream_t s, const LstmPlanesPlan &plan, size_t T, size_t B, size_t Bmax, size_t C, int dirs, const LstmResidentDir *dir,
                               unsigned *sync, unsigned *host_flag, unsigned *fault, float *exchange, size_t exchange_floats)
{
    for (int q = 0; q < dirs; ++q)
        if (!dir[q].Wrec || !dir[q].bias || !dir[q].peep || !dir[q].acts || !dir[q].c || !dir[q].ca || !dir[q].h) { set_last_error("resident LSTM: null operand"); return MYEA_E_INVALID; }
    PlaneKernelInfo *k = forward_kernel(C);
    if (!k) { set_last_error("resident LSTM: no kernel for %zu cells", C); return MYEA_E_UNSUPPORTED; }
    PlaneGeometry g;
    PlaneSync w;
    const int rc = prepare(s, plan, T, B, Bmax, C, dirs, sync, host_flag, fault, exchange, exchange_floats, (size_t)plan.rs * ((C + 31) / 32) * 3072 * kSlots, true, &g, &w);
    if (rc != MYEA_OK) return rc;
    hipLaunchKernelGGL(k->fn, dim3((unsigned)plan.grid), dim3((unsigned)(k->waves + 4) * 64u), forward_lds(k->waves, plan.rs), s, g, dir[0], dir[dirs > 1 ? 1 : 0], w);
    MYEA_HIP_TRY(hipGetLastError());
    return MYEA_OK;
}

size_t lstm_planes_sync_words() { return kSyncWords; }

int launch_lstm_planes_backward(hipStream_t s, const LstmPlanesPlan &plan, size_t T, size_t B, size_t Bmax, size_t C, int dirs, const LstmResidentDir *dir,
                                unsigned *sync, unsigned *host_flag, unsigned *fault, float *shares, size_t shares_floats)
{
    for (int q = 0; q < dirs; ++q)
        if (!dir[q].Wrec || !dir[q].peep || !dir[q].acts || !dir[q].c || !dir[q].ca || !dir[q].dh || !dir[q].dG || !dir[q].dc) { set_last_error("resident LSTM backward: null operand"); return MYEA_E_INVALID; }
    PlaneKernelInfo *k = backward_kernel(plan.members);
    if (!k) { set_last_error("resident LSTM backward: no kernel for %zu cells", C); return MYEA_E_UNSUPPORTED; }
    PlaneGeometry g;
    PlaneSync w;
    const int rc = prepare(s, plan, T, B, Bmax, C, dirs, sync, host_flag, fault, shares, shares_floats, (size_t)plan.rs * plan.members * plan.members * 1024 * 2, false, &g, &w);
    if (rc != MYEA_OK) return rc;
    hipLaunchKernelGGL(k->fn, dim3((unsigned)plan.grid), dim3((unsigned)(k->waves + 4) * 64u), backward_lds(plan.rs), s, g, dir[0], dir[dirs > 1 ? 1 : 0], w);
    MYEA_HIP_TRY(hipGetLastError());
    return MYEA_OK;
}

}  // namespace myea
