// Fused QKV projection for gfx950 (MI355X, CDNA4): the front end of the attention forward.
//
//   qkv[m][n] = sum_k x[m][k] w[k][n] (+ bias[n]),   m < M = B L,  n < N = 3 F,  F = R H
// written as the packed [B, L, 3, R H] tensor whose three slices fa_fwd_strided reads as q, k and v
// without a copy, with an optional rotary position encoding (rotate-half form) applied to the q and
// k slices before the one rounding to 16 bits.  The reference lists this front end as not done
// (reference README.md:137); its attention kernel takes q, k, v as three separate tensors
// (reference src/fused_attn_extention.cu:15-22).
//
// One kernel, one pass: a workgroup of eight wave64s owns a 256 x 256 tile of the output and walks
// the contraction in slices of 64.  The x and w slices are written into LDS by the loads themselves
// (direct-to-LDS loads: no staging registers, no LDS store instructions), into a ring of two
// 64 KB slots.  One load instruction of a wave fills 1 KB of consecutive LDS, lane l the 16 bytes
// at 16 l, and each lane is free to fetch any 16-byte chunk: the tiles stay row-major without
// padding, whole cache lines per wave on the global side, and the chunks of a row are permuted
// (XOR with a few bits of the row index) so that the operand reads touch every bank once:
//   x slot [256 rows][8 chunks]:  chunk c of row r sits at position c ^ ((r >> 1) & 7)
//          (16 consecutive rows of one logical chunk cover the 16 bank groups of 16 bytes);
//   w slot [64 rows][32 chunks]:  chunk c of contraction row k sits at c ^ (((k & 3) << 2) | (((k >> 3) & 1) << 1))
//          (the four rows a transpose read touches land in the four 64-byte quarters of the banks,
//          rows eight apart in different halves of a quarter).
// The products are computed transposed, C^T = W^T X^T, with v_mfma_f32_16x16x32_f16: the A operand
// W^T (16 outputs n x 32 k) comes from the row-major w slice through the LDS transpose read
// (ds_read_b64_tr_b16), the B operand X^T (32 k x 16 rows m) is a plain 16-byte read of a row of x.
// In the accumulator a lane then owns one output row m and, per 16 x 16 block, a run of four output
// features n: bias and rotation are applied in registers (the partner feature n + H/2 of a
// rotation sits in the same lane, or 32 lanes away at head_dim 16); the rounded rows then pass
// through a small per-wave LDS tile and leave as whole 256-byte row segments with streaming stores.
// The 16 x 16 x 32 instruction has the flops per clock of the 32 x 32 x 16 one with half the
// accumulator traffic per flop; on this chip, whose clock follows the switching activity, the
// same kernel written on 32 x 32 x 16 tiles measured 8.7 to 15 % slower on the same box.
//
// A wave owns 64 rows x 128 features (8 x 4 blocks of 16 x 16, 128 accumulator registers); its
// 128 features are whole heads for every head_dim up to 128.
#pragma once

#include "fused_attn_kernel.hpp"

namespace fa {
namespace qkv {

constexpr int kTileM = 256;
constexpr int kTileN = 256;
constexpr int kTileK = 64;    // contraction steps per slice (one ring slot)
constexpr int kWaves = 8;
constexpr int kBand = 4;      // row tiles per band of the tile order
constexpr int kSlots = 2;     // ring slots: one is read while the other is filled
constexpr int kRingHalves = kSlots * (kTileM + kTileN) * kTileK;                           // 128 KB
constexpr int kStageHalves = 16 * 128;      // per wave: 16 output rows of the wave's 128 features (4 KB)
constexpr int kLdsBytes = (kRingHalves + kWaves * kStageHalves) * (int)sizeof(_Float16);   // 160 KB

struct Params {
    const _Float16* x;       // [M, K]
    const _Float16* w;       // [K, N]
    const _Float16* bias;    // [N] or nullptr
    _Float16* out;           // [M, N]
    const float* rope_cos;   // [L, H / 2] or nullptr
    const float* rope_sin;
    int M, K, N;
    int F;                   // features per slice (N = 3 F)
    int L;                   // sequence length: position of row m is m % L
    int tiles_n;             // ceil(N / 256)
    int total_tiles;         // tiles_m * tiles_n
    int total_wgs;           // workgroups that take tiles: min(total_tiles, one per compute unit)
    int wgs_per_xcd;         // ceil(total_wgs / 8): the grid is 8 times this
    // small tiles: row tiles, and division by the tiles of a band, by the row tiles of the last band and by L
    int tiles_m;
    Divisor by_band, by_last, by_len;
};

__device__ __forceinline__ void dma16(uint32_t lds_addr, const void* base, uint32_t voff) {
    // M0 holds the LDS address of lane 0's 16 bytes.  Written in assembly so that the compiler
    // does not see an LDS write (it would wait for the load before the wave's next LDS read).
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :: "s"(lds_addr), "v"(voff), "s"(base) : "memory", "m0");
}
// ... and of lane 0's four bytes
__device__ __forceinline__ void dma4(uint32_t lds_addr, const void* base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :: "s"(lds_addr), "v"(voff), "s"(base) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }

template <int N>
using I = std::integral_constant<int, N>;

// HR = head_dim of the rotation (16, 32, 64, 128), or 0 for none.
template <int HR, bool BF>
__global__ __launch_bounds__(kWaves * 64, 2) void qkv_proj_kernel(const Params p) {
    constexpr int KS = kTileK;
    constexpr int NSLOT = kSlots;
    constexpr int CPRX = KS / 8;                        // 16-byte chunks per row of an x slot
    constexpr int LX = CPRX / 2;                        // x loads per wave and step
    constexpr int LW = KS / 16;                         // w loads per wave and step
    constexpr int XSLOT = kTileM * KS;                  // halves
    constexpr int WSLOT = KS * kTileN;
    constexpr int NSUB = KS / 32;                       // 32-wide contraction sub-steps per step
    extern __shared__ __attribute__((aligned(16))) _Float16 smem[];
    _Float16* const xs = smem;
    _Float16* const ws = smem + NSLOT * XSLOT;
    typedef short short8v __attribute__((ext_vector_type(8)));

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15;
    const int g4 = lane >> 4;
    const int wm = wave >> 1;
    const int wn = wave & 1;
    _Float16* const stage = smem + kRingHalves + wave * kStageHalves;     // this wave's output staging tile

    // A resident grid: workgroup `logical` takes the tiles logical, logical + G, logical + 2 G, ...
    // Workgroups are dealt round-robin to the XCDs, so they are renumbered first: one XCD (one L2)
    // then works on consecutive tiles, and the tiles are ordered in bands of four row tiles, feature
    // tile by feature tile inside a band: the 32 workgroups of an XCD cover about 4 x 8 tiles at a
    // time and share 4 row blocks of x and 8 column blocks of w in L2, instead of 1 and 32.
    const int wg = blockIdx.x;
    const int logical = (wg % kNumXcd) * p.wgs_per_xcd + wg / kNumXcd;
    if (logical >= p.total_wgs) return;
    const int tiles_m = p.total_tiles / p.tiles_n;
    auto tile_origin = [&](int tile, int& m0, int& n0) __attribute__((always_inline)) {
        const int band = tile / (kBand * p.tiles_n);
        const int in_band = tile - band * (kBand * p.tiles_n);
        const int band_rows = min(kBand, tiles_m - band * kBand);
        m0 = (band * kBand + in_band % band_rows) * kTileM;
        n0 = (in_band / band_rows) * kTileN;
    };

    // ---- the load stream -----------------------------------------------------------------------
    // Load instruction i of wave w fills the LDS positions (16-byte units) (w L + i) 64 + lane of a
    // slot; the lane fetches the chunk that belongs there: x position = row * 8 + (chunk ^ fx(row)),
    // w position = contraction row * 32 + (chunk ^ fw(row)).  Rows of x beyond M are read from row
    // M - 1 and feature chunks of w beyond N from chunk 0 (their results are never stored).  The
    // stream runs over all (tile, slice) pairs of the workgroup: the first slices of the next tile
    // are on their way while this one is finished.
    uint32_t xvo[LX], wvo[LW];
    const char* xsrc = nullptr;
    const char* wsrc = nullptr;
    int fetch_tile = logical, fetch_kt = 0;
    const int ksteps = p.K / KS;
    auto aim = [&]() __attribute__((always_inline)) {
        int m0, n0;
        tile_origin(fetch_tile, m0, n0);
#pragma unroll
        for (int i = 0; i < LX; ++i) {
            const int pos = (wave * LX + i) * 64 + lane;
            const int row = pos / CPRX;
            const int c = (pos % CPRX) ^ ((row >> 1) & 7);
            const int grow = min(m0 + row, p.M - 1) - m0;       // rows beyond M: never stored
            xvo[i] = ((uint32_t)grow * (uint32_t)p.K + (uint32_t)c * 8u) * 2u;
        }
#pragma unroll
        for (int i = 0; i < LW; ++i) {
            const int pos = (wave * LW + i) * 64 + lane;
            const int krow = pos >> 5;
            int c = (pos & 31) ^ (((krow & 3) << 2) | (((krow >> 3) & 1) << 1));
            if (n0 + c * 8 >= p.N) c = 0;                        // features beyond N: never stored
            wvo[i] = ((uint32_t)krow * (uint32_t)p.N + (uint32_t)c * 8u) * 2u;
        }
        xsrc = reinterpret_cast<const char*>(p.x + (int64_t)m0 * p.K);
        wsrc = reinterpret_cast<const char*>(p.w + n0);
    };
    const uint32_t xs_lds = (uint32_t)(uintptr_t)(FA_LDS void*)xs + (uint32_t)(wave * LX) * 1024u;
    const uint32_t ws_lds = (uint32_t)(uintptr_t)(FA_LDS void*)ws + (uint32_t)(wave * LW) * 1024u;
    // The LX + LW loads of a step are issued in two parts, one sub-step apart: 64 KB per step and
    // compute unit keep the texture path busy for half the step, and a wave that issues all its
    // loads at once waits at the issue port while the queue drains (measured: +3.5 % for two
    // parts; four parts, one per sub-step, lose that again because the last ones are issued too
    // late to land before the step ends).
    constexpr int NP = 2;
    constexpr int LPP = (LX + LW) / NP;              // loads per part
    static_assert((LX + LW) % NP == 0 && NP <= NSUB, "whole loads per part, at most one part per sub-step");
    auto issue_part = [&](int slot, auto part_c) __attribute__((always_inline)) {
        constexpr int PART = decltype(part_c)::value;
#pragma unroll
        for (int j = PART * LPP; j < (PART + 1) * LPP; ++j) {
            if (j < LX)
                dma16(xs_lds + (uint32_t)(slot * XSLOT * 2 + j * 1024), xsrc, xvo[j]);
            else
                dma16(ws_lds + (uint32_t)(slot * WSLOT * 2 + (j - LX) * 1024), wsrc, wvo[j - LX]);
        }
        if constexpr (PART == NP - 1) {
            xsrc += KS * 2;
            wsrc += (int64_t)KS * p.N * 2;
            if (++fetch_kt == ksteps) {
                fetch_kt = 0;
                fetch_tile += p.total_wgs;
                if (fetch_tile < p.total_tiles) aim();
            }
        }
    };
    auto issue = [&](int slot) __attribute__((always_inline)) {
        issue_part(slot, std::integral_constant<int, 0>{});
        issue_part(slot, std::integral_constant<int, 1>{});
    };

    // acc[nt][mt][r]: row m = m0 + wm 64 + mt 16 + c16, feature n = n0 + wn 128 + nt 16 + 4 g4 + r
    floatx4 acc[8][4];
    auto start_over = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < 8; ++nt)
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) acc[nt][mt] = floatx4{0.f, 0.f, 0.f, 0.f};
    };
    // The bias of a tile's features by a direct load into the wave's stage, which is idle until the tile ends: it has landed
    // with the first slice that is waited for, and takes no register meanwhile.
    auto request_bias = [&](int tile) __attribute__((always_inline)) {
        int m0, n0;
        tile_origin(tile, m0, n0);
        if (p.bias != nullptr) dma4((uint32_t)(uintptr_t)(FA_LDS void*)stage, p.bias, min(2u * (uint32_t)(n0 + wn * 128) + 4u * (uint32_t)lane, 2u * (uint32_t)p.N - 4u));
    };

    // ---- per-lane parts of the operand addresses (halves inside a slot) ---------------------------
    // B operand (x): row wm 64 + mt 16 + c16, logical chunk 4 s + g4 (k-slots 8 g4 ... of sub-step s are
    // contraction indices 32 s + 8 g4 ...).  The LDS serves the 16-byte reads of lanes 0-3, 12-15, 20-23
    // and 24-27 together (and 4-7, 8-11, 16-19, 28-31): with the chunk of row r at c ^ ((r >> 1) & 7)
    // and neighbouring chunks for g4 and g4 ^ 1 each such set of 16 lanes covers all banks once.
    int xrd[NSUB];
    {
        const int r0 = wm * 64 + c16;
        const int fx = (c16 >> 1) & 7;     // wm 64 and mt 16 do not reach these bits
#pragma unroll
        for (int s = 0; s < NSUB; ++s) xrd[s] = (r0 * CPRX + ((4 * s + g4) ^ fx)) * 8;
    }
    // A operand (w^T), transpose reads: lane s16 of the 16-lane group g4 points at contraction row
    // 32 s + 8 g4 + s16 / 4 (+ 4 for the second read), features 4 (s16 % 4) ... of the 16 of feature
    // block nt; lane j of the group receives four consecutive contraction rows of feature j, so the
    // two reads fill the k-slots 8 g4 ... 8 g4 + 7.  Chunk c of contraction row k sits at
    // c ^ (((k & 3) << 2) | (((k >> 3) & 1) << 1)): the four rows of a read land in the four 64-byte
    // quarters of the banks, and the rows of g4 and g4 ^ 1, eight apart, in different halves of a
    // quarter.  Feature block nt adds 2 nt to the chunk index, which commutes with that XOR: the
    // address of block nt is the address of block 0 XOR 16 nt (in halves).
    int wrd0;
    {
        const int kk = c16 >> 2;
        const int swz = (kk << 2) | ((g4 & 1) << 1);
        const int krow = 8 * g4 + kk;
        wrd0 = krow * kTileN + (wn * 16 + (swz | ((c16 & 3) >> 1))) * 8 + 4 * (c16 & 1);
    }

    // ---- end of a tile: bias, rotation, one rounding, whole-row stores; the accumulators start over ---
    // The rotation only reads the accumulators (results are formed in temporaries): done in place inside
    // the step loop it makes the compiler carry a second copy of all of them.
    auto finish_tile = [&](int done_tile) __attribute__((always_inline)) {
        int m0, n0;
        tile_origin(done_tile, m0, n0);
        const int nw = n0 + wn * 128;
        // What is read from memory, per 16-row block the distinct runs of the tables, is requested in one go ahead of its
        // use.  Requested where they are used, one wait behind the other, they and the bias took most of an
        // epilogue's time: M 16384 N 3072 K 1024 with tables 103.9 -> 92.5 us on the same box,
        // without them 90.3 -> 84.5, M 14400 N 768 K 256 17.5 -> 13.0; at K 5120 it is 1 %.
        // What is left of it is vector instructions, two waves' per SIMD, and the matrix core idle beside them.
        // The bias from LDS, widened once per run of features instead of once per row block, one decision per row block
        // instead of one per run whether it rotates (whose two sides met in register copies), and places in the stage one
        // XOR apart: with tables M 16384 N 3072 K 1024 92.7 -> 89.2 us, at head_dim 128 100.1 -> 93.8, M 8192 N 15360 K 5120
        // 943 -> 922, M 9000 N 4032 K 64 26.7 -> 24.2, M 8000 N 2304 K 768 41.2 -> 41.4; without tables 86.0 -> 85.5.
        constexpr int RUNS = HR == 0 ? 1 : HR <= 32 ? 1 : HR / 32;
        floatx4 cos4[RUNS], sin4[RUNS];
        const int at = HR > 0 ? m0 % p.L + wm * 64 + c16 : 0;
        auto request = [&](int mt) __attribute__((always_inline)) {
            if constexpr (HR > 0) {
                // position of the row in its sequence (rows beyond M: any)
                int pos = at + mt * 16;
                if (p.L < kTileM)
                    pos %= p.L;
                else
                    pos -= pos >= p.L ? p.L : 0;
#pragma unroll
                for (int i = 0; i < RUNS; ++i) {
                    const int64_t e = (int64_t)pos * (HR / 2) + (16 * i + 4 * g4) % (HR / 2);
                    cos4[i] = *reinterpret_cast<const floatx4*>(p.rope_cos + e);
                    sin4[i] = *reinterpret_cast<const floatx4*>(p.rope_sin + e);
                }
            }
        };
        request(0);
        // The bias comes last, on top of the finished sum and rounded once.  Accumulators that start at it round every
        // partial sum at its magnitude: M 4096 N 3840 K 5120 with a bias of 256, whose q and k a rotation by 45 degrees
        // brings back to 0.02, was 1.8e-4 (rms) off float64 that way and is 9.4e-6 off now, as on small tiles; one more matrix
        // instruction of bias times one, which does not round to nearest, 1.1e-5.
        if (p.bias != nullptr) {
            u16x4 bias4[8];
#pragma unroll
            for (int nt = 0; nt < 8; ++nt) bias4[nt] = *reinterpret_cast<const u16x4*>(stage + nt * 16 + 4 * g4);
            asm volatile("" ::: "memory");      // (the results pass through the same place)
#pragma unroll
            for (int nt = 0; nt < 8; ++nt) {
                floatx4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = BF ? bf16::elem_to_float(bias4[nt][e]) : elem_to_float(bias4[nt][e]);
#pragma unroll
                for (int mt = 0; mt < 4; ++mt) acc[nt][mt] += v;
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // The results leave through a private LDS tile of 16 rows x 128 features per wave, so that
        // every store instruction writes whole rows (16 lanes x 16 bytes = the wave's 256 bytes of a
        // row) as streaming stores.  A lane holds one row of a 16-row block and runs of four features;
        // chunk c (16 bytes) of stage row r sits at c ^ r, so that the run of feature block nt is the
        // first one's place XOR 32 nt bytes.
        const uint32_t stage0 = (uint32_t)(uintptr_t)(FA_LDS void*)stage;
        uint32_t place = stage0 + (uint32_t)(c16 * 256 + ((g4 >> 1) ^ c16) * 16 + 8 * (g4 & 1));
        auto store_run = [&](floatx4 v, int nt) __attribute__((always_inline)) {
            u16x4 hv;
#pragma unroll
            for (int e = 0; e < 4; ++e) hv[e] = BF ? bf16::float_to_elem(v[e]) : float_to_elem(v[e]);
            *(FA_LDS u32x2*)(uintptr_t)(place ^ (32u * nt)) = __builtin_bit_cast(u32x2, hv);
        };
        // (2 F is a multiple of 128: a wave's features are all of q and k, or all of v)
        const bool rotated = nw < 2 * p.F;
        const int l4 = lane >> 4, ch = lane & 15, n_out = nw + ch * 8;
        const uint32_t out_off = (uint32_t)l4 * (uint32_t)p.N * 2u + (uint32_t)ch * 16u;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            // (opaque, so that the places of all runs are not worked out ahead and held through the whole epilogue)
            asm volatile("" : "+v"(place));
            if (HR >= 32 && rotated) {
                // rotate-half: within a head, feature i < HR / 2 pairs with feature i + HR / 2:
                //   out[i] = y[i] cos_i - y[i + HR/2] sin_i,  out[i + HR/2] = y[i + HR/2] cos_i + y[i] sin_i
                // with cos_i, sin_i taken at the row's position.  Only the q and k slices (n < 2 F).  The
                // partner run sits in the same lane, HR / 32 feature blocks on.
                constexpr int D = HR >= 32 ? HR / 32 : 1;
#pragma unroll
                for (int pr = 0; pr < 4; ++pr) {
                    const int nt_a = (pr / D) * 2 * D + pr % D, nt_b = nt_a + D;
                    const floatx4 a = acc[nt_a][mt], b = acc[nt_b][mt], c4 = cos4[pr % D], s4 = sin4[pr % D];
                    store_run(a * c4 - b * s4, nt_a);
                    store_run(b * c4 + a * s4, nt_b);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else if (HR == 16 && rotated) {
                // head_dim 16: a head is one feature block and the partner of a run sits 32 lanes away
#pragma unroll
                for (int nt = 0; nt < 8; ++nt) {
                    const floatx4 a = acc[nt][mt];
                    floatx4 b;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float ae = a[e];      // (a bit cast taken straight from a vector element reads element 0)
                        b[e] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __builtin_bit_cast(int, ae)));
                    }
                    store_run(g4 < 2 ? a * cos4[0] - b * sin4[0] : a * cos4[0] + b * sin4[0], nt);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int nt = 0; nt < 8; ++nt) store_run(acc[nt][mt], nt);
            }
            if (mt < 3) request(mt + 1);
            // LDS operations of one wave complete in order; the waits keep the compiler from moving
            // the reads above the writes (and the next block's writes above these reads)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 4 * i + l4, row0 = m0 + wm * 64 + mt * 16 + 4 * i;
                const u32x4 w = *(FA_LDS const u32x4*)(uintptr_t)(stage0 + (uint32_t)(r * 256 + (ch ^ r) * 16));
                char* const out = reinterpret_cast<char*>(p.out + (int64_t)row0 * p.N + nw);
                if (row0 + l4 < p.M && n_out < p.N) __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(out + out_off));
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        if (done_tile + p.total_wgs < p.total_tiles) request_bias(done_tile + p.total_wgs);
        start_over();
    };

    const int my_tiles = (p.total_tiles - logical + p.total_wgs - 1) / p.total_wgs;
    const int total_steps = my_tiles * ksteps;
    int tile = logical, kt = 0;

    // Operand registers.  B (rows of x): the four fragments of a 32-wide sub-step, two sets.  A (w^T): the
    // eight fragments of a sub-step are used pair by pair (one unit = 2 A fragments x 4 B fragments = 8
    // matrix instructions), two pairs of registers: the reads of a pair are issued before the matrix
    // instructions of the pair before it, the B fragments of the next sub-step two units ahead.
    half8 wop[2][2], xop[2][4];
    auto load_a = [&](auto set_c, int slot, auto s_c, auto pair_c) __attribute__((always_inline)) {
        constexpr int SET = decltype(set_c)::value;
        constexpr int S = decltype(s_c)::value;
        constexpr int PAIR = decltype(pair_c)::value;
        const _Float16* const wb = ws + slot * WSLOT;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const _Float16* p0 = wb + (wrd0 ^ (16 * (2 * PAIR + e))) + (32 * S) * kTileN;
            const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FA_LDS short4v*)(p0));
            const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FA_LDS short4v*)(p0 + 4 * kTileN));
            const short8v both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            wop[SET][e] = __builtin_bit_cast(half8, both);
        }
    };
    auto load_b = [&](auto set_c, int slot, auto s_c) __attribute__((always_inline)) {
        constexpr int SET = decltype(set_c)::value;
        constexpr int S = decltype(s_c)::value;
        const _Float16* const xb = xs + slot * XSLOT;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt)
            xop[SET][mt] = *reinterpret_cast<const half8*>(xb + xrd[S] + mt * 16 * CPRX * 8);
    };
    auto multiply = [&](auto aset_c, auto bset_c, auto pair_c) __attribute__((always_inline)) {
        constexpr int ASET = decltype(aset_c)::value;
        constexpr int BSET = decltype(bset_c)::value;
        constexpr int PAIR = decltype(pair_c)::value;
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                if constexpr (BF)
                    acc[2 * PAIR + e][mt] = bf16::mfma16(wop[ASET][e], xop[BSET][mt], acc[2 * PAIR + e][mt]);
                else
                    acc[2 * PAIR + e][mt] = mfma16(wop[ASET][e], xop[BSET][mt], acc[2 * PAIR + e][mt]);
            }
    };

    // Step u reads slot u % 2 while the loads of step u + 1 fill the other one.  One barrier per
    // step, placed before the matrix instructions of the step's last unit: by then every wave has
    // the operands of that unit in registers, so the slot is free for the loads of step u + 2, and
    // the data of step u + 1 (each wave has waited for its own part) are visible to everybody, so
    // the operands of its first unit are requested before the last matrix instructions of step u
    // are issued.
    static_assert(NSLOT == 2, "the waits below assume that only the next step's loads are in flight");
    static_assert(NSUB == 2, "eight units per step");
    request_bias(logical);      // (loads complete in order: landed with the first slice)
    aim();
    issue(0);
    if (total_steps > 1) {
        issue(1);
        wait_loads<LX + LW>();      // loads complete in order: all but the second step's have landed
    } else {
        wait_loads<0>();
    }
    start_over();
    ring_barrier();
    load_a(I<0>{}, 0, I<0>{}, I<0>{});
    load_b(I<0>{}, 0, I<0>{});

    bool pending = false;      // the second part of the loads into the previous step's slot is still to be issued
    auto step = [&](int u, auto slot_c) __attribute__((always_inline)) {
        constexpr int SLOT = decltype(slot_c)::value;
        constexpr int PREV = (SLOT + NSLOT - 1) % NSLOT;
        // unit t (sub-step t / 4, fragment pair t % 4) uses A set t % 2 and B set (t / 4) % 2
        auto unit = [&](auto t_c) __attribute__((always_inline)) {
            constexpr int T = decltype(t_c)::value;
            load_a(I<(T + 1) & 1>{}, SLOT, I<(T + 1) / 4>{}, I<(T + 1) % 4>{});
            if constexpr (T == 1) load_b(I<1>{}, SLOT, I<1>{});
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (T == 1) {
                if (pending) issue_part(PREV, I<1>{});
            }
            multiply(I<T & 1>{}, I<(T / 4) & 1>{}, I<T % 4>{});
            __builtin_amdgcn_sched_barrier(0);
        };
        unit(I<0>{});
        unit(I<1>{});
        unit(I<2>{});
        unit(I<3>{});
        unit(I<4>{});
        unit(I<5>{});
        unit(I<6>{});
        // this wave's loads of step u + 1 have landed (the stores of an epilogue are waited for
        // with them), its reads of this step's slot have all returned
        wait_loads<0>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        ring_barrier();
        pending = u + NSLOT < total_steps;
        if (pending) issue_part(SLOT, I<0>{});
        // (at the end of a tile the operands of the next step are requested behind the epilogue, which
        // needs the registers)
        const bool last = kt + 1 == ksteps;
        if (u + 1 < total_steps && !last) {
            load_a(I<0>{}, (SLOT + 1) % NSLOT, I<0>{}, I<0>{});
            load_b(I<0>{}, (SLOT + 1) % NSLOT, I<0>{});
        }
        __builtin_amdgcn_sched_barrier(0);
        multiply(I<1>{}, I<1>{}, I<3>{});
        __builtin_amdgcn_sched_barrier(0);
        if (last) {
            finish_tile(tile);
            kt = 0;
            tile += p.total_wgs;
            __builtin_amdgcn_sched_barrier(0);
            if (u + 1 < total_steps) {
                load_a(I<0>{}, (SLOT + 1) % NSLOT, I<0>{}, I<0>{});
                load_b(I<0>{}, (SLOT + 1) % NSLOT, I<0>{});
            }
        } else {
            ++kt;
        }
    };
    for (int u = 0; u < total_steps; u += NSLOT) {
        step(u, I<0>{});
        if (u + 1 < total_steps) step(u + 1, I<1>{});
    }
}

// ---------------------------------------------------------------------------------------------
// Small-tile kernel: outputs that 256 x 256 tiles do not spread over the chip.
//
// Eight waves as KG contraction groups of WM x WN waves; a wave owns 16 MT rows x 16 NT features, a group the whole
// (16 MT WM) x (16 NT WN) tile, and with KG = 2 each group takes one 32-wide half of every slice: the
// wave tiles, and with them the products per byte read from LDS, are then twice as large as with eight waves
// side by side.  Slices of 64 in a ring of SLOTS slots, one barrier per slice, one tile per workgroup.  The
// slot layouts, the transposed product and the epilogue are those of the kernel above; w slots of 64
// features have half as many chunks per row, and the row's lowest bit selects the half of the banks itself.
//
// What bounds it: a 256 x 256 tile takes 1.3 to 1.5 us per slice of one compute unit, however many of them have
// one; a 128 x 256 tile takes 0.65 us, a 128 x 128 one 0.45, 64 x 128 (two per unit) 0.35 and 64 x 64 0.25, a
// mix of the 32 to 58 bytes per clock the direct loads deliver, the products and the barrier.  Same box,
// 256 x 256 tiles before, the shape that is picked now: M 512 N 15360 K 5120 113 -> 66 us, M 64 N 7680
// K 5120 101 -> 23, M 256 N 7680 K 2560 62 -> 18, M 2048 N 3072 K 1024 35 -> 20, M 128 N 1536 K 1024
// 30 -> 6.1 (geometric mean over 220 random shapes: 1.95x).  Rings of eight and six slots for the two
// smallest shapes, one workgroup per unit, were up to 1.9 times slower than two workgroups with short rings.
//
// The 16-feature blocks of a head are walked in an order that puts the two halves of a rotary pair next to
// each other (0, HR/32, 1, HR/32 + 1, ...): a wave with any even number of blocks has whole pairs, and a tile
// of 64 features may be half a head.
template <int MT, int NT, int WM, int WN, int KG, int SLOTS>
struct SmallTile {
    static_assert(WM * WN * KG == kWaves && (KG == 1 || (KG == 2 && MT % 2 == 0)) && NT % 2 == 0);
    static constexpr int TM = 16 * MT * WM, TN = 16 * NT * WN;
    static constexpr int XSLOT = TM * kTileK, WSLOT = kTileK * TN;       // halves
    static constexpr int LX = TM / 64, LW = TN / 64;                     // loads per wave and slice
    static constexpr int RING = SLOTS * (XSLOT + WSLOT) * 2;             // bytes
    static constexpr int OWN = MT / KG;                                  // 16-row blocks a wave finishes
    static constexpr int PART = KG == 1 ? 0 : kWaves * OWN * NT * 1024;  // accumulators handed over
    static constexpr int STAGE = kWaves * 16 * 16 * NT * 2;
    static constexpr int LDS = RING > PART + STAGE ? RING : PART + STAGE;
    static_assert(LDS <= 160 * 1024);
};

template <class F, int... J>
__device__ __forceinline__ void for_each_index(F f, std::integer_sequence<int, J...>) { (f(I<J>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void for_each_index(F f) { for_each_index(f, std::make_integer_sequence<int, N>{}); }

// Waits until at most min(left, MOST) slices of LOADS loads each are still under way.
template <int LOADS, int MOST>
__device__ __forceinline__ void wait_slices(int left) {
    if constexpr (MOST > 0) {
        if (left < MOST) return wait_slices<LOADS, MOST - 1>(left);
    }
    wait_loads<LOADS * MOST>();
}

template <int HR, bool BF, int MT, int NT, int WM, int WN, int KG, int SLOTS>
__global__ __launch_bounds__(kWaves * 64, MT * NT < 16 ? 4 : 2) void qkv_proj_small_kernel(const Params p) {
    using T = SmallTile<MT, NT, WM, WN, KG, SLOTS>;
    constexpr int TM = T::TM, TN = T::TN, LX = T::LX, LW = T::LW;
    constexpr int CPRX = kTileK / 8, CPRW = TN / 8;       // 16-byte chunks per row of a slot
    extern __shared__ __attribute__((aligned(16))) _Float16 smem[];
    typedef short short8v __attribute__((ext_vector_type(8)));

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15;
    const int g4 = lane >> 4;
    const int kg = wave / (WM * WN);
    const int wm = wave % (WM * WN) / WN;
    const int wn = wave % WN;

    const int wg = blockIdx.x;
    const int logical = (wg % kNumXcd) * p.wgs_per_xcd + wg / kNumXcd;
    if (logical >= p.total_wgs) return;
    // bands of 1024 rows, feature tile by feature tile inside a band, as above
    constexpr int BAND = kBand * kTileM / TM;
    const int band = p.by_band.of(logical);
    const int in_band = logical - band * (BAND * p.tiles_n);
    const int left = p.tiles_m - band * BAND, band_rows = min(BAND, left);
    const int col = left < BAND ? p.by_last.of(in_band) : in_band / BAND;
    const int m0 = (band * BAND + in_band - col * band_rows) * TM;
    const int n0 = col * TN;

    // first feature of the block at place b of the order described above
    auto feature_of = [](int b) __attribute__((always_inline)) {
        if constexpr (HR >= 64) {
            constexpr int HB = HR / 16;
            return 16 * (b / HB * HB + (b % HB >> 1) + (b & 1) * (HB / 2));
        }
        return 16 * b;
    };
    // place of chunk c of contraction row k in a w slot, less c
    auto w_swizzle = [](int k) __attribute__((always_inline)) {
        return CPRW >= 16 ? ((k & 3) << 2) | (((k >> 3) & 1) << 1) : (k & 2) << 1 | (((k >> 3) & 1) << 1);
    };

    // What the end of the tile needs from memory, a run's bias and the distinct runs of the tables for every row,
    // is requested in one go and waits in registers: requested where it is used, one load behind the
    // other, it made the end of a 128 x 256 tile take 10 us, as long as a dozen slices.
    constexpr int OWN = T::OWN;
    constexpr int RUNS = HR == 0 ? 0 : HR <= 32 ? 1 : NT / 2;
    const int b0 = n0 / 16 + wn * NT;
    u16x4 bias4[NT];
    floatx4 cos4[OWN][RUNS > 0 ? RUNS : 1], sin4[OWN][RUNS > 0 ? RUNS : 1];
    auto request = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int n = feature_of(b0 + nt) + 4 * g4;
            bias4[nt] = p.bias != nullptr && n < p.N ? *reinterpret_cast<const u16x4*>(p.bias + n) : u16x4{0, 0, 0, 0};
        }
        if constexpr (HR > 0) {
            const int at = m0 - p.by_len.of(m0) * p.L + 16 * (wm * MT + kg * OWN) + c16;
#pragma unroll
            for (int mt = 0; mt < OWN; ++mt) {
                // (rows beyond M: any row of the tables)
                int pos = at + 16 * mt;
                if (p.L < TM)
                    pos -= p.by_len.of(pos) * p.L;
                else
                    pos -= pos >= p.L ? p.L : 0;
#pragma unroll
                for (int i = 0; i < RUNS; ++i) {
                    const int64_t e = (int64_t)pos * (HR / 2) + (feature_of(b0 + 2 * i) + 4 * g4) % (HR / 2);
                    cos4[mt][i] = *reinterpret_cast<const floatx4*>(p.rope_cos + e);
                    sin4[mt][i] = *reinterpret_cast<const floatx4*>(p.rope_sin + e);
                }
            }
        }
    };
    uint32_t xvo[LX], wvo[LW];
#pragma unroll
    for (int i = 0; i < LX; ++i) {
        const int pos = (wave * LX + i) * 64 + lane;
        const int row = pos / CPRX;
        const int c = (pos % CPRX) ^ ((row >> 1) & 7);
        const int grow = min(m0 + row, p.M - 1) - m0;       // rows beyond M: never stored
        xvo[i] = ((uint32_t)grow * (uint32_t)p.K + (uint32_t)c * 8u) * 2u;
    }
#pragma unroll
    for (int i = 0; i < LW; ++i) {
        const int pos = (wave * LW + i) * 64 + lane;
        const int krow = pos / CPRW;
        const int c = (pos % CPRW) ^ w_swizzle(krow);
        int n = feature_of(n0 / 16 + (c >> 1)) + 8 * (c & 1);
        if (n >= p.N) n = 0;                                // features beyond N: never stored
        wvo[i] = ((uint32_t)krow * (uint32_t)p.N + (uint32_t)n) * 2u;
    }
    const char* xsrc = reinterpret_cast<const char*>(p.x + (int64_t)m0 * p.K);
    const char* wsrc = reinterpret_cast<const char*>(p.w);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(FA_LDS void*)smem;
    const uint32_t xs_lds = lds0 + (uint32_t)(wave * LX) * 1024u;
    const uint32_t ws_lds = lds0 + (uint32_t)(SLOTS * T::XSLOT * 2 + wave * LW * 1024);
    constexpr int LOADS = LX + LW;
    auto issue_one = [&](int slot, auto i_c) __attribute__((always_inline)) {
        constexpr int J = decltype(i_c)::value;
        if constexpr (J < LX)
            dma16(xs_lds + (uint32_t)(slot * T::XSLOT * 2 + J * 1024), xsrc, xvo[J]);
        else
            dma16(ws_lds + (uint32_t)(slot * T::WSLOT * 2 + (J - LX) * 1024), wsrc, wvo[J - LX]);
        if constexpr (J == LOADS - 1) {
            xsrc += kTileK * 2;
            wsrc += (int64_t)kTileK * p.N * 2;
        }
    };
    // loads FIRST ... END - 1 of a slice
    auto issue = [&](int slot, auto first_c, auto end_c) __attribute__((always_inline)) {
        constexpr int FIRST = decltype(first_c)::value;
        constexpr int COUNT = decltype(end_c)::value - FIRST;
        for_each_index<COUNT>([&](auto j_c) __attribute__((always_inline)) { issue_one(slot, I<FIRST + decltype(j_c)::value>{}); });
    };
    const int ksteps = p.K / kTileK;
    constexpr bool PIPE = KG == 1;
    for (int u = 0; u < min(PIPE ? SLOTS : SLOTS - 1, ksteps); ++u) issue(u, I<0>{}, I<LOADS>{});

    // acc[nt][mt][r]: row 16 (wm MT + mt) + c16 of the tile, feature 4 g4 + r of block wn NT + nt
    floatx4 acc[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = floatx4{0.f, 0.f, 0.f, 0.f};

    constexpr int NSUB = 2 / KG;       // 32-wide halves of a slice per group
    int xrd[NSUB];
#pragma unroll
    for (int s = 0; s < NSUB; ++s)
        xrd[s] = ((wm * MT * 16 + c16) * CPRX + ((4 * (s + kg) + g4) ^ ((c16 >> 1) & 7))) * 8;
    const int krow = 8 * g4 + (c16 >> 2);
    const int wrd0 = SLOTS * T::XSLOT + (32 * kg + krow) * TN + ((wn * 2 * NT + ((c16 & 3) >> 1)) ^ w_swizzle(krow)) * 8 + 4 * (c16 & 1);

    // Operands of a half slice.  Where a wave multiplies both halves, in two sets: those of the next half are
    // requested before the matrix instructions of this one.
    half8 xop[PIPE ? 2 : 1][MT], wop[PIPE ? 2 : 1][NT];
    auto load = [&](auto set_c, int slot, auto s_c) __attribute__((always_inline)) {
        constexpr int SET = decltype(set_c)::value;
        constexpr int S = decltype(s_c)::value;
        const _Float16* const xb = smem + slot * T::XSLOT;
        const _Float16* const wb = smem + slot * T::WSLOT;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) xop[SET][mt] = *reinterpret_cast<const half8*>(xb + xrd[S] + mt * 16 * kTileK);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const _Float16* const at = wb + (wrd0 ^ (16 * nt)) + 32 * S * TN;
            const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FA_LDS short4v*)(at));
            const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FA_LDS short4v*)(at + 4 * TN));
            const short8v both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            wop[SET][nt] = __builtin_bit_cast(half8, both);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // The loads into a slot go out one by one between the matrix instructions of a whole slice: a wave that
    // issues them all at once waits at the issue port while the queue drains, its matrix core idle.
    // HALF: 0 behind a barrier, 1 before the next one (if there is anything between).
    constexpr int GROUPS = NSUB * NT;
    auto multiply = [&](auto set_c, auto half_c, bool filling, auto fill_slot) __attribute__((always_inline)) {
        constexpr int SET = decltype(set_c)::value;
        constexpr int HALF = decltype(half_c)::value;
        auto group = [&](auto nt_c) __attribute__((always_inline)) {
            constexpr int nt = decltype(nt_c)::value;
            constexpr int GROUP = HALF * NT + nt;
            constexpr int FIRST = GROUP * LOADS / GROUPS, END = (GROUP + 1) * LOADS / GROUPS;
            if constexpr (END > FIRST) {
                if (filling) issue(fill_slot, I<FIRST>{}, I<END>{});
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                if constexpr (BF)
                    acc[nt][mt] = bf16::mfma16(wop[SET][nt], xop[SET][mt], acc[nt][mt]);
                else
                    acc[nt][mt] = mfma16(wop[SET][nt], xop[SET][mt], acc[nt][mt]);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        for_each_index<NT>(group);
    };

    // Rounds of the ring in which every load has a slice to fetch, with the slots known at compile time and no
    // decision in them (a wave issues an instruction every four or five clocks at best, and addresses and
    // branches took as long as the products), the rest one by one.  No more copies of a slice than
    // that: a short launch waits for its instructions, too.
    // step(slots of slices u, u + 1 and u - 1, whether slices u - 1 + AHEAD and u + AHEAD exist, slices behind the
    // one awaited)
    auto ring = [&](auto step) __attribute__((always_inline)) {
        constexpr int AHEAD = PIPE ? SLOTS : SLOTS - 1;        // the loads of slice u + AHEAD follow the barrier of slice u
        int u = 0;
        for (; u + SLOTS + AHEAD <= ksteps; u += SLOTS)
            for_each_index<SLOTS>([&](auto s_c) __attribute__((always_inline)) {
                constexpr int S = decltype(s_c)::value;
                step(s_c, I<(S + 1) % SLOTS>{}, I<(S + SLOTS - 1) % SLOTS>{}, S > 0 || u > 0, true, SLOTS);
            });
        for (int slot = 0; u < ksteps; ++u) {
            const int next = slot + 1 == SLOTS ? 0 : slot + 1, before = slot == 0 ? SLOTS - 1 : slot - 1;
            step(slot, next, before, u > 0 && u - 1 + AHEAD < ksteps, u + AHEAD < ksteps, ksteps - (PIPE ? 2 : 1) - u);
            slot = next;
        }
    };
    if constexpr (PIPE) {
        wait_slices<LOADS, SLOTS - 1>(ksteps - 1);
        ring_barrier();
        load(I<0>{}, I<0>{}, I<0>{});
        ring([&](auto slot, auto next, auto before, bool late, bool filling, int left) __attribute__((always_inline)) {
            load(I<1>{}, slot, I<1>{});
            multiply(I<0>{}, I<1>{}, late, before);
            // The operands of the slice's second half are in registers and this wave's loads of the next slice have
            // landed; behind the barrier that holds for everybody: the next slice may be read, and this
            // one's slot filled.
            wait_slices<LOADS, SLOTS - 2>(left);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            ring_barrier();
            // (behind the last slice: a slot that nobody uses any more, into registers that nobody uses)
            load(I<0>{}, next, I<0>{});
            multiply(I<1>{}, I<0>{}, filling, slot);
        });
    } else {
        ring([&](auto slot, auto, auto before, bool, bool filling, int left) __attribute__((always_inline)) {
            // This wave's loads of the slice have landed; behind the barrier everybody's have, and the slice before
            // has been read by all: its slot may be filled.
            wait_slices<LOADS, SLOTS - 2>(left);
            ring_barrier();
            load(I<0>{}, slot, I<0>{});
            multiply(I<0>{}, I<0>{}, filling, before);
            // (the reads of the slice have all returned: their results went into matrix instructions)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        });
    }
    request();
    __syncthreads();       // the ring is idle from here on

    // two groups: each finishes half of its rows and hands the sums of the other half over
    floatx4 own[NT][OWN];
    if constexpr (KG == 1) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < OWN; ++mt) own[nt][mt] = acc[nt][mt];
    } else {
        float* const part = reinterpret_cast<float*>(smem) + lane * 4;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < OWN; ++mt) {
                *reinterpret_cast<floatx4*>(part + ((wave * OWN + mt) * NT + nt) * 256) = kg == 0 ? acc[nt][mt + OWN] : acc[nt][mt];
                own[nt][mt] = kg == 0 ? acc[nt][mt] : acc[nt][mt + OWN];
            }
        __syncthreads();
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < OWN; ++mt)
                own[nt][mt] += *reinterpret_cast<const floatx4*>(part + (((wave ^ (WM * WN)) * OWN + mt) * NT + nt) * 256);
    }

    // bias, rotation, one rounding; whole rows leave through a private LDS tile of 16 rows (see above)
    _Float16* const stage = smem + T::PART / 2 + wave * (256 * NT);
    auto biased = [&](int nt, int mt) __attribute__((always_inline)) {
        floatx4 v = own[nt][mt];
        if (p.bias != nullptr) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += BF ? bf16::elem_to_float(bias4[nt][e]) : elem_to_float(bias4[nt][e]);
        }
        return v;
    };
    auto store_run = [&](floatx4 v, int nt) __attribute__((always_inline)) {
        u16x4 hv;
#pragma unroll
        for (int e = 0; e < 4; ++e) hv[e] = BF ? bf16::float_to_elem(v[e]) : float_to_elem(v[e]);
        *reinterpret_cast<u32x2*>(stage + c16 * (16 * NT) + ((2 * nt + (g4 >> 1)) ^ (c16 & (2 * NT - 1))) * 8 + 4 * (g4 & 1)) = __builtin_bit_cast(u32x2, hv);
    };
#pragma unroll
    for (int mt = 0; mt < OWN; ++mt) {
        const int mb = m0 + 16 * (wm * MT + kg * OWN + mt);
        if constexpr (HR >= 32) {
#pragma unroll
            for (int nt = 0; nt < NT; nt += 2) {
                floatx4 a = biased(nt, mt);
                floatx4 b = biased(nt + 1, mt);
                if (feature_of(b0 + nt) < 2 * p.F) {
                    const floatx4 c4 = cos4[mt][nt / 2 % RUNS], s4 = sin4[mt][nt / 2 % RUNS];
                    const floatx4 ra = a * c4 - b * s4;
                    const floatx4 rb = b * c4 + a * s4;
                    a = ra;
                    b = rb;
                }
                store_run(a, nt);
                store_run(b, nt + 1);
            }
        } else {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                floatx4 a = biased(nt, mt);
                if constexpr (HR == 16) {
                    // a head is one block and the partner of a run sits 32 lanes away
                    floatx4 b;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float ae = a[e];
                        b[e] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __builtin_bit_cast(int, ae)));
                    }
                    if (16 * (b0 + nt) < 2 * p.F) a = g4 < 2 ? a * cos4[mt][0] - b * sin4[mt][0] : a * cos4[mt][0] + b * sin4[mt][0];
                }
                store_run(a, nt);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < NT / 2; ++i) {
            const int r = i * (32 / NT) + lane / (2 * NT), ch = lane % (2 * NT);
            const u32x4 w = *reinterpret_cast<const u32x4*>(stage + r * (16 * NT) + (ch ^ (r & (2 * NT - 1))) * 8);
            const int n = feature_of(b0 + (ch >> 1)) + 8 * (ch & 1);
            if (mb + r < p.M && n < p.N)
                __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(p.out + (int64_t)(mb + r) * p.N + n));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
}

}  // namespace qkv
}  // namespace fa
