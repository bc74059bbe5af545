// Fused multi-head attention forward for gfx950 (MI355X, CDNA4).
//
// One kernel computes O = softmax(Q K^T * scale) V per (batch, head) without ever
// writing the L x L score matrix to memory.  It replaces, as a single pass, the
// reference's attention_kernel and every threadblock_* helper it calls
// (reference include/fused_attn.cuh:48-538 and :605-858).
//
// Five kernels share the pieces in this file:
//   fwd_kernel_split     (fused_attn_split.inc) waves of a workgroup share out the keys of 16 query rows:
//                        small grids
//   fwd_kernel_group     (fused_attn_split.inc) eight waves that share key tiles in LDS and run free between
//                        one barrier per tile: in-between grids, and large ones the next two
//                        would fill badly
//   fwd_kernel_pingpong  (fused_attn_kernel_impl.inc) eight waves in two groups that alternate vector and
//                        matrix phases, 32 x 32 matrix tiles
//   fwd_kernel_pp16      (fused_attn_kernel_impl.inc) the same phases, 16 x 16 matrix tiles
//   (qkv_proj_kernel     qkv_proj_kernel.hpp: the projection in front of them)
// all of them streaming K and V through LDS in tiles and computing, per 32 keys,
//   S^T = K_sub * Q^T        v_mfma_f32_*_{f16,bf16}, Q held in registers
//   online softmax on S^T    f32
//   O^T += V_sub^T * P^T     V^T fetched with ds_read_b64_tr_b16
//
// Why the transposed products: in the 32x32 accumulator layout lane l owns column
// (l % 32) -- one query -- and 16 of the 32 rows (keys); lane l^32 owns the other 16.
// A softmax row therefore lives in one lane pair, so row max / row sum need 15 in-lane
// ops and a single v_permlane32_swap.  The packed 16-bit P^T registers are, as they stand,
// a valid B operand of the second product provided the A operand (V^T) enumerates keys
// in the same order, which the transpose-read from the V tile provides.
//
// MFMA operand maps of fwd_kernel_pingpong (g = lane / 32, ln = lane % 32; fwd_kernel_pp16 gives the 16 x 16 ones):
//   A (32 x 16): lane holds row ln,   k = 8 g + i          (i = 0..7)
//   B (16 x 32): lane holds col ln,   k = 8 g + i
//   C (32 x 32): lane holds col ln,   row = 8 (r / 4) + 4 g + r % 4   (r = 0..15)
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fa {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));    // at any 16-bit element
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));

#define FA_LDS __attribute__((address_space(3)))

// Division of numbers below 2^31 by d <= 2^31 - 1: the high half of n * mul, shifted (mul = 0: d is 1).  mul is
// floor(2^(31 + s) / d) + 1 with s = ceil(log2 d), which exceeds 2^(31 + s) / d by at most 1 <= 2^s / d, so that
// n * mul / 2^(31 + s) exceeds n / d by at most n / (2^31 d) < 1 / d and has the same whole part.  (It fits 32 bits: d is
// above 2^(s - 1), hence 2^(31 + s) / d below 2^32 by at least 2^32 / d > 2.)
struct Divisor {
    uint32_t mul;
    uint32_t shift;
    __device__ __forceinline__ int of(int n) const { return mul == 0 ? n : (int)(__umulhi((uint32_t)n, mul) >> shift); }
};

inline Divisor divisor(int64_t d) {
    if (d <= 1) return {0, 0};
    uint32_t s = 0;
    while (((int64_t)1 << s) < d) ++s;
    return {(uint32_t)(((uint64_t)1 << (31 + s)) / (uint64_t)d + 1), s - 1};
}

struct FwdParams {
    const _Float16* q;
    const _Float16* k;
    const _Float16* v;
    const _Float16* mask;  // additive [B, L, L] or nullptr
    _Float16* o;
    float* lse;            // optional [B, R, L] natural-log row sums of exp(scores), or nullptr
    int64_t stride_b;      // q, k, v: elements between batches
    int64_t stride_h;      // ... between heads
    int64_t stride_l;      // ... between sequence positions
    int64_t ostride_b;     // the same three for o
    int64_t ostride_h;
    int64_t ostride_l;
    int B, R, L;
    int n_qtiles;          // workgroups per (batch, head): ceil(L / queries per workgroup), or half of
                           // that (rounded up) when a causal workgroup takes a pair of query tiles
    int total_wgs;         // B * R * n_qtiles
    int wgs_per_xcd;       // ceil(total_wgs / 8)
    int heads_per_xcd;     // causal eight-wave launches: 0 = every workgroup takes the pair of query tiles
                           // (t, n - 1 - t) of one head; > 0 = resident grid, the heads of an XCD's
                           // workgroups (B * R / 8 of them) dealt out tile by tile, see the kernel
    int waves;             // key-split kernel: waves per workgroup
    float scale_log2e;     // scale * log2(e)
    float bias;            // bias of the reference of the exponentials, log2 units (see kBiasMin)
};

// The split and group kernels', apart from the tile kernels': fields added to those changed the compiler's order of the tile
// kernels' instructions, B1 R32 L16384 H128 +1.1 % and B4 R16 L4096 H64 +1.6 % of the time; behind what they read, with
// the same instructions, the second of these stayed (256.9 -> 261.0 us); apart, 253.9 and 254.3.
struct SplitParams : FwdParams {
    Divisor by_qtiles;     // division by n_qtiles and by R
    Divisor by_heads;
    // what a score may be above the reference, in raw scores (the limit of one probability in fp16, and in bf16 what
    // keeps the sum of 32 of them below kTripSum), and log2(e) / scale_log2e
    float leash, mask_scale;
};

constexpr int kNumXcd = 8;

// Kernel variants.
constexpr int kPlain = 0;    // no mask
constexpr int kAdditive = 1; // additive [B, L, L] mask
constexpr int kCausal = 2;   // key index <= query index, key tiles above the diagonal skipped
constexpr int kCausalDealt = 3;   // tile kernels only: causal with the query tiles dealt out to a resident grid
constexpr int kAdditiveRagged = 4;   // tile kernels only: additive mask, L no multiple of eight

template <int H>
struct Geometry {
    static constexpr int KS = H / 16;                    // k-steps of the QK^T product
    static constexpr int HV = H < 32 ? 32 : H;           // V columns held in LDS (zero padded)
    static constexpr int DB = HV / 32;                   // 32-row blocks of O^T
};

// NaN-propagating maximum: lowers to v_maximum3_f32 without the input canonicalisation that
// fmaxf needs in IEEE mode.
__device__ __forceinline__ float fmax2(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// Exchanges a value between lanes l and l^32.  v_permlane32_swap(a, b) leaves, in lanes < 32,
// (a[l], a[l + 32]) and, in lanes >= 32, (b[l - 32], b[l]); with a = b = x every lane holds its own
// value and its partner's.  The two results are copied to scalars before the bit cast: applying
// __builtin_bit_cast directly to a vector element reads element 0 for both.
__device__ __forceinline__ float pair_max(float x) {
    const uint32_t xb = __builtin_bit_cast(uint32_t, x);
    const u32x2 r = __builtin_amdgcn_permlane32_swap(xb, xb, false, false);
    const uint32_t r0 = r[0], r1 = r[1];
    return fmax2(__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1));
}

// ... and the same with lanes l and l^16.
__device__ __forceinline__ float quad_max(float x) {
    const uint32_t xb = __builtin_bit_cast(uint32_t, x);
    const u32x2 r = __builtin_amdgcn_permlane16_swap(xb, xb, false, false);
    const uint32_t r0 = r[0], r1 = r[1];
    return fmax2(__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1));
}

__device__ __forceinline__ float pair_sum(float x) {
    const uint32_t xb = __builtin_bit_cast(uint32_t, x);
    const u32x2 r = __builtin_amdgcn_permlane32_swap(xb, xb, false, false);
    const uint32_t r0 = r[0], r1 = r[1];
    return __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
}

__device__ __forceinline__ uint32_t pack_rtz(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
}

// The eight 16-bit values of `v` moved down by n places (n >= 8: nothing of interest is left).
__device__ __forceinline__ u32x4 drop_halves(u32x4 v, uint32_t n) {
    if (n & 4) v = u32x4{v[2], v[3], 0u, 0u};
    if (n & 2) v = u32x4{v[1], v[2], v[3], 0u};
    if (n & 1) v = u32x4{(v[0] >> 16) | (v[1] << 16), (v[1] >> 16) | (v[2] << 16), (v[2] >> 16) | (v[3] << 16), v[3] >> 16};
    return v;
}

// Bias (log2 units) of the reference the exponentials are taken against, in every kernel
// (FwdParams::bias), and the largest sum of a query's 32 probabilities of one sub-tile that the
// eight-wave kernel's fast path accepts.  A key at the reference maximum gets the probability
// 2^-bias.  The probabilities are rounded to fp16 before the second product (normal numbers down
// to 2^-14, subnormals down to 2^-24), so a weight more than 24 - bias log2 units below the row
// maximum is lost: a tail of L small weights loses at most L 2^-(24 - bias) of the row.  The
// launcher picks bias = 11 - ceil(log2 L), between kBiasMin and kBiasMax, which keeps that share
// at or below 2^-13 = 1.2e-4 whatever the sequence length; what is left of the fp16 range is the
// leash of the speculative reference, which may lag the true maximum by 15 + bias log2 units before
// the check sends the wave down the slow path: 14 units at L = 4096, 12 at 16384, 10 at 65536.
// bf16 probabilities have the exponents of float32 and lose nothing at the bottom.  What the bias is limited by
// there is O, which is summed in float32 before it is divided by the row sum: at 2^14 its last bit,
// 2^-149, is still below a bf16 subnormal's, 2^-133, once divided (2^16 was measured to cost values
// around 2^-120 precision).  The leash is 29 units, and the sums of a sub-tile stay below kTripSum
// all the same, so that values up to 2^128 / (kTripSum L / 32) pass whatever the scores do.  (Raising
// kTripSum to 2^32 instead gives the same leash and infinities from values of 2^91 on, where scores rise
// that far; without the longer leash scores with a spread of N(0, 3) inputs take 1.03 to 1.3 times as long.)
constexpr float kBiasMin = -8.0f;
constexpr float kBiasMax = 6.0f;
constexpr float kTripSum = 32768.f;
constexpr float kBiasBf16 = 14.0f;

// O^T[.][nb] *= alpha, in place.  Written as one instruction per register with the register tied
// as input and output, so that the rarely taken rescale does not make the compiler keep a second
// copy of the accumulators (and copy them on the common path).  The leading wait covers the
// matrix-core results the multiplies read.
template <int DB, int NQB>
__device__ __forceinline__ void scale_accumulators(floatx16 (&o)[DB][NQB], int nb, float alpha) {
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float e = o[db][nb][r];
            asm volatile("v_mul_f32 %0, %1, %0" : "+v"(e) : "v"(alpha));
            o[db][nb][r] = e;
        }
    }
}

// Ring tiles of the ping-pong kernel are chunk-major: a 64-key tile of H columns is stored as H / 8
// columns of 64 rows x 16 bytes, column c at c * kColStride halves.  One direct-to-LDS load of a
// wave (64 lanes x 16 bytes, contiguous in LDS) fills one column, lane = key row.  The 64-byte pad
// between columns spreads the four columns touched by a transpose read over all banks.
constexpr int kColStride = 64 * 8 + 32;
template <int H>
constexpr int ring_tile_k() { return (H / 8) * kColStride; }
template <int H>
constexpr int ring_tile_v() { return (Geometry<H>::HV / 8) * kColStride; }
// Per-lane part of the K operand address in a ring tile: row (sub * 32 + lane % 32) of column
// lane / 32; k-step kk adds 2 kk columns.
__device__ __forceinline__ const _Float16* k_ring_ptr(const _Float16* ks, int sub, int lane) {
    return ks + (lane >> 5) * kColStride + (sub * 32 + (lane & 31)) * 8;
}

// Per-lane part of the transpose-read address in a ring tile.  Inside each group of 16 lanes, lane j
// receives, for i = 0..3, element (j % 4) of the 8-byte row fetched by lane 4 i + j / 4: four consecutive
// keys of one head-dim column.  Lane s of a 16-lane group points at row key0 + s / 4, halves 4 (s % 4) ... of the
// 32-byte span that starts at column 2 * ((lane / 16) % 2); head-dim block db adds 4 db columns.
__device__ __forceinline__ const _Float16* v_ring_ptr(const _Float16* vs, int sub, int lane) {
    const int s16 = lane & 15;
    return vs + (2 * ((lane >> 4) & 1) + ((s16 & 3) >> 1)) * kColStride +
           (sub * 32 + 4 * (lane >> 5) + (s16 >> 2)) * 8 + 4 * (s16 & 1);
}

template <int H, int NQB>
constexpr int lds_bytes_pingpong() {
    return 3 * (ring_tile_k<H>() + ring_tile_v<H>()) * (int)sizeof(_Float16);
}

// Additive-mask variant of the ping-pong kernel: behind the rings every wave has a private slab
// for the mask values of its 32 NQB queries and the 32 keys of one sub-tile (row stride
// kMaskSubStr halves: 64 bytes of mask plus 16 of padding).
constexpr int kMaskSubStr = 40;
template <int H, int NW, int NQB>
constexpr int lds_bytes_pingpong_masked() {
    return lds_bytes_pingpong<H, NQB>() + NW * 32 * NQB * kMaskSubStr * (int)sizeof(_Float16);
}

// Split and group kernels.  The launch's parameters in one go: left to itself the compiler loads them in three rounds, each behind a branch.
__device__ __forceinline__ void load_args(const SplitParams& p) {
    asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.stride_b), "s"(p.stride_h), "s"(p.stride_l), "s"(p.R), "s"(p.L), "s"(p.n_qtiles),
                 "s"(p.total_wgs), "s"(p.wgs_per_xcd), "s"(p.by_qtiles.mul), "s"(p.by_qtiles.shift), "s"(p.by_heads.mul), "s"(p.by_heads.shift));
}

// What the launcher has worked out for the softmax (see SplitParams).
struct SplitConstants {
    float c, bias, leash, mask_scale;
    __device__ __forceinline__ explicit SplitConstants(const SplitParams& p) : c(p.scale_log2e), bias(p.bias), leash(p.leash), mask_scale(p.mask_scale) {}
};

// Key-split kernel: LDS of one wave (slabs of the 32 keys it works on and their mask values; at the end
// its share of 16 rows of O in float32, rows padded by 16 bytes against bank conflicts), and of a
// workgroup (plus m and l of every row).
constexpr int kSplitMaxWaves = 4;
constexpr int kRawBuffer = 0x00027000;     // word 3 of a raw buffer resource: no stride, no swizzle, 32-bit data format
template <int H>
constexpr int split_row_floats() { return H + 4; }
template <int H, bool MASK>
constexpr int split_wave_bytes() {
    constexpr int part = 16 * split_row_floats<H>() * 4, slabs = 2 * 32 * H * 2 + (MASK ? 1024 : 0);
    return part > slabs ? part : slabs;
}
template <int H, bool MASK>
constexpr int split_lds_bytes(int waves) { return waves * (split_wave_bytes<H, MASK>() + 16 * 8); }

// Group kernel: sub-tiles of 32 keys per key group and key tile (two where one group would otherwise pass a
// barrier per sub-tile: +2 %), and ring slots (two where three would cost a resident workgroup: with the mask slabs
// behind them a compute unit would hold two workgroups instead of three at head_dim 64, and the wait for a tile's
// mask values is one for everything under way in any case).
template <int H, int GK>
constexpr int group_sub() { return GK == 1 && H <= 64 ? 2 : 1; }
template <int H, int GK, bool MASK>
constexpr int group_slots() { return (GK == 2 && H == 128) || MASK ? 2 : 3; }
template <int H, int GK, bool MASK>
constexpr int group_ring_bytes() { return group_slots<H, GK, MASK>() * GK * group_sub<H, GK>() * 2 * 32 * H * 2; }
// What the second key group's wave of a row group hands to the first one's: O as the lanes hold it, m and l.
template <int H, int NQ>
constexpr int group_part_bytes() { return NQ * (H / 16 * 1024 + 512); }
// LDS: the ring of key tiles and the mask slabs, later the rows of O on their way out or, with two key groups,
// the second one's shares (whichever is larger).
template <int H, int NQ, int GK, bool MASK>
constexpr int group_lds_bytes() {
    constexpr int ring = group_ring_bytes<H, GK, MASK>() + (MASK ? 8 * group_sub<H, GK>() * NQ * 1024 : 0), part = GK == 1 ? 8 * 16 * (H + 8) * 2 : 8 / GK * group_part_bytes<H, NQ>();
    return ring > part ? ring : part;
}
// Waves per SIMD that the group kernel's registers are to last for.  16-row waves: six, three workgroups per compute unit.
// Masked launches with the two that three ring slots left room for: B2 R12 L2048 H64 bias (768 workgroups) took
// 52.7 us instead of 44.3, B16 R12 L381 padding (576) 21.0 instead of 18.6, B14 R8 L576 (bf16) 23.2 instead of 20.0.
// Launches without a mask stay below the 80 registers of six by themselves: 260 shapes, plain and causal, take the
// time that they take with a bound of four (1.000 in the mean for one and for two key groups).  At head_dim 16 and 32
// without a mask eight, four workgroups: two sub-tiles at a time (split_two) take 65 registers if they are let.
template <int H, int NQ, bool MASK>
constexpr int group_waves_per_simd() { return NQ == 1 && H <= 32 && !MASK ? 8 : NQ == 1 && H <= 64 ? 6 : NQ == 1 || H <= 64 ? 4 : 2; }
// (written in assembly so that the compiler does not see an LDS write, see RingLoader)
__device__ __forceinline__ void group_dma16(uint32_t lds_addr, const _Float16* base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(voff), "s"(base) : "memory", "m0");
}

// Barrier between the phases of the ping-pong kernel.  It does not wait for the wave's own LDS
// reads: nothing is handed from wave to wave through LDS stores (the rings are written by
// direct-to-LDS loads, which their issuer waits for with vmcnt), and every read of a ring slot is
// consumed by a matrix instruction at least one barrier before the loads that overwrite the slot
// are issued.  The scheduling barriers keep the compiler from moving matrix or vector
// instructions of one phase into the next.
__device__ __forceinline__ void ring_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

// One group's share of a 64-key ring tile, fetched straight into LDS.  Wave w of the group (NWG
// waves) owns the columns w * NP ... w * NP + NP - 1; lane l fetches the 16 bytes of key row l.
// Rows at or beyond L are read from row L - 1 instead: their scores are masked to -inf, or belong
// to sub-tiles that are never consumed, and a probability of exactly zero times a finite V row
// contributes nothing.  Tiles starting at or beyond `limit` are not fetched at all (limit <= L).
// The loads are asynchronous: the issuing wave waits for vmcnt before the barrier that hands the
// tile to its readers.
template <int H, int NWG>
struct RingLoader {
    static constexpr int CPR = H / 8;
    static constexpr int NP = (CPR + NWG - 1) / NWG;
    int col0;
    uint32_t lane_off;   // byte offset of this lane's row inside a full tile

    __device__ __forceinline__ void init(int wave_in_group, int64_t stride_l, int lane) {
        col0 = wave_in_group * NP;
        lane_off = (uint32_t)lane * (uint32_t)stride_l * 2u;
    }
    // The load is written in assembly so that the compiler does not see an LDS write: it would
    // otherwise wait for the load before the next LDS read of the wave.  M0 holds the LDS address
    // of lane 0's 16 bytes; lane l lands 16 l bytes further on.
    static __device__ __forceinline__ void dma16(uint32_t lds_addr, const _Float16* base, uint32_t voff) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :: "s"(lds_addr), "v"(voff), "s"(base) : "memory", "m0");
    }
    __device__ __forceinline__ void issue(const _Float16* src, int64_t stride_l, int key0, int limit, int L,
                                          _Float16* tile, int lane) const {
        issue_at(src + (int64_t)key0 * stride_l + col0 * 8, stride_l, key0, limit, L, tile, lane);
    }
    // `base` = src + key0 * stride_l + 8 * col0, kept by callers that walk the tiles in order
    __device__ __forceinline__ void issue_at(const _Float16* base, int64_t stride_l, int key0, int limit, int L,
                                             _Float16* tile, int lane) const {
        if (key0 >= limit) return;
        uint32_t voff = lane_off;
        if (key0 + 64 > L) voff = (uint32_t)(min(key0 + lane, L - 1) - key0) * (uint32_t)stride_l * 2u;
        const uint32_t lds0 = (uint32_t)(uintptr_t)(FA_LDS void*)tile + (uint32_t)col0 * (kColStride * 2);
#pragma unroll
        for (int i = 0; i < NP; ++i)
            if (CPR % NWG == 0 || col0 + i < CPR) dma16(lds0 + i * (kColStride * 2), base + i * 8, voff);
    }
};

__device__ __forceinline__ void wait_ring_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

}  // namespace fa

// The kernels proper are written once and compiled for both element types: fp16 in namespace fa,
// bf16 in namespace fa::bf16.  All 16-bit data travel as bit patterns (half8 / u32x4 registers,
// _Float16 pointers for address arithmetic); only the few operations that interpret them differ.
#define FA_ELEM_BF16 0
#include "fused_attn_kernel_impl.inc"
#include "fused_attn_split.inc"
#undef FA_ELEM_BF16
#define FA_ELEM_BF16 1
#include "fused_attn_kernel_impl.inc"
#include "fused_attn_split.inc"
#undef FA_ELEM_BF16
