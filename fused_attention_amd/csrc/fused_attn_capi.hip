// C ABI of libfused_attn_gfx950.so: argument validation, launch geometry and the launch
// itself.  Host counterpart of launch_attention_kernel (reference
// include/fused_attn.cuh:860-894): picks the workgroup shape, sizes the dynamic LDS block,
// builds the grid and launches on the caller's stream.
#include "fused_attn_kernel.hpp"
#include "qkv_proj_kernel.hpp"

#include "../../include/fused_attn.h"

#include <mutex>
#include <utility>
#include <vector>

namespace {

constexpr int kKeyTile = 64;     // keys per LDS tile
constexpr int kNumCu = 256;      // compute units of one MI355X

// Launch shape: wave64s per workgroup and blocks of 32 query rows per wave.
struct Shape {
    int waves;
    int nqb;
    int rows() const { return waves * 32 * nqb; }
};

// The tile kernels' shapes (fwd_kernel_pingpong, fwd_kernel_pp16); pick_variant below weighs that launch, where
// the problem fills the chip well enough for one, against the key-split and group kernels, which take
// everything else:
//   {8, 2}  eight 64-row waves share one K/V stream, 512 queries per workgroup, one resident per
//           compute unit: head_dim <= 64 (with head_dim 128 a 64-row wave would need the whole
//           register file of a SIMD);
//   {8, 1}  the same with 32-row waves, 256 queries per workgroup: head_dim 128, without additive mask, and
//           causal launches at head_dim 64 that fill one round of pairs of such tiles, not of larger ones;
//   {0, 0}  no tile kernel.
int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// How well a shape uses the chip, in 1/1024: the share of the (rounds x slots) grid of resident
// workgroup slots that the problem's workgroups occupy, times the share of each workgroup's query
// rows that exist (the last workgroup of a sequence may be mostly empty).
int64_t usage(int64_t heads, int64_t L, int64_t rows, int64_t slots) {
    const int64_t per_head = ceil_div(L, rows);
    const int64_t wgs = heads * per_head;
    // in floating point: the products overflow 64 bits for the largest accepted shapes
    const double filled = (double)wgs / ((double)ceil_div(wgs, slots) * (double)slots);
    const double rows_used = (double)L / ((double)per_head * (double)rows);
    return (int64_t)(1024.0 * filled * rows_used);
}

// Causal launches of the eight-wave kernel.  Query tile t of a head costs t + 1 key blocks.  The
// plain schedule gives every workgroup the pair (t, n - 1 - t), n + 1 blocks, and the grid runs
// ceil(pairs / 256) rounds of them; a last round that is mostly empty costs as much as a full one,
// and in a lone part-filled round the idle compute units could have taken the small tiles.
// The dealt schedule (kernel: p.heads_per_xcd > 0) keeps 32 workgroups resident per XCD and deals
// the tiles of the XCD's heads out in descending cost, serpentine over the workgroups; it needs
// B * R to be a multiple of 8 so that the XCDs carry equal loads.  Time in key blocks of the
// busiest workgroup under either schedule; the dealt one is taken when it saves 8 % or more
// (measured: 5 to 17 % faster then, against 11 to 28 % fewer blocks).
struct CausalPlan {
    bool dealt;
    int64_t blocks;       // key blocks the busiest workgroup walks through
};

CausalPlan plan_causal_walk(int64_t heads, int64_t n, int64_t H);

// One causal launch asks for its plan twice (shape choice, then grid), and a serving loop asks for
// the same few plans over and over: the last results are kept per host thread.
CausalPlan plan_causal(int64_t heads, int64_t n, int64_t H) {
    struct Entry {
        int64_t heads, n, H;
        CausalPlan plan;
    };
    constexpr int kEntries = 8;
    thread_local Entry cache[kEntries] = {};
    thread_local int next = 0;
    for (const Entry& e : cache)
        if (e.heads == heads && e.n == n && e.H == H) return e.plan;
    const CausalPlan plan = plan_causal_walk(heads, n, H);
    cache[next] = Entry{heads, n, H, plan};
    next = (next + 1) % kEntries;
    return plan;
}

CausalPlan plan_causal_walk(int64_t heads, int64_t n, int64_t H) {
    const int64_t pairs = heads * ceil_div(n, 2);
    const CausalPlan paired{false, ceil_div(pairs, kNumCu) * (n + 1)};
    constexpr int kPerXcd = kNumCu / fa::kNumXcd;
    // head_dim below 64: dealing the tiles out spreads an XCD's workgroups over more heads at a
    // time than its L2 holds K and V for, and measures slower than the part-filled round
    if (H < 64 || heads % fa::kNumXcd != 0) return paired;
    const int64_t hx = heads / fa::kNumXcd;
    const int64_t items = hx * n;
    if (items > (int64_t)1 << 22) return paired;     // the walk below is linear in the items
    int64_t load[kPerXcd] = {};
    for (int64_t j0 = 0, round = 0; j0 < items; j0 += kPerXcd, ++round)
        for (int w = 0; w < kPerXcd; ++w) {
            const int64_t j = j0 + ((round & 1) ? kPerXcd - 1 - w : w);
            if (j < items) load[w] += n - j / hx;
        }
    int64_t worst = 0;
    for (int w = 0; w < kPerXcd; ++w) worst = load[w] > worst ? load[w] : worst;
    return worst * 100 <= paired.blocks * 92 ? CausalPlan{true, worst} : paired;
}

// mask_chunks: an additive mask whose rows hold a 16-byte chunk at least and stay below 2^24 values (the
// ping-pong kernel keeps 32-bit byte offsets inside the 64 mask rows of a wave).
Shape pick_shape(int64_t B, int64_t R, int64_t L, int64_t H, bool has_mask, bool mask_chunks,
                 bool causal) {
    const int64_t heads = B * R;
    // head_dim 128 with a mask: the group kernel was the faster one on 843 of 861 random shapes, by up to 33 %,
    // and at most 7 % slower on the others
    if (has_mask && (!mask_chunks || H > 64)) return {0, 0};
    // Taken into account when the workgroups fill the chip well enough: usage of 0.55 in a lone round, 0.7
    // in a part-filled second round, 0.6 from two rounds on (a lone round may be emptier than the tail of
    // several, because idle units leave the busy ones more of the power budget).  A causal workgroup
    // takes two query tiles (see the kernel).
    const Shape tile = H > 64 ? Shape{8, 1} : Shape{8, 2};
    const int64_t rows = tile.rows() * (causal ? 2 : 1);
    const int64_t wgs = heads * ceil_div(L, rows);
    if (causal) {
        // with the dealt schedule: useful key blocks over the blocks the 256 compute units are held for
        const int64_t n = ceil_div(L, tile.rows());
        const CausalPlan plan = plan_causal(heads, n, H);
        if (plan.dealt) {
            const double held = (double)plan.blocks * kNumCu;
            const double useful = (double)heads * (double)n * (double)(n + 1) / 2.0;
            const double rows_used = (double)L / ((double)n * (double)tile.rows());
            if (1024.0 * useful / held * rows_used >= 614.0) return tile;
        }
    }
    const int64_t used = usage(heads, L, rows, kNumCu);
    if (wgs >= 2 * kNumCu ? used >= 614 : used >= (wgs <= kNumCu ? 560 : 717)) return tile;
    // One round of pairs of 256-query tiles: of 500 random causal shapes at head_dim 64 it is the fastest on a
    // quarter, by up to 26 % (B1 R32 L4096 103 -> 91 us, B3 R12 L3394 93.8 -> 77.8, B2 R40 L999 29.1 -> 24.1), and
    // the choice with it loses 1.3 % against the best kernel of each, without it 4.8 %.  (At head_dim 16 and 32
    // the group kernel is never more than 3 % behind it; plain launches, 214 shapes: 7 % at most, on 9 of them.)
    if (causal && H == 64 && heads * ceil_div(L, 512) <= kNumCu && usage(heads, L, 512, kNumCu) >= 560) return {8, 1};
    return {0, 0};
}

// Dynamic LDS above 64 KiB has to be opted into per kernel function and per device: done on the
// first launch of that kernel on that device.
hipError_t allow_large_lds(const void* kernel, int bytes) {
    static std::mutex lock;
    static std::vector<std::pair<const void*, int>> done;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> guard(lock);
    for (const auto& d : done)
        if (d.first == kernel && d.second == dev) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) done.emplace_back(kernel, dev);
    return e;
}

// BF selects the bf16 instantiation (namespace fa::bf16) of the same kernel source.
template <int H, int NW, int NQB, int WPE, int MODE, bool BF>
hipError_t launch_pingpong(const fa::FwdParams& p, hipStream_t stream) {
    constexpr int lds = MODE == fa::kAdditive || MODE == fa::kAdditiveRagged ? fa::lds_bytes_pingpong_masked<H, NW, NQB>() : fa::lds_bytes_pingpong<H, NQB>();
    auto kernel = BF ? fa::bf16::fwd_kernel_pingpong<H, NW, NQB, WPE, MODE> : fa::fwd_kernel_pingpong<H, NW, NQB, WPE, MODE>;
    if constexpr (lds > 64 * 1024) {
        const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kernel), lds);
        if (e != hipSuccess) return e;
    }
    const int grid = p.wgs_per_xcd * fa::kNumXcd;
    // the launch's own status, not the thread's sticky last error (which may stem from the caller's code)
    fa::FwdParams params = p;
    void* args[] = {&params};
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(grid), dim3(NW * 64), args, lds, stream);
}

// The eight-wave kernel with its products written as 16 x 16 tiles (fwd_kernel_pp16), head_dim 64
// (64-row waves) and 128 (32-row waves).
// Plain launches: on a full chip the clock follows the switching activity and the 16 x 16 x 32
// instruction moves half as many accumulator registers per flop; where part of the chip idles the
// clock is not held back and its 36 (34) matrix instructions per sub-tile instead of 20 (18) cost
// more than they save, and a part-filled last round takes that from the whole launch.  Measured on
// the same box, by workgroups, head_dim 64: 256 +2.9 and +3.6 %, 480 +1.1 %, 512 +3.5 %; 192 -5 to
// -9 %, 384 -3.4 and -4.6 %, 448 -0.7 %, 640 -1.0 %, 1152 -0.8 %.  head_dim 128: 224 +3.4 %, 256
// +3.1 %, 480 +2.5 %, 512 +2.1 %, 1280 +3.1 %, 2048 +5.2 %; 192 -0.3 %, 384 -2.0 %, 448 +1.3 %, 640
// -0.9 %, 800 -0.2 %, 1088 +0.1 %, 1600 -0.9 %.  Taken when the last round is at least seven
// eighths full.
// Causal launches in pairs of tiles or dealt out: there the gain is the kernel's deal of 16-query
// blocks to the waves, which does not depend on the clock, and only an emptier single round loses
// (head_dim 64: 144 pairs -4.3 %, 160 -6.2 %, 192 -1.4 and +1.3 %, 200 -0.6 %; 240 +3.6 %, 256
// +5.5 %, 400 +1.4 %, 960 +4.5 and +7.5 %, 1152 +5.4 %, dealt +3.2 to +4.7 %; head_dim 128: 1024
// pairs +5.1 and +5.4 %, dealt +4.2 %): taken from seven eighths of a round on.
bool use_tiles16(int64_t H, Shape sh, const fa::FwdParams& p, bool causal) {
    if (H < 64 || (H == 64 && sh.nqb != 2)) return false;
    if (8 * (int64_t)p.total_wgs < 7 * kNumCu) return false;
    if (causal) return true;            // (a dealt launch is a whole resident grid)
    if (H == 64 && p.total_wgs < kNumCu) return false;     // (224 and 240 workgroups: +1.6 and +2.5 % at L = 4096, -1.4 % at L = 1024)
    const int last = p.total_wgs % kNumCu;
    return last == 0 || 8 * last >= 7 * kNumCu;
}

template <int H, bool BF, int MODE>
hipError_t launch_pp16(const fa::FwdParams& p, hipStream_t stream) {
    constexpr int lds = fa::lds_bytes_pingpong<H, 2>();
    auto kernel = BF ? fa::bf16::fwd_kernel_pp16<H, 8, true, MODE> : fa::fwd_kernel_pp16<H, 8, true, MODE>;
    if constexpr (lds > 64 * 1024) {
        const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kernel), lds);
        if (e != hipSuccess) return e;
    }
    fa::FwdParams params = p;
    void* args[] = {&params};
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(p.wgs_per_xcd * fa::kNumXcd), dim3(8 * 64), args,
                           lds, stream);
}

template <int H, bool BF>
hipError_t launch_pp16_mode(int mode, const fa::FwdParams& p, hipStream_t stream) {
    switch (mode) {
        case fa::kPlain: return launch_pp16<H, BF, fa::kPlain>(p, stream);
        case fa::kCausal: return launch_pp16<H, BF, fa::kCausal>(p, stream);
        case fa::kCausalDealt: return launch_pp16<H, BF, fa::kCausalDealt>(p, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_tiles16(int64_t H, int mode, bool bf16, const fa::FwdParams& p, hipStream_t stream) {
    if (H == 64) return bf16 ? launch_pp16_mode<64, true>(mode, p, stream) : launch_pp16_mode<64, false>(mode, p, stream);
    if (H == 128) return bf16 ? launch_pp16_mode<128, true>(mode, p, stream) : launch_pp16_mode<128, false>(mode, p, stream);
    return hipErrorInvalidValue;
}

template <int H, int MODE, bool BF>
hipError_t dispatch_shape(Shape sh, const fa::FwdParams& p, hipStream_t stream) {
    constexpr bool MASK = MODE == fa::kAdditive || MODE == fa::kAdditiveRagged;
    // the dealt causal schedule exists at head_dim 64 and 128 only (plan_causal never asks for it elsewhere),
    // and no masked launch at head_dim 128 (pick_shape)
    if constexpr ((MODE == fa::kCausalDealt && H < 64) || (MASK && H > 64))
        return hipErrorInvalidValue;
    else if constexpr (H == 64 && (MODE == fa::kCausal || MODE == fa::kCausalDealt))
        return sh.nqb == 1 ? launch_pingpong<H, 8, 1, 2, MODE, BF>(p, stream) : launch_pingpong<H, 8, 2, 2, MODE, BF>(p, stream);
    else
        return launch_pingpong<H, 8, (H > 64 ? 1 : 2), 2, MODE, BF>(p, stream);
}

template <int MODE, bool BF>
hipError_t dispatch_head_dim(int64_t H, Shape sh, const fa::FwdParams& p, hipStream_t stream) {
    switch (H) {
        case 16: return dispatch_shape<16, MODE, BF>(sh, p, stream);
        case 32: return dispatch_shape<32, MODE, BF>(sh, p, stream);
        case 64: return dispatch_shape<64, MODE, BF>(sh, p, stream);
        case 128: return dispatch_shape<128, MODE, BF>(sh, p, stream);
        default: return hipErrorInvalidValue;
    }
}

template <int MODE>
hipError_t dispatch(int64_t H, Shape sh, const fa::FwdParams& p, hipStream_t stream, bool bf16) {
    return bf16 ? dispatch_head_dim<MODE, true>(H, sh, p, stream) : dispatch_head_dim<MODE, false>(H, sh, p, stream);
}

// Which kernel runs a problem: a tile kernel (the launch of pick_shape), the key-split kernel (`waves` share out
// the keys of 16 query rows), or the group kernel with 16 NQ rows per wave and GK key groups (kGroup<NQ><GK>).
enum VariantKind { kTile, kSplit, kGroup11, kGroup12, kGroup21 };
struct Variant {
    VariantKind kind;
    int waves;
};

fa::SplitParams split_params(const fa::FwdParams& p, bool bf16) {
    // (two divisions by run-time numbers are 0.05 to 0.1 us at the start of a workgroup)
    fa::SplitParams params{p, fa::divisor(p.n_qtiles), fa::divisor(p.R), 0.f, 0.f};
    params.leash = ((bf16 ? 10.f : 15.f) + p.bias) / p.scale_log2e;
    params.mask_scale = 1.4426950408889634f / p.scale_log2e;
    return params;
}

// The key-split kernel (16 query rows per workgroup).
template <int H, int MODE, bool BF>
hipError_t launch_split(const fa::FwdParams& p, hipStream_t stream) {
    constexpr int WPE = H <= 64 ? 4 : 2;
    auto kernel = BF ? fa::bf16::fwd_kernel_split<H, MODE, WPE> : fa::fwd_kernel_split<H, MODE, WPE>;
    constexpr int most = fa::split_lds_bytes<H, MODE == fa::kAdditive>(fa::kSplitMaxWaves);
    if constexpr (most > 64 * 1024) {
        const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kernel), most);
        if (e != hipSuccess) return e;
    }
    fa::SplitParams params = split_params(p, BF);
    void* args[] = {&params};
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(p.wgs_per_xcd * fa::kNumXcd), dim3(p.waves * 64), args,
                           fa::split_lds_bytes<H, MODE == fa::kAdditive>(p.waves), stream);
}

// The group kernel: 16 NQ query rows per wave, GK key groups.
template <int H, int NQ, int GK, int MODE, bool BF>
hipError_t launch_group(const fa::FwdParams& p, hipStream_t stream) {
    constexpr int lds = fa::group_lds_bytes<H, NQ, GK, MODE == fa::kAdditive>();
    static_assert(lds <= 160 * 1024, "fits a compute unit");
    constexpr int WPE = fa::group_waves_per_simd<H, NQ, MODE == fa::kAdditive>();
    auto kernel = BF ? fa::bf16::fwd_kernel_group<H, NQ, GK, MODE, WPE> : fa::fwd_kernel_group<H, NQ, GK, MODE, WPE>;
    if constexpr (lds > 64 * 1024) {
        const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kernel), lds);
        if (e != hipSuccess) return e;
    }
    fa::SplitParams params = split_params(p, BF);
    void* args[] = {&params};
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(p.wgs_per_xcd * fa::kNumXcd), dim3(8 * 64), args, lds, stream);
}

// 32 rows per wave at head_dim 128: without mask and causal flag only (with one of them it was the fastest kernel
// on none of 2100 random shapes)
template <int H, int MODE>
constexpr bool group21_offered() { return H <= 64 || MODE == fa::kPlain; }

template <int H, int MODE, bool BF>
hipError_t dispatch_variant(const Variant& v, const fa::FwdParams& p, hipStream_t stream) {
    switch (v.kind) {
        case kSplit: return launch_split<H, MODE, BF>(p, stream);
        case kGroup11: return launch_group<H, 1, 1, MODE, BF>(p, stream);
        case kGroup12: return launch_group<H, 1, 2, MODE, BF>(p, stream);
        case kGroup21:
            if constexpr (group21_offered<H, MODE>()) return launch_group<H, 2, 1, MODE, BF>(p, stream);
            return hipErrorInvalidValue;
        default: return hipErrorInvalidValue;
    }
}

template <int MODE, bool BF>
hipError_t dispatch_variant_head_dim(int64_t H, const Variant& v, const fa::FwdParams& p, hipStream_t stream) {
    switch (H) {
        case 16: return dispatch_variant<16, MODE, BF>(v, p, stream);
        case 32: return dispatch_variant<32, MODE, BF>(v, p, stream);
        case 64: return dispatch_variant<64, MODE, BF>(v, p, stream);
        case 128: return dispatch_variant<128, MODE, BF>(v, p, stream);
        default: return hipErrorInvalidValue;
    }
}

template <bool BF>
hipError_t dispatch_variant_mode(int64_t H, int mode, const Variant& v, const fa::FwdParams& p, hipStream_t stream) {
    switch (mode) {
        case fa::kPlain: return dispatch_variant_head_dim<fa::kPlain, BF>(H, v, p, stream);
        case fa::kCausal: return dispatch_variant_head_dim<fa::kCausal, BF>(H, v, p, stream);
        case fa::kAdditive: return dispatch_variant_head_dim<fa::kAdditive, BF>(H, v, p, stream);
        default: return hipErrorInvalidValue;
    }
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }

struct Strides {
    int64_t b, h, l;
};

bool strides_ok(const Strides& s, int64_t H) {
    return s.l >= H && s.h >= 0 && s.b >= 0 && (s.l % 8) == 0 && (s.h % 8) == 0 && (s.b % 8) == 0;
}

bool extent_ok(const Strides& s, int64_t B, int64_t R, int64_t L) {
    constexpr int64_t kMaxElems = (int64_t)1 << 62;
    return !(L > kMaxElems / s.l || (s.h > 0 && R > kMaxElems / s.h) || (s.b > 0 && B > kMaxElems / s.b));
}

int validate(const void* q, const void* k, const void* v, const void* mask, void* out, int64_t B,
             int64_t R, int64_t L, int64_t H, const Strides& in, const Strides& os,
             fa::FwdParams* p, float scale, Shape* shape, bool causal, void* lse) {
    const int64_t stride_b = in.b, stride_h = in.h, stride_l = in.l;
    if (q == nullptr || k == nullptr || v == nullptr || out == nullptr) return FA_ERR_NULL_POINTER;
    if (!fa_fwd_query(H)) return FA_ERR_BAD_HEAD_DIM;
    if (B < 1 || R < 1 || L < 1) return FA_ERR_BAD_SHAPE;
    // the kernels track the row maximum of the raw scores, which is the maximum of the scaled ones
    // only for a positive scale, and they divide the additive mask by the scale
    if (!(scale > 0.f) || scale > 3.0e38f) return FA_ERR_BAD_SCALE;
    if (!strides_ok(in, H) || !strides_ok(os, H)) return FA_ERR_BAD_STRIDE;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out)) return FA_ERR_MISALIGNED;
    if (mask != nullptr && (reinterpret_cast<uintptr_t>(mask) & 1u) != 0) return FA_ERR_MISALIGNED;
    constexpr int64_t kMaxInt = 0x7fffffff;
    if (L > kMaxInt - 4096 || B > kMaxInt || R > kMaxInt || B * R > kMaxInt) return FA_ERR_TOO_LARGE;
    // the tile loaders keep 32-bit byte offsets inside a 64-key tile
    if (stride_l > ((int64_t)1 << 24)) return FA_ERR_TOO_LARGE;
    *shape = pick_shape(B, R, L, H, mask != nullptr,
                        L >= 8 && L <= ((int64_t)1 << 24), causal);
    int64_t n_qtiles = 0, total = 0;       // (no tile kernel: use_variant fills in the launch)
    p->heads_per_xcd = 0;
    if (shape->waves != 0) {
        n_qtiles = ceil_div(L, shape->rows());
        // Pairs of query tiles for causal launches, and for masked ones (see the kernel) when the pairs, two tiles
        // long, need no more time on the chip than the tiles in rounds of their own
        const int64_t pairs = ceil_div(n_qtiles, 2);
        if (causal) {
            const CausalPlan plan = plan_causal(B * R, n_qtiles, H);
            n_qtiles = pairs;
            if (plan.dealt) {
                p->heads_per_xcd = (int)(B * R / fa::kNumXcd);
                total = kNumCu;                                       // a resident grid
            }
        } else if (mask != nullptr && 2 * ceil_div(B * R * pairs, kNumCu) <= ceil_div(B * R * n_qtiles, kNumCu)) {
            n_qtiles = pairs;
        }
        if (total == 0) total = B * R * n_qtiles;
        if (total > kMaxInt - 8) return FA_ERR_TOO_LARGE;
    }
    if (!extent_ok(in, B, R, L) || !extent_ok(os, B, R, L)) return FA_ERR_TOO_LARGE;

    p->q = static_cast<const _Float16*>(q);
    p->k = static_cast<const _Float16*>(k);
    p->v = static_cast<const _Float16*>(v);
    p->mask = static_cast<const _Float16*>(mask);
    p->o = static_cast<_Float16*>(out);
    p->lse = static_cast<float*>(lse);
    p->stride_b = stride_b;
    p->stride_h = stride_h;
    p->stride_l = stride_l;
    p->ostride_b = os.b;
    p->ostride_h = os.h;
    p->ostride_l = os.l;
    p->B = (int)B;
    p->R = (int)R;
    p->L = (int)L;
    p->n_qtiles = (int)n_qtiles;
    p->total_wgs = (int)total;
    p->wgs_per_xcd = (int)((total + fa::kNumXcd - 1) / fa::kNumXcd);
    p->scale_log2e = scale * 1.4426950408889634f;
    p->bias = fa_fwd_reference_bias(L);
    return FA_OK;
}

// Time of a launch of the key-split or the group kernel, in microseconds: fits over 6700 calls drawn from the ranges of
// perf/cases.py (B 1..32, R 4..40, L 32..16384, every head_dim; plain, causal, padding and bias, N(0, 1) and N(0, 3), which no
// estimate can tell apart beforehand), every kernel that is offered timed on MI355X with three sets of buffers in turn,
// causal ones in part behind a producer of q, k and v.  What counts is the order of the estimates, so that is what
// was fitted: the time lost against the best kernel of each call, with a share of the estimates' own error.  Choosing the
// smallest one loses 0.9 % on these calls, more than 3 % on 10 % of them, and 0.9 % on 600 left out of the fit (the fit
// before, of the kernels as they were then: 1.9, 20 and 1.7 %).  Two things in the fit are not measured times.  The 93 problems
// whose kernel the tests name were held where they are, by a penalty: without it the loss is 0.6 % (B8 R12 L1024 H64: 32.2 us
// on the tile kernel, 30.4 on 16-row waves of the group kernel).  And the times of two key groups behind a producer were taken
// 1.1 times as long: the producer that was timed is a copy, and behind the projection, whose stores pass L2, K and V
// are read twice as often from further away (measured on one call, B1 R40 L512 H128 causal: 12.6 us against 12.9 alone, 2 us
// more in the block).
// Against the choice before, of all 7271 calls 794 take over 3 % less time and 69 over 3 % more, scattered over the ranges; the
// furthest, timed again: B1 R16 L9344 H64 causal 209 -> 252 us (two key groups before, the tile kernel now), B11 R12 L397 H128
// causal 19.8 -> 23.7 (two key groups, 16 rows), B6 R40 L2924 H16 padding 584 -> 697 (tile, 16 rows).  Other weights in the fit move
// them elsewhere (10 to 15 of 1000 calls outside a fit, with eight times the weight on calls that get slower or without the
// tests' problems): estimates of four terms cannot tell these calls from their neighbours.
//   split:  kLaunch + a ceil(sub-tiles / waves)              the longest wave
//                   + b sub-tiles of all workgroups / 256    one compute unit's share of the work
//                   + c k                                    start and merge
//   group:  kLaunch + a (sub-tiles + (rounds - 1) mean) / GK      the longest chain of workgroups
//                   + b mean w / GK                               w = workgroups per compute unit, taken
//                                                                 half way between the mean and
//                                                                 the most (k) of any
//                   + s sub-tiles min(k, resident) / GK           the longest one's neighbours
//                   + c k
// with sub-tiles of 32 keys, a causal tile's mean being about half of them, and rounds = k over the
// workgroups resident per compute unit (a zero: the times do not tell that term from the others).
struct Cost {
    float a, b, c;
};
struct GroupCost {
    float a, b, s, c;
};
constexpr float kLaunch = 3.2f;
// [head_dim 16, 32, 64, 128][plain, causal, mask]
constexpr Cost kCostSplit2[4][3] = {
    {{0.0758f, 0.034f, 0.0884f}, {0.106f, 0.0478f, 0.0936f}, {0.155f, 0.0632f, 0.0567f}},
    {{0.125f, 0.0612f, 0.0286f}, {0.109f, 0.0801f, 0.0968f}, {0.174f, 0.069f, 0.0605f}},
    {{0.182f, 0.0718f, 0.132f}, {0.223f, 0.0592f, 0.258f}, {0.231f, 0.0895f, 0.145f}},
    {{0.397f, 0.104f, 0.467f}, {0.292f, 0.153f, 0.617f}, {0.475f, 0.174f, 0.486f}},
};
constexpr Cost kCostSplit4[4][3] = {
    {{0.0218f, 0.0416f, 0.127f}, {0.0372f, 0.0455f, 0.179f}, {0.0635f, 0.064f, 0.085f}},
    {{0.0423f, 0.0474f, 0.132f}, {0.0355f, 0.05f, 0.197f}, {0.0395f, 0.0632f, 0.129f}},
    {{0.0881f, 0.0792f, 0.183f}, {0.0541f, 0.0716f, 0.367f}, {0.157f, 0.0995f, 0.194f}},
    {{0.321f, 0.2f, 0.434f}, {0.183f, 0.148f, 0.758f}, {0.538f, 0.213f, 0.39f}},
};
constexpr GroupCost kCostGroup11[4][3] = {
    {{0.101f, 0.132f, 0.0418f, 0.308f}, {0.115f, 0.126f, 0.0555f, 0.572f}, {0.14f, 0.182f, 0.0665f, 0.367f}},
    {{0.0976f, 0.144f, 0.014f, 0.32f}, {0.101f, 0.129f, 0.0366f, 0.468f}, {0.103f, 0.249f, 0.013f, 0.368f}},
    {{0.121f, 0.221f, 0.0445f, 0.389f}, {0.12f, 0.21f, 0.0548f, 0.527f}, {0.17f, 0.291f, 0.0665f, 0.315f}},
    {{0.261f, 0.356f, 0.0547f, 0.72f}, {0.324f, 0.344f, 0.00125f, 0.747f}, {0.409f, 0.406f, 0.0119f, 0.441f}},
};
constexpr GroupCost kCostGroup12[4][3] = {
    {{0.18f, 0.145f, 0.00668f, 0.451f}, {0.179f, 0.131f, 0.00861f, 0.834f}, {0.0817f, 0.32f, 0.000997f, 0.395f}},
    {{0.126f, 0.161f, 0.0165f, 0.448f}, {0.143f, 0.162f, 0.00435f, 0.931f}, {0.0562f, 0.31f, 0.00126f, 0.363f}},
    {{0.17f, 0.243f, 0.015f, 0.717f}, {0.109f, 0.247f, 0.024f, 1.35f}, {0.183f, 0.368f, 0.012f, 0.581f}},
    {{0.219f, 0.423f, 0.00546f, 1.59f}, {0.142f, 0.457f, 0.00095f, 2.27f}, {0.327f, 0.534f, 0.028f, 1.35f}},
};
constexpr GroupCost kCostGroup21[4][3] = {
    {{0.101f, 0.239f, 0.103f, 0.233f}, {0.0673f, 0.286f, 0.103f, 0.0705f}, {0.13f, 0.558f, 0.054f, 0.216f}},
    {{0.117f, 0.267f, 0.0574f, 0.438f}, {0.242f, 0.247f, 0.0506f, 0.0534f}, {0.21f, 0.523f, 0.0417f, 0.21f}},
    {{0.195f, 0.362f, 0.0865f, 1.11f}, {0.344f, 0.34f, 0.063f, 0.196f}, {0.481f, 0.522f, 0.0506f, 0.365f}},
    {{0.656f, 0.436f, 0.00707f, 1.2f}, {}, {}},
};

struct GroupShape {
    VariantKind kind;
    int nq, gk;
    // workgroups per compute unit, by head_dim (without a mask; the estimates were fitted with these)
    int resident[4];
    const GroupCost (*cost)[3];
};
constexpr GroupShape kGroups[] = {
    {kGroup11, 1, 1, {4, 4, 3, 2}, kCostGroup11},
    {kGroup12, 1, 2, {4, 4, 3, 2}, kCostGroup12},
    {kGroup21, 2, 1, {3, 3, 2, 1}, kCostGroup21},
};

// The same for the eight-wave tile kernels that are left beside them: 64-row waves at head_dim 16 to 64,
// 32-row waves at 128.  One workgroup per compute unit: a per sub-tile of a round, b per sub-tile of the mean
// compute unit (idle units leave the others a higher clock), c per round.
constexpr Cost kCostTile[4][3] = {       // [head_dim][plain, causal, mask], fwd_kernel_pingpong
    {{0.585f, 0.0251f, 2.44f}, {0.621f, 0.0232f, 3.88f}, {0.852f, 0.102f, 3.31f}},
    {{0.587f, 0.0616f, 2.17f}, {0.589f, 0.0622f, 2.86f}, {1.02f, 0.0687f, 2.33f}},
    {{0.502f, 0.394f, 4.71f}, {0.537f, 0.217f, 17.3f}, {1.16f, 0.213f, 9.3f}},
    {{0.39f, 0.506f, 4.64f}, {0.591f, 0.203f, 8.23f}, {}},
};
constexpr Cost kCostTile16[2][2] = {     // [head_dim 64, 128][plain, causal], fwd_kernel_pp16
    {{0.519f, 0.34f, 7.48f}, {0.548f, 0.357f, 5.95f}},
    {{0.174f, 0.683f, 6.67f}, {0.57f, 0.289f, 6.49f}},
};

// ... and for causal launches of 32-row waves at head_dim 64 (500 random shapes that fit one round of them)
constexpr Cost kCostTile256 = {0.52f, 0.0564f, 4.93f};
// Causal launches with their tiles dealt out: a per sub-tile of the busiest workgroup, b per sub-tile of the mean
// one, s per sub-tile of the mean one and head of its XCD, up to the 32 that its workgroups can be on at a
// time (each head's K and V then serve one workgroup instead of many: half as long again at B17 R40 L1635 H128),
// c per tile of a workgroup.  64-row and 32-row waves at head_dim 64, 32-row waves at 128.
constexpr GroupCost kCostDealt[3] = {{0.506f, 0.381f, 0.00144f, 2.25f}, {0.153f, 0.293f, 0.0184f, 0.793f}, {0.0864f, 0.73f, 0.0046f, 4.77f}};

float ceil_f(float x) {
    const float t = (float)(int64_t)x;
    return t < x ? t + 1.f : t;
}

// `tile` and `p` hold the launch of the tile kernels (validate).
Variant pick_variant(int64_t B, int64_t R, int64_t L, int64_t H, bool has_mask, bool causal, const Shape& tile,
                     const fa::FwdParams& p) {
    const int h = H == 16 ? 0 : H == 32 ? 1 : H == 64 ? 2 : 3;
    const int m = has_mask ? 2 : causal ? 1 : 0;
    const float heads = (float)(B * R), nsub = (float)ceil_div(L, 32);
    Variant best{kGroup11, 8};
    float least = 3.0e38f;
    auto offer = [&](VariantKind kind, int waves, float us) {
        if (us < least) {
            least = us;
            best = Variant{kind, waves};
        }
    };
    // short sequences only: the fit ends at 2048, and the vector cache bounds the kernel on long ones
    if (L <= 2048) {
        const float wgs = heads * (float)ceil_div(L, 16) / kNumCu;
        const float mean = causal ? 0.5f * (nsub + 0.5f) : nsub;
        for (int waves = 2; waves <= (nsub > 2.f ? 4 : 2); waves += 2) {
            const Cost& t = waves == 2 ? kCostSplit2[h][m] : kCostSplit4[h][m];
            offer(kSplit, waves, kLaunch + t.a * ceil_f(nsub / (float)waves) + t.b * wgs * mean + t.c * ceil_f(wgs));
        }
    }
    for (const GroupShape& g : kGroups) {
        if (g.nq == 2 && H == 128 && m != 0) continue;         // (group21_offered)
        if (has_mask && L < 8) continue;                       // (SplitMask::load_any)
        const int rows = 16 * g.nq * (8 / g.gk);
        const float wgs = heads * (float)ceil_div(L, rows) / kNumCu, k = ceil_f(wgs);
        const float mean = causal ? 0.5f * (nsub + (float)rows / 32.f) : nsub;
        const float rounds = ceil_f(wgs / (float)g.resident[h]);
        const GroupCost& t = g.cost[h][m];
        const float shared = k < (float)g.resident[h] ? k : (float)g.resident[h];
        offer(g.kind, 8, kLaunch + t.c * k + (t.a * (nsub + (rounds - 1.f) * mean) + t.b * mean * 0.5f * (wgs + k) + t.s * nsub * shared) / (float)g.gk);
    }
    if (tile.waves != 0) {
        const float n = (float)ceil_div(L, tile.rows()), steps = (float)tile.rows() / 32.f;     // sub-tiles per block
        if (causal && p.heads_per_xcd > 0) {
            const float hx = (float)p.heads_per_xcd, worst = (float)plan_causal(B * R, (int64_t)n, H).blocks * steps;
            const float mean = 0.5f * n * (n + 1.f) * heads * steps / kNumCu;
            const GroupCost& t = kCostDealt[H == 128 ? 2 : tile.nqb == 1 ? 1 : 0];
            offer(kTile, 8, kLaunch + t.a * worst + mean * (t.b + t.s * (hx < 32.f ? hx : 32.f)) +
                                t.c * ceil_f(hx * n * fa::kNumXcd / kNumCu));
            return best;
        }
        // a pair of tiles per workgroup: causal ones, and masked ones where the grid says so
        const float u = (float)p.total_wgs / kNumCu, chain = causal ? (n + 1.f) * steps : nsub * ceil_f(n / (float)p.n_qtiles);
        const Cost& t = H == 64 && tile.nqb == 1 ? kCostTile256
                        : !has_mask && use_tiles16(H, tile, p, causal) ? kCostTile16[h - 2][causal ? 1 : 0] : kCostTile[h][m];
        const float rounds = ceil_f(u);
        offer(kTile, 8, kLaunch + chain * (t.a * rounds + t.b * u) + t.c * rounds);
    }
    return best;
}

// The launch of a key-split or group kernel in place of the tile kernels' one.
int use_variant(const Variant& v, fa::FwdParams* p) {
    int64_t rows = 16;
    for (const GroupShape& g : kGroups)
        if (g.kind == v.kind) rows = 16 * g.nq * (8 / g.gk);
    const int64_t per_head = ceil_div(p->L, rows), total = (int64_t)p->B * p->R * per_head;
    if (total > 0x7fffffff - 8) return FA_ERR_TOO_LARGE;
    p->n_qtiles = (int)per_head;
    p->total_wgs = (int)total;
    p->wgs_per_xcd = (int)ceil_div(total, fa::kNumXcd);
    p->heads_per_xcd = 0;
    p->waves = v.waves;
    return FA_OK;
}

// The launch fa_fwd makes for a problem on dense tensors, without making it.
int describe_launch(int64_t B, int64_t R, int64_t L, int64_t H, int flags, int has_mask, Shape* shape, Variant* v, fa::FwdParams* p) {
    if ((flags & ~(FA_FLAG_CAUSAL | FA_FLAG_BF16)) != 0) return FA_ERR_BAD_FLAGS;
    const bool causal = (flags & FA_FLAG_CAUSAL) != 0;
    if (causal && has_mask) return FA_ERR_BAD_FLAGS;
    // validate() only looks at the pointers' alignment
    void* const fake = reinterpret_cast<void*>(static_cast<uintptr_t>(4096));
    const Strides dense{L * R * H, H, R * H};
    const int rc = validate(fake, fake, fake, has_mask ? fake : nullptr, fake, B, R, L, H, dense, dense, p, 1.0f, shape, causal, nullptr);
    if (rc != FA_OK) return rc;
    *v = pick_variant(B, R, L, H, has_mask != 0, causal, *shape, *p);
    return v->kind != kTile ? use_variant(*v, p) : FA_OK;
}

}  // namespace

extern "C" {

int fa_fwd_query(int64_t H) { return (H == 16 || H == 32 || H == 64 || H == 128) ? 1 : 0; }

// 11 - ceil(log2 L): a tail of L small weights then loses at most 2^-13 of a row (see kBiasMin)
float fa_fwd_reference_bias(int64_t L) {
    int log2_len = 0;
    while (log2_len < 62 && ((int64_t)1 << log2_len) < L) ++log2_len;
    const float bias = 11.0f - (float)log2_len;
    return bias < fa::kBiasMin ? fa::kBiasMin : (bias > fa::kBiasMax ? fa::kBiasMax : bias);
}

const char* fa_strerror(int status) {
    switch (status) {
        case FA_OK: return "success";
        case FA_ERR_NULL_POINTER: return "fa_fwd: q, k, v and out must be non-null device pointers";
        case FA_ERR_BAD_HEAD_DIM: return "fa_fwd: head_dim must be 16, 32, 64 or 128";
        case FA_ERR_BAD_SHAPE:
            return "fa_fwd: B, R and L must be at least 1 (fa_qkv_proj: and the feature counts multiples of 64)";
        case FA_ERR_BAD_STRIDE:
            return "fa_fwd: strides must be non-negative multiples of 8 elements and stride_l >= head_dim";
        case FA_ERR_MISALIGNED: return "fa_fwd: q, k, v and out must be 16-byte aligned";
        case FA_ERR_TOO_LARGE: return "fa_fwd: problem size exceeds the supported index range";
        case FA_ERR_BAD_FLAGS: return "fa_fwd_ex: unknown flag, or FA_FLAG_CAUSAL together with a mask";
        case FA_ERR_BAD_SCALE: return "fa_fwd: scale must be finite and positive";
        default: break;
    }
    if (status > 0) return hipGetErrorString(static_cast<hipError_t>(status));
    return "fa_fwd: unknown status";
}

int fa_fwd_strided(const void* q, const void* k, const void* v, const void* mask, void* out, void* lse,
                   int64_t B, int64_t R, int64_t L, int64_t H, int64_t stride_b, int64_t stride_h,
                   int64_t stride_l, int64_t out_stride_b, int64_t out_stride_h, int64_t out_stride_l,
                   float scale, int flags, void* stream) {
    if ((flags & ~(FA_FLAG_CAUSAL | FA_FLAG_BF16)) != 0) return FA_ERR_BAD_FLAGS;
    const bool causal = (flags & FA_FLAG_CAUSAL) != 0;
    const bool bf16 = (flags & FA_FLAG_BF16) != 0;
    if (causal && mask != nullptr) return FA_ERR_BAD_FLAGS;
    if (lse != nullptr && (reinterpret_cast<uintptr_t>(lse) & 3u) != 0) return FA_ERR_MISALIGNED;
    fa::FwdParams p;
    Shape shape{0, 0};
    const int rc = validate(q, k, v, mask, out, B, R, L, H, Strides{stride_b, stride_h, stride_l},
                            Strides{out_stride_b, out_stride_h, out_stride_l}, &p, scale, &shape, causal, lse);
    if (rc != FA_OK) return rc;
    if (bf16) p.bias = fa::kBiasBf16;
    const Variant variant = pick_variant(B, R, L, H, mask != nullptr, causal, shape, p);
    const int rcv = variant.kind != kTile ? use_variant(variant, &p) : FA_OK;
    // A grid of 2^32 threads or more does not fit the dispatch packet (head_dim 16, L = 43: from 11 million heads
    // on): such a problem runs as two, halves of the batch or of the heads.
    const int64_t threads = (int64_t)p.wgs_per_xcd * fa::kNumXcd * 64 * (variant.kind == kSplit ? variant.waves : 8);
    if (rcv != FA_OK && B * R == 1) return rcv;
    if ((rcv != FA_OK || threads > 0xffffffffll) && B * R > 1) {
        const int64_t B1 = B > 1 ? B / 2 : 1, R1 = B > 1 ? R : R / 2;
        const int64_t in = B > 1 ? B1 * stride_b : R1 * stride_h, to = B > 1 ? B1 * out_stride_b : R1 * out_stride_h;
        auto at = [](const void* ptr, int64_t elements) { return static_cast<const uint16_t*>(ptr) + elements; };
        const int first = fa_fwd_strided(q, k, v, mask, out, lse, B1, R1, L, H, stride_b, stride_h, stride_l, out_stride_b,
                                         out_stride_h, out_stride_l, scale, flags, stream);
        if (first != FA_OK) return first;
        return fa_fwd_strided(at(q, in), at(k, in), at(v, in), mask != nullptr && B > 1 ? at(mask, B1 * L * L) : mask,
                              const_cast<uint16_t*>(at(out, to)), lse != nullptr ? static_cast<float*>(lse) + B1 * R1 * L : nullptr,
                              B > 1 ? B - B1 : 1, B > 1 ? R : R - R1, L, H, stride_b, stride_h, stride_l, out_stride_b,
                              out_stride_h, out_stride_l, scale, flags, stream);
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipError_t e;
    if (variant.kind != kTile) {
        const int mode = causal ? fa::kCausal : mask != nullptr ? fa::kAdditive : fa::kPlain;
        e = bf16 ? dispatch_variant_mode<true>(H, mode, variant, p, s) : dispatch_variant_mode<false>(H, mode, variant, p, s);
    } else if (mask == nullptr && use_tiles16(H, shape, p, causal))
        e = launch_tiles16(H, causal ? (p.heads_per_xcd > 0 ? fa::kCausalDealt : fa::kCausal) : fa::kPlain, bf16, p, s);
    else if (causal && p.heads_per_xcd > 0)
        e = dispatch<fa::kCausalDealt>(H, shape, p, s, bf16);
    else if (causal)
        e = dispatch<fa::kCausal>(H, shape, p, s, bf16);
    else if (mask != nullptr && L % 8 != 0)
        e = dispatch<fa::kAdditiveRagged>(H, shape, p, s, bf16);
    else if (mask != nullptr)
        e = dispatch<fa::kAdditive>(H, shape, p, s, bf16);
    else
        e = dispatch<fa::kPlain>(H, shape, p, s, bf16);
    return static_cast<int>(e);
}

int fa_fwd_plan(int64_t B, int64_t R, int64_t L, int64_t H, int flags, int has_mask, int* plan) {
    if (plan == nullptr) return FA_ERR_NULL_POINTER;
    fa::FwdParams p;
    Shape shape{0, 0};
    Variant v{kTile, 0};
    const int rc = describe_launch(B, R, L, H, flags, has_mask, &shape, &v, &p);
    if (rc != FA_OK) return rc;
    const bool tile = v.kind == kTile;
    plan[0] = v.waves;
    plan[1] = tile ? 32 * shape.nqb : v.kind == kGroup21 ? 32 : 16;
    plan[2] = p.wgs_per_xcd * fa::kNumXcd;
    plan[3] = p.total_wgs;
    plan[4] = p.n_qtiles;
    plan[5] = p.heads_per_xcd;
    plan[6] = !tile || (!has_mask && use_tiles16(H, shape, p, (flags & FA_FLAG_CAUSAL) != 0)) ? 16 : 32;
    return FA_OK;
}

int fa_fwd_variant(int64_t B, int64_t R, int64_t L, int64_t H, int flags, int has_mask, int* variant) {
    if (variant == nullptr) return FA_ERR_NULL_POINTER;
    fa::FwdParams p;
    Shape shape{0, 0};
    Variant v{kTile, 0};
    const int rc = describe_launch(B, R, L, H, flags, has_mask, &shape, &v, &p);
    if (rc != FA_OK) return rc;
    int rows = v.kind == kTile ? shape.rows() : 16, groups = v.kind == kSplit ? v.waves : 1;
    for (const GroupShape& g : kGroups)
        if (g.kind == v.kind) {
            rows = 16 * g.nq * (8 / g.gk);
            groups = g.gk;
        }
    variant[0] = v.kind == kTile ? 0 : v.kind == kSplit ? 1 : 2;
    variant[1] = v.waves;
    variant[2] = rows;
    variant[3] = groups;
    variant[4] = p.wgs_per_xcd * fa::kNumXcd;
    variant[5] = p.total_wgs;
    variant[6] = p.n_qtiles;
    return FA_OK;
}

int fa_fwd_ex(const void* q, const void* k, const void* v, const void* mask, void* out, void* lse,
              int64_t B, int64_t R, int64_t L, int64_t H, int64_t stride_b, int64_t stride_h,
              int64_t stride_l, float scale, int flags, void* stream) {
    return fa_fwd_strided(q, k, v, mask, out, lse, B, R, L, H, stride_b, stride_h, stride_l, stride_b, stride_h,
                          stride_l, scale, flags, stream);
}

int fa_fwd(const void* q, const void* k, const void* v, const void* mask, void* out, int64_t B,
           int64_t R, int64_t L, int64_t H, int64_t stride_b, int64_t stride_h, int64_t stride_l,
           float scale, void* stream) {
    return fa_fwd_ex(q, k, v, mask, out, nullptr, B, R, L, H, stride_b, stride_h, stride_l, scale, 0,
                     stream);
}

int fa_fwd_timed_ex(const void* q, const void* k, const void* v, const void* mask, void* out, void* lse,
                    int64_t B, int64_t R, int64_t L, int64_t H, int64_t stride_b, int64_t stride_h,
                    int64_t stride_l, int64_t out_stride_b, int64_t out_stride_h, int64_t out_stride_l,
                    float scale, int flags, void* stream, int iters, float* ms_per_launch) {
    if (ms_per_launch == nullptr) return FA_ERR_NULL_POINTER;
    if (iters < 1) return FA_ERR_BAD_SHAPE;
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipError_t e = hipEventCreate(&e0);
    if (e != hipSuccess) return static_cast<int>(e);
    e = hipEventCreate(&e1);
    if (e != hipSuccess) {
        (void)hipEventDestroy(e0);
        return static_cast<int>(e);
    }
    int rc = FA_OK;
    e = hipEventRecord(e0, s);
    if (e != hipSuccess) rc = static_cast<int>(e);
    for (int i = 0; i < iters && rc == FA_OK; ++i)
        rc = fa_fwd_strided(q, k, v, mask, out, lse, B, R, L, H, stride_b, stride_h, stride_l, out_stride_b,
                            out_stride_h, out_stride_l, scale, flags, stream);
    if (rc == FA_OK) {
        e = hipEventRecord(e1, s);
        if (e == hipSuccess) e = hipEventSynchronize(e1);
        float ms = 0.f;
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
        if (e == hipSuccess)
            *ms_per_launch = ms / (float)iters;
        else
            rc = static_cast<int>(e);
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return rc;
}

int fa_fwd_timed(const void* q, const void* k, const void* v, const void* mask, void* out, int64_t B,
                 int64_t R, int64_t L, int64_t H, int64_t stride_b, int64_t stride_h,
                 int64_t stride_l, float scale, void* stream, int iters, float* ms_per_launch) {
    return fa_fwd_timed_ex(q, k, v, mask, out, nullptr, B, R, L, H, stride_b, stride_h, stride_l, stride_b,
                           stride_h, stride_l, scale, 0, stream, iters, ms_per_launch);
}

}  // extern "C"

namespace {
template <int HR, bool BF>
hipError_t launch_qkv(const fa::qkv::Params& p, hipStream_t stream) {
    auto kernel = fa::qkv::qkv_proj_kernel<HR, BF>;
    constexpr int kQkvLds = fa::qkv::kLdsBytes;
    constexpr int kQkvThreads = fa::qkv::kWaves * 64;
    const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kernel), kQkvLds);
    if (e != hipSuccess) return e;
    fa::qkv::Params params = p;
    void* args[] = {&params};
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(p.wgs_per_xcd * fa::kNumXcd),
                           dim3(kQkvThreads), args, kQkvLds, stream);
}

// Tiles and grid of the projection kernel for an M x N output.
int qkv_geometry(int64_t M, int64_t N, fa::qkv::Params* p) {
    constexpr int64_t kMaxInt = 0x7fffffff;
    const int64_t tiles_m = ceil_div(M, fa::qkv::kTileM);
    p->tiles_n = (int)ceil_div(N, fa::qkv::kTileN);
    if (tiles_m * p->tiles_n > kMaxInt - 8) return FA_ERR_TOO_LARGE;
    p->total_tiles = (int)(tiles_m * p->tiles_n);
    // a resident grid, one workgroup per compute unit, each walking through its share of the tiles
    p->total_wgs = p->total_tiles < kNumCu ? p->total_tiles : kNumCu;
    p->wgs_per_xcd = (int)ceil_div(p->total_wgs, fa::kNumXcd);
    return FA_OK;
}

// The small-tile kernel's shapes (SmallTile): 16-row and 16-feature blocks per wave, waves per group, groups, slots.
using Tile128x256 = fa::qkv::SmallTile<4, 4, 2, 4, 1, 3>;
using Tile128x128 = fa::qkv::SmallTile<4, 4, 2, 2, 2, 3>;
using Tile64x128 = fa::qkv::SmallTile<2, 4, 2, 2, 2, 3>;
using Tile64x64 = fa::qkv::SmallTile<2, 2, 2, 2, 2, 4>;

// Which kernel runs a projection: 0 the 256 x 256 one, otherwise the small-tile kernel with a shape of kQkvTiles.
enum QkvKind { kQkvWhole, kQkv128x256, kQkv128x128, kQkv64x128, kQkv64x64, kQkvKinds };
struct QkvTile {
    int tm, tn;
};
constexpr QkvTile kQkvTiles[kQkvKinds] = {{fa::qkv::kTileM, fa::qkv::kTileN},
                                          {Tile128x256::TM, Tile128x256::TN},
                                          {Tile128x128::TM, Tile128x128::TN},
                                          {Tile64x128::TM, Tile64x128::TN},
                                          {Tile64x64::TM, Tile64x64::TN}};

template <int HR, bool BF, int MT, int NT, int WM, int WN, int KG, int SLOTS>
hipError_t launch_qkv_small(fa::qkv::SmallTile<MT, NT, WM, WN, KG, SLOTS>, const fa::qkv::Params& p, hipStream_t stream) {
    constexpr int lds = fa::qkv::SmallTile<MT, NT, WM, WN, KG, SLOTS>::LDS;
    auto kernel = fa::qkv::qkv_proj_small_kernel<HR, BF, MT, NT, WM, WN, KG, SLOTS>;
    const hipError_t e = allow_large_lds(reinterpret_cast<const void*>(kernel), lds);
    if (e != hipSuccess) return e;
    fa::qkv::Params params = p;
    void* args[] = {&params};
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(p.wgs_per_xcd * fa::kNumXcd), dim3(fa::qkv::kWaves * 64),
                           args, lds, stream);
}

template <int HR, bool BF>
hipError_t dispatch_qkv_kind(QkvKind kind, const fa::qkv::Params& p, hipStream_t stream) {
    switch (kind) {
        case kQkvWhole: return launch_qkv<HR, BF>(p, stream);
        case kQkv128x256: return launch_qkv_small<HR, BF>(Tile128x256{}, p, stream);
        case kQkv128x128: return launch_qkv_small<HR, BF>(Tile128x128{}, p, stream);
        case kQkv64x128: return launch_qkv_small<HR, BF>(Tile64x128{}, p, stream);
        case kQkv64x64: return launch_qkv_small<HR, BF>(Tile64x64{}, p, stream);
        default: return hipErrorInvalidValue;
    }
}

template <bool BF>
hipError_t dispatch_qkv(int64_t rope_head_dim, QkvKind kind, const fa::qkv::Params& p, hipStream_t stream) {
    switch (rope_head_dim) {
        case 0: return dispatch_qkv_kind<0, BF>(kind, p, stream);
        case 16: return dispatch_qkv_kind<16, BF>(kind, p, stream);
        case 32: return dispatch_qkv_kind<32, BF>(kind, p, stream);
        case 64: return dispatch_qkv_kind<64, BF>(kind, p, stream);
        case 128: return dispatch_qkv_kind<128, BF>(kind, p, stream);
        default: return hipErrorInvalidValue;
    }
}

// Time of a projection in microseconds, fitted on 2853 random shapes (M 32..16384, N 192..15360, K 64..5120, both
// types, with and without tables) on MI355X: half of the estimates are within 3.6 %, and choosing the smallest
// one loses 0.12 % against the best kernel of each shape (over 3 % for 41 of them, 18 % at most).  (A fit over
// 300 of them that favoured the 256 x 256 kernel by 4 %: 0.25 %, 72 shapes, 51 %; of 59 shapes that those 4 %
// decided, 31 went to the slower kernel.)  With k workgroups on the busiest of the 256 compute units, w on the mean
// one and rounds = k over the resident ones:
//   launch + K / 64 (round rounds + busiest k + mean w) + (start + start_rope) rounds + (end + end_rope) k
struct QkvCost {
    int resident;
    float launch, round, busiest, mean, start, end, start_rope, end_rope;
};
constexpr QkvCost kQkvCost[kQkvKinds] = {
    {1, 0.84f, 1.04f, 0.f, 0.542f, 5.85f, 0.f, 2.84f, 0.f},
    {1, 0.43f, 0.514f, 0.f, 0.308f, 4.61f, 0.f, 2.14f, 0.f},
    {1, 1.29f, 0.303f, 0.f, 0.143f, 3.04f, 0.f, 0.961f, 0.f},
    {2, 2.54f, 0.0987f, 0.11f, 0.134f, 0.f, 0.919f, 0.0769f, 0.5f},
    {2, 2.74f, 0.0456f, 0.0856f, 0.0836f, 0.f, 0.536f, 0.0806f, 0.381f},
};

QkvKind pick_qkv(int64_t M, int64_t N, int64_t K, bool rope) {
    QkvKind best = kQkvWhole;
    float least = 3.0e38f;
    const float slices = (float)(K / fa::qkv::kTileK);
    for (int kind = 0; kind < kQkvKinds; ++kind) {
        const QkvCost& c = kQkvCost[kind];
        const float mean = (float)ceil_div(M, kQkvTiles[kind].tm) * (float)ceil_div(N, kQkvTiles[kind].tn) / kNumCu;
        // (a grid of less than 2^32 threads: the dispatch packet holds no more)
        if (kind != kQkvWhole && mean > (float)(0xffffffffu / (64 * fa::qkv::kWaves) / kNumCu - 1)) continue;
        const float busiest = ceil_f(mean), rounds = ceil_f(mean / (float)c.resident);
        float us = c.launch + slices * (c.round * rounds + c.busiest * busiest + c.mean * mean) + c.start * rounds + c.end * busiest;
        if (rope) us += c.start_rope * rounds + c.end_rope * busiest;
        if (us < least) {
            least = us;
            best = (QkvKind)kind;
        }
    }
    return best;
}

// The launch of a small-tile kernel in place of the 256 x 256 one's.
int use_qkv_kind(QkvKind kind, fa::qkv::Params* p) {
    if (kind == kQkvWhole) return FA_OK;
    const QkvTile t = kQkvTiles[kind];
    const int64_t tiles_n = ceil_div(p->N, t.tn), tiles_m = ceil_div(p->M, t.tm), tiles = tiles_m * tiles_n;
    if (tiles > 0x7fffffff - 8) return FA_ERR_TOO_LARGE;
    const int64_t band = (int64_t)fa::qkv::kBand * fa::qkv::kTileM / t.tm;
    p->tiles_m = (int)tiles_m;
    p->by_band = fa::divisor(band * tiles_n);
    p->by_last = fa::divisor(tiles_m % band != 0 ? tiles_m % band : band);
    p->by_len = fa::divisor(p->L);
    p->tiles_n = (int)tiles_n;
    p->total_tiles = (int)tiles;
    p->total_wgs = (int)tiles;
    p->wgs_per_xcd = (int)ceil_div(tiles, fa::kNumXcd);
    return FA_OK;
}
}  // namespace

extern "C" {

int fa_qkv_proj(const void* x, const void* w, const void* bias, void* qkv, int64_t B, int64_t L, int64_t F_in,
                int64_t R, int64_t H, const float* rope_cos, const float* rope_sin, int flags, void* stream) {
    if ((flags & ~FA_FLAG_BF16) != 0) return FA_ERR_BAD_FLAGS;
    if (x == nullptr || w == nullptr || qkv == nullptr) return FA_ERR_NULL_POINTER;
    if ((rope_cos == nullptr) != (rope_sin == nullptr)) return FA_ERR_NULL_POINTER;
    if (!fa_fwd_query(H)) return FA_ERR_BAD_HEAD_DIM;
    if (B < 1 || L < 1 || R < 1 || F_in < 1) return FA_ERR_BAD_SHAPE;
    constexpr int64_t kMaxInt = 0x7fffffff;
    if (B > kMaxInt || L > kMaxInt || R > kMaxInt || B * L > kMaxInt - 2 * fa::qkv::kTileM) return FA_ERR_TOO_LARGE;
    const int64_t F = R * H;
    // the contraction is walked in whole steps of 64, and the three slices start on 64-feature boundaries
    if (F_in % fa::qkv::kTileK != 0 || F % 64 != 0) return FA_ERR_BAD_SHAPE;
    // the loaders keep 32-bit byte offsets inside a tile: 256 rows of x, 64 rows of w
    if (F_in > ((int64_t)1 << 22) || F > ((int64_t)1 << 22)) return FA_ERR_TOO_LARGE;
    if (!aligned16(x) || !aligned16(w) || !aligned16(qkv) || !aligned16(rope_cos) || !aligned16(rope_sin) ||
        (reinterpret_cast<uintptr_t>(bias) & 7u) != 0)
        return FA_ERR_MISALIGNED;
    fa::qkv::Params p;
    p.x = static_cast<const _Float16*>(x);
    p.w = static_cast<const _Float16*>(w);
    p.bias = static_cast<const _Float16*>(bias);
    p.out = static_cast<_Float16*>(qkv);
    p.rope_cos = rope_cos;
    p.rope_sin = rope_sin;
    p.M = (int)(B * L);
    p.K = (int)F_in;
    p.N = (int)(3 * F);
    p.F = (int)F;
    p.L = (int)L;
    const int rc = qkv_geometry(B * L, 3 * F, &p);
    if (rc != FA_OK) return rc;
    const QkvKind kind = pick_qkv(B * L, 3 * F, F_in, rope_cos != nullptr);
    const int rck = use_qkv_kind(kind, &p);
    if (rck != FA_OK) return rck;
    const int64_t hr = rope_cos != nullptr ? H : 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const hipError_t e = (flags & FA_FLAG_BF16) != 0 ? dispatch_qkv<true>(hr, kind, p, s) : dispatch_qkv<false>(hr, kind, p, s);
    return static_cast<int>(e);
}

int fa_qkv_proj_plan(int64_t B, int64_t L, int64_t F_in, int64_t R, int64_t H, int* plan) {
    if (plan == nullptr) return FA_ERR_NULL_POINTER;
    if (!fa_fwd_query(H)) return FA_ERR_BAD_HEAD_DIM;
    if (B < 1 || L < 1 || R < 1 || F_in < 1) return FA_ERR_BAD_SHAPE;
    constexpr int64_t kMaxInt = 0x7fffffff;
    if (B > kMaxInt || L > kMaxInt || R > kMaxInt || B * L > kMaxInt - 2 * fa::qkv::kTileM) return FA_ERR_TOO_LARGE;
    const int64_t F = R * H;
    if (F_in % fa::qkv::kTileK != 0 || F % 64 != 0) return FA_ERR_BAD_SHAPE;
    if (F_in > ((int64_t)1 << 22) || F > ((int64_t)1 << 22)) return FA_ERR_TOO_LARGE;
    fa::qkv::Params p;
    const int rc = qkv_geometry(B * L, 3 * F, &p);
    if (rc != FA_OK) return rc;
    plan[0] = p.wgs_per_xcd * fa::kNumXcd;
    plan[1] = p.total_wgs;
    plan[2] = p.total_tiles;
    plan[3] = p.tiles_n;
    return FA_OK;
}

int fa_qkv_proj_variant(int64_t B, int64_t L, int64_t F_in, int64_t R, int64_t H, int rope, int* variant) {
    int plan[4];
    if (variant == nullptr) return FA_ERR_NULL_POINTER;
    int rc = fa_qkv_proj_plan(B, L, F_in, R, H, plan);
    if (rc != FA_OK) return rc;
    fa::qkv::Params p;
    p.M = (int)(B * L);
    p.N = (int)(3 * R * H);
    p.L = (int)L;
    rc = qkv_geometry(p.M, p.N, &p);
    if (rc != FA_OK) return rc;
    const QkvKind kind = pick_qkv(p.M, p.N, F_in, rope != 0);
    rc = use_qkv_kind(kind, &p);
    if (rc != FA_OK) return rc;
    variant[0] = kQkvTiles[kind].tm;
    variant[1] = kQkvTiles[kind].tn;
    variant[2] = p.wgs_per_xcd * fa::kNumXcd;
    variant[3] = p.total_wgs;
    variant[4] = p.total_tiles;
    variant[5] = p.tiles_n;
    return FA_OK;
}

}  // extern "C"
