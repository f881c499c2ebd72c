// flash_attn.hip -- fused attention forward for gfx950 with the paper's
// score programs inside the tile loop: the attention-side integration site
// the reference reaches through its FA4 fork (src/sfu_repro/fa4.py:454-752,
// extras/paper/manuscript/main.tex:483-509), whose kernel is not part of the
// reference tree.
//
// Modes (AttnMode): softmax with hardware exp2 (v_exp_f32), the B5 D2 "safe",
// FA4 D3 or PWL2 exp2 polynomial (every exponent, or four of every ROUTE);
// tanh softcap (B2) cap*tanh(s/cap) with FP32 hardware tanh or the D4 BF16
// program, followed by the hardware softmax; sigmoid attention
// p = sigmoid(s + bias) with hardware exp/rcp, the B3 direct D3 or B3-D2
// program (fitted for n = 4096) or the BF16 sigmoid D3-D6 programs,
// unnormalised O = P V.
//
// Layout: Q, O [B, Hq, S, D] and K, V [B, Hkv, S, D] at any element strides
// with a contiguous head dimension (D 64 or 128), BF16, grouped-query heads
// (Hq a multiple of Hkv), any S (the last block may be partial), optional causal mask.
// s = q.k * scale.
//
// Design (all-transposed MFMA formulation, v_mfma_f32_32x32x16_bf16):
//  * a block of 4 or 8 waves owns 32 queries per wave, held as the B operand
//    Q^T (fragments of 8 BF16 per lane);
//  * 64-key tiles of K and V move from memory straight into rings of LDS
//    tiles (load_to_lds, swizzled rows): K three and V two tiles ahead with 8
//    waves, both one ahead with 4, both two ahead at head_dim 64; Q takes the
//    same way once, through the V ring;
//  * S^T = K Q^T: lane (h, c) of a wave accumulates 16 keys x query c for
//    each 32-key tile, so every per-query reduction is lane-local plus one
//    exchange with lane c + 32;
//  * O^T = V^T P^T: the S^T accumulator registers become the P^T fragments
//    with no data movement by numbering the MFMA k index in the order the
//    accumulator holds the keys; the V^T fragments come from the row-major V
//    tile in the same order through gfx950's transposing LDS reads
//    (ds_read_b64_tr_b16, two per fragment), and O^T keeps each lane on its
//    own query, so the online-softmax rescale is lane-local too;
//  * one barrier per tile.  With 8 waves, two to a SIMD, waves 0-3 meet it
//    ahead of S and waves 4-7 ahead of O += P V, so the two waves of a SIMD
//    stay half a tile apart and one's MFMAs meet the other's score program;
//  * O leaves through LDS, whole rows to memory;
//  * causal blocks run from the heaviest query block down.
//
// What bounds it: the score program's issue slots next to the matrix cores
// (head_dim 128, causal, S 4096, 32 query heads: 4,160 MFMAs of 32 cycles a
// SIMD, 65 us of its time at 2.05 GHz), and the power budget: the clock is
// 2.05 GHz here and 1.8 GHz where MFMAs run back to back.
#include <hip/hip_runtime.h>

#include "flash_attn.hpp"
#include "spline_ops_hip.h"

namespace pt {

struct AttnParams {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    uint16_t* o;
    uint16_t* o2;  // the same rows at strides o2s, or null
    float* lse;  // [B, Hq, S] natural-log partition function, or null
    AttnStrides qs, ks, vs, os, o2s;
    int64_t hq, hkv, seq;
    int64_t kv_len;  // keys 0 .. kv_len - 1 are real, the rest padding (masked)
    float scale;     // s = q.k * scale
    float cap;       // softcap
    float sig_bias;  // sigmoid attention: p = sigmoid(s + sig_bias)
    int causal;
    int route;       // exp2 route of the kRouteRuntime instantiations
    uint32_t rmask;  // and its periodic mask (routes up to 32)
    int group;       // query heads per KV head
    int wide;        // a row stride too large for 32-bit lane offsets
};

// Launch constants of the score programs, in VGPRs (vgpr()).
struct ScoreConsts {
    float scale;    // s = q.k * scale
    float sl;       // softmax modes: log2 e times the unit of the exponents
    float cap, inv_cap, bias;
    float tanh[SoftcapConsts::T::P.deg + 1];  // softcap D4
};

template <int MODE>
__device__ __forceinline__ ScoreConsts score_consts(const AttnParams& p) {
    ScoreConsts c;
    c.scale = vgpr(p.scale);
    c.sl = vgpr(attn_is_plain_softmax(MODE) ? p.scale * kLog2e : kLog2e);
    c.cap = vgpr(p.cap);
    c.inv_cap = vgpr(1.0f / p.cap);
    c.bias = vgpr(p.sig_bias);
#pragma unroll
    for (int i = 1; i <= SoftcapConsts::T::P.deg; ++i) c.tanh[i] = vgpr(bf16_value(SoftcapConsts::T::P.c[i]));
    return c;
}

// Softmax scores of 16 accumulator registers (one 32-key tile), in the
// units the caller's exponent FMA scales by sl: the raw dot products for
// plain softmax (sl = scale * log2 e), the capped score y for the softcap
// modes (sl = log2 e, so the product by log2 e is the exponent FMA's own).
// The D4 program runs on BF16 pairs: u = bf16(bf16(s) * (1/cap)),
// y = bf16(cap * TANH_D4_BF16(u)), the B2 program on the BF16 score.
template <int MODE>
__device__ __forceinline__ void softmax_exponents(const f32x16_t& acc, const ScoreConsts& k, float (&x)[16]) {
    if constexpr (MODE == kAttnSoftcapD4) {
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            const uint32_t u = pack_bf(rbf(acc[r] * k.scale) * k.inv_cap, rbf(acc[r + 1] * k.scale) * k.inv_cap);
            float t0, t1;
            SoftcapConsts::T::eval2(u, k.tanh, t0, t1);
            x[r] = rbf(t0 * k.cap);
            x[r + 1] = rbf(t1 * k.cap);
        }
    } else {
        static_assert(MODE == kAttnSoftcapNative, "plain softmax keeps the raw dot products");
#pragma unroll
        for (int r = 0; r < 16; ++r)
            x[r] = k.cap * native_lane<kTanh, kFwd>(acc[r] * k.scale * k.inv_cap);
    }
}

// Exponent slot i (kt * 16 + r) of the tile takes the mode's polynomial
// (FA4's routed exp2, four lanes per group of exp2_emu_freq,
// src/sfu_repro/fa4.py:313-353): i % ROUTE < 4 for a template route (ROUTE 4
// routes all), bit i of the tile's mask rmask (tile_route_mask) for
// kRouteRuntime (wave-uniform, so the decision is a scalar branch).  The slot
// is a function of the key index alone (16 bit5 + 4 bits3..4 + bits0..1),
// which the backward evaluates to route the same keys.
template <int ROUTE>
__device__ __forceinline__ bool slot_routed(int i, uint32_t rmask) {
    if constexpr (ROUTE == kRouteRuntime) return (rmask >> i) & 1u;
    else return ROUTE >= 4 && i % ROUTE < 4;
}

// exp2 of a softmax exponent (x <= 8 under the lazy rescale) in slot i.
template <int MODE, int ROUTE>
__device__ __forceinline__ float softmax_exp2(float x, int i, uint32_t rmask) {
    if constexpr (attn_has_exp2_program(MODE))
        if (slot_routed<ROUTE>(i, rmask)) return exp2_lane<attn_exp2_kind<MODE>()>(x);
    return __builtin_amdgcn_exp2f(x);
}

// Two exponents, slots i (even) and i + 1: the routing groups of four start
// at even slots (the route is even), so one decision routes both, and the
// packed FP16 program evaluates them with one instruction per step.
template <int MODE, int ROUTE>
__device__ __forceinline__ void softmax_exp2_pair(float x0, float x1, int i, uint32_t rmask, float& y0, float& y1) {
    if (slot_routed<ROUTE>(i, rmask)) {
        exp2_pair<attn_exp2_kind<MODE>()>(x0, x1, y0, y1);
    } else {
        y0 = __builtin_amdgcn_exp2f(x0);
        y1 = __builtin_amdgcn_exp2f(x1);
    }
}

// Sigmoid-attention probabilities of two scores, before their rounding to
// BF16: the only consumer is the conversion to the BF16 operand of the P V
// product, which performs the programs' final rounding.
template <int MODE>
__device__ __forceinline__ void sigmoid_prob2(float s0, float s1, float bias, float& p0, float& p1) {
    if constexpr (MODE == kAttnSigmoidB3) {
        float dy;
        b3_lane<false, true, true>(rbf(s0), p0, dy);
        b3_lane<false, true, true>(rbf(s1), p1, dy);
    } else if constexpr (MODE == kAttnSigmoidB3D2) {
        float dy;
        b3_d2_lane(rbf(s0), p0, dy);
        b3_d2_lane(rbf(s1), p1, dy);
    } else if constexpr (MODE >= kAttnSigmoidD3 && MODE <= kAttnSigmoidD6) {
        BF16Prog<kSigmoid, kFwd, MODE - kAttnSigmoidD3 + 3>::open2(pack_bf(s0 + bias, s1 + bias), p0, p1);
    } else {
        p0 = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-(s0 + bias) * kLog2e));
        p1 = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-(s1 + bias) * kLog2e));
    }
}

// Rescale threshold of the online softmax (log2 units): the running maximum
// m is only moved when a tile raises it by more than this, so exponents stay
// <= 8 and P <= 256; O and l carry the same stale m, so the final O / l is
// unchanged.  Most tiles skip the 64-register rescale of O.
constexpr float kRescaleThreshold = 8.0f;

// Accumulator register r of 32-key tile kt holds key k0 + kt*32 + 8*(r/4) +
// 4h + r%4; diag = k0 + 4h - klast, with klast the last key the query may
// see (itself under the causal mask, at most the last real key), so the key
// is masked when diag + that offset > 0.
template <bool MASKED>
__device__ __forceinline__ bool key_masked(int diag, int kt, int r) {
    return MASKED && diag + kt * 32 + 8 * (r >> 2) + (r & 3) > 0;
}

// Softmax modes: exponents x of the tile (plain softmax keeps the raw dot
// products and folds the scale into the exp2 argument, sl; softcap modes
// transform first), masked keys to -inf, and the lazy online-max update,
// which rescales O and l when this tile raises the maximum by more than the
// threshold.  Sigmoid modes have no state to update.
template <int MODE, bool MASKED, int HD>
__device__ __forceinline__ void tile_softmax_state(const ScoreConsts& k, const f32x16_t (&sacc)[2], float (&x)[2][16],
                                                   f32x16_t (&oacc)[HD / 32], float& m, float& l, int diag) {
    if constexpr (!attn_is_sigmoid(MODE)) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            if constexpr (attn_is_plain_softmax(MODE)) {
#pragma unroll
                for (int r = 0; r < 16; ++r) x[kt][r] = sacc[kt][r];
            } else {
                softmax_exponents<MODE>(sacc[kt], k, x[kt]);
            }
        }
        // max over four independent chains
        float mx[4] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (key_masked<MASKED>(diag, kt, r)) x[kt][r] = -__builtin_inff();
                mx[r & 3] = __builtin_fmaxf(mx[r & 3], x[kt][r]);
            }
        const float mt =
            half_max(__builtin_fmaxf(__builtin_fmaxf(mx[0], mx[1]), __builtin_fmaxf(mx[2], mx[3]))) * k.sl;
        // lanes c and c + 32 hold the same query and take the same decision
        const bool move = mt > m + kRescaleThreshold;
        // scheduling fences around the rare rescale: without them the
        // scheduler interleaves it with the surrounding code and the register
        // allocator then copies all of O on the common no-rescale path
        __builtin_amdgcn_sched_barrier(0);
        if (__any(move)) {
            const float m_use = move ? mt : m;
            const float alpha = __builtin_amdgcn_exp2f(m - m_use);
            m = m_use;
            l *= alpha;
#pragma unroll
            for (int dt = 0; dt < HD / 32; ++dt) oacc[dt] *= alpha;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Eight probabilities (keys kt*32 + 8cc + {0..3, 4..7} of the accumulator
// layout) as the BF16 B operand of one O^T MFMA; softmax modes add them to
// the four row-sum chains ls.
template <int MODE, int ROUTE, bool MASKED>
__device__ __forceinline__ bf16x8_t tile_probs8(const ScoreConsts& k, const f32x16_t (&sacc)[2],
                                                const float (&x)[2][16], int kt, int cc, float m, int diag,
                                                uint32_t rmask, float (&ls)[4]) {
    float pr[8];
    if constexpr (attn_is_sigmoid(MODE)) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const int r = 8 * cc + e;
            sigmoid_prob2<MODE>(sacc[kt][r] * k.scale, sacc[kt][r + 1] * k.scale, k.bias, pr[e], pr[e + 1]);
            pr[e] = key_masked<MASKED>(diag, kt, r) ? 0.0f : pr[e];
            pr[e + 1] = key_masked<MASKED>(diag, kt, r + 1) ? 0.0f : pr[e + 1];
        }
    } else if constexpr (exp2_is_f16(attn_exp2_kind<MODE>())) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const int r = 8 * cc + e;
            float ev0, ev1;
            softmax_exp2_pair<MODE, ROUTE>(__builtin_fmaf(x[kt][r], k.sl, -m), __builtin_fmaf(x[kt][r + 1], k.sl, -m),
                                           kt * 16 + r, rmask, ev0, ev1);
            pr[e] = key_masked<MASKED>(diag, kt, r) ? 0.0f : ev0;
            pr[e + 1] = key_masked<MASKED>(diag, kt, r + 1) ? 0.0f : ev1;
            ls[e & 3] += pr[e];
            ls[(e + 1) & 3] += pr[e + 1];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int r = 8 * cc + e;
            const float ev = softmax_exp2<MODE, ROUTE>(__builtin_fmaf(x[kt][r], k.sl, -m), kt * 16 + r, rmask);
            // v_exp_f32(-inf) is 0; the polynomial programs clamp at -127
            pr[e] = (attn_has_exp2_program(MODE) && key_masked<MASKED>(diag, kt, r)) ? 0.0f : ev;
            ls[e & 3] += pr[e];
        }
    }
    bf16x8_t pf;
#pragma unroll
    for (int e = 0; e < 8; ++e) pf[e] = (__bf16)pr[e];
    return pf;
}

// Shape of the forward: waves (32 queries each) per block and tiles per LDS
// ring.  head_dim 128: 8 waves that share each staged tile, one block per CU
// with four tiles of K and of V in 130 KiB, or two independent 4-wave blocks
// with two tiles each (fwd_waves picks); head_dim 64: three independent
// 4-wave blocks per CU, three tiles each in 50 KiB.
template <int HD, int W>
struct FwdShape {
    static constexpr int kWaves = W;
    static constexpr int kRing = HD == 64 ? 3 : W == 8 ? 4 : 2;
    static constexpr int kBlockQ = 32 * kWaves;
    static constexpr int kRowB = HD * 2;                      // bytes per row
    static constexpr int kTileB = lds_row<HD>(kAttnBlockK);  // bytes per staged tile
    static constexpr int kChunks = RowLoader<HD>::kChunks, kLoadRows = RowLoader<HD>::kLoadRows;
    static constexpr int kLoads = kAttnBlockK / kLoadRows / kWaves;  // per wave, tile and operand
    static_assert(lds_row<HD>(kBlockQ) <= kRing * kTileB, "Q passes through the V ring");
};

// Waves per SIMD the register allocation is held to: 2 at head_dim 128 (256
// VGPRs), 3 at head_dim 64 (168), where three 4-wave blocks share a CU.
template <int HD>
constexpr int fwd_waves_per_eu() { return HD == 64 ? 3 : 2; }

constexpr bool attn_is_softcap(int mode) { return mode == kAttnSoftcapNative || mode == kAttnSoftcapD4; }

// The kernel's own order of issue (priority while a wave only issues the S
// MFMAs, LDS reads a fixed number ahead of the products) against the
// compiler's: the softcap and sigmoid modes at head_dim 64 run faster the
// latter way (S 4096, 32 heads, causal / not, with the order: hardware sigmoid
// 106 / 200 us, sigmoid D3 127 / 237, B3-D2 125 / 231; without: 104 / 191, 124 /
// 221, 123 / 225).
template <int MODE, int HD>
constexpr bool fwd_ordered() { return HD != 64 || attn_is_plain_softmax(MODE); }

// Each 16 keys' products right behind their probabilities, which then hold 4
// VGPRs instead of 16: the polynomial softmax, B3 and softcap D4 at head_dim 64
// (S 4096, 32 heads, causal / not, against all products behind all
// probabilities: B3 130 / 236 us against 132 / 236, B3-D2 123 / 225 against 125
// / 224, while sigmoid D3 loses, 126 / 226 against 124 / 221, and hardware
// softcap, 168 / 303 against 166 / 299; softcap D4 spills the other way, the
// polynomial softmax is within 3 % either way).
template <int MODE, int HD>
constexpr bool fwd_fused() {
    return HD == 64 && (attn_has_exp2_program(MODE) || MODE == kAttnSigmoidB3 || MODE == kAttnSigmoidB3D2 ||
                        MODE == kAttnSoftcapD4);
}

// Grid (q_heads, ceil(S / (32 W)), batch), W waves of 32 queries per block:
// blockIdx.y runs over query blocks, heaviest first under the causal mask,
// and the head index varies fastest, so the first wave of resident blocks
// takes the longest query blocks of every head.
//
// Any S: rows past the last real key are staged as zeros (their probability
// is 0), queries past the sequence take a row of zeros and store nothing, and
// a wave with no query at all only stages.
template <int MODE, int ROUTE, int HD, int W>
__global__ void __launch_bounds__(64 * W)
    __attribute__((amdgpu_waves_per_eu(fwd_waves_per_eu<HD>()))) flash_fwd_kernel(AttnParams p) {
    using F = FwdShape<HD, W>;
    constexpr int kRing = F::kRing, kRowB = F::kRowB, kTileB = F::kTileB;
    constexpr bool kSigmoid = attn_is_sigmoid(MODE);
    constexpr bool kLate = W == 8;  // the second wave of each SIMD runs half a tile behind
    constexpr bool kOrdered = fwd_ordered<MODE, HD>(), kFused = fwd_fused<MODE, HD>();
    constexpr int kAheadV = kLate ? kRing - 2 : kRing - 1, kInFlight = kLate ? kRing - 3 : kRing - 2;
    constexpr int kC = HD / 16, kD = HD / 32;
    // K ring, V ring
    __shared__ __align__(1024) unsigned char smem[2 * kRing * kTileB];
    constexpr uint32_t kV = kRing * kTileB;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int h = lane >> 5, c32 = lane & 31;
    const int seq = (int)p.seq, klim = (int)p.kv_len - 1;  // the last real key
    const int nqb = (seq + F::kBlockQ - 1) / F::kBlockQ;
    const int head = blockIdx.x, b = blockIdx.z;
    const int qb = p.causal ? nqb - 1 - (int)blockIdx.y : (int)blockIdx.y;
    const int kvh = (int)((uint32_t)head / (uint32_t)p.group);
    const uint16_t* qp = p.q + b * p.qs.b + head * p.qs.h;
    const uint16_t* kp = p.k + b * p.ks.b + kvh * p.ks.h;
    const uint16_t* vp = p.v + b * p.vs.b + kvh * p.vs.h;
    const int q0 = qb * F::kBlockQ + wave * 32;  // first query of this wave
    const int qrow = q0 + c32;                   // this lane's query
    const bool qin = qrow < seq;

    // the last visible key of this lane's query, and of the wave's queries
    const int klast = p.causal && qrow < klim ? qrow : klim;
    const int whi = p.causal && q0 + 31 < klim ? q0 + 31 : klim;
    // key tiles of the block and of this wave (none without a query)
    const int ktiles = klim / kAttnBlockK + 1;
    const int ncausal = p.causal ? (qb + 1) * (F::kBlockQ / kAttnBlockK) : ktiles;
    const int nkb = ncausal < ktiles ? ncausal : ktiles;
    const int nw = q0 < seq ? whi / kAttnBlockK + 1 : 0;

    // ---- staging: load j of a wave moves rows kLoadRows (W j + wave) ..
    const RowLoader<HD> loader(lane, p.wide);
    const TileReader<HD> reader(lane);
    auto load_tile = [&](uint32_t lds, const uint16_t* base, int64_t stride, int t) {
#pragma unroll
        for (int j = 0; j < F::kLoads; ++j) {
            const int r = F::kLoadRows * (j * W + wave);
            loader.load(lds + lds_row<HD>(r), F::kLoadRows * wave, base, stride, t * kAttnBlockK + r, klim);
        }
    };
    auto load_k = [&](int t) { load_tile(lds0 + (uint32_t)(t % kRing * kTileB), kp, p.ks.s, t); };
    auto load_v = [&](int t) { load_tile(lds0 + kV + (uint32_t)(t % kRing * kTileB), vp, p.vs.s, t); };

    // ---- prologue: K(0), Q through the V ring, the K tiles ahead
    load_k(0);
#pragma unroll
    for (int j = 0; j < 32 / F::kLoadRows; ++j) {
        const int r = F::kLoadRows * (j * W + wave);
        loader.load(lds0 + kV + lds_row<HD>(r), F::kLoadRows * wave, qp, p.qs.s, qb * F::kBlockQ + r, seq - 1);
    }
#pragma unroll
    for (int t = 1; t < kRing - 1; ++t)
        if (t < nkb) load_k(t);

    const ScoreConsts k = score_consts<MODE>(p);
    f32x16_t oacc[kD];
#pragma unroll
    for (int dt = 0; dt < kD; ++dt) oacc[dt] = (f32x16_t){};
    float m = -__builtin_inff(), l = 0.0f;

    wait_loads<0>();
    block_barrier();
    bf16x8_t qf[kC];
#pragma unroll
    for (int c = 0; c < kC; ++c) qf[c] = reader.row_frag(smem + kV + lds_row<HD>(wave * 32), c);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    block_barrier();  // every wave has its Q fragments: the V ring is free
#pragma unroll
    for (int t = 0; t < kAheadV; ++t)
        if (t < nkb) load_v(t);

    // sync(i): K(i), V(i) and older tiles have landed for every wave, and every
    // wave is done with tile i - 1, late waves but for its P V.  Loads K of
    // kRing - 1 tiles ahead over K(i - 1), V as far ahead over V(i - 1), or one
    // tile less over V(i - 2) where late waves still read V(i - 1).  The loads
    // of kRing - 2 tiles (one less with late waves) may still be in flight.
    auto sync = [&](int i) {
        if (kInFlight > 0 && i > 0 && i + kInFlight + (kLate ? 1 : 0) < nkb) wait_loads<2 * F::kLoads * kInFlight>();
        else wait_loads<0>();
        block_barrier();
        if (i + kRing - 1 < nkb) load_k(i + kRing - 1);
        if (i + kAheadV < nkb) load_v(i + kAheadV);
    };
    // S^T = K Q^T of tile i: two 32-key accumulators, independent chains
    // interleaved, six fragments read ahead where two waves run in step
    f32x16_t s[2];
    auto scores = [&](int i) {
        const uint32_t tile = (uint32_t)(i % kRing * kTileB);
        if constexpr (kOrdered) __builtin_amdgcn_sched_barrier(0);
        if constexpr (!kLate && kOrdered) __builtin_amdgcn_s_setprio(1);  // the other blocks keep the VALU busy meanwhile
        s[0] = s[1] = (f32x16_t){};
#pragma unroll
        for (int c = 0; c < kC; ++c)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) s[kt] = mfma32(reader.row_frag(smem + tile + lds_row<HD>(kt * 32), c), qf[c], s[kt]);
        if constexpr (kLate) {
            __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
            for (int g = 0; g < 2 * kC - 6; ++g) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
        }
        if constexpr (!kLate && kOrdered) __builtin_amdgcn_s_setprio(0);
        if constexpr (kOrdered) __builtin_amdgcn_sched_barrier(0);
    };
    // O^T += V^T P^T of the 16 keys g
    bf16x8_t pf[4];
    auto accumulate8 = [&](uint32_t tile, int g) {
#pragma unroll
        for (int dt = 0; dt < kD; ++dt)
            oacc[dt] = mfma32(reader.col_frag(smem + tile + lds_row<HD>(16 * g), dt), pf[g], oacc[dt]);
    };
    // probabilities of tile i (masked: it holds the causal diagonal of the
    // wave's queries or keys past the last) as the B operands of P V
    auto probabilities = [&](auto masked_c, int i) {
        constexpr bool MASKED = decltype(masked_c)::value;
        const int diag = i * kAttnBlockK - klast + 4 * h;
        const uint32_t rmask = ROUTE == kRouteRuntime ? tile_route_mask(p.route, p.rmask, i) : 0u;
        float x[2][16];
        float ls[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        tile_softmax_state<MODE, MASKED, HD>(k, s, x, oacc, m, l, diag);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            pf[g] = tile_probs8<MODE, ROUTE, MASKED>(k, s, x, g >> 1, g & 1, m, diag, rmask, ls);
            if constexpr (kFused) accumulate8(kV + (uint32_t)(i % kRing * kTileB), g);
        }
        if constexpr (!kSigmoid) l += (ls[0] + ls[1]) + (ls[2] + ls[3]);
    };
    // the products of tile i, three fragments read ahead
    auto accumulate = [&](int i) {
        if constexpr (!kFused) {
            if constexpr (kOrdered) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int g = 0; g < 4; ++g) accumulate8(kV + (uint32_t)(i % kRing * kTileB), g);
            if constexpr (kOrdered) {
                __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
                for (int g = 0; g < 4 * kD - 3; ++g) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                }
                __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    // Late waves (the second wave of each SIMD) meet sync(i + 1) between the
    // score program and P V of tile i, the others ahead of S(i + 1).
    const bool late = kLate && wave >= 4;
    sync(0);
    int i = 0;
    for (; i + 1 < nw; ++i) {
        scores(i);
        probabilities(std::integral_constant<bool, false>{}, i);
        if (late) sync(i + 1);
        accumulate(i);
        if (!late) sync(i + 1);
    }
    int synced = i;  // sync(0) .. sync(synced) met
    if (nw > 0) {  // the wave's last tile
        scores(i);
        probabilities(std::integral_constant<bool, true>{}, i);
        if (late && i + 1 < nkb) sync(++synced);
        accumulate(i);
    }
    while (synced + 1 < nkb) sync(++synced);
    if (nw == 0) return;

    // ---- normalise and store: oacc[dt][r] = O^T[dt*32 + 8*(r/4) + 4h + r%4][qrow]
    // through LDS, so that whole rows reach memory.  After sync(nkb - 1) the
    // other waves read K(nkb - 1), V(nkb - 1) and V(nkb - 2) only: wave w
    // takes part w % 2 of free K tile w / 2, the last two waves a free V tile.
    float inv = 1.0f;
    if constexpr (!kSigmoid) {
        l = half_sum(l);
        inv = 1.0f / l;
        // log sum exp(s') with s' the (capped) scaled score: m and log2(l) are
        // in log2 units
        if (p.lse != nullptr && h == 0 && qin)
            p.lse[((int64_t)b * p.hq + head) * seq + qrow] = (m + __builtin_log2f(l)) * kLn2;
    }
    const int part = wave >> 1;  // 32 rows are half a tile
    const uint32_t slot = part < kRing - 1 ? (uint32_t)((nkb + part) % kRing * kTileB)
                                           : kV + (uint32_t)(nkb % kRing * kTileB);
    unsigned char* orows = smem + slot + (wave & 1) * 32 * kRowB;
#pragma unroll
    for (int dt = 0; dt < kD; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<u32x2_t*>(orows + c32 * kRowB + ((dt * 4 + g) ^ (c32 & (F::kChunks - 1))) * 16 + h * 8) =
                (u32x2_t){pack_bf(oacc[dt][4 * g] * inv, oacc[dt][4 * g + 1] * inv),
                          pack_bf(oacc[dt][4 * g + 2] * inv, oacc[dt][4 * g + 3] * inv)};
    __builtin_amdgcn_wave_barrier();  // LDS accesses of one wave complete in order
    uint16_t* op = p.o + b * p.os.b + head * p.os.h;
    uint16_t* o2p = p.o2 != nullptr ? p.o2 + b * p.o2s.b + head * p.o2s.h : nullptr;
#pragma unroll
    for (int j = 0; j < 32 / F::kLoadRows; ++j) {
        const int r = j * F::kLoadRows + loader.lr;
        const u32x4_t w =
            *reinterpret_cast<const u32x4_t*>(orows + r * kRowB + (loader.lc ^ (r & (F::kChunks - 1))) * 16);
        if (q0 + r < seq) {
            *reinterpret_cast<u32x4_t*>(op + (q0 + r) * p.os.s + loader.lc * 8) = w;
            if (o2p != nullptr) *reinterpret_cast<u32x4_t*>(o2p + (q0 + r) * p.o2s.s + loader.lc * 8) = w;
        }
    }
}

}  // namespace pt

using namespace pt;

namespace {

// any even route >= 4 (FA4's validation, src/sfu_repro/fa4.py:226-233);
// the ones without a template instantiation take kRouteRuntime
bool route_supported(int route) { return route >= 4 && route % 2 == 0; }

// LDS that a block asks for beyond its tiles, so that two of them share a CU
// instead of three: causal softcap at head_dim 64 in grids of two to four
// blocks a CU, of which each batch element has one a CU and more.  Three to a
// CU then hold three quarters of the grid and more from the start, so that
// little is left to even out their unequal lengths; two leave more (the light
// blocks of what runs first make room for heavy ones).  Hardware softcap /
// softcap D4, three against two to a CU: S 3072, 32 heads 108 / 136 against 100 /
// 123 us; S 4096 164 / 205 against 161 / 193; 4 x 1024 63 / 76 against 58 / 68;
// 3 x 2048, 16 heads 117 / 144 against 90 / 110; worst, 3 x 1280, 65.6 / 77.9
// against 65.0 / 80.6.  Outside the rule three win: S 4608 192 / 240 against 199
// / 247; 4 x 1500, 16 heads (0.75 a CU and batch element) 68 / 80 against 80 /
// 96; S 4096 without the mask 295 / 366 against 306 / 380.
template <int MODE, int HD, int W>
unsigned fwd_spare_lds(const AttnParams& prm, int64_t batch) {
    using F = FwdShape<HD, W>;
    if (HD != 64 || !attn_is_softcap(MODE) || !prm.causal) return 0;
    const int64_t cus = device_shape().cus, each = prm.hq * ((prm.seq + F::kBlockQ - 1) / F::kBlockQ);
    if (each < cus || batch * each <= 2 * cus || batch * each > 4 * cus) return 0;
    return 160 * 1024 / 3 + 1024 - 2 * F::kRing * F::kTileB;  // a third of the CU's LDS, and more
}

template <int MODE, int ROUTE, int HD, int W>
void launch_fwd_shape(const AttnParams& prm, int64_t batch, hipStream_t st) {
    constexpr int kBlockQ = FwdShape<HD, W>::kBlockQ;
    const dim3 grid((unsigned)prm.hq, (unsigned)((prm.seq + kBlockQ - 1) / kBlockQ), (unsigned)batch);
    hipLaunchKernelGGL((flash_fwd_kernel<MODE, ROUTE, HD, W>), grid, dim3(64 * W), (fwd_spare_lds<MODE, HD, W>(prm, batch)),
                       st, prm);
}

// Waves per head_dim-128 block.  One 8-wave block per CU stages each tile once
// for 256 queries; two 4-wave blocks per CU are half the size and leave less
// of the chip idle in a round that is not full.  8 waves are taken where their
// blocks make an even number of whole rounds (causal blocks are dispatched
// heaviest first, so two rounds add up to equal loads) and from ten rounds on.
// Time with 4 waves over time with 8, by rounds of 8-wave blocks (32 heads over
// 8, S = 2048 rounds; hardware softmax / D2 at 4 of 12 / softcap D4 / sigmoid
// D3):
//   rounds   causal                       without the mask
//   1        0.89  0.88  0.81  0.79       1.03  1.04  1.12  1.03
//   1.5      0.95  0.92  0.96  0.90       0.91  0.89  0.88  0.83
//   1.75     0.99  1.02  1.07  1.05       1.01  1.03  1.10  1.00
//   1.88     1.02  1.05  1.09  1.08       1.02  1.03  1.09  1.01
//   2        0.99  1.04  1.07  1.06       1.01  1.03  1.09  1.01
//   2.12     0.98  0.98  1.02  0.99       0.93  0.91  0.91  0.85
//   2.5      0.98  0.95  0.98  0.92       0.94  0.93  0.93  0.88
//   3        0.98  0.95  0.97  0.92       1.02  1.03  1.07  1.01
//   4        1.00  1.02  1.04  0.95       1.02  1.03  1.07  0.99
//   5        0.99  0.98  1.02  0.92       1.02  1.03  1.07  0.99
//   6        1.01  0.99  1.04  0.96       1.02  1.03  1.06  0.99
//   10       1.01  1.01  1.04  0.98       1.03  1.02  1.06  1.00
//   11       1.00  1.00  1.03  0.97       1.05  1.02  1.06  1.00
// So the rule is on the right side at one round causal, at two, and between
// whole rounds at a half and less.  It leaves up to 1.12 (softcap) where a
// second round is nearly full (62 heads, 1.94: softmax 0.96, softcap 1.14) and
// at odd whole rounds without the mask, and costs the sigmoid modes up to 5 %
// at four causal rounds and more.
int fwd_waves(const AttnParams& prm, int64_t batch) {
    const int64_t blocks = batch * prm.hq * ((prm.seq + 255) / 256), cus = device_shape().cus;
    return blocks % (2 * cus) == 0 || blocks >= 10 * cus ? 8 : 4;
}

template <int MODE, int ROUTE>
void launch_fwd(const AttnParams& prm, int64_t batch, hipStream_t st, int hd) {
    if (hd == 64) launch_fwd_shape<MODE, ROUTE, 64, 4>(prm, batch, st);
    else if (fwd_waves(prm, batch) == 8) launch_fwd_shape<MODE, ROUTE, 128, 8>(prm, batch, st);
    else launch_fwd_shape<MODE, ROUTE, 128, 4>(prm, batch, st);
}

template <int MODE>
void launch_routed(const AttnParams& prm, int64_t batch, hipStream_t st, int route, int hd) {
    switch (route) {
        case 6: launch_fwd<MODE, 6>(prm, batch, st, hd); break;
        case 8: launch_fwd<MODE, 8>(prm, batch, st, hd); break;
        case 10: launch_fwd<MODE, 10>(prm, batch, st, hd); break;
        case 12: launch_fwd<MODE, 12>(prm, batch, st, hd); break;
        case 16: launch_fwd<MODE, 16>(prm, batch, st, hd); break;
        case 20: launch_fwd<MODE, 20>(prm, batch, st, hd); break;
        case 24: launch_fwd<MODE, 24>(prm, batch, st, hd); break;
        case 32: launch_fwd<MODE, 32>(prm, batch, st, hd); break;
        case 4: launch_fwd<MODE, 4>(prm, batch, st, hd); break;
        default: launch_fwd<MODE, kRouteRuntime>(prm, batch, st, hd); break;
    }
}

bool stride_ok(const AttnStrides& t) { return t.b >= 0 && t.h >= 0 && t.s >= 0 && t.s % 8 == 0 && t.h % 8 == 0 && t.b % 8 == 0; }

}  // namespace

extern "C" int launch_flash_attention_fwd_two_outputs_bf16(void* out, void* out2, float* lse, const void* q,
                                                           const void* k, const void* v, int64_t batch,
                                                           int64_t q_heads, int64_t kv_heads, int64_t seq,
                                                           int64_t valid_keys, int64_t head_dim,
                                                           const int64_t* strides, int mode, int exp2_route,
                                                           int causal, float scale, float cap,
                                                           float sigmoid_bias, void* stream) {
    if (batch < 0 || q_heads <= 0 || kv_heads <= 0 || seq < 0 || (head_dim != 64 && head_dim != 128) || !strides)
        return hipErrorInvalidValue;
    if (seq > 0 && (valid_keys < 1 || valid_keys > seq)) return hipErrorInvalidValue;
    if (q_heads % kv_heads != 0 || mode < 0 || mode >= kAttnModes) return hipErrorInvalidValue;
    if ((mode == kAttnSoftcapNative || mode == kAttnSoftcapD4) && !(cap > 0.0f && cap <= __FLT_MAX__))
        return hipErrorInvalidValue;
    if (attn_has_exp2_program(mode) && !route_supported(exp2_route)) return hipErrorInvalidValue;
    const int hd = (int)head_dim;
    // the B3 programs are fitted for n = 4096 (src/sfu_repro/fa4.py:404-413;
    // autonumerics_zero/evolution/fit_flash_sigmoid_exp2_d2.py)
    if ((mode == kAttnSigmoidB3 || mode == kAttnSigmoidB3D2) && seq != 4096) return hipErrorInvalidValue;
    const AttnStrides st[4] = {{strides[0], strides[1], strides[2]}, {strides[3], strides[4], strides[5]},
                               {strides[6], strides[7], strides[8]}, {strides[9], strides[10], strides[11]}};
    for (const AttnStrides& t : st)
        if (!stride_ok(t)) return hipErrorInvalidValue;
    AttnStrides st2{};
    if (out2) st2 = {strides[12], strides[13], strides[14]};
    if (!stride_ok(st2)) return hipErrorInvalidValue;
    if (batch == 0 || seq == 0) return hipSuccess;
    if (!out || !q || !k || !v || !aligned16(out) || !aligned16(q) || !aligned16(k) || !aligned16(v))
        return hipErrorInvalidValue;
    if (out2 && !aligned16(out2)) return hipErrorInvalidValue;
    if (lse && (reinterpret_cast<uintptr_t>(lse) & 3)) return hipErrorInvalidValue;
    if (attn_is_sigmoid(mode)) lse = nullptr;  // sigmoid attention has no partition function
    const int64_t qblocks = (seq + kAttnBlockQ - 1) / kAttnBlockQ;  // the last one may be partial
    if (batch > 65535 || qblocks > 65535 || q_heads > 0x7fffffff) return hipErrorInvalidValue;
    AttnParams prm{(const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (uint16_t*)out,
                   (uint16_t*)out2, lse, st[0], st[1], st[2], st[3], st2, q_heads, kv_heads, seq, valid_keys, scale,
                   cap > 0.0f ? cap : 1.0f, sigmoid_bias, causal != 0, exp2_route, host_route_mask(exp2_route),
                   (int)(q_heads / kv_heads), 0};
    // staging adds up to 7 rows to a wave's address as a 32-bit byte offset
    for (int i = 0; i < 3; ++i) prm.wide |= st[i].s > (int64_t(1) << 27);
    hipStream_t hst = hs(stream);
    switch (mode) {
        case kAttnSoftmaxNative: launch_fwd<kAttnSoftmaxNative, 0>(prm, batch, hst, hd); break;
        case kAttnSoftmaxExp2D2: launch_routed<kAttnSoftmaxExp2D2>(prm, batch, hst, exp2_route, hd); break;
        case kAttnSoftmaxExp2D3: launch_routed<kAttnSoftmaxExp2D3>(prm, batch, hst, exp2_route, hd); break;
        case kAttnSoftmaxExp2Pwl2: launch_routed<kAttnSoftmaxExp2Pwl2>(prm, batch, hst, exp2_route, hd); break;
        case kAttnSoftmaxExp2Pwl2Safe:
            launch_routed<kAttnSoftmaxExp2Pwl2Safe>(prm, batch, hst, exp2_route, hd);
            break;
        case kAttnSoftmaxExp2Pwl2SafeF16:
            launch_routed<kAttnSoftmaxExp2Pwl2SafeF16>(prm, batch, hst, exp2_route, hd);
            break;
        case kAttnSoftmaxExp2Pwl1Safe: launch_routed<kAttnSoftmaxExp2Pwl1Safe>(prm, batch, hst, exp2_route, hd); break;
        case kAttnSoftmaxExp2Pwl1SafeF16:
            launch_routed<kAttnSoftmaxExp2Pwl1SafeF16>(prm, batch, hst, exp2_route, hd);
            break;
        case kAttnSoftmaxExp2Pwl2SafeBF16:
            launch_routed<kAttnSoftmaxExp2Pwl2SafeBF16>(prm, batch, hst, exp2_route, hd);
            break;
        case kAttnSoftmaxExp2D2NoClamp:
            launch_routed<kAttnSoftmaxExp2D2NoClamp>(prm, batch, hst, exp2_route, hd);
            break;
        case kAttnSoftmaxExp2D2SafeF16:
            launch_routed<kAttnSoftmaxExp2D2SafeF16>(prm, batch, hst, exp2_route, hd);
            break;
        case kAttnSoftmaxExp2D2SafeBF16:
            launch_routed<kAttnSoftmaxExp2D2SafeBF16>(prm, batch, hst, exp2_route, hd);
            break;
        case kAttnSoftmaxExp2Pwl2F16: launch_routed<kAttnSoftmaxExp2Pwl2F16>(prm, batch, hst, exp2_route, hd); break;
        case kAttnSoftcapNative: launch_fwd<kAttnSoftcapNative, 0>(prm, batch, hst, hd); break;
        case kAttnSoftcapD4: launch_fwd<kAttnSoftcapD4, 0>(prm, batch, hst, hd); break;
        case kAttnSigmoidNative: launch_fwd<kAttnSigmoidNative, 0>(prm, batch, hst, hd); break;
        case kAttnSigmoidB3: launch_fwd<kAttnSigmoidB3, 0>(prm, batch, hst, hd); break;
        case kAttnSigmoidB3D2: launch_fwd<kAttnSigmoidB3D2, 0>(prm, batch, hst, hd); break;
        case kAttnSigmoidD3: launch_fwd<kAttnSigmoidD3, 0>(prm, batch, hst, hd); break;
        case kAttnSigmoidD3 + 1: launch_fwd<kAttnSigmoidD3 + 1, 0>(prm, batch, hst, hd); break;
        case kAttnSigmoidD3 + 2: launch_fwd<kAttnSigmoidD3 + 2, 0>(prm, batch, hst, hd); break;
        case kAttnSigmoidD6: launch_fwd<kAttnSigmoidD6, 0>(prm, batch, hst, hd); break;
    }
    return hipGetLastError();
}

extern "C" int launch_flash_attention_fwd_strided_keys_bf16(void* out, float* lse, const void* q,
                                                            const void* k, const void* v, int64_t batch,
                                                            int64_t q_heads, int64_t kv_heads, int64_t seq,
                                                            int64_t valid_keys, int64_t head_dim,
                                                            const int64_t* strides, int mode, int exp2_route,
                                                            int causal, float scale, float cap,
                                                            float sigmoid_bias, void* stream) {
    return launch_flash_attention_fwd_two_outputs_bf16(out, nullptr, lse, q, k, v, batch, q_heads, kv_heads, seq,
                                                       valid_keys, head_dim, strides, mode, exp2_route, causal,
                                                       scale, cap, sigmoid_bias, stream);
}

extern "C" int launch_flash_attention_fwd_strided_bf16(void* out, float* lse, const void* q,
                                                       const void* k, const void* v, int64_t batch,
                                                       int64_t q_heads, int64_t kv_heads, int64_t seq,
                                                       int64_t head_dim, const int64_t* strides,
                                                       int mode, int exp2_route, int causal,
                                                       float scale, float cap, float sigmoid_bias,
                                                       void* stream) {
    return launch_flash_attention_fwd_strided_keys_bf16(out, lse, q, k, v, batch, q_heads, kv_heads, seq, seq,
                                                        head_dim, strides, mode, exp2_route, causal, scale,
                                                        cap, sigmoid_bias, stream);
}

extern "C" int launch_flash_attention_fwd_bf16(void* out, const void* q, const void* k,
                                               const void* v, int64_t batch, int64_t q_heads,
                                               int64_t kv_heads, int64_t seq, int64_t head_dim,
                                               int mode, int causal, float scale, float cap,
                                               void* stream) {
    if (mode < 0 || mode > kAttnSigmoidB3) return hipErrorInvalidValue;
    const int64_t hs_ = seq * head_dim;  // [B, H, S, D] contiguous
    const int64_t strides[12] = {q_heads * hs_, hs_, head_dim, kv_heads * hs_, hs_, head_dim,
                                 kv_heads * hs_, hs_, head_dim, q_heads * hs_, hs_, head_dim};
    return launch_flash_attention_fwd_strided_bf16(out, nullptr, q, k, v, batch, q_heads, kv_heads,
                                                   seq, head_dim, strides, mode, 4, causal, scale,
                                                   cap, -__builtin_logf((float)seq), stream);
}
