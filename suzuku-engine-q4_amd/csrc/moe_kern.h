// Routed-expert decode / verify-window kernels and their launch templates,
// shared by the translation units that instantiate them per weight type
// (moe_decode.hip: IQ3_S and Q8_0, plus the host entry points;
// moe_fmt_gu.hip / moe_fmt_dn.hip: the other formats of formats.h).
// Routed-expert decode (1 token) and verify window (2..8 tokens) over
// experts resident at base + slot*stride (gate/up IQ3_S, Q8_0, IQ2_S,
// IQ2_XXS, IQ2_XS, IQ3_XXS, IQ4_XS; down IQ3_S, Q8_0, IQ4_NL, Q2_0, IQ2_S).
//
// Two launches per layer, 1024-thread blocks:
//   moe_gu_k  the intermediate rows of the unique experts are split into one
//             contiguous share per block; h[u][t][r] =
//             silu(gate_r . q8(x_t)) * (up_r . q8(x_t)) goes out as fp32.
//   moe_dn_k  each block owns a few output rows: it quantizes every selected
//             h[u][t] (q8, 32-value groups) into LDS, dots its rows of every
//             expert's down matrix and writes y[t][r] += sum_u w[u][t] *
//             (down_u[r] . q8(h[u][t])) in a fixed order -- deterministic, no
//             atomics.
// Each unique expert's rows are read once per launch and dotted with every
// token that selected it (the verify window's reuse; reference
// q4_hip_moe_exec_win src/q4_rocm.cu:7444-7531, CPU twin
// q4_cpuex_dispatch_win src/q4_cpuexp.c:2618-2753).
//
// Weights go from global memory straight into registers (moe_unit.h): a lane
// holds a 64-value unit of a row, and a wave computes it as soon as its own
// loads are back, so no weight passes through LDS and no wave waits for
// another after the one barrier behind the prologue (codebook tables and q8
// activations in LDS).  The first weights are asked for only behind that
// prologue: its loads, and its instructions' fetches, would otherwise queue
// behind the weight stream (decode layer 13.2 -> 11.4 us).
#pragma once
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "moe_unit.h"
#include "mmvq_engine.h"
#include "route_wave.h"
#include "q4mi_internal.h"

namespace q4mi {

constexpr uint32_t kMaxU = 64;    // unique experts per call (reference bound n<=64)
constexpr uint32_t kMaxT = 8;     // tokens per call
constexpr uint32_t kT = 1024;     // threads per block
constexpr uint32_t kW = kT / 64;  // waves per block
constexpr uint32_t kDnRowsMax = 32;   // most output rows of a down block
constexpr int kSrcDev = 0, kSrcHost = 1, kSrcLogits = 2;   // list source of a launch
struct HostList {
    int32_t id[kMaxU];
    float w[kMaxU];
};

struct ListSrc {
    const int32_t *es;   // device ids (null: use the HostList argument)
    const float *ew;     // device weights
    const int32_t *nh;   // device per-token counts (null: n_fixed)
    uint32_t stride;     // entries between tokens in es/ew
    uint32_t n_tok;
    uint32_t n_fixed;    // count per token when nh is null / host list length
    uint32_t unique;     // host list already deduplicated (one token)
    // One token's router logits in place of the lists (lg non-null): the
    // plan's entries are route_k's top-k of lg [n_exp] plus, with shared >= 0,
    // expert `shared` at weight sg[0] (or 1); gate/up block 0 writes them to
    // o_ids / o_wts / o_nh (row 0, topk + 1 entries) as route_k would.
    const float *lg;
    const float *sg;
    int32_t *o_ids;
    float *o_wts;
    int32_t *o_nh;
    uint32_t n_exp, topk;
    int32_t shared;
};

// What the down launch needs of a device list, written by gate/up block 0.
struct __align__(16) Plan {
    uint32_t nu;
    uint32_t nsel;                  // selected (u, t) pairs
    uint32_t pad[2];
    int32_t uid[kMaxU];
    uint32_t sel[kMaxU];            // token bitmask per unique expert
    uint32_t pslot[kMaxU];          // first pair slot of u (slots in (u, t) order)
    uint32_t prow[kMaxU];           // pair slot -> h row u * kMaxT + t
    float w[kMaxT][kMaxU];          // routing weight of (token, unique expert)
};

// One (token, pick) entry of the flattened lists per lane, token-major, and
// the unique expert it belongs to.
struct PlanLane {
    bool valid, first;   // in the lists / first appearance of its id
    int32_t id;
    float w;
    uint32_t tok, u;
};

// Wave 0 of a gate/up block: the lists' unique experts (first-appearance order
// over (token, pick)) into P->nu, uid, sel.  ht: 4.5 KB of LDS.
// LG: the source holds one token's router logits (ListSrc::lg) instead of
// the lists; a separate instantiation, so that the other kernels do not
// carry the top-k code (their start-up runs with a cold instruction cache).
template <bool LG>
__device__ PlanLane build_plan(Plan *P, const ListSrc &s, uint32_t lane, uint32_t *ht) {
    uint32_t E = 0, tok = 0;
    int32_t id = -1;
    float w = 0.f;
    if constexpr (LG) {
        // one token's router logits: route_k's top-k (same code, same
        // picks and weights) and the shared entry after them; gate/up block
        // 0 also writes them out as route_k's lists
        int32_t *s_id = (int32_t *)(ht + 1024);
        float *s_p = (float *)(ht + 1024 + 64);
        const uint32_t tk = route_wave<8>(s.lg, s.n_exp, s.topk, lane, s_id, s_p);
        float sk = 0.f;
        for (uint32_t k = 0; k < tk; k++) sk += s_p[k];
        const float inv2 = sk > 0.f ? __fdiv_rn(1.f, sk) : 0.f;
        const uint32_t nsh = s.shared >= 0 ? 1u : 0u;
        E = s.topk + nsh;
        if (lane < s.topk) {
            id = lane < tk ? s_id[lane] : -1;
            w = lane < tk ? (sk > 0.f ? s_p[lane] * inv2 : s_p[lane]) : 0.f;
        } else if (lane == s.topk && nsh) {
            id = s.shared;
            w = s.sg ? s.sg[0] : 1.f;
        }
        if (s.o_ids && blockIdx.x == 0) {
            if (lane < E) {
                s.o_ids[lane] = id;
                s.o_wts[lane] = w;
            }
            if (lane == 0 && s.o_nh) s.o_nh[0] = (int32_t)E;
        }
    } else {
        // lane -> (token, pick) of the flattened lists, token-major
        // every token's count in one load (lane t holds token t's), then
        // read back lane by lane: one memory round trip, not one per token
        const int cnt_l = lane < s.n_tok ? (s.nh ? s.nh[lane] : (int)s.n_fixed) : 0;
        // the entries are loaded in the same round trip as the counts, assuming
        // each token has at most CAP = 64 / (n_tok rounded up to a power of two)
        // of them (lane l: token l / CAP, entry l % CAP; within the lists' rows);
        // a longer list loads them again once the counts are known
        const uint32_t cap_sh = s.n_tok <= 1 ? 6u : s.n_tok == 2 ? 5u : s.n_tok <= 4 ? 4u : 3u;
        const uint32_t st = lane >> cap_sh, sr = lane & ((1u << cap_sh) - 1u);
        int32_t sid = -1;
        float sw = 0.f;
        if (st < s.n_tok && sr < s.stride) {
            sid = s.es[(size_t)st * s.stride + sr];
            sw = s.ew[(size_t)st * s.stride + sr];
        }
        uint32_t rem = 0;
        bool found = false;
        for (uint32_t t = 0; t < s.n_tok; t++) {
            int c = __builtin_amdgcn_readlane(cnt_l, t);
            if (c < 0) c = 0;
            if ((uint32_t)c > s.stride) c = (int)s.stride;
            if (!found && lane < E + (uint32_t)c) {
                found = true;
                tok = t;
                rem = lane - E;
            }
            E += (uint32_t)c;
        }
        if (E > kMaxU) E = kMaxU;
        if (__ballot(lane < E && rem >= (1u << cap_sh)) == 0) {
            const int src = (int)((tok << cap_sh) + rem);
            const int32_t gid = __shfl(sid, src);
            const float gw = __shfl(sw, src);
            if (lane < E) {
                id = gid;
                w = gw;
            }
        } else if (lane < E) {
            id = s.es[(size_t)tok * s.stride + rem];
            w = s.ew[(size_t)tok * s.stride + rem];
        }
    }
    const bool valid = lane < E && id >= 0;
    // First occurrence of each id, through a 1024-bucket table in LDS (ht,
    // 4 KB of LDS not yet in use): every valid lane takes the minimum
    // lane of its bucket; that lane holds the first occurrence of the id
    // unless it holds another id of the same bucket (ids 1024 apart), which
    // only the exact pass over the lanes (v_readlane per lane) settles.
    const uint64_t vmask = __ballot(valid);
    const uint32_t hb = (uint32_t)id & 1023u;
    if (valid) ht[hb] = 0xFFFFFFFFu;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    if (valid) atomicMin(&ht[hb], lane);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    const uint32_t mlane = valid ? ht[hb] : lane;
    const bool clash = valid && __shfl(id, (int)mlane) != id;
    uint32_t first_j = (valid && !clash) ? mlane : lane;
    if (__builtin_expect(__ballot(clash) != 0, 0)) {
        first_j = lane;
        for (uint32_t j = 0; j < E; j++) {
            if (!((vmask >> j) & 1ull)) continue;
            const int32_t idj = __builtin_amdgcn_readlane(id, j);
            if (idj == id && j < first_j) first_j = j;
        }
    }
    const bool first = valid && first_j == lane;
    const uint64_t fm = __ballot(first);
    const uint32_t u = (uint32_t)__popcll(fm & ((1ull << first_j) - 1ull));
    P->sel[lane] = 0;
    const uint32_t nu = (uint32_t)__popcll(fm);
    if (lane == 0) P->nu = nu;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if (first) P->uid[u] = id;
    if (valid) atomicOr(&P->sel[u], 1u << tok);
    return PlanLane{valid, first, id, w, tok, u};
}

// ... and the rest of the plan (pair slots, weights), by the wave that
// publishes it.
__device__ inline void finish_plan(Plan *P, const PlanLane &l, uint32_t lane) {
    const uint32_t nu = P->nu;
#pragma unroll
    for (uint32_t t = 0; t < kMaxT; t++) P->w[t][lane] = 0.f;
    if (lane >= nu) P->uid[lane] = -1;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if (l.valid) atomicAdd(&P->w[l.tok][l.u], l.w);   // a token's repeated id adds its weights
    // pair slots: pslot[u] = sum over v < u of popcount(sel[v]), counted
    // per token bit with a ballot and mbcnt (no cross-lane round trips)
    const uint32_t sl = lane < nu ? P->sel[lane] : 0u;
    uint32_t below = 0, nsel = 0;
#pragma unroll
    for (uint32_t t = 0; t < kMaxT; t++) {
        const uint64_t b = __ballot((sl >> t) & 1u);
        below += __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32),
                                           __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
        nsel += (uint32_t)__popcll(b);
    }
    if (lane < nu) {
        P->pslot[lane] = below;
        uint32_t k = below;
        for (uint32_t t = 0; t < kMaxT; t++)
            if ((sl >> t) & 1u) P->prow[k++] = lane * kMaxT + t;
    }
    if (lane == 0) P->nsel = nsel;
}

struct MoeArgs {
    const uint8_t *base;
    uint64_t stride, og, ou, od;
    uint64_t stride_d;  // bytes between experts' down matrices (= stride when packed)
    uint32_t K;       // in_dim (gate/up columns)
    uint32_t n_ff;
    uint32_t n_embd;
    uint32_t rb_gu, rb_dn;
    uint32_t tpe, tpe_inv;   // gate/up: tasks per expert, ceil(2^32 / tpe)
    uint32_t nsel_cap;       // down: q8(h) rows the LDS holds
    uint32_t dn_rows;        // down: output rows per block
    const float *x;   // [n_tok][K]
    float *h;         // [kMaxU][kMaxT][n_ff] fp32 h
    float *y;         // [n_tok][n_embd], accumulated
    ListSrc src;
    Plan *gplan;      // device list: the plan gate/up block 0 publishes for down
    HostList hl;      // host list (src.unique), read in place from the kernel arguments
};

// The kernel's own argument block (kernel parameters start at offset 0 of
// the kernarg segment).  Uniform reads through it are scalar loads: a host
// list's ids and weights are read where they are used.
typedef const __attribute__((address_space(4))) MoeArgs *KArgs;
__device__ inline KArgs kargs() { return (KArgs)__builtin_amdgcn_kernarg_segment_ptr(); }

__host__ __device__ inline size_t al16(size_t v) { return (v + 15) & ~(size_t)15; }

// silu(g) * u in fp64: 2^f on [-1/2, 1/2] by its Taylor series in f ln 2 to
// the tenth power (error below 3e-13), the reciprocal by one Newton step on
// the hardware's.
__device__ inline double silu_mul(double g, double u) {
    const double t = fmin(fmax(g * -1.4426950408889634, -1100.0), 1100.0);
    const double n = rint(t), x = (t - n) * 0.6931471805599453;
    double p = 1.0 / 3628800;
    p = fma(p, x, 1.0 / 362880);
    p = fma(p, x, 1.0 / 40320);
    p = fma(p, x, 1.0 / 5040);
    p = fma(p, x, 1.0 / 720);
    p = fma(p, x, 1.0 / 120);
    p = fma(p, x, 1.0 / 24);
    p = fma(p, x, 1.0 / 6);
    p = fma(p, x, 0.5);
    p = fma(p, x, 1.0);
    p = fma(p, x, 1.0);
    const double d = 1.0 + ldexp(p, (int)n);
    const double r0 = __builtin_amdgcn_rcp(d), r = fma(fma(-d, r0, 1.0), r0, r0);
    return g * (d < __builtin_inf() ? r : 0.0) * u;
}

// ------------------------------------------------------------- gate / up
// What bounds it: a one-token launch (hidden 2048, 11 experts, 9.9 MB) is the
// launch itself (1.7 us), the prologue (activations in, q8 codes and tables
// in LDS, 1.6 us) and one burst of weights with its decode behind it; a
// window's is its table lookups (random LDS banks), the decode's VALU and the
// L1 path in about equal parts.  Measured per launch (kernel trace), copying rows
// through an LDS ring / this kernel: one token 7.1 / 6.7 us, 4 tokens (36 MB)
// 16.8 / 13.0 us, 4 tokens at hidden 2560 IQ2_S (43 MB) 24.6 / 19.5 us.
// One block of 16 waves per CU: two blocks of 64-register waves repeat the
// prologue and took 19.0 us for the 4-token launch.
//
// Sums and silu are taken in fp64, at fp32's instruction rate: h is then the
// correctly rounded one but for about 1e-9 of it, so that its q8 codes in the
// down launch, which an fp32 sum's error moves now and then (about one code in
// 200,000), are those of exact arithmetic.  fp64 adds 0.2 us at one token and
// 0.3 to 0.9 at four, which the times above include.
//
// A wave's task is RPW = 64 / LPR intermediate rows of one expert: LPR lanes
// per row with UPL units each (unit li + LPR m), first the gate rows, then
// the up rows of the same lanes.  A block takes a contiguous share of the
// tasks, its waves every kW-th task of it.
//
// LDS: [tables] Plan | x codes [n_tok][K] | x scales [n_tok][K/32] | out
//
// Share of block `bid` of `nblk`: tasks [share_lo(bid), share_lo(bid + 1)).
__device__ inline uint32_t share_lo(uint32_t PT, uint32_t bid, uint32_t nblk) {
    // the first PT % nblk blocks take one task more (one 32-bit division:
    // a 64-bit one is ~100 scalar instructions of start-up code)
    const uint32_t q = PT / nblk, r = PT % nblk;
    return bid * q + min(bid, r);
}

// Share of block `bid` when the blocks split the tasks by work: a task of
// unique expert u costs 3 + (tokens that picked u) -- one decode of its rows
// shared by all of them, one dot per token -- so the blocks holding an
// expert every token picked (the shared expert) get fewer tasks.  Every
// wave computes the same value (lane u: expert u, sel = its token mask).
__device__ inline void share_weighted(uint32_t sel, uint32_t nu, uint32_t tpe, uint32_t bid,
                                      uint32_t nblk, uint32_t lane, uint32_t &p0, uint32_t &p1) {
    const uint32_t c = lane < nu ? 3u + (uint32_t)__popc(sel) : 0u;
    const uint32_t incl = q4mi_wave_incl_scan(c);
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    auto at = [&](uint32_t b) -> uint32_t {
        if (b >= nblk) return nu * tpe;
        // target in units of 1/tpe of an expert's cost: t = total * tpe * b /
        // nblk (< 2^32: total <= 64 * 11, tpe <= 1024, b < 4096)
        const uint32_t t = total * tpe * b / nblk;
        // expert u0 = number of experts whose whole cost ends at or before t
        const uint64_t done = __ballot(incl * tpe <= t && lane < nu);
        const uint32_t u0 = (uint32_t)__popcll(done);
        if (u0 >= nu) return nu * tpe;
        const uint32_t ex = (uint32_t)__builtin_amdgcn_readlane((int)(incl - c), (int)u0);
        const uint32_t cu = (uint32_t)__builtin_amdgcn_readlane((int)c, (int)u0);
        const uint32_t into = (t - ex * tpe) / cu;   // tasks of u0 before t
        return u0 * tpe + min(into, tpe);
    };
    p0 = at(bid);
    p1 = at(bid + 1);
}

// Finished (row, token) results of a wave, kept until a whole wave of them
// can take silu together (one lane per result instead of one lane per row).
template <int NT, int RPW>
struct GuOut {
    static constexpr uint32_t kCap = 64 + NT * RPW;
    double g[kCap], u[kCap];
    uint32_t dst[kCap];
};

template <uint32_t TY, int NT, int LPR, int UPL, int SRC>
__global__ __launch_bounds__(kT) void moe_gu_k(MoeArgs a) {
    using U = Unit<TY>;
    using Raw = typename U::Raw;
    constexpr uint32_t RPW = 64 / LPR;
    static_assert(UPL == 1 || !U::kEven || U::step(LPR) % 4 == 0, "units of a lane share their shifts");
    extern __shared__ __align__(16) uint8_t smem[];
    const LPtr tab = 0;   // the tables are the start of LDS
    Plan *P = (Plan *)(smem + U::kTabBytes);
    int8_t *xq = (int8_t *)(P + 1);
    constexpr uint32_t kUnits = LPR * UPL, K = 64 * kUnits;   // a row's units, columns
    double *xd = (double *)(xq + NT * K);
    auto *outs = (GuOut<NT, RPW> *)(xd + NT * (K / 32));
    const uint32_t tid = threadIdx.x, lane = tid & 63u, bid = blockIdx.x, nblk = gridDim.x;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const KArgs ka = kargs();
    constexpr bool uniq = SRC == kSrcHost;
    // prologue loads ahead of the weight stream: activations, codebook
    constexpr uint32_t kOpt = 8u * kUnits;     // octs per token
    const uint32_t no = a.src.n_tok * kOpt;
    Oct v0 = {};
    if (tid < no) v0 = ld_oct(a.x, tid);
    const uint32_t code = U::code(tid, kT);

    // this lane's unit fields within a task's rows
    const uint32_t li = lane % LPR, slot = lane / LPR;
    const typename U::Offs of = U::offs(slot * a.rb_gu, li);
    int32_t idv = -1;
    uint32_t selv = 0;
    uint32_t T0 = 0, T1 = 0, T = 0;
    // row base of task t's gate (which 0) or up (1) rows
    auto rows_of = [&](uint32_t t, int which) __attribute__((always_inline)) {
        const uint32_t u = __umulhi(t, a.tpe_inv), r0 = (t - u * a.tpe) * RPW;
        const int32_t id = uniq ? ka->hl.id[u] : __builtin_amdgcn_readlane(idv, u);
        return uniform_ptr(a.base + (uint64_t)(uint32_t)id * a.stride + (which ? a.ou : a.og) +
                           (uint64_t)(r0 * a.rb_gu));
    };
    // The wave's units in the order it takes them: per task the gate rows'
    // UPL units, then the up rows'.  One unit is held in registers, and its
    // registers are refilled with the next one's fields as soon as they are
    // decoded: sixteen waves' units fill the CU's L1 path, and more in flight
    // only delays every wave's first unit (4-token window, us per layer with
    // 1 / 2 / 4 units in flight: 22.1 / 22.6 / 25.8).
    Raw s;
    uint32_t lT = 0, lw = 0, lm = 0;      // next unit to load: task, half, unit
    GPtr lb = nullptr;                    // its rows
    auto load = [&]() __attribute__((always_inline)) {
        const bool ok = lT < T1;
        if (ok && (UPL == 1 || lm == 0)) lb = rows_of(lT, lw);
        U::load(s, lb + U::step(LPR) * lm, of, ok);
        if (ok && ++lm == UPL) {
            lm = 0;
            lT += lw ? kW : 0u;
            lw ^= 1u;
        }
    };
    auto first_load = [&]() __attribute__((always_inline)) {
        lT = T;
        if (T < T1) load();
    };
    if constexpr (uniq) {
        const uint32_t PT = a.src.n_fixed * a.tpe;
        T0 = share_lo(PT, bid, nblk);
        T1 = share_lo(PT, bid + 1, nblk);
        T = T0 + wave;
    }
    PlanLane pl = {};
    if (!uniq && wave == 0) pl = build_plan<SRC == kSrcLogits>(P, a.src, lane, (uint32_t *)outs);
    // q8 of x (codes by units), the codebook tables
    auto quant_x = [&](const Oct &v, uint32_t i) __attribute__((always_inline)) {
        const uint32_t t = NT == 1 ? 0u : i / kOpt, o = i - t * kOpt;
        quant_oct(v, o, kUnits, xq + t * K, xd + t * (2u * kUnits));
    };
    if (tid < no) quant_x(v0, tid);
    for (uint32_t i = tid + kT; i < no; i += kT) quant_x(ld_oct(a.x, i), i);
    U::init(smem, code, tid, kT);
    if (uniq) first_load();
    bar();
    if constexpr (!uniq) {
        const uint32_t nu = P->nu;
        idv = lane < nu ? P->uid[lane] : -1;
        selv = lane < nu ? P->sel[lane] : 0u;
        if (NT == 1) {
            T0 = share_lo(nu * a.tpe, bid, nblk);
            T1 = share_lo(nu * a.tpe, bid + 1, nblk);
        } else {
            share_weighted(selv, nu, a.tpe, bid, nblk, lane, T0, T1);
        }
        T0 = __builtin_amdgcn_readfirstlane(T0);
        T1 = __builtin_amdgcn_readfirstlane(T1);
        T = T0 + wave;
        first_load();
        if (bid == 0 && wave == 0) {   // the down launch reuses this plan
            finish_plan(P, pl, lane);
            constexpr uint32_t n = sizeof(Plan) / 16;
#pragma unroll
            for (uint32_t i = 0; i < n; i += 64)
                if (i + lane < n) ((uint4 *)a.gplan)[i + lane] = ((const uint4 *)P)[i + lane];
        }
    }

    GuOut<NT, RPW> &out = outs[wave];
    uint32_t cnt = 0;
    auto flush = [&]() __attribute__((always_inline)) {
        for (uint32_t i = lane; i < cnt; i += 64) {
            a.h[out.dst[i]] = (float)silu_mul(out.g[i], out.u[i]);
        }
        cnt = 0;
    };
    auto finish = [&](uint32_t t0, uint32_t u, uint32_t sel, const double (&g)[NT],
                      const double (&up)[NT]) __attribute__((always_inline)) {
        const uint32_t r = (t0 - u * a.tpe) * RPW + slot;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            if (NT > 1 && !((sel >> t) & 1u)) continue;
            const double gs = q4mi_rsum<LPR>(g[t]), us = q4mi_rsum<LPR>(up[t]);
            if (li == LPR - 1) {
                out.g[cnt + slot] = gs;
                out.u[cnt + slot] = us;
                out.dst[cnt + slot] = (u * kMaxT + t) * a.n_ff + r;
            }
            cnt += RPW;
        }
        if (cnt >= 64) flush();
    };
    if (T < T1) {
        double g[NT], acc[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) acc[t] = 0.0;
        uint32_t up = 0, um = 0;              // half, unit of the one to compute
        uint32_t u = __umulhi(T, a.tpe_inv);
        uint32_t sel = uniq ? 1u : (uint32_t)__builtin_amdgcn_readlane((int)selv, u);
        while (T < T1) {
            const uint32_t un = li + LPR * um;
            UnitW w;
            U::decode(tab, s, of, w);
            if (!U::kRawW) {
                unit_consumed(w);
                load();
            }
#pragma unroll
            for (int t = 0; t < NT; t++)
                if (NT == 1 || ((sel >> t) & 1u))
                    acc[t] = unit_dot64<TY>(w, xq + t * K, xd + t * (2u * kUnits), kUnits, un, acc[t]);
            if (U::kRawW) load();
            if (UPL == 1 || ++um == UPL) {
                um = 0;
                if (!up) {
#pragma unroll
                    for (int t = 0; t < NT; t++) g[t] = acc[t];
                } else {
                    finish(T, u, sel, g, acc);
                    T += kW;
                    u = min(__umulhi(T, a.tpe_inv), kMaxU - 1);
                    sel = uniq ? 1u : (uint32_t)__builtin_amdgcn_readlane((int)selv, u);
                }
                up ^= 1u;
#pragma unroll
                for (int t = 0; t < NT; t++) acc[t] = 0.0;
            }
        }
    }
    flush();
}

// ---------------------------------------------------------------- down
// What bounds it: the prologue (every block quantizes every selected h row)
// and, behind it, the weights' decode as above.  Measured per launch, copying
// rows through an LDS ring / this kernel: one token 6.6 / 4.9 us, 4 tokens
// (hidden 2048, 18 MB) 15.9 / 9.1 us, 4 tokens at hidden 2560 IQ4_NL 20.8 /
// 14.5 us.
//
// A block owns dn_rows output rows.  Its waves form dn_rows / (rows per wave)
// row slices; the waves of a slice take every kES-th expert each, their lanes
// the slice's rows, UPR units (lanes) per row.  A wave adds w[u][t] times its
// lanes' partial dots over its experts in registers; the block then joins
// the lanes and the waves through LDS in a fixed order.
//
// LDS: [tables] | h codes [nsel_cap][n_ff] | h scales | parts [kW][NT][]
template <uint32_t TY, int NT, int UPR, int SRC>
__global__ __launch_bounds__(kT) void moe_dn_k(MoeArgs a) {
    using U = Unit<TY>;
    using Raw = typename U::Raw;
    constexpr bool uniq = SRC == kSrcHost;
    constexpr uint32_t RPW = 64 / UPR;                 // rows a wave can hold
    constexpr bool kPow2 = (UPR & (UPR - 1)) == 0;
    constexpr uint32_t NV = kPow2 ? 1u : (uint32_t)UPR;   // partial sums per row and wave
    constexpr uint32_t n_ff = 64u * UPR, opr = 8u * UPR;   // h values, octs per row
    extern __shared__ __align__(16) uint8_t smem[];
    const LPtr tab = 0;   // the tables are the start of LDS
    int8_t *hq = (int8_t *)(smem + U::kTabBytes);
    float *hd = (float *)(hq + (size_t)a.nsel_cap * n_ff);
    float *part = hd + (size_t)a.nsel_cap * (2u * UPR);   // [kW][NT][RPW * NV]
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r0 = blockIdx.x * a.dn_rows, nr = min(a.dn_rows, a.n_embd - r0);
    const uint32_t nslice = (a.dn_rows + RPW - 1) / RPW;   // row slices of the block
    const uint32_t rps = (a.dn_rows + nslice - 1) / nslice;   // rows per slice (<= RPW)
    const uint32_t slice = wave % nslice, es = wave / nslice, ES = kW / nslice;
    const uint32_t nt = a.src.n_tok;
    const KArgs ka = kargs();

    // device lists: the plan of this call's gate/up launch, lane u holding
    // expert u's fields (and pair slot u's h row)
    int32_t idv = -1;
    uint32_t nu = 0, nsel = 0, selv = 0, psv = 0, prv = 0;
    float wv[NT];
    if constexpr (!uniq) {
        const Plan *P = a.gplan;
        nu = P->nu;
        nsel = P->nsel;
        idv = P->uid[lane];
        selv = P->sel[lane];
        psv = P->pslot[lane];
        prv = P->prow[lane];
#pragma unroll
        for (int t = 0; t < NT; t++) wv[t] = P->w[t][lane];
    } else {
        nu = nsel = a.src.n_fixed;
    }
    // old y of this thread's output (16 lanes per output, the last one stores)
    const uint32_t o16 = tid >> 4, nout = nt * nr;
    const bool owner = (tid & 15u) == 15u;
    auto y_at = [&](uint32_t o) -> float * {
        const uint32_t t = o / nr;
        return a.y + (size_t)t * a.n_embd + r0 + (o - t * nr);
    };
    float yv = 0.f;
    if (owner && o16 < nout) yv = *y_at(o16);
    const uint32_t code = U::code(tid, kT);

    // h rows this wave quantizes: pair slots wave, wave + kW, ..., OJ octs per
    // lane and row
    constexpr uint32_t OJ = (opr + 63) / 64, kB = OJ == 1 ? 3 : 2;
    Oct hv[kB][OJ];
    auto load_rows = [&](uint32_t q) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t k = 0; k < kB; k++)
            if (q + k * kW < nsel) {
                const uint32_t s = q + k * kW;
                const uint32_t row = uniq ? s * kMaxT : (uint32_t)__builtin_amdgcn_readlane((int)prv, s);
#pragma unroll
                for (uint32_t j = 0; j < OJ; j++)
                    if (opr % 64 == 0 || lane + 64 * j < opr)
                        hv[k][j] = ld_oct(a.h + (size_t)row * n_ff, lane + 64 * j);
            }
    };
    auto quant_rows = [&](uint32_t q) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t k = 0; k < kB; k++)
            if (q + k * kW < nsel) {
                const uint32_t s = q + k * kW;
#pragma unroll
                for (uint32_t j = 0; j < OJ; j++)
                    if (opr % 64 == 0 || lane + 64 * j < opr)
                        quant_oct(hv[k][j], lane + 64 * j, UPR, hq + s * n_ff, hd + s * (2u * UPR));
            }
    };

    // the lane's row of the slice and unit of the row
    const uint32_t slot = lane / UPR, un = lane % UPR;
    const uint32_t rr = slice * rps + slot;             // row within the block
    const bool act = es < ES && slot < rps && rr < nr;
    // (idle lanes read the block's first row)
    const typename U::Offs of = U::offs((act ? rr : 0u) * a.rb_dn, un);
    Raw s;                                              // (one unit in flight, as above)
    // (past the last expert: one dword line of the last one's rows, so that
    // every wait knows how many loads are behind it)
    GPtr lb = nullptr;
    auto load_w = [&](uint32_t u) __attribute__((always_inline)) {
        const bool ok = u < nu;
        if (ok) {
            const int32_t id = uniq ? ka->hl.id[u] : __builtin_amdgcn_readlane(idv, u);
            lb = uniform_ptr(a.base + (uint64_t)(uint32_t)id * a.stride_d + a.od +
                             (uint64_t)(r0 * a.rb_dn));
        }
        U::load(s, lb, of, ok);
    };
    const bool work = es < ES && es < nu;
    load_rows(wave);
    U::init(smem, code, tid, kT);
    quant_rows(wave);
    if (work) load_w(es);
    for (uint32_t q = wave + kB * kW; q < nsel; q += kB * kW) {
        load_rows(q);
        quant_rows(q);
    }
    bar();

    float acc[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t] = 0.f;
    if (work) {
        for (uint32_t u = es; u < nu; u += ES) {
            const uint32_t sel = uniq ? 1u : (uint32_t)__builtin_amdgcn_readlane((int)selv, u);
            uint32_t ps = uniq ? u : (uint32_t)__builtin_amdgcn_readlane((int)psv, u);
            UnitW w;
            U::decode(tab, s, of, w);
            if (!U::kRawW) {
                unit_consumed(w);
                load_w(u + ES);
            }
#pragma unroll
            for (int t = 0; t < NT; t++) {
                if (!uniq && !((sel >> t) & 1u)) continue;
                const float f = unit_dot<TY>(w, hq + ps * n_ff, hd + ps * (2u * UPR), UPR, un, 0.f);
                const float wt = uniq ? ka->hl.w[u]
                                      : __builtin_bit_cast(float, __builtin_amdgcn_readlane(
                                            __builtin_bit_cast(int, wv[t]), u));
                acc[t] = fmaf(wt, f, acc[t]);
                ps++;
            }
            if (U::kRawW) load_w(u + ES);
        }
    }
    // join: a row's lanes (by DPP where their count is a power of two), then
    // its waves in es order
#pragma unroll
    for (int t = 0; t < NT; t++) {
        float *j = part + ((size_t)wave * NT + t) * (RPW * NV);
        if constexpr (kPow2) {
            const float v = q4mi_rsum<UPR>(acc[t]);
            if (un == UPR - 1) j[slot] = v;
        } else {
            if (slot < RPW) j[slot * NV + un] = acc[t];
        }
    }
    bar();
    for (uint32_t o = o16; o < nout; o += kT / 16) {
        const uint32_t t = o / nr, row = o - t * nr;
        const uint32_t sl = row / rps, sr = row - sl * rps;
        float v = 0.f;
        for (uint32_t i = tid & 15u; i < ES * NV; i += 16) {
            const uint32_t w = i / NV, p = i - w * NV;
            v += part[(((size_t)w * nslice + sl) * NT + t) * (RPW * NV) + sr * NV + p];
        }
        v = q4mi_rsum<16>(v);
        if (owner) {
            float *y = y_at(o);
            *y = (o == o16 ? yv : *y) + v;
        }
    }
}

// ------------------------------------------------------------------ host
constexpr size_t kLdsCap = 160 * 1024;

template <class Kern>
static bool moe_launch(Kern kern, const MoeArgs &a, uint32_t grid, size_t lds, DynLds &st,
                       const char *name) {
    if (!dyn_lds_ok((const void *)kern, lds, kLdsCap, st, name)) return false;
    kern<<<dim3(grid), dim3(kT), lds, stream()>>>(a);
    return launch_ok(name);
}

// bytes build_plan uses at its scratch: the 1024-bucket table, then (router
// logits) one token's 64 picks and probabilities
constexpr size_t kPlanTable = 4096 + 512;

template <uint32_t TY, int NT, int LPR, int UPL, int SRC>
static bool launch_gu(const MoeArgs &a) {
    constexpr uint32_t RPW = 64 / LPR;
    static DynLds state;
    MoeArgs b = a;
    b.tpe = a.n_ff / RPW;
    b.tpe_inv = (uint32_t)((0x100000000ull + b.tpe - 1) / b.tpe);
    const size_t fixed = al16(Unit<TY>::kTabBytes + sizeof(Plan) + (size_t)NT * a.K +
                              (size_t)NT * (a.K / 32) * 8);
    const size_t lds = fixed + std::max(sizeof(GuOut<NT, RPW>) * kW, kPlanTable);
    return moe_launch(moe_gu_k<TY, NT, LPR, UPL, SRC>, b, (uint32_t)cu_count(), lds, state,
                      "moe_gu_k");
}

template <uint32_t TY, int NT, int UPR, int SRC>
static bool launch_dn(const MoeArgs &a, uint32_t nu_host) {
    constexpr uint32_t RPW = 64 / UPR, NV = (UPR & (UPR - 1)) == 0 ? 1u : (uint32_t)UPR;
    static DynLds state;
    MoeArgs b = a;
    // rows per block: one block per CU, but no fewer rows than a wave holds
    // (up to 8)
    const uint32_t cus = (uint32_t)cu_count();
    b.dn_rows = std::min(kDnRowsMax, std::max((a.n_embd + cus - 1) / cus, std::min(8u, RPW)));
    b.nsel_cap = nu_host ? nu_host : kMaxU;   // selected pairs (<= 64)
    const size_t hb = (size_t)b.nsel_cap * a.n_ff + (size_t)b.nsel_cap * (a.n_ff / 32) * 4;
    const size_t lds = Unit<TY>::kTabBytes + hb + (size_t)kW * NT * RPW * NV * 4;
    return moe_launch(moe_dn_k<TY, NT, UPR, SRC>, b, (a.n_embd + b.dn_rows - 1) / b.dn_rows, lds,
                      state, "moe_dn_k");
}

template <uint32_t TY, int NT, int LPR, int UPL>
static bool gu_src(const MoeArgs &a) {
    if constexpr (NT == 1) {
        if (a.src.lg) return launch_gu<TY, NT, LPR, UPL, kSrcLogits>(a);
        if (a.src.unique) return launch_gu<TY, NT, LPR, UPL, kSrcHost>(a);
    } else if (a.src.lg || a.src.unique) {
        set_error("moe_gu_k: host lists and router logits take one token");
        return false;
    }
    return launch_gu<TY, NT, LPR, UPL, kSrcDev>(a);
}

// Gate/up lanes per row x units per lane, by the row's 64-value units.
template <uint32_t TY, int NT>
static bool gu_dispatch(const MoeArgs &a) {
    switch (a.K / 64) {
    case 4: return gu_src<TY, NT, 4, 1>(a);
    case 8: return gu_src<TY, NT, 8, 1>(a);
    case 16: return gu_src<TY, NT, 16, 1>(a);
    case 32: return gu_src<TY, NT, 32, 1>(a);
    case 64: return gu_src<TY, NT, 32, 2>(a);
    case 128: return gu_src<TY, NT, 32, 4>(a);
    case 40: return gu_src<TY, NT, 8, 5>(a);
    case 10:   // 640 columns: Q8_0 alone has whole-dword rows there
        if constexpr (TY == Q4MI_T_Q8_0) return gu_src<TY, NT, 2, 5>(a);
    }
    set_error("moe_gu_k: K=%u not covered", a.K);
    return false;
}

template <uint32_t TY, int NT, int UPR>
static bool dn_src(const MoeArgs &a, uint32_t nu_host) {
    if constexpr (NT == 1) {
        if (a.src.unique) return launch_dn<TY, NT, UPR, kSrcHost>(a, nu_host);
    } else if (a.src.unique) {
        set_error("moe_dn_k: host lists take one token");
        return false;
    }
    return launch_dn<TY, NT, UPR, kSrcDev>(a, nu_host);
}

template <uint32_t TY, int NT>
static bool dn_dispatch(const MoeArgs &a, uint32_t nu_host) {
    switch (a.n_ff / 64) {
    case 4: return dn_src<TY, NT, 4>(a, nu_host);
    case 8: return dn_src<TY, NT, 8>(a, nu_host);
    case 10: return dn_src<TY, NT, 10>(a, nu_host);
    case 16: return dn_src<TY, NT, 16>(a, nu_host);
    }
    set_error("moe_dn_k: n_ff=%u not covered", a.n_ff);
    return false;
}

// Dispatch of the types instantiated outside moe_decode.hip (moe_fmt_*.hip).
bool moe_fmt_gu(uint32_t ty, int nt, const MoeArgs &a);
bool moe_fmt_dn(uint32_t ty, int nt, const MoeArgs &a, uint32_t nu_host);

}  // namespace q4mi
