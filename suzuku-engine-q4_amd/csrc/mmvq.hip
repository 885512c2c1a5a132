// Dense decode MMVQ: y[t][r] = scale * (W_r . q8(x_t)) for 1..8 tokens over
// IQ3_S, Q8_0, IQ4_NL, Q2_0, IQ2_S or Q6_K weight rows.  C ABI: q4_mmvq_n and friends (reference
// src/q4_mmvq.cu:266-349, src/q4.h:914-927) plus q4mi_mmvq, which takes
// already-quantized activations and can export the per-group int32 sums.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

#include "mmvq_engine.h"
#include "moe_unit.h"
#include "q4mi_internal.h"

namespace q4mi {

// Optional build (-DQ4MI_GTRACE): thread 0 of each of the first 1024 blocks
// records wall-clock phase timestamps (10 ns ticks) of the last call.
#ifdef Q4MI_GTRACE
static __device__ unsigned long long g_gtr[1024 * 8];
#define Q4MI_GTR(k) do { if (threadIdx.x == 0 && blockIdx.x < 1024) g_gtr[blockIdx.x * 8 + (k)] = wall_clock64(); } while (0)
#else
#define Q4MI_GTR(k) do { } while (0)
#endif

bool quant8_launch(const float *x, const int32_t *ids, uint64_t rows, uint32_t cols,
                   int8_t *q, float *d, int32_t *bs);

// XF: fp32 activations xf [nt][K], quantized by every block into LDS
// behind its weight tile (the q8 codes and scales of q8_quant_k, bit for
// bit), so a call needs no separate quantize launch; else xq / xd hold them.
// (Two instantiations: the in-block quantizer's batched loads take 32
// registers, which the pre-quantized kernel does not pay for.)
template <class F, int NT, int TPR, int GPT, bool XF, int NTHR>
__global__ __launch_bounds__(NTHR) void mmvq_k(const uint8_t *__restrict__ W, uint32_t rows,
                                              uint32_t K, uint32_t rb, uint32_t R,
                                              const float *__restrict__ xf,
                                              const int8_t *__restrict__ xq,
                                              const float *__restrict__ xd, uint32_t nt,
                                              float *__restrict__ y, float scale,
                                              int32_t *__restrict__ sums) {
    extern __shared__ __align__(16) uint8_t smem[];
    void *tab = smem;
    uint8_t *tile = smem + F::kTabBytes;
    const uint32_t tid = threadIdx.x;
    const uint32_t r0 = blockIdx.x * R;
    const uint32_t nr = min(R, rows - r0);
    const uint32_t G = K / 32;
    // Tables first, then the tile's copies, then the x loads: a wave's VMEM
    // operations complete in issue order, so loads issued behind the copies
    // return when the copies have landed (measured: copies first, or copies
    // from fewer waves while the others build the table and quantize, are
    // slower for IQ3_S 4096 x 4096).
    Q4MI_GTR(0);
    F::init(tab, tid, NTHR);
    Q4MI_GTR(1);
    stage_tile_issue(tile, W + (size_t)r0 * rb, nr * rb, tid, NTHR);
    Q4MI_GTR(2);
    const uint32_t hid = tid, nh = NTHR;
    const uint32_t gi = tid % TPR;
    XRegs<NT, GPT> x;
    // pre-quantized codes: loaded while the tile copy is in flight
    if constexpr (!XF) load_xregs<NT, GPT, TPR>(x, xq, xd, K, nt, gi);
    if constexpr (XF) {
        // 8 lanes per 32-value group, nh / 8 groups per pass; the loads of
        // kB passes are issued before any is used (a load issued behind the
        // tile copies returns only when they have landed, so one wait must
        // cover all of them)
        int8_t *lq = (int8_t *)(tile + ((R * rb + 15u) & ~15u));
        float *ld = (float *)(lq + (size_t)NT * K);
        // kB passes per round: one round covers a short x at any block size
        // (a larger kB is start-up code that such a call skips)
        constexpr int kB = NTHR >= 1024 ? 2 : NTHR >= 512 ? 4 : 8;
        const uint32_t ng = nt * G, step = nh / 8, sub = hid & 7u;
        for (uint32_t g0 = hid >> 3; g0 < ng; g0 += kB * step) {
            float4 v[kB];
#pragma unroll
            for (int k = 0; k < kB; k++) {
                const uint32_t gid = g0 + k * step;
                if (gid < ng) {
                    const uint32_t t = gid / G, g = gid % G;
                    v[k] = *(const float4 *)(xf + (size_t)t * K + 32u * g + 4u * sub);
                }
            }
#pragma unroll
            for (int k = 0; k < kB; k++) {
                const uint32_t gid = g0 + k * step;
                if (gid < ng) {   // uniform per 8-lane team
                    const uint32_t t = gid / G, g = gid % G;
                    float dd;
                    int bsum;
                    const uint32_t packed = q4mi_quant_team8(v[k], &dd, &bsum);
                    *(uint32_t *)(lq + (size_t)t * K + 32u * g + 4u * sub) = packed;
                    if (sub == 0) ld[gid] = dd;
                }
            }
        }
    }
    if constexpr (XF) {
        xq = (const int8_t *)(tile + ((R * rb + 15u) & ~15u));
        xd = (const float *)(xq + (size_t)NT * K);
    }
    Q4MI_GTR(3);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    Q4MI_GTR(4);
    __syncthreads();
    Q4MI_GTR(5);
    if constexpr (XF) load_xregs<NT, GPT, TPR>(x, xq, xd, K, nt, gi);
    for (uint32_t rr = tid / TPR; rr < nr; rr += NTHR / TPR) {
        float acc[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) acc[t] = 0.f;
        int32_t *srow = sums ? sums + (size_t)(r0 + rr) * G : nullptr;
        row_dot<F, NT, GPT, TPR>(tab, tile, (const uint32_t *)tile, rr * rb, gi, x, acc, srow,
                                 (size_t)rows * G);
        reduce_acc<TPR, NT>(acc);
        if (gi == TPR - 1) {
#pragma unroll
            for (int t = 0; t < NT; t++)
                if ((uint32_t)t < nt) y[(size_t)t * rows + r0 + rr] = scale * acc[t];
        }
    }
    Q4MI_GTR(6);
}

// a = {its lower half, b's lower half}, b = {a's upper half, its upper half}.
template <class T>
__device__ inline void swap_halves(T &a, T &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a),
                                                    __builtin_bit_cast(uint32_t, b), false, false);
    const uint32_t r0 = r[0], r1 = r[1];
    a = __builtin_bit_cast(T, r0);
    b = __builtin_bit_cast(T, r1);
}
// The sum of two neighbouring groups of a row, one pair per lane.
template <uint32_t TY>
__device__ inline float pair_sum(const float (&acc)[2], uint32_t li) {
    if constexpr (TY != Q4MI_T_Q6_K) return acc[1] + acc[0];
    // lanes 2k, 2k + 1 hold groups 4k, 4k + 2 and 4k + 1, 4k + 3
    const float keep = li & 1u ? acc[1] : acc[0], give = li & 1u ? acc[0] : acc[1];
    return keep + q4mi_team8_swap<0xB1>(give);
}

// The same products with the weights in registers (moe_unit.h), the kernel of
// most calls (unit_ok).  What bounds it: up to about 20 MB the launch, its
// prologue (codes and tables, 1.6 us) and the first loads' latency; above,
// the L1 path and, at several tokens, the codes' LDS reads.  Tile kernel /
// this one, us: IQ3_S 4096 x 4096 at 1 / 4 / 8 tokens 5.7 / 4.2, 13.0 / 6.5,
// 11.5 / 9.4; IQ3_S 151936 x 2048 58.7 / 29.6, 56.7 / 45.3, 91.2 / 66.5.
//
// 1024-thread blocks, each with a contiguous share of the rows; a wave's task
// is RPW = 64 / LPR rows, LPR lanes per row with UPL units each, and its
// registers are refilled with the next unit as soon as one is decoded.  The
// block holds the tokens' q8 codes in LDS, quantized there from fp32 x (XF)
// or laid out from xq / xd.
//
// A row's sum is the tile kernel's, bit for bit (so it depends neither on nt
// or XF nor on the weights' address): its lane i holds groups i, i + TPR, ...,
// adds them in that order by fp32 multiply-adds, and the lanes are joined as a
// tree over their index.  Here a lane's units hold two such chains, joined
// first.  Rows of 128 and 256 groups (TPR = 64) over 64 lanes put a chain's
// groups into lanes l and l + 32: the halves of the wave swap one unit group's
// sum and scale each (kFold), so that the lower lanes hold the chains of the
// first groups of units l, l + 32, ... and the upper ones those of the second.
// A Q6_K unit's groups lie two apart, so neighbouring lanes exchange one chain
// (pair_sum).  With a lane's own groups added first instead, IQ3_S at 4096
// columns had 8.0e-8 of error against 64 bits, not 7.7e-8.
//
// The grid size is an argument: reading gridDim makes the runtime fill 248
// bytes of hidden arguments at every launch (host time of a call, IQ3_S 1024 x
// 2048: 4.51 us with them, 4.21 without; the tile kernel, which never had
// them, 4.22).
//
// LDS (from offset 0): [tables] | x codes [NT][K] | x scales [NT][K/32]
template <uint32_t TY, int NT, int LPR, int UPL, bool XF>
__global__ __launch_bounds__(1024) void mmvq_u_k(const uint8_t *__restrict__ W, uint32_t rows,
                                                 uint32_t rb, const float *__restrict__ xf,
                                                 const int8_t *__restrict__ xq,
                                                 const float *__restrict__ xd, uint32_t nt,
                                                 float *__restrict__ y, float scale,
                                                 int32_t *__restrict__ sums, uint32_t nblk) {
    using U = Unit<TY>;
    constexpr uint32_t RPW = 64 / LPR, kUnits = LPR * UPL, K = 64 * kUnits, kOpt = 8 * kUnits;
    constexpr uint32_t kNT = 1024, kNW = kNT / 64;
    static_assert(UPL == 1 || !U::kEven || U::step(LPR) % 4 == 0, "units of a lane share their shifts");
    extern __shared__ __align__(16) uint8_t smem[];
    const LPtr tab = 0;
    int8_t *lq = (int8_t *)(smem + U::kTabBytes);
    float *ld = (float *)(lq + NT * K);
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t no = nt * kOpt;
    const uint32_t code = U::code(tid, kNT);
    for (uint32_t i = tid; i < no; i += kNT) {
        const uint32_t t = NT == 1 ? 0u : i / kOpt, o = i - t * kOpt;
        if constexpr (XF) {
            quant_oct<TY>(ld_oct(xf, i), o, kUnits, lq + t * K, ld + t * (K / 32));
        } else {
            *(uint2 *)(lq + t * K + code_at<TY>(o, kUnits)) = ((const uint2 *)xq)[i];
            const uint32_t g = o >> 2;
            if ((o & 3u) == 0)
                ld[t * (K / 32) + 2u * group_unit<TY>(g) + group_half<TY>(g)] = xd[t * (K / 32) + g];
        }
    }
    U::init(smem, code, tid, kNT);

    // this lane's units within a task's rows (rows past the matrix repeat its
    // last one)
    const uint32_t li = lane % LPR, slot = lane / LPR;
    const typename U::Offs of = U::offs(min(slot, rows - 1u) * rb, li);
    const uint32_t PT = (rows + RPW - 1) / RPW, rlast = rows > RPW ? rows - RPW : 0u;
    const uint32_t q = PT / nblk, r = PT % nblk, b = blockIdx.x;
    const uint32_t T1 = b * q + min(b, r) + q + (b < r ? 1u : 0u);
    uint32_t T = b * q + min(b, r) + wave;
    constexpr int D = UPL > 1 ? 2 : 1;
    typename U::Raw s[D];
    uint32_t lT = T, lm = 0;      // next unit to load
    GPtr lb = nullptr;
    auto load = [&](typename U::Raw &s) __attribute__((always_inline)) {
        const bool ok = lT < T1;
        if (ok && (UPL == 1 || lm == 0)) lb = uniform_ptr(W + (uint64_t)min(lT * RPW, rlast) * rb);
        U::load(s, lb + U::step(LPR) * lm, of, ok);
        if (ok && ++lm == UPL) {
            lm = 0;
            lT += kNW;
        }
    };
    if (T < T1) {
#pragma unroll
        for (int k = 0; k < D; k++) {
            load(s[k]);
            asm volatile("" ::: "memory");
        }
    }
    bar();
    if (T >= T1) return;
    constexpr bool kFold = LPR == 64;
    // token t's codes of unit un (the lane's um-th) and the scales they go with
    auto load_x = [&](UnitX &x, int t, uint32_t un, uint32_t um) __attribute__((always_inline)) {
        load_unit_q(x.q, lq + t * K, kUnits, un);
        const float *d = ld + t * (K / 32);
        if constexpr (kFold) {
            d += 2u * ((li & 31u) + 64u * um) + (li >> 5);
            x.d = make_float2(d[0], d[64]);
        } else {
            x.d = *(const float2 *)(d + 2u * un);
        }
    };
    // one or two tokens' codes of the lane's unit stay in registers
    constexpr bool kXR = UPL == 1 && NT <= 2;
    UnitX xr[kXR ? NT : 1];
    if constexpr (kXR) {
#pragma unroll
        for (int t = 0; t < NT; t++) load_x(xr[t], t, li, 0);
    }
    float acc[NT][2];
#pragma unroll
    for (int t = 0; t < NT; t++) acc[t][0] = acc[t][1] = 0.f;
    uint32_t um = 0;
    while (T < T1) {
#pragma unroll
        for (int k = 0; k < D; k++) {
            const uint32_t un = li + LPR * um;
            const uint32_t row = min(T * RPW, rlast) + slot;
            UnitW w;
            if (k == 0 || T < T1) {
                U::decode(tab, s[k], of, w);
                if (!U::kRawW) unit_consumed(w);
                if (kFold) swap_halves(w.d[0], w.d[1]);
            }
            if (!U::kRawW) load(s[k]);
            if (k == 0 || T < T1) {
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    if (NT > 2 && (uint32_t)t >= nt) continue;
                    UnitX xl;
                    if constexpr (!kXR) load_x(xl, t, un, um);
                    const UnitX &x = kXR ? xr[kXR ? t : 0] : xl;
                    int sm[2];
                    unit_sums<TY>(w, x.q, sm);
                    int c[2] = {sm[0], sm[1]};
                    if (kFold) swap_halves(c[0], c[1]);
                    float &a0 = acc[t][0], &a1 = acc[t][kFold ? 0 : 1];
                    a0 = fmaf((float)c[0], w.d[0] * x.d.x, a0);
                    a1 = fmaf((float)c[1], w.d[1] * x.d.y, a1);
                    if (!XF && sums && slot < rows) {
                        int32_t *o = sums + ((size_t)t * rows + row) * (K / 32);
                        o[unit_group<TY>(un, 0)] = sm[0];
                        o[unit_group<TY>(un, 1)] = sm[1];
                    }
                }
                if (UPL == 1 || ++um == UPL) {
                    um = 0;
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        if (kFold) {
                            acc[t][1] = acc[t][0];
                            swap_halves(acc[t][0], acc[t][1]);
                        }
                        const float v = q4mi_rsum<kFold ? 32 : LPR>(pair_sum<TY>(acc[t], li));
                        if (li == LPR - 1 && (uint32_t)t < nt && slot < rows)
                            y[(size_t)t * rows + row] = scale * v;
                        acc[t][0] = acc[t][1] = 0.f;
                    }
                    T += kNW;
                }
            }
            if (U::kRawW) {
                asm volatile("" ::: "memory");
                load(s[k]);
            }
        }
    }
}

template <uint32_t TY, int NT, int LPR, int UPL, bool XF>
static bool unit_launch(const uint8_t *W, uint32_t rows, const float *xf, const int8_t *xq,
                        const float *xd, uint32_t nt, float *y, float scale, int32_t *sums) {
    constexpr uint32_t K = 64 * LPR * UPL, RPW = 64 / LPR;
    const auto kern = mmvq_u_k<TY, NT, LPR, UPL, XF>;
    const size_t lds = Unit<TY>::kTabBytes + (size_t)NT * K + (size_t)NT * (K / 32) * 4;
    static DynLds state;
    if (!dyn_lds_ok((const void *)kern, lds, 160 * 1024, state, "mmvq_u_k")) return false;
    // one block per CU (each task at least one row set); the types without
    // tables to build take up to four times as many for a tall matrix, which
    // the CUs then share by their actual rate (151936 x 2048, 1 / 4 tokens,
    // one block per CU and four: Q8_0 64.1 / 67.2 and 60.0 / 66.1 us, IQ4_NL
    // 36.8 / 51.1 and 34.9 / 45.4, Q2_0 26.3 / 42.3 and 22.9 / 35.5)
    const uint32_t tasks = (rows + RPW - 1) / RPW, cus = (uint32_t)cu_count();
    const uint32_t most = Unit<TY>::kTabBytes ? 1u : 4u;
    const uint32_t grid = std::min(cus * std::max(1u, std::min(most, tasks / (64u * cus))), tasks);
    kern<<<dim3(grid), dim3(1024), lds, stream()>>>(W, rows, (uint32_t)q4mi_row_bytes(TY, K), xf, xq,
                                                    xd, nt, y, scale, sums, grid);
    return launch_ok("mmvq_u_k");
}

template <uint32_t TY, int NT>
static bool unit_nt(const uint8_t *W, uint32_t rows, uint32_t K, const float *xf, const int8_t *xq,
                    const float *xd, uint32_t nt, float *y, float scale, int32_t *sums) {
    const auto go = [&](auto lpr, auto upl) {
        constexpr int L = decltype(lpr)::value, P = decltype(upl)::value;
        return xf ? unit_launch<TY, NT, L, P, true>(W, rows, xf, xq, xd, nt, y, scale, sums)
                  : unit_launch<TY, NT, L, P, false>(W, rows, xf, xq, xd, nt, y, scale, sums);
    };
    // 4096 and 8192 columns: 64 lanes a row, or 32 with twice the units (the
    // same bits).  64 give the waves more tasks and swap sums (kFold) per unit
    // and token; 32 are faster from three tokens on where there are four (Q6_K,
    // whose units take more registers: eight) rows a wave and more.  64 / 32
    // lanes, us, 4 tokens at 4096 columns: IQ3_S 4096 rows 6.5 / 7.0, 16384 13.1
    // / 13.2, 32768 21.8 / 20.5; Q2_0 16384 12.4 / 11.4; Q6_K 24576 22.7 / 23.8,
    // 32768 30.8 / 29.5, 50000 46.1 / 43.0.  Q8_0 (no table, 68 bytes a unit)
    // always takes 32.
    constexpr bool kMay32 = TY == Q4MI_T_Q8_0 || NT > 2, kMay64 = TY != Q4MI_T_Q8_0;
    const bool l32 = !kMay64 || rows >= (TY == Q4MI_T_Q6_K ? 32768u : 16384u);
    using std::integral_constant;
#define Q4MI_L(L, P) go(integral_constant<int, L>(), integral_constant<int, P>())
    switch (K / 64) {
    case 4: return Q4MI_L(4, 1);
    case 8: return Q4MI_L(8, 1);
    case 16: return Q4MI_L(16, 1);
    case 32: return Q4MI_L(32, 1);
    case 64:
        if constexpr (kMay32)
            if (l32) return Q4MI_L(32, 2);
        if constexpr (kMay64) return Q4MI_L(64, 1);
        break;
    case 128:
        if constexpr (kMay32)
            if (l32) return Q4MI_L(32, 4);
        if constexpr (kMay64) return Q4MI_L(64, 2);
        break;
    case 40: return Q4MI_L(8, 5);
    case 10:   // 640 columns: not of the 256-value superblock types
        if constexpr (TY == Q4MI_T_Q8_0 || TY == Q4MI_T_IQ4_NL || TY == Q4MI_T_Q2_0)
            return Q4MI_L(2, 5);
    }
#undef Q4MI_L
    set_error("mmvq: K=%u not covered", K);
    return false;
}

template <uint32_t TY>
static bool unit_any(const uint8_t *W, uint32_t rows, uint32_t K, const float *xf, const int8_t *xq,
                     const float *xd, uint32_t nt, float *y, float scale, int32_t *sums) {
    if (nt == 1) return unit_nt<TY, 1>(W, rows, K, xf, xq, xd, nt, y, scale, sums);
    if (nt == 2) return unit_nt<TY, 2>(W, rows, K, xf, xq, xd, nt, y, scale, sums);
    if (nt <= 4) return unit_nt<TY, 4>(W, rows, K, xf, xq, xd, nt, y, scale, sums);
    return unit_nt<TY, 8>(W, rows, K, xf, xq, xd, nt, y, scale, sums);
}

// Which kernel.  The register path takes rows that are whole dwords (others,
// e.g. IQ3_S at 256 columns, keep the tile kernel's 2-byte copies), and is
// the faster one over 480 calls (six types, 500-50000 rows, 1024-4096
// columns, 1-8 tokens: 0.67 of the tile kernel's time in the geometric mean)
// but for the tall Q8_0 matrices at one or two tokens, where the tile
// kernel's many short blocks stream closer to the memory's rate.  Tile /
// register kernel, us, over 0.7-1.5 GB of distinct matrices (runs differ by 1 to 2 %):
//   1 token, columns      1024          2048          4096          8192
//     112 MB          23.1 / 23.7   22.7 / 22.7   23.3 / 21.6   23.6 / 22.6
//     144 MB          27.8 / 29.0   27.5 / 27.5   27.9 / 27.3   28.7 / 27.7
//     208 MB          38.4 / 42.0   37.4 / 39.8   38.1 / 39.2   38.5 / 39.0
//     331 MB          58.1 / 63.2   58.1 / 61.5   58.3 / 59.0   57.8 / 60.6
//   2 tokens
//     144 MB          28.8 / 29.5   29.0 / 28.3   31.0 / 28.8   32.0 / 28.5
//     208 MB          39.8 / 42.4   39.5 / 41.0   42.1 / 41.3   42.9 / 40.3
//     331 MB          61.2 / 64.1   60.4 / 61.3   63.4 / 62.0   63.9 / 62.0
//     500 MB          89.0 / 97.0   87.7 / 91.7   92.8 / 90.4   92.1 / 91.1
static bool unit_ok(uint32_t ty, const uint8_t *W, uint64_t rows, uint64_t K, uint32_t nt) {
    const uint64_t rb = q4mi_row_bytes(ty, K), bytes = rows * rb;
    if (((uintptr_t)W & 3u) || rb % 4) return false;
    if (ty != Q4MI_T_Q8_0 || nt > 2) return true;
    return bytes < (160ull << 20) || (nt == 2 && K > 2560);
}

// weight bytes per row tile
static uint32_t tile_target(uint32_t ty) {
    return ty == Q4MI_T_Q8_0 || ty == Q4MI_T_Q6_K ? 24576u : 14336u;
}

template <class F, int NT>
static bool mmvq_launch_nt(const uint8_t *W, uint32_t rows, uint32_t K, const float *xf,
                           const int8_t *xq, const float *xd, uint32_t nt, float *y,
                           float scale, int32_t *sums) {
    const uint32_t G = K / 32;
    const RowLayout L = layout_for(G);
    const uint32_t rb = (uint32_t)q4mi_row_bytes(F::kType, K);
    const size_t xlds = xf ? (size_t)NT * K + (size_t)NT * (K / 32) * 4 : 0;
    auto lds_of = [&](uint32_t r) {
        return F::kTabBytes + (((size_t)r * rb + 15) & ~(size_t)15) + xlds + 64;
    };
    uint32_t nthr = 256;
    uint32_t R = L.tpr ? tile_rows(rb, L.tpr, tile_target(F::kType)) : 1;
    // fp32 x (the short matrices): a 1024-thread block per 1024 / tpr rows
    // (one row per wave) while that still fills the CUs, else 512 threads
    // per 512 / tpr rows.  The compute after a tile lands is then a quarter
    // (a half) of a 256-thread block's, whose waves take four rows each
    // (IQ3_S 4096 x 4096: 256 blocks of 16 rows, 6.2 against 7.1 us).  Several
    // tokens' x registers fit 1024-thread blocks (128 VGPRs) only at one
    // token, 512-thread blocks up to two.
    if (xf && L.tpr) {
        const uint32_t cus = (uint32_t)cu_count();
        for (uint32_t n = 1024; n >= 512; n /= 2) {
            const uint32_t r = n / (uint32_t)L.tpr;
            if ((n == 1024 ? NT == 1 : NT <= 2) && (rows + r - 1) / r >= cus && lds_of(r) <= 65536) {
                nthr = n;
                R = r;
                break;
            }
        }
    }
    // pre-quantized x at one token (the tall matrices, many tiles per CU):
    // 512-thread blocks of one row per wave (Q8_0 151936 x 2048: 59.8 against
    // 61.2 us, 8-row tiles either way)
    if (!xf && NT == 1 && L.tpr) {
        const uint32_t r = 512u / (uint32_t)L.tpr;
        if ((rows + r - 1) / r >= 4u * (uint32_t)cu_count() && lds_of(r) <= 65536) {
            nthr = 512;
            R = r;
        }
    }
#ifdef Q4MI_KNOBS
    if (getenv("Q4MI_GEMV_NTHR") && L.tpr && NT == 1 && xf) {
        nthr = (uint32_t)atoi(getenv("Q4MI_GEMV_NTHR"));
        R = tile_rows(rb, L.tpr, getenv("Q4MI_GEMV_TILE") ? (uint32_t)atoi(getenv("Q4MI_GEMV_TILE"))
                                                          : tile_target(F::kType), nthr);
    }
#endif
    const size_t lds = lds_of(R);
    const dim3 grid((rows + R - 1) / R), blk(nthr);
#define Q4MI_L(T, P)                                                                     \
    if (L.tpr == T && L.gpt == P) {                                                      \
        const auto args = [&](auto kern) {                                               \
            kern<<<grid, blk, lds, stream()>>>(W, rows, K, rb, R, xf, xq, xd, nt, y, scale, sums); \
        };                                                                               \
        if constexpr (NT == 1) {                                                         \
            if (xf && nthr == 1024) args(mmvq_k<F, NT, T, P, true, 1024>);              \
            else if (xf && nthr == 512) args(mmvq_k<F, NT, T, P, true, 512>);           \
            else if (xf) args(mmvq_k<F, NT, T, P, true, 256>);                          \
            else if (nthr == 512) args(mmvq_k<F, NT, T, P, false, 512>);                 \
            else args(mmvq_k<F, NT, T, P, false, 256>);                                 \
        } else if constexpr (NT == 2) {                                                  \
            if (xf && nthr == 512) args(mmvq_k<F, NT, T, P, true, 512>);                \
            else if (xf) args(mmvq_k<F, NT, T, P, true, 256>);                          \
            else args(mmvq_k<F, NT, T, P, false, 256>);                                 \
        } else {                                                                         \
            if (xf) args(mmvq_k<F, NT, T, P, true, 256>);                               \
            else args(mmvq_k<F, NT, T, P, false, 256>);                                 \
        }                                                                                \
        return launch_ok("mmvq_k");                                                      \
    }
    Q4MI_L(8, 1) Q4MI_L(16, 1) Q4MI_L(32, 1) Q4MI_L(64, 1) Q4MI_L(64, 2) Q4MI_L(64, 4)
    Q4MI_L(16, 5) Q4MI_L(4, 5)
#undef Q4MI_L
    set_error("mmvq: K=%u not covered", K);
    return false;
}

template <class F>
static bool mmvq_launch(const uint8_t *W, uint32_t rows, uint32_t K, const float *xf,
                        const int8_t *xq, const float *xd, uint32_t nt, float *y, float scale,
                        int32_t *sums) {
    if (nt == 1) return mmvq_launch_nt<F, 1>(W, rows, K, xf, xq, xd, nt, y, scale, sums);
    if (nt == 2) return mmvq_launch_nt<F, 2>(W, rows, K, xf, xq, xd, nt, y, scale, sums);
    if (nt <= 4) return mmvq_launch_nt<F, 4>(W, rows, K, xf, xq, xd, nt, y, scale, sums);
    return mmvq_launch_nt<F, 8>(W, rows, K, xf, xq, xd, nt, y, scale, sums);
}

// IQ3_S, Q8_0, IQ4_NL, Q2_0, IQ2_S, Q6_K with 8..256 groups per row (a
// whole number of blocks).
bool mmvq_covered(uint32_t ty, uint64_t K) {
    switch (ty) {
    case Q4MI_T_IQ3_S: case Q4MI_T_Q8_0: case Q4MI_T_IQ4_NL: case Q4MI_T_Q2_0:
    case Q4MI_T_IQ2_S: case Q4MI_T_Q6_K: break;
    default: return false;
    }
    if (!q4mi_row_bytes(ty, K) || K > 8192) return false;
    return layout_for((uint32_t)(K / 32)).tpr != 0;
}

// one launch for the type: pre-quantized (xq, xd) or fp32 x (xf)
static bool mmvq_any(uint32_t ty, const uint8_t *W, uint64_t rows, uint64_t K, const float *xf,
                     const int8_t *xq, const float *xd, uint32_t nt, float *y, float scale,
                     int32_t *sums) {
    const uint32_t r = (uint32_t)rows, k = (uint32_t)K;
    if (unit_ok(ty, W, rows, K, nt)) {
        switch (ty) {
        case Q4MI_T_IQ3_S: return unit_any<Q4MI_T_IQ3_S>(W, r, k, xf, xq, xd, nt, y, scale, sums);
        case Q4MI_T_Q8_0: return unit_any<Q4MI_T_Q8_0>(W, r, k, xf, xq, xd, nt, y, scale, sums);
        case Q4MI_T_IQ4_NL: return unit_any<Q4MI_T_IQ4_NL>(W, r, k, xf, xq, xd, nt, y, scale, sums);
        case Q4MI_T_Q2_0: return unit_any<Q4MI_T_Q2_0>(W, r, k, xf, xq, xd, nt, y, scale, sums);
        case Q4MI_T_IQ2_S: return unit_any<Q4MI_T_IQ2_S>(W, r, k, xf, xq, xd, nt, y, scale, sums);
        case Q4MI_T_Q6_K: return unit_any<Q4MI_T_Q6_K>(W, r, k, xf, xq, xd, nt, y, scale, sums);
        }
    }
    switch (ty) {
    case Q4MI_T_IQ3_S: return mmvq_launch<FmtIQ3S>(W, r, k, xf, xq, xd, nt, y, scale, sums);
    case Q4MI_T_Q8_0: return mmvq_launch<FmtQ80>(W, r, k, xf, xq, xd, nt, y, scale, sums);
    case Q4MI_T_IQ4_NL: return mmvq_launch<FmtIQ4NL>(W, r, k, xf, xq, xd, nt, y, scale, sums);
    case Q4MI_T_Q2_0: return mmvq_launch<FmtQ20>(W, r, k, xf, xq, xd, nt, y, scale, sums);
    case Q4MI_T_IQ2_S: return mmvq_launch<FmtIQ2S>(W, r, k, xf, xq, xd, nt, y, scale, sums);
    case Q4MI_T_Q6_K: return mmvq_launch<FmtQ6K>(W, r, k, xf, xq, xd, nt, y, scale, sums);
    }
    set_error("mmvq: type %u not covered", ty);
    return false;
}

bool mmvq_q8(uint32_t ty, const uint8_t *W, uint64_t rows, uint64_t K, const int8_t *xq,
             const float *xd, uint32_t nt, float *y, float scale, int32_t *sums) {
    return mmvq_any(ty, W, rows, K, nullptr, xq, xd, nt, y, scale, sums);
}

// Activations quantized inside the tile kernel's blocks: used while the codes
// of the padded token count fit 16 KB of LDS beside the tile and the call has at
// most 1024 row tiles.  Every block re-reads and re-quantizes all of x, so
// a tall matrix (Q8_0 151936 x 2048: 18992 tiles) is faster with one quantize
// launch (measured: 56.5 against 70.8 us at 1 token), a short one (IQ3_S 4096 x
// 4096: 512 tiles) without it (7.97 against 7.32 us).
static bool mmvq_fused_fits(uint32_t ty, uint64_t rows, uint64_t K, uint32_t nt) {
    const uint32_t ntp = nt == 1 ? 1 : nt == 2 ? 2 : nt <= 4 ? 4 : 8;
    if ((uint64_t)ntp * K > 16384) return false;
    const RowLayout L = layout_for((uint32_t)(K / 32));
    const uint32_t rb = (uint32_t)q4mi_row_bytes(ty, K);
    const uint32_t R = tile_rows(rb, L.tpr, tile_target(ty));
    return (rows + R - 1) / R <= 1024;
}

static bool mmvq_f32(uint32_t ty, const uint8_t *W, uint64_t rows, uint64_t K, const float *x,
                     uint32_t nt, float *y, float scale) {
    return mmvq_any(ty, W, rows, K, x, nullptr, nullptr, nt, y, scale, nullptr);
}

static int g_on = -1;
static const float *g_hold = nullptr;
static const float *g_cur_x = nullptr;
static uint64_t g_cur_k = 0;
static uint32_t g_cur_n = 0;

}  // namespace q4mi

using namespace q4mi;

extern "C" {

/* Q4_MMVQ=0 turns the int8 GEMV off (callers keep another path); any
 * other value or unset: on. */
int q4_mmvq_on(void) {
    if (g_on < 0) {
        const char *e = getenv("Q4_MMVQ");
        g_on = (e && e[0] == '0') ? 0 : 1;
    }
    return g_on;
}
void q4_mmvq_set(int v) { g_on = v; }
/* Kept for ABI shape: this library has no verify-only policy. */
void q4_mmvq_verify(int on) { (void)on; }

/* Allocate the activation buffers (call outside any stream capture). */
void q4_mmvq_warm(void) { (void)ensure_xq((size_t)8 * 8192); }

void q4_mmvq_hold(const float *d_x) {
    g_hold = d_x;
    g_cur_x = nullptr;
}
void q4_mmvq_release(void) {
    g_hold = nullptr;
    g_cur_x = nullptr;
}

/* y[t*nrows + r] = scale * dot(W row r, q8(x[t])), t < n (1..8).  Types:
 * IQ3_S, Q8_0, IQ4_NL, Q2_0, IQ2_S, Q6_K; ncols a whole number of blocks with
 * ncols/32 in {8,16,20,32,64,80,128,256}.  false = not covered; nothing
 * launched. */
bool q4_mmvq_n(uint32_t ty, const uint8_t *d_w, uint64_t nrows, uint64_t ncols,
               const float *d_x, float *d_y, float scale, uint32_t n) {
    if (!q4_mmvq_on() || n < 1 || n > 8 || !d_w || !d_x || !d_y || !nrows ||
        nrows > 0x7fffffffu || !mmvq_covered(ty, ncols)) {
        set_error("q4_mmvq_n: not covered");
        return false;
    }
    if ((uintptr_t)d_x % 16 == 0 && (unit_ok(ty, d_w, nrows, ncols, n) || mmvq_fused_fits(ty, nrows, ncols, n))) {
        // every block quantizes x itself: no quantize launch, no held codes
        g_cur_x = nullptr;
        return mmvq_f32(ty, d_w, nrows, ncols, d_x, n, d_y, scale);
    }
    if (!ensure_xq((size_t)8 * 8192)) return false;
    Scratch &s = lib_scratch();
    const bool reuse = g_hold && g_hold == d_x && g_cur_x == d_x && g_cur_k == ncols &&
                       g_cur_n >= n;
    if (!reuse) {
        if (!quant8_launch(d_x, nullptr, n, (uint32_t)ncols, s.xq, s.xd, nullptr))
            return false;
        g_cur_x = d_x;
        g_cur_k = ncols;
        g_cur_n = n;
    }
    return mmvq_q8(ty, d_w, nrows, ncols, s.xq, s.xd, n, d_y, scale, nullptr);
}

/* Pre-quantized variant: xq [n][ncols] int8, xd [n][ncols/32] fp32 (the
 * q4mi_quant8 layout).  d_sums (optional) receives the exact int32 group
 * sums, d_sums[(t*nrows + r)*(ncols/32) + g] = (2s+1) * sum w*q. */
bool q4mi_mmvq(uint32_t ty, const uint8_t *d_w, uint64_t nrows, uint64_t ncols,
               const int8_t *d_xq, const float *d_xd, uint32_t n, float *d_y, float scale,
               int32_t *d_sums) {
    if (n < 1 || n > 8 || !d_w || !d_xq || !d_xd || !d_y || !nrows || nrows > 0x7fffffffu ||
        !mmvq_covered(ty, ncols) || ((uintptr_t)d_xq & 15)) {
        set_error("q4mi_mmvq: not covered");
        return false;
    }
    return mmvq_q8(ty, d_w, nrows, ncols, d_xq, d_xd, n, d_y, scale, d_sums);
}

}  // extern "C"

#ifdef Q4MI_GTRACE
/* GEMV trace build only: the phase timestamps [1024 blocks][8] of the last
 * call. */
extern "C" bool q4mi_gtrace_read(unsigned long long *dst) {
    if (hipDeviceSynchronize() != hipSuccess) return false;
    return hipMemcpyFromSymbol(dst, HIP_SYMBOL(q4mi::g_gtr), sizeof(q4mi::g_gtr)) == hipSuccess;
}
#endif
