// Partial-pivoting LU panel with the rows held in registers (lu::Panel,
// src/lapack_like/factor/LU/Panel.hpp:15-60; pivot choice as blas::MaxInd,
// src/core/imports/blas/MaxInd.hpp:26-46).
//
// A panel of up to 128 columns is factored 32 columns at a time. Per 32-column block:
//   rpanel_kernel         the block's columns over all rows below the diagonal, 1024 rows per
//                         workgroup, two rows of 32 entries per thread in VGPRs;
//   panel_solve_kernel    the block's row interchanges in the panel's other columns and
//                         U12 = L11^-1 A12 for the columns to its right;
//   panel_update_kernel   A22 -= L21 U12 inside the panel.
// Every entry receives its updates one FMA at a time in step order, and the pivots are the
// first entries of largest magnitude, so the factors are bitwise those of lu::Panel.
//
// What bounds it: the chain of column steps (search, exchange, scale, update); a step moves a
// few hundred bytes. With the rows in LDS and the candidates exchanged through memory across
// all XCDs (lu_panel.hip) a step takes 4.7-5.2 us at any height: the LDS traffic of the rank-1
// update and two trips to memory. In registers the update costs only its FMAs, so a workgroup
// carries 1024 rows instead of 128, and 32 workgroups -- one XCD -- hold the 32768 rows of the
// tallest panel: their exchange stays in that XCD's L2 (0.95 us for a record and the winner's
// row, against 2.0-2.6 us through memory), and a panel of at most 1024 rows needs none.
// Measured per 128-column FP64 panel, all launches: 610 -> 215 us up to 1024 rows (a 32-column
// block 42 us, its solve 5 us, its update 6-10 us), 612 -> 375 us at 16384 rows (block 76-100 us).
// A block step is now about 2000 cycles of dependent work per workgroup (search 430, two
// barriers and the row's trip through LDS 900, division and scaling 300, FMAs 150-600), and
// 2500 more for the exchange with more than one workgroup.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "elx_common.hpp"
#include "exchange.hpp"
#include "wave.hpp"

namespace {

using elx::xchg::ld16;
using elx::xchg::mix32;
using elx::xchg::st16;
using elx::xchg::u4;
using elx::wv::bcast_lane;
using elx::wv::row_bcast;
using elx::wv::static_for;

constexpr int NTMAX = 512;                 // 8 waves: two per SIMD, 256 VGPRs each
constexpr int WS = 32;                     // columns per block
constexpr int RPT = 2;                     // rows per thread (two named halves of the code)
constexpr int RWG = NTMAX * RPT;           // rows per workgroup
constexpr int GMAX = 32;                   // workgroups (one XCD's CUs)
constexpr int NC = WS / 8;                 // 8-column chunks of a row
constexpr int WPANEL = 128;                // widest panel
constexpr int ROWLD = WS + 1;              // a row in LDS and the reciprocal of its pivot entry
constexpr int SPIN_LIMIT = 1 << 20;        // bounded wait: every wave exits

template <typename T>
struct RArgs {
    i64 mp;  // rows of the block (from its diagonal down)
    int w;   // columns, <= WS
    T* A;
    i64 lda;
    int32_t* dests;
    i64 goff;               // global index of the block's first row
    int2* spairs;           // 2 WS moves of this block (positions relative to its first row)
    const int32_t* orig_in; // row each panel position came from (null: the panel's first block)
    int32_t* orig_out;
    int c0;                 // the block's first column in the panel
    int W;                  // the panel's columns
    int last;               // the panel's last block
    int2* pairs;            // 2 W moves of the whole panel (positions relative to its first row)
    int32_t* info;
    int32_t* done;          // steps completed (fewer than w after an exactly zero pivot)
    int G;
    uint32_t seq_base;
    u4* uarea;              // uncached: [2][G] records, then [2][G][WS + 1] row entries
                            // and the pivot's reciprocal
    u4* xarea;              // the same in ordinary memory
};

template <int CTRL>
__device__ __forceinline__ uint32_t dpp32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t lane32(uint32_t v, int l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}

// The order key of a candidate magnitude: its bits (non-negative floats order like their bit
// patterns) as hi = high word + 1, 0 for no candidate, and lo.
struct Key {
    uint32_t hi, lo;
};
__device__ __forceinline__ Key key_of(double v, bool live) {
    const uint64_t b = (uint64_t)__double_as_longlong(fabs(v));
    return (live && v == v) ? Key{(uint32_t)(b >> 32) + 1u, (uint32_t)b} : Key{0u, 0u};
}
__device__ __forceinline__ Key key_of(float v, bool live) {
    return (live && v == v) ? Key{__float_as_uint(fabsf(v)) + 1u, 0u} : Key{0u, 0u};
}
__device__ __forceinline__ uint64_t key64(Key k) { return ((uint64_t)k.hi << 32) | k.lo; }
// the key of an exact zero
__device__ __forceinline__ bool key_is_zero(Key k) { return k.hi == 1u && k.lo == 0u; }

// Largest (smallest) value over the wave, or over lanes 0..7 with FEW: one DPP instruction per
// butterfly step.
template <bool FEW>
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    v = max(v, dpp32<0xB1>(v));   // quad_perm [1,0,3,2]
    v = max(v, dpp32<0x4E>(v));   // quad_perm [2,3,0,1]
    v = max(v, dpp32<0x141>(v));  // row_half_mirror
    if constexpr (FEW) return lane32(v, 0);
    v = max(v, dpp32<0x140>(v));  // row_mirror
    return max(max(lane32(v, 0), lane32(v, 16)), max(lane32(v, 32), lane32(v, 48)));
}
// The lane holding the largest key, ties to the smallest label; lane 0 when every key is 0.
// The high words alone decide unless two of them are equal.
template <bool FEW>
__device__ __forceinline__ int wave_argmax(Key k, uint32_t lbl) {
    const uint32_t mh = wave_max<FEW>(k.hi);
    uint64_t hit = __ballot(k.hi == mh);
    if (hit & (hit - 1)) {
        if (mh == 0) return 0;
        const bool in = k.hi == mh;
        const uint32_t ml = wave_max<FEW>(in ? k.lo : 0u);
        const bool in2 = in && k.lo == ml;
        const uint32_t nl = wave_max<FEW>(in2 ? ~lbl : 0u);
        hit = __ballot(in2 && ~lbl == nl);
    }
    return __ffsll((unsigned long long)hit) - 1;
}

__device__ __forceinline__ void bits_of(double v, uint32_t& lo, uint32_t& hi) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    lo = (uint32_t)b;
    hi = (uint32_t)(b >> 32);
}
__device__ __forceinline__ void bits_of(float v, uint32_t& lo, uint32_t& hi) {
    lo = __float_as_uint(v);
    hi = 0u;
}
__device__ __forceinline__ void value_of(u4 c, double& v) {
    v = __longlong_as_double((long long)(((uint64_t)c[1] << 32) | c[0]));
}
__device__ __forceinline__ void value_of(u4 c, float& v) { v = __uint_as_float(c[0]); }

__device__ __forceinline__ uint32_t xcc_id() {
    uint32_t x;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
    return x & 0xFu;
}

// MULTI: G > 1 workgroups, those with blockIdx % 8 == 0 of a grid of 8 G dealt round-robin over
// the XCDs. Column 0 is exchanged through uncached memory and its records carry each
// workgroup's XCD; once every reader has seen that all are the same (all readers see the same
// records, so all decide alike) the later columns go through that XCD's L2, otherwise they too
// go through uncached memory. Records and row entries are tagged as in exchange.hpp; both are
// double-buffered by column parity (a workgroup publishes column c + 2 only after it has read
// every record of column c + 1, each of which was published after its writer had read column
// c's row).
// NT: threads. A block of at most 128 (512) rows runs in 1 (4) waves: fewer waves to wait for at
// the barriers and a SIMD of its own for each.
template <typename T, bool MULTI, int NT>
__global__ __launch_bounds__(NT) void rpanel_kernel(RArgs<T> p) {
    constexpr int NW = NT / 64;
    __shared__ __align__(16) uint4 rec[2][NW];   // a wave's candidate: key, label
    __shared__ T rows[2][ROWLD];                 // the best candidate's row and reciprocal
    __shared__ T grow[2][ROWLD];                 // the winner's (MULTI)
    __shared__ int meta[2][4];                   // pivot position, winning workgroup, status

    if (MULTI && (blockIdx.x & 7) != 0) return;
    const int g = MULTI ? (int)(blockIdx.x >> 3) : 0, t = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, w = p.w;
    const uint32_t xcc = MULTI ? xcc_id() : 0u;
    if (*p.info != 0) {
        // an earlier block met an exactly zero pivot (or gave up): nothing changes any more
        if (g == 0) {
            if (t < 2 * WS) p.spairs[t] = int2{-1, -1};
            if (t < w) p.dests[t] = (int32_t)(p.goff + t);
            if (t == 0) *p.done = 0;
        }
        return;
    }

    T a[RPT][WS];
    int lbl[RPT], org[RPT];
    const i64 r0 = (i64)g * (NT * RPT) + t;
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const i64 r = r0 + q * NT;
        const bool ok = r < p.mp;
        lbl[q] = ok ? (int)r : -1;
        org[q] = ok ? (p.orig_in ? p.orig_in[p.c0 + r] : (int)(p.c0 + r)) : -1;
        const T* row = p.A + r;
#pragma unroll
        for (int j = 0; j < WS; ++j) a[q][j] = (ok && j < w) ? row[(i64)j * p.lda] : T(0);
    }
    // every load has landed before the first record goes out: a workgroup stores its rows only
    // after it has seen every other's records
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    const uint32_t nrec = 2u * (uint32_t)p.G, nunit = nrec * (2u + WS);
    bool l2 = false, stopped = false, aborted = false;
    int steps = 0, dest = lane;  // lane c: the pivot position of column c
    const int ngroups = (w + 7) / 8;
#pragma unroll 1
    for (int gi = 0; gi < NC; ++gi) {
        static_for<0, 8>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            const int c = gi * 8 + s;
            const int par = c & 1;
            // The search and the exchange change no row; the update below runs in straight line
            // under the rows' own masks, so the rows stay in fixed registers (a uniform branch
            // around it made the compiler copy them at every step).
            bool live = false;
            int piv = 0, wrow = -1;
            const T* us = MULTI ? grow[par] : rows[par];
            if (c < w && !stopped) {
                // each wave's candidate, the first of largest magnitude among its live rows, with
                // its row and reciprocal (the division runs beside the search)
                const Key k0 = key_of(a[0][s], lbl[0] >= c), k1 = key_of(a[1][s], lbl[1] >= c);
                const bool second = key64(k1) > key64(k0) || (key64(k1) == key64(k0) && lbl[1] < lbl[0]);
                const Key k = second ? k1 : k0;
                const uint32_t kl = (uint32_t)(second ? lbl[1] : lbl[0]);
                const T kinv = T(1) / (second ? a[1][s] : a[0][s]);
                const int cl = wave_argmax<false>(k, kl);
                const bool cq = __builtin_amdgcn_readlane(second ? 1 : 0, cl) != 0;
                if (lane == cl) rec[par][wave] = uint4{k.hi, k.lo, kl, 0u};
                __syncthreads();
                // the best of the NW waves, found alike by every wave; its lane writes the row
                // (a store of one lane takes the LDS as long as one of 64: 16 of them per step)
                const uint4 wr = rec[par][lane & (NW - 1)];
                const Key wk = lane < NW ? Key{wr.x, wr.y} : Key{0u, 0u};
                const int bw = wave_argmax<true>(wk, wr.z);
                Key bk = Key{lane32(wk.hi, bw), lane32(wk.lo, bw)};
                if (wave == bw && lane == cl) {
                    T* row = rows[par];
                    row[WS] = kinv;
                    // the chunks still to be updated; two separate bodies (the markers keep them
                    // from being merged into one with a select per word)
                    auto put = [&](auto qc) {
                        constexpr int q = decltype(qc)::value;
                        static_for<s, 8>([&](auto jc) { row[decltype(jc)::value] = a[q][decltype(jc)::value]; });
                        static_for<1, NC>([&](auto kc) {
                            constexpr int k = decltype(kc)::value;
                            if (gi + k < ngroups)
                                static_for<8 * k, 8 * k + 8>(
                                    [&](auto jc) { row[decltype(jc)::value] = a[q][decltype(jc)::value]; });
                        });
                    };
                    if (cq) {
                        put(std::integral_constant<int, 1>{});
                        asm volatile("; row 1");
                    } else {
                        put(std::integral_constant<int, 0>{});
                        asm volatile("; row 0");
                    }
                }
                piv = (int)lane32(wr.z, bw);
                int gw = g;
                if constexpr (MULTI) {
                    if (wave == bw) {
                        // the row lane cl just wrote, read by the others of this wave
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                        const uint32_t seq = p.seq_base + (uint32_t)c;
                        const bool have = bk.hi != 0;
                        const bool mine = lane >= s && lane <= WS;  // lane WS: the reciprocal
                        // one store of the row (a lane per entry), one of the record
                        if (have && mine) {
                            uint32_t lo, hi;
                            bits_of(rows[par][lane], lo, hi);
                            u4 v = u4{lo, hi, (uint32_t)lane, 0u};
                            v[3] = seq ^ mix32(v[0], v[1], v[2]);
                            const uint32_t at = nrec + (uint32_t)((par * p.G + g) * (WS + 1) + lane);
                            if (l2) st16<elx::xchg::kXcdStore>(p.xarea, nunit, at, v);
                            else st16(p.uarea, nunit, at, v);
                        }
                        const uint32_t at = (uint32_t)(par * p.G + lane);
                        if (lane == g) {
                            u4 v = u4{bk.lo, bk.hi, (have ? (uint32_t)piv : 0x3FFFFFu) | (xcc << 24), 0u};
                            v[3] = seq ^ mix32(v[0], v[1], v[2]);
                            if (l2) st16<elx::xchg::kXcdStore>(p.xarea, nunit, at, v);
                            else st16(p.uarea, nunit, at, v);
                        }
                        Key rk = Key{0u, 0u};
                        uint32_t rl = 0xFFFFFFFFu, rx = xcc;
                        bool got = lane >= p.G, ok = true;
                        int spins = 0;
                        while (true) {
                            asm volatile("" ::: "memory");  // the load stays in the loop
                            if (!got) {
                                const u4 r = l2 ? ld16<elx::xchg::kXcdLoad>(p.xarea, nunit, at)
                                                : ld16(p.uarea, nunit, at);
                                if (r[3] == (seq ^ mix32(r[0], r[1], r[2]))) {
                                    got = true;
                                    rk = Key{r[1], r[0]};
                                    rl = r[2] & 0xFFFFFFu;
                                    rx = r[2] >> 24;
                                }
                            }
                            if (__all(got ? 1 : 0)) break;
                            if (++spins > SPIN_LIMIT) {
                                ok = false;
                                break;
                            }
                        }
                        const int win = wave_argmax<false>(rk, rl);
                        const Key gk = Key{lane32(rk.hi, win), lane32(rk.lo, win)};
                        const bool same = __all(rx == xcc ? 1 : 0);
                        if (ok && gk.hi != 0) {
                            const uint32_t rat = nrec + (uint32_t)((par * p.G + win) * (WS + 1) + lane);
                            bool in = !mine;
                            T v = T(0);
                            spins = 0;
                            while (true) {
                                asm volatile("" ::: "memory");
                                if (!in) {
                                    const u4 r = l2 ? ld16<elx::xchg::kXcdLoad>(p.xarea, nunit, rat)
                                                    : ld16(p.uarea, nunit, rat);
                                    if (r[2] == (uint32_t)lane && r[3] == (seq ^ mix32(r[0], r[1], r[2]))) {
                                        in = true;
                                        value_of(r, v);
                                    }
                                }
                                if (__all(in ? 1 : 0)) break;
                                if (++spins > SPIN_LIMIT) {
                                    ok = false;
                                    break;
                                }
                            }
                            if (mine) grow[par][lane] = v;
                        }
                        if (lane == 0) {
                            meta[par][0] = (int)lane32(rl, win);
                            meta[par][1] = win;
                            // 0 gave up, 1 no usable pivot, 2 a pivot; + 2 on one XCD
                            meta[par][2] = !ok ? 0 : ((gk.hi == 0 || key_is_zero(gk)) ? 1 : 2) + (same ? 2 : 0);
                        }
                    }
                    __syncthreads();
                    piv = __builtin_amdgcn_readfirstlane(meta[par][0]);
                    gw = __builtin_amdgcn_readfirstlane(meta[par][1]);
                    const int st = __builtin_amdgcn_readfirstlane(meta[par][2]);
                    aborted = st == 0;
                    if (c == 0) l2 = st > 2;
                    live = st == 2 || st == 4;
                } else {
                    __syncthreads();
                    live = bk.hi != 0 && !key_is_zero(bk);
                }
                // no candidate, or an exactly zero pivot: lu::Panel throws
                // SingularMatrixException here (Panel.hpp:52-53), the pivot being the current row
                // and every earlier step applied
                stopped = !live;
                if (live) steps = c + 1;
                if (live && lane == c) dest = piv;
                // the register row (0 or 1) of this lane that won, if any
                if (wave == bw && gw == g && lane == cl) wrow = cq ? 1 : 0;
            }
            const T u0 = us[lane & 15], u1 = us[16 + (lane & 15)], inv = us[WS];
            T l[RPT];
            bool act[RPT];
            static_for<0, RPT>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                int L = lbl[q];
                L = !live ? L : (wrow == q ? c : (L == c ? piv : L));
                lbl[q] = L;
                act[q] = live && L > c;
                l[q] = T(0);
                if (act[q]) {
                    l[q] = a[q][s] * inv;
                    a[q][s] = l[q];
                }
            });
            // the entry broadcasts run with every lane on (a DPP source lane must be active), the
            // FMAs only on the live rows
            static_for<0, NC>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                if (gi + k < ngroups) {
                    constexpr int e0 = (k == 0) ? s + 1 : 0;
                    T ub[8];
                    static_for<e0, 8>([&](auto ec) {
                        constexpr int e = decltype(ec)::value, j = 8 * k + e;
                        ub[e] = row_bcast<j & 15>(j < 16 ? u0 : u1);
                    });
                    static_for<0, RPT>([&](auto qc) {
                        constexpr int q = decltype(qc)::value;
                        if (act[q])
                            static_for<e0, 8>([&](auto ec) {
                                constexpr int e = decltype(ec)::value, j = 8 * k + e;
                                a[q][j] = __builtin_fma(-l[q], ub[e], a[q][j]);
                            });
                    });
                }
            });
        });
        // the finished chunk to the end: after NC rotations every entry is back in its place
        static_for<0, RPT>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            T f[8];
            static_for<0, 8>([&](auto ec) { f[decltype(ec)::value] = a[q][decltype(ec)::value]; });
            static_for<0, WS - 8>([&](auto jc) { a[q][decltype(jc)::value] = a[q][decltype(jc)::value + 8]; });
            static_for<0, 8>([&](auto ec) { a[q][WS - 8 + decltype(ec)::value] = f[decltype(ec)::value]; });
        });
    }

    if (aborted) {
        // a peer never arrived: the block's columns stay as they were
        if (t < 2 * WS) p.spairs[t] = int2{-1, -1};
        if (t < w) p.dests[t] = (int32_t)(p.goff + t);
        if (t == 0) {
            *p.done = 0;
            atomicCAS(p.info, 0, -1);
        }
        return;
    }
    if (g == 0) {
        if (t < w) p.dests[t] = (int32_t)(p.goff + dest);
        if (t == 0) {
            *p.done = steps;
            if (steps < w) atomicCAS(p.info, 0, (int32_t)(p.goff + steps + 1));
        }
    }
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const i64 r = r0 + q * NT;
        if (r >= p.mp) continue;
        const int L = lbl[q], phys = (int)r, o = org[q];
        T* row = p.A + L;
#pragma unroll
        for (int j = 0; j < WS; ++j)
            if (j < w) row[(i64)j * p.lda] = a[q][j];
        if (L < WS) p.spairs[L] = (L != phys) ? int2{L, phys} : int2{-1, -1};
        if (phys < WS) p.spairs[WS + phys] = (L >= WS) ? int2{L, phys} : int2{-1, -1};
        // the panel's list: a position's row is final once its block is done
        const int pos = p.c0 + L;
        if (L < w) {
            p.pairs[pos] = (pos != o) ? int2{pos, o} : int2{-1, -1};
            if (o < p.W) p.pairs[p.W + o] = int2{-1, -1};
        } else if (p.last) {
            if (o < p.W) p.pairs[p.W + o] = int2{pos, o};
        } else {
            p.orig_out[pos] = o;
        }
    }
    // a block shorter than WS rows leaves no stale moves behind
    if (g == 0 && t < WS && t >= p.mp) {
        p.spairs[t] = int2{-1, -1};
        p.spairs[WS + t] = int2{-1, -1};
    }
}

// The block's interchanges in the panel columns left and right of it and, on the right,
// U12 = L11^-1 A12: x_i = fma(-l_ik, x_k, x_i) for k in turn, the panel's own order. A wave
// takes CW columns; lane i < 32 holds row i of the block, the other lanes the rows that the
// block's moves carry out of it. All of a column's sources are loaded before its first store.
// `done` < 32 (an exactly zero pivot) applies the completed steps only.
constexpr int CW = 2;
template <typename T>
__global__ __launch_bounds__(256) void panel_solve_kernel(T* P, i64 lda, i64 mp, int c0, int w, int W,
                                                          const int2* __restrict__ spairs,
                                                          const int32_t* __restrict__ done) {
    const int lane = threadIdx.x & 63;
    const int steps = *done;
    // columns [0, c0) and [c0 + w, W), CW per wave
    const int nl = (c0 + CW - 1) / CW;
    const int u = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
    const bool right = u >= nl;
    const int j0 = right ? c0 + w + (u - nl) * CW : u * CW, jend = right ? W : c0;
    if (j0 >= jend) return;
    int2 mv = spairs[lane];
    if (mv.x < 0 || mv.y < 0 || mv.x >= mp || mv.y >= mp) mv = int2{-1, -1};
    const bool top = lane < 32 && lane < mp;
    const int src = mv.x >= 0 ? mv.y : (top ? lane : -1);
    const int dst = mv.x >= 0 ? mv.x : (top ? lane : -1);
    T* D = P + c0;  // the block's first row, panel column 0
    T x[CW];
#pragma unroll
    for (int q = 0; q < CW; ++q) x[q] = (src >= 0 && j0 + q < jend) ? D[src + (i64)(j0 + q) * lda] : T(0);
    if (right) {
        // row `lane` of L11, strictly below the diagonal
        T l[WS];
#pragma unroll
        for (int k = 0; k < WS; ++k)
            l[k] = (lane < 32 && lane > k && k < steps && lane < mp) ? D[lane + (i64)(c0 + k) * lda] : T(0);
        static_for<0, WS>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            if (k < steps) {
#pragma unroll
                for (int q = 0; q < CW; ++q) {
                    const T xk = bcast_lane(x[q], k);
                    if (lane < 32 && lane > k) x[q] = __builtin_fma(-l[k], xk, x[q]);
                }
            }
        });
    }
#pragma unroll
    for (int q = 0; q < CW; ++q)
        if (dst >= 0 && j0 + q < jend) D[dst + (i64)(j0 + q) * lda] = x[q];
}

// A22 -= L21 U12 inside the panel: rank 32 on the matrix cores (bit for bit the FMA chain over k),
// a 16 x 16 tile of A22 per wave, every operand loaded straight into its lane before the first
// product. One memory latency and 8 products: at these sizes the launch is latency-bound (a row
// per thread with U12 through the scalar cache took 6-13 us, this 4-9).
constexpr int UR = 64, UC = 16;  // rows, columns per workgroup
template <typename T>
__global__ __launch_bounds__(256) void panel_update_kernel(const T* __restrict__ L, const T* __restrict__ U,
                                                           T* __restrict__ C, i64 lda, i64 rows, int cols,
                                                           const int32_t* __restrict__ done) {
    typedef elx::wv::Mfma4<T> MF;
    const int steps = *done;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, kq = lane >> 4;
    const i64 r = (i64)blockIdx.x * UR + wave * 16 + l16;
    const int j0 = (int)blockIdx.y * UC;
    if (steps <= 0) return;
    const bool rin = r < rows, jin = j0 + l16 < cols;
    T l[WS / 4], u[WS / 4];
#pragma unroll
    for (int kk = 0; kk < WS / 4; ++kk) {
        const int k = 4 * kk + kq;
        l[kk] = (rin && k < steps) ? L[r + (i64)k * lda] : T(0);
        u[kk] = (jin && k < steps) ? U[k + (i64)(j0 + l16) * lda] : T(0);
    }
    // D(j, r): lanes run down the columns of A22
    typename MF::acc c;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int j = j0 + MF::row(kq, q);
        c[q] = (rin && j < cols) ? C[r + (i64)j * lda] : T(0);
    }
    if (steps == WS) {
#pragma unroll
        for (int kk = 0; kk < WS / 4; ++kk) c = MF::run(u[kk], -l[kk], c);
    } else {
        // a block that stopped: only its completed steps (a zero operand would meet infinities)
        for (int k = 0; k < steps; ++k) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = j0 + MF::row(kq, q);
                if (rin && j < cols) c[q] = __builtin_fma(-L[r + (i64)k * lda], U[k + (i64)j * lda], c[q]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int j = j0 + MF::row(kq, q);
        if (rin && j < cols) C[r + (i64)j * lda] = c[q];
    }
}

template <typename T>
elx_status_t rpanel(hipStream_t s, i64 mp, i64 W, T* P, i64 lda, int32_t* dests, i64 goff,
                    int2* pairs, int32_t* info) {
    ELX_ARG(W >= 1 && W <= WPANEL && mp >= W && mp <= (i64)RWG * GMAX);
    elx::ProfScope prof_(s, elx::kKPanel, 2.0 * (double)mp * (double)W * sizeof(T));
    // work space: done, spairs, two row-origin arrays
    const size_t ints = (size_t)((mp + 63) / 64 * 64);
    void* ws = nullptr;
    ELX_CHECK(elx::scratch_get(elx::kSlotRPanel, 256 + 2 * WS * sizeof(int2) + 2 * ints * sizeof(int32_t), &ws));
    int32_t* done = static_cast<int32_t*>(ws);
    int2* spairs = reinterpret_cast<int2*>(static_cast<char*>(ws) + 256);
    int32_t* orig[2];
    orig[0] = reinterpret_cast<int32_t*>(spairs + 2 * WS);
    orig[1] = orig[0] + ints;
    elx::RPanelSync* sync = nullptr;
    if (mp > RWG) ELX_CHECK(elx::rpanel_sync_get(sizeof(u4) * 2 * GMAX * (2 + WS), &sync));
    int which = 0;
    for (i64 c0 = 0; c0 < W; c0 += WS) {
        const int w = (int)std::min<i64>(WS, W - c0);
        RArgs<T> a;
        a.mp = mp - c0;
        a.w = w;
        a.A = P + c0 + c0 * lda;
        a.lda = lda;
        a.dests = dests + c0;
        a.goff = goff + c0;
        a.spairs = spairs;
        a.orig_in = c0 ? orig[which ^ 1] : nullptr;
        a.orig_out = orig[which];
        which ^= 1;
        a.c0 = (int)c0;
        a.W = (int)W;
        a.last = (c0 + w == W) ? 1 : 0;
        a.pairs = pairs;
        a.info = info;
        a.done = done;
        a.G = (int)((a.mp + RWG - 1) / RWG);
        if (a.G == 1) {
            a.seq_base = 0;
            a.uarea = a.xarea = nullptr;
            if (a.mp <= 64 * RPT)
                hipLaunchKernelGGL((rpanel_kernel<T, false, 64>), dim3(1), dim3(64), 0, s, a);
            else if (a.mp <= 256 * RPT)
                hipLaunchKernelGGL((rpanel_kernel<T, false, 256>), dim3(1), dim3(256), 0, s, a);
            else
                hipLaunchKernelGGL((rpanel_kernel<T, false, NTMAX>), dim3(1), dim3(NTMAX), 0, s, a);
            ELX_HIP(hipGetLastError());
        } else {
            a.seq_base = (uint32_t)((++sync->epoch) * WS);
            a.uarea = static_cast<u4*>(sync->uarea);
            a.xarea = static_cast<u4*>(sync->xarea);
            // an ordinary launch (a cooperative one costs 11 us before and after it on this
            // stream): at most one workgroup per CU of one XCD waits on others, each gets its
            // CU as soon as earlier work drains, and every wait is bounded
            hipLaunchKernelGGL((rpanel_kernel<T, true, NTMAX>), dim3(8 * (unsigned)a.G), dim3(NTMAX), 0, s, a);
            ELX_HIP(hipGetLastError());
        }
        const int nr = (int)(W - c0 - w);
        const int units = (int)((c0 + CW - 1) / CW) + (nr + CW - 1) / CW;
        if (units > 0) {
            hipLaunchKernelGGL(panel_solve_kernel<T>, dim3((units + 3) / 4), dim3(256), 0, s, P, lda,
                               mp - c0, (int)c0, w, (int)W, spairs, done);
            ELX_HIP(hipGetLastError());
        }
        const i64 rows = mp - c0 - w;
        if (nr > 0 && rows > 0) {
            const T* L = P + (c0 + w) + c0 * lda;
            T* C = P + (c0 + w) + (c0 + w) * lda;
            const T* U = P + c0 + (c0 + w) * lda;
            hipLaunchKernelGGL(panel_update_kernel<T>, dim3((unsigned)((rows + UR - 1) / UR), (nr + UC - 1) / UC),
                               dim3(256), 0, s, L, U, C, lda, rows, nr, done);
            ELX_HIP(hipGetLastError());
        }
    }
    return ELX_SUCCESS;
}

}  // namespace

namespace elx {

// One XCD holds the panel when its CUs carry it at 1024 rows each.
bool rpanel_fits(i64 mp, i64 w) {
    const DeviceInfo& di = device_info();
    return w >= 1 && w <= WPANEL && mp >= w &&
           mp <= (i64)RWG * std::min<i64>(GMAX, std::max(di.num_cus / 8, 1));
}

elx_status_t launch_rpanel(hipStream_t s, i64 mp, i64 w, double* A, i64 lda, int32_t* dests,
                           i64 goff, int2* pairs, int32_t* info) {
    return rpanel<double>(s, mp, w, A, lda, dests, goff, pairs, info);
}
elx_status_t launch_rpanel(hipStream_t s, i64 mp, i64 w, float* A, i64 lda, int32_t* dests,
                           i64 goff, int2* pairs, int32_t* info) {
    return rpanel<float>(s, mp, w, A, lda, dests, goff, pairs, info);
}

}  // namespace elx
