// Triangular solves of any order with a few right-hand sides: the substitution phase of
// lu::SolveAfter and cholesky::SolveAfter (src/lapack_like/factor/LU/SolveAfter.hpp:66-92,
// Cholesky/SolveAfter.hpp:15-43), left side, all orientations.
//
// One persistent launch per 16 right-hand sides (and up to 8 such groups side by side) instead of
// a diagonal solve and a GEMM per 128 rows: at 1 to 16 columns each of those kernels was one
// dependent chain on a mostly idle chip (20-38 us for the diagonal block, 29 us for an update
// whose 128 x 128 tiles held 1 to 16 used columns), 256 pairs of them in an n = 16384 solve.
// Here a workgroup takes one 128-row block after another; a block's rows take the products with
// the earlier blocks' solutions as those are published, then the block's triangle is solved 16
// rows at a time: wave w holds rows 16 w .. 16 w + 15 of all 16 vectors in one MFMA accumulator,
// wave s solves its 16 x 16 triangle, and the waves below it update on the matrix cores. What
// bounds it is that chain per block: 8 dependent 16-row solves, and the hand-off of the block's
// solution through memory, in FP64 (FP32) 19 (12) us with a unit diagonal, 21 (14) without one, 28 (21)
// for 5 to 16 vectors; the matrix is read once, half a tile ahead. FP64, per triangle, the pairs of kernels
// before -> this one: n = 16384 15 -> 2.7 ms with one right-hand side, 8.9 -> 3.6 ms with 16; n = 1024
// 0.52 -> 0.18 ms.
//
// Every entry is updated in the order of the blocked substitution: block by block, one FMA per
// unknown of an earlier block in ascending column order, then the steps of its own block; the
// result is that of trsm_block_kernel and the GEMM kernels bit for bit.
// The hand-off is through uncached memory in tagged 16-byte units (exchange.hpp): a unit holds
// eight bytes of the solution, the launch's epoch and a hash, so a reader needs no flag or store
// completion. The epoch lives in device memory and the last workgroup advances it. The area is one
// per device and each launch waits for the one before it; inside a capture, and where the area
// cannot be had, the caller's blocked sequence runs instead.
// The blocks are dealt out in order by a counter, so a block waits only on blocks that running
// workgroups hold, never on one that has yet to get its place on the chip, whatever else runs
// there. Every wait is bounded all the same (ELX_SOLVE_SPIN_LIMIT polls, 2^20 unless set, some
// seconds): one that runs out turns the solution into NaN and, where the caller has an info word,
// that into -1.
#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <type_traits>

#include "elx_common.hpp"
#include "exchange.hpp"
#include "wave.hpp"

using namespace elx::wv;
using elx::xchg::ld16;
using elx::xchg::mix32;
using elx::xchg::st16;
using elx::xchg::u4;

namespace {

constexpr int BS = 128, SB = 16, NW = BS / SB, CNT = 64 * NW;  // block, sub-block, waves, threads
constexpr int NV = 16;                                         // right-hand sides per group
constexpr int MAX_GROUPS = 8;
constexpr int SPIN_LIMIT = 1 << 20;  // polls of a wait

// Eight bytes of a row of the solution: entries PER*q .. of its 16 vectors.
template <typename T>
struct Unit;
template <>
struct Unit<double> {
    static constexpr int PER = 1;
    __device__ static void pack(const double* v, uint32_t& a, uint32_t& b) {
        const uint64_t x = (uint64_t)__double_as_longlong(v[0]);
        a = (uint32_t)x;
        b = (uint32_t)(x >> 32);
    }
    __device__ static void unpack(uint32_t a, uint32_t b, double* v) {
        v[0] = __longlong_as_double((long long)(((uint64_t)b << 32) | a));
    }
};
template <>
struct Unit<float> {
    static constexpr int PER = 2;
    __device__ static void pack(const float* v, uint32_t& a, uint32_t& b) {
        a = __float_as_uint(v[0]);
        b = __float_as_uint(v[1]);
    }
    __device__ static void unpack(uint32_t a, uint32_t b, float* v) {
        v[0] = __uint_as_float(a);
        v[1] = __uint_as_float(b);
    }
};

template <typename T>
struct ChainArgs {
    i64 n, nrhs;
    const T* A;
    i64 lda;
    T* B;
    i64 ldb;
    int mtrans, back;
    int32_t* info;   // may be null: non-zero stops the solve, a wait that runs out sets -1
    u4* area;        // [groups][nblk][BS * NV / PER] units
    uint32_t* ctrl;  // epoch, workgroups finished, blocks dealt out, waits lost
    int groups;      // of 16 right-hand sides
    int spin_limit;
};

// The exchange loads are plain intrinsics to the compiler: without this a poll loop's load could
// be taken out of the loop.
__device__ __forceinline__ void reread() { asm volatile("" ::: "memory"); }

// NR: vectors per lane in a triangle solve: 4, or 1 where the group has at most 4 vectors.
template <typename T, bool UNIT, int NR>
__global__ __launch_bounds__(CNT) void solve_chain_kernel(ChainArgs<T> p) {
    typedef Mfma4<T> MF;
    constexpr int PER = Unit<T>::PER, UNITS = BS * NV / PER, UPT = UNITS / CNT, RU = NV / PER;
    __shared__ T xs[2][BS * NV];           // an earlier block's solution, [k][v]
    __shared__ T xd[BS][NV + 1];           // this block's
    __shared__ T tiles[NW][SB][SB + 1];
    __shared__ uint32_t s_item;
    if (p.info && *p.info != 0) return;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int l16 = lane & 15, kq = lane >> 4;
    const int nblk = (int)((p.n + BS - 1) / BS);
    const uint32_t epoch = p.ctrl[0] + 1u;  // never the tag of memory that is zero
    const uint32_t count = (uint32_t)nblk * UNITS;
    // Logical forward problem: the backward forms walk both matrices from their ends, over the
    // same 128-row blocks from the top (so the partial block comes first: rows before lo do not
    // exist and are those of the identity).
    const i64 sgn = p.back ? -1 : 1, np = (i64)nblk * BS;
    const i64 lo = p.back ? np - p.n : 0, hi = p.back ? np : p.n;
    const i64 si = sgn * (p.mtrans ? p.lda : 1), sj = sgn * (p.mtrans ? 1 : p.lda), ei = sgn;
    const T* __restrict__ M0 = p.back ? p.A - (np - 1) * (si + sj) : p.A;
    // within an earlier block the products go up the matrix's own columns either way
    const int kfirst = p.back ? BS - 1 - kq : kq;
    const i64 sk = p.back ? -sj : sj;
    // the vector that a lane solves in its register r: the first four in registers 0
    auto vcol = [&](int r) { return kq + 4 * r; };
    bool lost = false;

    const int items = nblk * p.groups;
    for (;;) {
        // the next block, the groups of right-hand sides side by side
        if (t == 0) s_item = atomicAdd(&p.ctrl[2], 1u);
        __syncthreads();
        const int item = __builtin_amdgcn_readfirstlane((int)s_item);
        if (item >= items) break;
        const int b = item / p.groups, group = item - b * p.groups;
        const i64 v0 = (i64)group * NV;
        const int nv = (int)((p.nrhs - v0) < NV ? (p.nrhs - v0) : NV);
        const u4* area = p.area + (size_t)group * count;
        T* X0 = (p.back ? p.B - (np - 1) * ei : p.B) + v0 * p.ldb;
        const i64 i0 = (i64)b * BS, iw = i0 + SB * wave;  // the block's and this wave's first row
        const i64 il = iw + l16;
        const bool rin = il >= lo && il < hi;
        const T* __restrict__ Mr = M0 + (rin ? il : lo) * si;  // this lane's row
        typename MF::acc acc;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const i64 i = iw + MF::row(kq, r);
            acc[r] = (i >= lo && i < hi && l16 < nv) ? X0[i * ei + l16 * p.ldb] : T(0);
        }
        // the block's own triangle: operands left of this wave's sub-block, its rows and diagonal
        T md[NW - 1][4], mrow[SB], dg = T(1);
        auto load_diag = [&]() {
#pragma unroll
            for (int s = 0; s < NW - 1; ++s)
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
                    md[s][kk] = (s < wave && rin && i0 + SB * s + 4 * kk + kq >= lo)
                                    ? Mr[(i0 + SB * s + 4 * kk + kq) * sj]
                                    : T(0);
#pragma unroll
            for (int k = 0; k < SB; ++k)
                mrow[k] = (k < l16 && rin && iw + k >= lo) ? Mr[(iw + k) * sj] : T(0);
            if (!UNIT && rin) dg = Mr[il * sj];
        };

        // products with the earlier blocks, half a tile at a time; the next half, and before the
        // last block the triangle, is loaded while a solution is awaited
        constexpr int H = BS / 8;  // operands per half
        auto load_half = [&](int kb, int h, T(&m)[H]) {
#pragma unroll
            for (int kk = 0; kk < H; ++kk) {
                const int k = h * (BS / 2) + 4 * kk;
                const bool in = rin && (kb > 0 || !p.back || kfirst - k >= lo);
                m[kk] = in ? Mr[((i64)kb * BS + kfirst) * sj + k * sk] : T(0);
            }
        };
        auto multiply = [&](int kb, int h, const T(&m)[H]) {
            const T* x = xs[kb & 1] + h * (BS / 2) * NV + kq * NV + l16;
#pragma unroll
            for (int kk = 0; kk < H; ++kk) acc = MF::run(m[kk], -x[4 * kk * NV], acc);
        };
        // a unit's place in LDS: rows in the order of the products
        auto slot = [&](int q) { return (p.back ? BS - 1 - q / RU : q / RU) * NV + (q % RU) * PER; };
        auto await = [&](int kb) {
            T* x = xs[kb & 1];
            const uint32_t at = (uint32_t)kb * UNITS;
            int spins = 0;
            // one lane per wave watches the block's last unit, then every thread reads its own
            if (lane == 0 && !lost) {
                while (ld16(area, count, at + UNITS - 1)[2] != epoch && spins < p.spin_limit) {
                    ++spins;
                    reread();
                }
            }
            bool got[UPT];
#pragma unroll
            for (int u = 0; u < UPT; ++u) got[u] = false;
            spins = 0;
            while (true) {
                reread();
                u4 r[UPT];
#pragma unroll
                for (int u = 0; u < UPT; ++u) r[u] = ld16(area, count, at + t + CNT * u);
                bool all = true;
#pragma unroll
                for (int u = 0; u < UPT; ++u) {
                    const uint32_t id = at + t + CNT * u;
                    if (!got[u] && r[u][2] == epoch && r[u][3] == mix32(r[u][0], r[u][1] ^ id, epoch)) {
                        got[u] = true;
                        Unit<T>::unpack(r[u][0], r[u][1], x + slot(t + CNT * u));
                    }
                    all = all && got[u];
                }
                if (__all(all ? 1 : 0)) break;
                if (lost || ++spins > p.spin_limit) {
                    lost = true;
#pragma unroll
                    for (int u = 0; u < UPT; ++u)
                        if (!got[u])
                            for (int e = 0; e < PER; ++e) x[slot(t + CNT * u) + e] = T(__builtin_nan(""));
                    break;
                }
            }
            __syncthreads();
        };
        T ma[H] = {}, mb[H];
        if (b > 0) load_half(0, 0, ma);
        for (int kb = 0; kb + 1 < b; ++kb) {
            await(kb);
            load_half(kb, 1, mb);
            multiply(kb, 0, ma);
            load_half(kb + 1, 0, ma);
            multiply(kb, 1, mb);
        }
        load_diag();
        if (b > 0) {
            await(b - 1);
            load_half(b - 1, 1, mb);
            multiply(b - 1, 0, ma);
            multiply(b - 1, 1, mb);
        }

        // the block's triangle, 16 rows at a time: wave s updates with the sub-blocks above it as
        // they are solved (one barrier each), solves its own and publishes it while the waves
        // below go on
        const T dr = UNIT ? T(1) : T(1) / dg;
        const int nsub = (int)((hi - i0 < BS ? hi - i0 : BS) + SB - 1) / SB;
        static_for<0, NW - 1>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            if (s < wave && s < nsub) {
                __syncthreads();
#pragma unroll
                for (int kk = 0; kk < 4; ++kk) acc = MF::run(md[s][kk], -xd[SB * s + 4 * kk + kq][l16], acc);
            }
        });
        if (wave < nsub) {
            // S(v, i): lane l16 holds entry i, register r vector vcol(r)
            T(*tile)[SB + 1] = tiles[wave];
            T x[NR];
#pragma unroll
            for (int r = 0; r < 4; ++r) tile[MF::row(kq, r)][l16] = acc[r];
            wave_lds_sync();
            // every lane divides its entry at each step; the step's own is lane k's, whose entry is
            // final but for that division
            auto solve = [&](auto divide) {
#pragma unroll
                for (int r = 0; r < NR; ++r) x[r] = tile[l16][vcol(r)];
                static_for<0, SB>([&](auto kc) {
                    constexpr int k = decltype(kc)::value;
                    T xk[NR];
#pragma unroll
                    for (int r = 0; r < NR; ++r) xk[r] = row_bcast<k>(divide(x[r]));
                    if (l16 > k) {
#pragma unroll
                        for (int r = 0; r < NR; ++r) x[r] = __builtin_fma(-mrow[k], xk[r], x[r]);
                    }
                });
            };
            if constexpr (UNIT) {
                solve([](T v) { return v; });
            } else {
                solve([&](T v) { return quot(v, dg, dr); });
                bool ok = divisor_ok(dg);
#pragma unroll
                for (int r = 0; r < NR; ++r) ok = ok && dividend_ok(x[r]);
                if (__all(ok ? 1 : 0)) {
#pragma unroll
                    for (int r = 0; r < NR; ++r) x[r] = quot(x[r], dg, dr);
                } else {
                    solve([&](T v) { return v / dg; });
#pragma unroll
                    for (int r = 0; r < NR; ++r) x[r] = x[r] / dg;
                }
            }
#pragma unroll
            for (int r = 0; r < NR; ++r) xd[SB * wave + l16][vcol(r)] = x[r];
            if (NR < 4) {
#pragma unroll
                for (int r = NR; r < 4; ++r) xd[SB * wave + l16][vcol(r)] = T(0);
            }
        }
        for (int s = wave; s < nsub; ++s) {
            __syncthreads();
            if (s == wave && b + 1 < nblk) {
#pragma unroll
                for (int u = 0; u < SB * RU / 64; ++u) {
                    const int q = lane + 64 * u, row = SB * wave + q / RU;
                    const uint32_t id = (uint32_t)b * UNITS + SB * wave * RU + q;
                    T v[PER];
#pragma unroll
                    for (int e = 0; e < PER; ++e) v[e] = xd[row][(q % RU) * PER + e];
                    uint32_t lo32, hi32;
                    Unit<T>::pack(v, lo32, hi32);
                    st16(area, count, id, u4{lo32, hi32, epoch, mix32(lo32, hi32 ^ id, epoch)});
                }
            }
        }
        // the solution in place of the right-hand sides
        for (int idx = t; idx < BS * NV; idx += CNT) {
            const int i = idx & (BS - 1), v = idx >> 7;
            if (i0 + i >= lo && i0 + i < hi && v < nv) X0[(i0 + i) * ei + v * p.ldb] = xd[i][v];
        }
        if (item == items - 1) break;  // the launch ends with this block: it does not ask for another
        __syncthreads();
    }
    // the last workgroup to finish opens the next launch's epoch and its count of blocks, and reports a
    // lost wait (not before: a workgroup that starts late still has to find the info word as it was)
    if (lost && lane == 0) {
        atomicOr(&p.ctrl[3], 1u);
        __threadfence();
    }
    __syncthreads();
    if (t == 0 && atomicAdd(&p.ctrl[1], 1u) == gridDim.x - 1) {
        if (atomicExch(&p.ctrl[3], 0u) != 0u && p.info) *p.info = -1;
        p.ctrl[1] = 0u;
        p.ctrl[2] = 0u;
        p.ctrl[0] = epoch;
    }
}

template <typename T>
elx_status_t chain_impl(hipStream_t s, int uplo, int orient, int diag, i64 n, i64 nrhs, const T* A, i64 lda,
                        T* B, i64 ldb, int32_t* info, bool* taken) {
    const elx::DeviceInfo& di = elx::device_info();
    const i64 nblk = (n + BS - 1) / BS;
    const size_t units = (size_t)nblk * (BS * NV / Unit<T>::PER);
    const i64 most = std::min<i64>(MAX_GROUPS, (nrhs + NV - 1) / NV);
    ELX_ARG(units < ((size_t)1 << 27));
    *taken = false;
    // Inside a capture the caller's blocked sequence runs: a replay on one stream could meet a solve
    // on another, or a forked branch of its own graph, in the one hand-off area. A status that
    // cannot be had (another stream's capture forbids the call) counts as a capture.
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    const hipError_t se = hipStreamIsCapturing(s, &st);
    if (se != hipSuccess) (void)hipGetLastError();
    if (se != hipSuccess || st != hipStreamCaptureStatusNone) return ELX_SUCCESS;
    elx::ChainSync* sync = nullptr;
    ELX_CHECK(elx::chain_sync_get(&sync));
    std::lock_guard<std::mutex> lk(sync->mu);
    if (!elx::chain_area(*sync, units * sizeof(u4) * (size_t)most, s)) return ELX_SUCCESS;
    ELX_HIP(hipStreamWaitEvent(s, sync->last, 0));
    elx::ProfScope prof_(s, elx::kKTrsm, (double)n * (double)n * (double)nrhs);
    ChainArgs<T> a;
    a.n = n;
    a.A = A;
    a.lda = lda;
    a.ldb = ldb;
    a.mtrans = orient != elx::kNormal ? 1 : 0;
    a.back = ((uplo == elx::kLower) != (a.mtrans != 0)) ? 0 : 1;
    a.info = info;
    const char* limit = std::getenv("ELX_SOLVE_SPIN_LIMIT");
    a.spin_limit = limit ? std::min(std::max(std::atoi(limit), 0), 1 << 30) : SPIN_LIMIT;
    a.area = static_cast<u4*>(sync->area);
    a.ctrl = static_cast<uint32_t*>(sync->ctrl);
    for (i64 v = 0; v < nrhs; v += NV * MAX_GROUPS) {
        a.nrhs = std::min<i64>(nrhs - v, NV * MAX_GROUPS);
        a.B = B + v * ldb;
        const i64 groups = (a.nrhs + NV - 1) / NV;
        const dim3 grid((unsigned)std::min<i64>(nblk * groups, di.num_cus));
        a.groups = (int)groups;
        auto go = [&](auto ut, auto rt) {
            constexpr bool U = decltype(ut)::value;
            constexpr int R = decltype(rt)::value;
            hipLaunchKernelGGL((solve_chain_kernel<T, U, R>), grid, dim3(CNT), 0, s, a);
        };
        const std::integral_constant<int, 1> one;
        const std::integral_constant<int, 4> four;
        const std::true_type yes;
        const std::false_type no;
        if (a.nrhs <= 4) diag == elx::kUnit ? go(yes, one) : go(no, one);
        else diag == elx::kUnit ? go(yes, four) : go(no, four);
        ELX_HIP(hipGetLastError());
    }
    ELX_HIP(hipEventRecord(sync->last, s));
    *taken = true;
    return ELX_SUCCESS;
}

}  // namespace

namespace elx {

elx_status_t launch_solve_chain(hipStream_t s, int uplo, int orient, int diag, i64 n, i64 nrhs,
                                const double* A, i64 lda, double* B, i64 ldb, int32_t* info,
                                bool* taken) {
    return chain_impl<double>(s, uplo, orient, diag, n, nrhs, A, lda, B, ldb, info, taken);
}
elx_status_t launch_solve_chain(hipStream_t s, int uplo, int orient, int diag, i64 n, i64 nrhs,
                                const float* A, i64 lda, float* B, i64 ldb, int32_t* info,
                                bool* taken) {
    return chain_impl<float>(s, uplo, orient, diag, n, nrhs, A, lda, B, ldb, info, taken);
}

}  // namespace elx
