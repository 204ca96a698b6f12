// Triangular solves with an order <= 128 triangle and any number of vectors.
#include <algorithm>
#include <type_traits>

#include "elx_common.hpp"
#include "wave.hpp"

using namespace elx::wv;

namespace {

// ---------------------------------------------------------------------------------------
// Triangular solves M x = b for many independent vectors with an order <= 128 triangle.
// Left side: the vectors are columns of B and M = op(A). Right side (X op(A) = B): the
// vectors are rows of B and M = op(A)^T. Every entry is updated as the reference BLAS dtrsm
// does: in forward and column-oriented backward substitution x_i -= M(i,j) x_j for j in turn,
// one FMA each; division by the diagonal on the left side, multiplication by its reciprocal on
// the right side.
//
// A wave solves 16 vectors in registers, with the backward forms run as forward ones on
// reversed indices. The order is cut into 16-entry blocks: the block's 16 x 16 triangle is
// solved with an entry per lane (x_k reaches the other 15 lanes of a vector by a DPP
// broadcast), x goes through the wave's own LDS tile into operand layout, and the later blocks
// are updated on the matrix cores, whose products are the same FMA chains in the same order,
// so the results are the scalar code's bit for bit. No workgroup barrier; the triangle is read
// straight from the caches in operand layout. Divisions are quotients by the reciprocal where the
// operands allow it (wave.hpp), else the block is solved again with plain ones. What bounds it: per
// wave 8 dependent block solves of 16 steps and 28 tile products, and the fetch of their straight-line
// code: FP64 17-27 us (right side) and 11-24 us (left) from 64 to 16384 vectors, 9 us for one (left,
// non-unit), one wave per SIMD; with 16 lanes per vector, all 128 steps dependent and 132 KB of LDS
// per 16 vectors, it took 52 us per 4096 vectors (240 us at 16256) and 20 us for one.
//
// maxbits (may be null): the largest |entry| written is folded into *maxbits (the bits of a
// non-negative float, atomic max), for the exponent of a low-precision product that follows.
// ---------------------------------------------------------------------------------------
constexpr int TBLK = 16, TNB = 8;  // entries per block, blocks
// FULL: order 128, no bounds on the order (the loads are then unconditional and go out together).
// NR: vectors per lane, 4, or (left side) 1 where there are at most 4 vectors in all: the steps' code,
// which a few waves fetch as they go through it once, is a quarter as long (FP64, left, non-unit, one
// vector, launch included: order 128 25.4 -> 18.9 us, order 64 20.3 -> 17.5).
template <typename T, bool RIGHT, bool UNIT, bool FULL, int NR>
__global__ __launch_bounds__(256) void trsm_block_kernel(int m, i64 nvec, const T* __restrict__ A,
                                                         i64 lda, T* B, i64 ldb, int mtrans, int back,
                                                         const int32_t* __restrict__ stop,
                                                         unsigned* maxbits) {
    typedef Mfma4<T> MF;
    __shared__ T tiles[4][TBLK][TBLK + 1];
    if (stop && *stop != 0) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l16 = lane & 15, kq = lane >> 4;
    const i64 v0 = ((i64)blockIdx.x * 4 + wave) * TBLK;
    if (v0 >= nvec) return;
    T(*tile)[TBLK + 1] = tiles[wave];
    // strides of M's logical rows and columns, and of an entry and a vector of B; the backward
    // forms walk both from their ends
    const i64 sgn = back ? -1 : 1;
    const i64 si = sgn * (mtrans ? lda : 1), sj = sgn * (mtrans ? 1 : lda);
    const i64 ei = sgn * (RIGHT ? ldb : 1), ev = RIGHT ? 1 : ldb;
    const T* __restrict__ M0 = back ? A - (i64)(m - 1) * (si + sj) : A;
    T* X0 = back ? B - (i64)(m - 1) * ei : B;
    const T* __restrict__ Ml = M0 + l16 * si;            // row l16 of M
    const T* __restrict__ Mk = Ml + kq * sj;             // and column kq: operand layout
    const bool vin = v0 + l16 < nvec;
    // the vectors: LEFT D(v, i), its row MF::row(kq, r) vector kq + 4 r; RIGHT D(i, v), so that lanes
    // run along the contiguous index
    typename MF::acc acc[TNB];
#pragma unroll
    for (int b = 0; b < TNB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = TBLK * b + (RIGHT ? MF::row(kq, r) : l16);
            const i64 v = v0 + (RIGHT ? l16 : kq + 4 * r);
            acc[b][r] = (r < NR && (FULL || i < m) && (RIGHT ? vin : v < nvec)) ? X0[i * ei + v * ev] : T(0);
        }
    if (NR < 4) {  // the rows of the tile that no vector takes
#pragma unroll
        for (int r = NR; r < 4; ++r) tile[MF::row(kq, r)][l16] = T(0);
    }
    float mx = 0.0f;
    // a block's triangle (row l16), diagonal and the operands M(i, k) of the later blocks, loaded
    // one block ahead
    T mrow[2][TBLK], dgv[2], mop[2][TNB][4];
    auto load = [&](auto bc) {
        constexpr int b = decltype(bc)::value, p = b & 1;
        const int ii = TBLK * b + l16;
#pragma unroll
        for (int k = 0; k < TBLK; ++k)
            mrow[p][k] = (FULL || ii < m) && (FULL || k < l16) ? Ml[TBLK * b * si + (TBLK * b + k) * sj] : T(0);
        dgv[p] = (!UNIT && (FULL || ii < m)) ? Ml[TBLK * b * si + ii * sj] : T(1);
        static_for<b + 1, TNB>([&](auto nc) {
            constexpr int nb = decltype(nc)::value;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
                mop[p][nb][kk] = (FULL || TBLK * nb + l16 < m)
                                     ? Mk[TBLK * nb * si + (TBLK * b + 4 * kk) * sj]
                                     : T(0);
        });
    };
    load(std::integral_constant<int, 0>{});
    static_for<0, TNB>([&](auto bc) {
        constexpr int b = decltype(bc)::value, p = b & 1;
        if (FULL || TBLK * b < m) {
            if constexpr (b + 1 < TNB) load(std::integral_constant<int, b + 1>{});
            const T dg = dgv[p], dr = UNIT ? T(1) : T(1) / dg;
            // S(v, i): lane l16 holds entry i, register r the vector of the tile's row MF::row(kq, r)
            T x[NR];
            if (RIGHT) {
#pragma unroll
                for (int r = 0; r < 4; ++r) tile[MF::row(kq, r)][l16] = acc[b][r];
                wave_lds_sync();
#pragma unroll
                for (int r = 0; r < NR; ++r) x[r] = tile[l16][MF::row(kq, r)];
                wave_lds_sync();
            } else {
#pragma unroll
                for (int r = 0; r < NR; ++r) x[r] = acc[b][r];
            }
            // a lane's entry is final (but for its own diagonal) once the earlier ones are applied;
            // every lane scales its entry at each step, and the step's own is lane k's
            auto substitute = [&](auto scale) {
                static_for<0, TBLK>([&](auto kc) {
                    constexpr int k = decltype(kc)::value;
                    T xk[NR];
#pragma unroll
                    for (int r = 0; r < NR; ++r) xk[r] = row_bcast<k>(scale(x[r]));
                    if (l16 > k) {
#pragma unroll
                        for (int r = 0; r < NR; ++r) x[r] = __builtin_fma(-mrow[p][k], xk[r], x[r]);
                    }
                });
            };
            if constexpr (UNIT) {
                substitute([](T v) { return v; });
            } else if constexpr (RIGHT) {
                substitute([&](T v) { return v * dr; });
#pragma unroll
                for (int r = 0; r < NR; ++r) x[r] = x[r] * dr;
            } else {
                substitute([&](T v) { return quot(v, dg, dr); });
                bool ok = divisor_ok(dg);
#pragma unroll
                for (int r = 0; r < NR; ++r) ok = ok && dividend_ok(x[r]);
                if (__all(ok ? 1 : 0)) {
#pragma unroll
                    for (int r = 0; r < NR; ++r) x[r] = quot(x[r], dg, dr);
                } else {
#pragma unroll
                    for (int r = 0; r < NR; ++r) x[r] = acc[b][r];
                    substitute([&](T v) { return v / dg; });
#pragma unroll
                    for (int r = 0; r < NR; ++r) x[r] = x[r] / dg;
                }
            }
            if (maxbits) {
#pragma unroll
                for (int r = 0; r < NR; ++r) mx = fmaxf(mx, (float)fabs(x[r]));
            }
            // into operand layout: X(v = l16, k = kq + 4 kk)
            T xop[4];
#pragma unroll
            for (int r = 0; r < NR; ++r) tile[MF::row(kq, r)][l16] = x[r];
            wave_lds_sync();
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) xop[kk] = tile[l16][kq + 4 * kk];
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = TBLK * b + (RIGHT ? kq + 4 * r : l16);
                const i64 v = v0 + (RIGHT ? l16 : kq + 4 * r);
                if ((FULL || i < m) && (RIGHT ? vin : v < nvec)) {
                    if constexpr (RIGHT) X0[i * ei + v * ev] = xop[r];
                    else if (r < NR) X0[i * ei + v * ev] = x[r < NR ? r : 0];
                }
            }
            // b_i -= m_ik x_k as fma(m_ik, -x_k, b_i): the same number
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) xop[kk] = -xop[kk];
            static_for<b + 1, TNB>([&](auto nc) {
                constexpr int nb = decltype(nc)::value;
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
                    acc[nb] = RIGHT ? MF::run(mop[p][nb][kk], xop[kk], acc[nb])
                                    : MF::run(xop[kk], mop[p][nb][kk], acc[nb]);
            });
        }
    });
    if (maxbits) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
        if (lane == 0) atomicMax(maxbits, __float_as_uint(mx));
    }
}

// The transposed backward forms as the reference BLAS computes them: each x_i a dot product in
// ascending k from its nearest entry on, which is one dependent chain per vector, m (m - 1) / 2 FMAs
// and m quotients. Four waves bring the triangle (packed by its rows) and the vectors to LDS, then
// one wave solves, a vector per lane: 16 rows at a time, their solutions and those of the next 16
// in registers, the operands read ahead of the chain. Columns past the order are zero and so are their
// unknowns: such terms leave a sum as it is. Left, unit, 64 vectors: order 64 47 us (FP64) and 56
// (FP32), order 128 124 and 156 us; with each row fetched through the scalar cache as its step began
// 84, 88, 222 and 233, and with 16 lanes per vector 69, 120, 210 and 410.
// Only a direct Trsm of order <= 128 asks for this order; the solves of larger systems and of
// factored ones run their diagonal blocks through trsm_block_kernel.
constexpr int DNT = 64, DB = 16;  // vectors per workgroup, rows per block
template <typename T>
__global__ __launch_bounds__(256) void trsm_dot_kernel(int m, i64 nvec, const T* __restrict__ A, i64 lda,
                                                       T* B, i64 ldb, int right, int unit,
                                                       const int32_t* __restrict__ stop) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int nb = (m + DB - 1) / DB, mp = nb * DB;
    T* xs = reinterpret_cast<T*>(smem_raw);  // xs[i * DNT + v], mp rows
    T* tri = xs + mp * DNT;                  // M(i, k) = A(k, i), k >= i, at row(i)[k]
    auto row = [&](int i) { return tri + (i * mp - i * (i - 1) / 2 - i); };
    T* inv = tri + mp * (mp + 1) / 2;        // 1 / M(i, i)
    if (stop && *stop != 0) return;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const i64 v0 = (i64)blockIdx.x * DNT;
    const int nv = (int)((nvec - v0) < DNT ? (nvec - v0) : DNT);
#pragma unroll 4
    for (int i = wave; i < m; i += 4)
        for (int k = i + lane; k < mp; k += 64) row(i)[k] = k < m ? A[k + i * lda] : T(0);
    if (!unit && t < m) inv[t] = T(1) / A[t + t * lda];
    // a vector per lane (right) or down the columns (left): coalesced either way
#pragma unroll 4
    for (int idx = t; idx < mp * DNT; idx += 256) {
        const int i = right ? idx / DNT : idx % mp, v = right ? idx % DNT : idx / mp;
        xs[i * DNT + v] = (v < nv && i < m) ? (right ? B[v0 + v + (i64)i * ldb] : B[i + (v0 + v) * ldb]) : T(0);
    }
    __syncthreads();
    if (wave == 0) {
        T xi[DB], xn[DB];               // this block's solutions and the next one's
        T ri[DB], rn[DB], bi, dr;       // a row's entries beside them, its right-hand side and inverse diagonal
        T xb[2][DB], rb[2][DB];         // blocks further on
        auto row_ahead = [&](int i, bool more) __attribute__((always_inline)) {
            const T* r = row(i);
            const int k0 = i / DB * DB;
            bi = xs[i * DNT + t];
            if (!unit) dr = inv[i];
#pragma unroll
            for (int u = 0; u < DB; ++u) ri[u] = r[k0 + u];  // those left of the diagonal are not used
            if (more) {
#pragma unroll
                for (int u = 0; u < DB; ++u) rn[u] = r[k0 + DB + u];
            }
        };
        row_ahead(m - 1, false);
        for (int ib = nb - 1; ib >= 0; --ib) {
            const bool more = ib + 1 < nb;
            static_for<0, DB>([&](auto rc) __attribute__((always_inline)) {
                constexpr int r = DB - 1 - decltype(rc)::value;
                const int i = ib * DB + r;
                if (i >= m) {
                    xi[r] = T(0);
                    return;
                }
                const T* rp = row(i);
                auto fetch = [&](int kb, T(&x)[DB], T(&w)[DB]) __attribute__((always_inline)) {
#pragma unroll
                    for (int u = 0; u < DB; ++u) {
                        x[u] = xs[(kb * DB + u) * DNT + t];
                        w[u] = rp[kb * DB + u];
                    }
                };
                T acc = bi;
                const T d = ri[r], di = dr;
                if (ib + 2 < nb) fetch(ib + 2, xb[0], rb[0]);
#pragma unroll
                for (int u = r + 1; u < DB; ++u) acc = __builtin_fma(-ri[u], xi[u], acc);
                if (more) {
#pragma unroll
                    for (int u = 0; u < DB; ++u) acc = __builtin_fma(-rn[u], xn[u], acc);
                }
                if (i > 0) row_ahead(i - 1, r > 0 ? more : true);
                for (int kb = ib + 2; kb < nb; kb += 2) {
                    if (kb + 1 < nb) fetch(kb + 1, xb[1], rb[1]);
#pragma unroll
                    for (int u = 0; u < DB; ++u) acc = __builtin_fma(-rb[0][u], xb[0][u], acc);
                    if (kb + 1 >= nb) break;
                    if (kb + 2 < nb) fetch(kb + 2, xb[0], rb[0]);
#pragma unroll
                    for (int u = 0; u < DB; ++u) acc = __builtin_fma(-rb[1][u], xb[1][u], acc);
                }
                if (!unit) {
                    if (right) acc = acc * di;
                    else if (__all(divisor_ok(d) && dividend_ok(acc) ? 1 : 0)) acc = quot(acc, d, di);
                    else acc = acc / d;
                }
                xi[r] = acc;
                xs[i * DNT + t] = acc;
            });
#pragma unroll
            for (int u = 0; u < DB; ++u) xn[u] = xi[u];
        }
    }
    __syncthreads();
    for (int idx = t; idx < m * DNT; idx += 256) {
        const int i = right ? idx / DNT : idx % m, v = right ? idx % DNT : idx / m;
        if (v < nv) {
            if (right) B[v0 + v + (i64)i * ldb] = xs[i * DNT + v];
            else B[i + (v0 + v) * ldb] = xs[i * DNT + v];
        }
    }
}

}  // namespace

namespace elx {

// dot_order: the transposed backward forms in the reference BLAS's order (see trsm_dot_kernel).
template <typename T>
static elx_status_t trsm_small_impl(hipStream_t s, int side, int uplo, int orient, int diag,
                                    i64 m, i64 n, const T* A, i64 lda, T* B, i64 ldb,
                                    const int32_t* stop, bool dot_order, unsigned* maxbits = nullptr) {
    if (m <= 0 || n <= 0) return ELX_SUCCESS;
    const bool right = (side == kRight);
    const i64 order = right ? n : m;
    const i64 nvec = right ? m : n;
    ELX_ARG(order <= 128);
    const bool trans = (orient != kNormal);
    const bool lower = (uplo == kLower);
    // Left: M = op(A). Right: M = op(A)^T.
    const bool mtrans = right ? !trans : trans;
    const bool lower_eff = lower != mtrans;
    const int unit = diag == kUnit ? 1 : 0, mt = mtrans ? 1 : 0;
    ProfScope prof_(s, kKTrsm, (double)order * (double)order * (double)nvec);
    if (!lower_eff && mtrans && dot_order) {
        auto bytes = [](size_t m) {
            m = (m + DB - 1) / DB * DB;
            return sizeof(T) * (m * DNT + m * (m + 1) / 2 + m);
        };
        if (bytes((size_t)order) > (64 << 10)) {  // 133 KB at order 128 in FP64
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&trsm_dot_kernel<T>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes(128));
            (void)hipGetLastError();
        }
        hipLaunchKernelGGL(trsm_dot_kernel<T>, dim3(cdiv(nvec, DNT)), dim3(256), bytes((size_t)order), s,
                           (int)order, nvec, A, lda, B, ldb, right ? 1 : 0, unit, stop);
        ELX_HIP(hipGetLastError());
        return ELX_SUCCESS;
    }
    const dim3 grid(cdiv(nvec, 4 * TBLK));
    const int back = lower_eff ? 0 : 1;
    auto go_n = [&](auto rt, auto ut, auto nt) {
        constexpr bool R = decltype(rt)::value, U = decltype(ut)::value;
        constexpr int N = decltype(nt)::value;
        if (order == TBLK * TNB)
            hipLaunchKernelGGL((trsm_block_kernel<T, R, U, true, N>), grid, dim3(256), 0, s, (int)order,
                               nvec, A, lda, B, ldb, mt, back, stop, maxbits);
        else
            hipLaunchKernelGGL((trsm_block_kernel<T, R, U, false, N>), grid, dim3(256), 0, s, (int)order,
                               nvec, A, lda, B, ldb, mt, back, stop, maxbits);
    };
    auto go = [&](auto rt, auto ut) {
        if constexpr (!decltype(rt)::value) {
            if (nvec <= 4) return go_n(rt, ut, std::integral_constant<int, 1>{});
        }
        go_n(rt, ut, std::integral_constant<int, 4>{});
    };
    const std::true_type yes;
    const std::false_type no;
    if (right) unit ? go(yes, yes) : go(yes, no);
    else unit ? go(no, yes) : go(no, no);
    ELX_HIP(hipGetLastError());
    return ELX_SUCCESS;
}

elx_status_t launch_trsm_small(hipStream_t s, int side, int uplo, int orient, int diag, i64 m,
                               i64 n, const double* A, i64 lda, double* B, i64 ldb,
                               const int32_t* stop, bool dot_order) {
    return trsm_small_impl<double>(s, side, uplo, orient, diag, m, n, A, lda, B, ldb, stop, dot_order);
}

elx_status_t launch_trsm_small(hipStream_t s, int side, int uplo, int orient, int diag, i64 m,
                               i64 n, const float* A, i64 lda, float* B, i64 ldb,
                               const int32_t* stop, bool dot_order) {
    return trsm_small_impl<float>(s, side, uplo, orient, diag, m, n, A, lda, B, ldb, stop, dot_order);
}

elx_status_t launch_trsm_small_f32(hipStream_t s, int side, int uplo, int orient, int diag,
                                   i64 m, i64 n, const float* A, i64 lda, float* B, i64 ldb,
                                   unsigned* maxbits) {
    return trsm_small_impl<float>(s, side, uplo, orient, diag, m, n, A, lda, B, ldb, nullptr, false,
                                  maxbits);
}

}  // namespace elx
