// Row permutation, small triangular solve and unblocked Cholesky kernels.
#include <algorithm>
#include <type_traits>

#include "elx_common.hpp"
#include "wave.hpp"

using namespace elx::wv;

namespace {

// ---------------------------------------------------------------------------------------
// Row moves: the net effect of one panel's swap sequence on the columns outside the panel
// (PB.PermuteRows(AB0) / PB.PermuteRows(AB2), src/lapack_like/factor/LU.cpp:136-137).
// One wave per column. All sources of a column are read (and staged in LDS) before any
// destination is written, so overlapping source/destination rows are safe. A move whose
// source or destination lies outside the `rows` rows below r0 is skipped, so a list that a
// panel left unwritten can never reach past the column.
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ int2 move_in_range(int2 p, i64 rows) {
    return (p.x >= 0 && p.y >= 0 && p.x < rows && p.y < rows) ? p : int2{-1, -1};
}

template <typename T>
__global__ __launch_bounds__(256) void row_moves_kernel(const int2* __restrict__ pairs,
                                                        int npairs, T* A, i64 lda, i64 r0,
                                                        i64 rows, i64 c0, i64 c1, i64 c2,
                                                        i64 c3, const int32_t* __restrict__ stop) {
    __shared__ T stage[4][256];
    __shared__ int2 pr[256];
    if (stop && *stop != 0) return;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    for (int i = t; i < 256; i += 256)
        pr[i] = (i < npairs) ? move_in_range(pairs[i], rows) : int2{-1, -1};
    __syncthreads();
    const i64 n1 = c1 - c0, total = n1 + (c3 - c2);
    const i64 cidx = (i64)blockIdx.x * 4 + wave;
    const bool active = cidx < total;
    T* col = nullptr;
    if (active) {
        const i64 j = (cidx < n1) ? (c0 + cidx) : (c2 + (cidx - n1));
        col = A + r0 + j * lda;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = lane + 64 * q;
            if (pr[i].x >= 0) stage[wave][i] = col[pr[i].y];
        }
    }
    __syncthreads();
    if (active) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = lane + 64 * q;
            if (pr[i].x >= 0) col[pr[i].x] = stage[wave][i];
        }
    }
}

// The same moves for an fp32 matrix stored row by row (row i contiguous at A + i*lda), as the
// mixed-precision factorization keeps its working copy: each move is a contiguous segment
// copy. A workgroup owns a 64-column slice of every moved row; wave w reads the slice of moves
// 32w .. 32w+31 (a float per lane, 256 contiguous bytes per move), and all writes follow one
// barrier, so overlapping sources and destinations are safe. Moves outside the `rows` rows
// below r0 are skipped.
__global__ __launch_bounds__(512) void row_moves_rowmajor_kernel(const int2* __restrict__ pairs,
                                                                 int npairs, float* A, i64 lda,
                                                                 i64 r0, i64 rows, i64 c0, i64 c1,
                                                                 i64 c2, i64 c3) {
    __shared__ int2 pr[256];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (t < 256) pr[t] = (t < npairs) ? move_in_range(pairs[t], rows) : int2{-1, -1};
    __syncthreads();
    const i64 s1 = (c1 - c0 + 63) / 64;  // slices of the first range
    const i64 sl = blockIdx.x;
    const i64 col = (sl < s1) ? (c0 + sl * 64 + lane) : (c2 + (sl - s1) * 64 + lane);
    const bool in = (sl < s1) ? (col < c1) : (col < c3);
    float v[32];
#pragma unroll
    for (int q = 0; q < 32; ++q) {
        const int2 p = pr[wave * 32 + q];
        v[q] = (in && p.x >= 0) ? A[(r0 + p.y) * lda + col] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 32; ++q) {
        const int2 p = pr[wave * 32 + q];
        if (in && p.x >= 0) A[(r0 + p.x) * lda + col] = v[q];
    }
}

// ---------------------------------------------------------------------------------------
// Explicit permutation of a swap sequence (Permutation::ExplicitVector,
// src/lapack_like/perm/Permutation.cpp:731-745). The swaps are sequential by nature; one
// thread replays them on an LDS copy of the index vector when it fits, else in global
// memory.
// ---------------------------------------------------------------------------------------
constexpr int kSwapChunk = 1024;  // swap destinations staged in LDS per round
__global__ __launch_bounds__(256) void swaps_to_perm_kernel(const int32_t* __restrict__ dests,
                                                            i64 nswaps, i64 size, int32_t* perm,
                                                            int inverse, int in_lds) {
    extern __shared__ int32_t sp[];
    __shared__ int32_t dq[kSwapChunk];
    const int t = threadIdx.x;
    int32_t* p = in_lds ? sp : perm;
    for (i64 i = t; i < size; i += 256) p[i] = (int32_t)i;
    // The swaps are applied one after another by one thread; the whole workgroup first stages
    // each chunk of destinations (in application order) in LDS, so the dependent chain waits
    // on no global load.
    for (i64 c0 = 0; c0 < nswaps; c0 += kSwapChunk) {
        const int cn = (int)((nswaps - c0) < kSwapChunk ? (nswaps - c0) : kSwapChunk);
        __syncthreads();  // p initialised, or the previous chunk applied
        for (int u = t; u < cn; u += 256) dq[u] = dests[inverse ? (nswaps - 1 - (c0 + u)) : (c0 + u)];
        __syncthreads();
        if (t == 0) {
#pragma unroll 4
            for (int u = 0; u < cn; ++u) {
                const i64 j = inverse ? (nswaps - 1 - (c0 + u)) : (c0 + u);
                const i64 d = dq[u];
                if (d != j && d >= 0 && d < size) {
                    const int32_t a = p[j];
                    p[j] = p[d];
                    p[d] = a;
                }
            }
        }
    }
    __syncthreads();
    if (in_lds)
        for (i64 i = t; i < size; i += 256) perm[i] = p[i];
}

template <typename T>
__global__ void gather_rows_kernel(const int32_t* __restrict__ perm, i64 m, i64 n,
                                   const T* __restrict__ Bin, i64 ldin, T* __restrict__ Bout,
                                   i64 ldout) {
    const i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    const i64 j = blockIdx.y;
    if (i >= m || j >= n) return;
    Bout[i + j * ldout] = Bin[(i64)perm[i] + j * ldin];
}

// ---------------------------------------------------------------------------------------
// Unblocked Cholesky of an n x n (n <= 128) diagonal block in one workgroup, in LDS.
// Lower: cholesky::LowerVariant3Unblocked (src/lapack_like/factor/Cholesky/LowerVariant3.hpp:
// 15-41): alpha = sqrt(a_jj) (a_jj <= 0 -> NonHPD), a21 *= 1/alpha, dsyr('L', -1, a21).
// Upper: UpperVariant3Unblocked (UpperVariant3.hpp:15-46) on the row instead of the column,
// factored as its transpose; fma(x, -y, a) and fma(y, -x, a) are the same number. The dsyr
// update is a(i,l) = fma(x_i, -x_l, a(i,l)), skipped when x_l == 0, as in the reference BLAS.
//
// Schedule (potf2_fast): 16 columns at a time, right-looking. Wave 0 factors the 16 x 16
// diagonal block with a row per lane (pivots by readlane, multipliers by a DPP broadcast
// within the lanes of the block), two waves solve the rows below it (a row per lane), and all
// waves apply the rank-16 update to the 16 x 16 tiles right of it on the matrix cores. Every
// entry receives exactly the unblocked algorithm's FMAs in column order, so the result is the
// same bit for bit. What bounds it is the chain of 128 pivots (square root, reciprocal, scale,
// one FMA: about 450 cycles each): 245 -> 69 us (FP64) and 206 -> 71 us (FP32) per 128 x 128
// block against the 32-column schedule below, whose block column went through one wave.
//
// The skip of a zero multiplier matters only beside an infinity or NaN (0 * inf), and the state
// at a non-positive pivot is the unblocked algorithm's at that column. Both are left to the
// general schedule (potf2_general), which starts again from the untouched block: 32 columns at
// a time, all threads bring the block column up to date with the columns to its left, wave 0
// factors it in registers (lane q holds rows q and q + 64), and on a failure the block columns
// to the right receive the updates of the finished columns.
// ---------------------------------------------------------------------------------------
constexpr int PT = 512;  // threads of the diagonal-block Cholesky

// The clean case; false (to every thread) at a pivot that is not positive or an entry that is
// not finite. S holds the block's lower triangle, S[r + c*LD]. sbad: two flags, zero on entry,
// each written between barriers where the other one is read.
template <typename T>
__device__ __forceinline__ bool potf2_fast(T* S, int n, int LD, T* sinv, int* sbad) {
    typedef Mfma4<T> MF;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int l16 = lane & 15, kq = lane >> 4;
    for (int c0 = 0; c0 < n; c0 += 16) {
        const int nt = (n - c0 + 15) / 16;  // tile rows from the diagonal one down
        if (wave == 0) {
            // rows and columns past the end are those of the identity
            T a[16];
#pragma unroll
            for (int c = 0; c < 16; ++c)
                a[c] = (c0 + l16 < n && c <= l16) ? S[(c0 + l16) + (c0 + c) * LD] : (c == l16 ? T(1) : T(0));
            bool bad = false;
            T myinv = T(0);
            static_for<0, 16>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                const T ajj = bcast_lane(a[j], j);
                bad = bad || !(ajj > T(0));
                const T alpha = sqrt(ajj);
                const T inv = T(1) / alpha;
                const T x = l16 > j ? inv * a[j] : (l16 == j ? alpha : a[j]);
                a[j] = x;
                if (l16 == j) myinv = inv;
                static_for<j + 1, 16>([&](auto cc) {
                    constexpr int c = decltype(cc)::value;
                    a[c] = __builtin_fma(x, -row_bcast<c>(x), a[c]);
                });
            });
#pragma unroll
            for (int c = 0; c < 16; ++c)
                if (c <= l16) bad = bad || !finite(a[c]);
            if (lane < 16) {
                sinv[lane] = myinv;
#pragma unroll
                for (int c = 0; c < 16; ++c)
                    if (c0 + lane < n && c <= lane) S[(c0 + lane) + (c0 + c) * LD] = a[c];
            }
            if (__any(bad ? 1 : 0) && lane == 0) sbad[0] = 1;
        }
        __syncthreads();
        if (sbad[0]) return false;
        if (nt == 1) break;
        if (wave < 2) {
            const int r = c0 + 16 + wave * 64 + lane;
            T l11[16], a[16];
            const bool in = r < n;
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                l11[k] = S[(c0 + l16) + (c0 + k) * LD];  // a full block: rows below it exist
                a[k] = in ? S[r + (c0 + k) * LD] : T(0);
            }
            const T inv = sinv[l16];
            bool bad = false;
            static_for<0, 16>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                a[k] = row_bcast<k>(inv) * a[k];
                bad = bad || !finite(a[k]);
                static_for<k + 1, 16>([&](auto cc) {
                    constexpr int c = decltype(cc)::value;
                    a[c] = __builtin_fma(a[k], -row_bcast<c>(l11[k]), a[c]);
                });
            });
            if (in) {
#pragma unroll
                for (int k = 0; k < 16; ++k) S[r + (c0 + k) * LD] = a[k];
            }
            if (__any(bad ? 1 : 0) && lane == 0) sbad[1] = 1;
        }
        __syncthreads();
        if (sbad[1]) return false;
        // tiles (bi, bj), 1 <= bj <= bi < nt: C(r, c) -= X(r, :) X(c, :)^T
        int q = 0;
        for (int bi = 1; bi < nt; ++bi)
            for (int bj = 1; bj <= bi; ++bj, ++q) {
                if (q % (PT / 64) != wave) continue;
                const int r = c0 + 16 * bi + l16, ca = c0 + 16 * bj + l16;
                typename MF::acc acc;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int c = c0 + 16 * bj + MF::row(kq, u);
                    acc[u] = (r < n && c <= r) ? S[r + c * LD] : T(0);
                }
#pragma unroll
                for (int k = 0; k < 16; k += 4) {
                    const T xc = ca < n ? S[ca + (c0 + k + kq) * LD] : T(0);
                    const T xr = r < n ? S[r + (c0 + k + kq) * LD] : T(0);
                    acc = MF::run(-xc, xr, acc);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int c = c0 + 16 * bj + MF::row(kq, u);
                    if (r < n && c <= r) S[r + c * LD] = acc[u];
                }
            }
        __syncthreads();
    }
    return true;
}

// Any block: returns the first column with a non-positive pivot, or -1.
template <typename T>
__device__ __noinline__ int potf2_general(T* S, int n, int LD, int upper, int* s_fail) {
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    if (t == 0) *s_fail = -1;
    __syncthreads();
    // (1) entries (r, c) of block column J, c in [c0, c1), r >= c: FMAs of columns [0, jmax)
    auto left_update = [&](int c0, int c1, int jmax) {
        const int h = n - c0, w = c1 - c0;
        for (int idx = t; idx < h * w; idx += PT) {
            const int r = c0 + idx % h, c = c0 + idx / h;
            if (r < c) continue;
            T acc = S[r + c * LD];
#pragma unroll 4
            for (int j = 0; j < jmax; ++j) {
                const T x = S[r + j * LD], y = S[c + j * LD];
                if ((upper ? x : y) != T(0)) acc = __builtin_fma(x, -y, acc);
            }
            S[r + c * LD] = acc;
        }
    };
    int fail = -1;
    for (int c0 = 0; c0 < n; c0 += 32) {
        const int c1 = min(n, c0 + 32);
        if (c0 > 0) {
            left_update(c0, c1, c0);
            __syncthreads();
        }
        // (2) the block column in wave 0's registers: rows c0 + q and c0 + 64 + q of lane q
        if (wave == 0) {
            T rw[2][32];
#pragma unroll
            for (int sl = 0; sl < 2; ++sl) {
                const int r = c0 + 64 * sl + lane;
#pragma unroll
                for (int cc = 0; cc < 32; ++cc)
                    rw[sl][cc] = (r < n && c0 + cc < c1 && r >= c0 + cc) ? S[r + (c0 + cc) * LD] : T(0);
            }
            int f = -1;
#pragma unroll
            for (int jj = 0; jj < 32; ++jj) {
                const int cj = c0 + jj;
                if (cj < c1 && f < 0) {
                    T alpha = bcast_lane(rw[0][jj], jj);
                    if (alpha <= T(0)) {
                        f = cj;
                    } else {
                        alpha = sqrt(alpha);
                        const T inv = T(1) / alpha;
#pragma unroll
                        for (int sl = 0; sl < 2; ++sl) {
                            const int r = c0 + 64 * sl + lane;
                            if (r == cj) rw[sl][jj] = alpha;
                            else if (r > cj) rw[sl][jj] = inv * rw[sl][jj];
                        }
#pragma unroll
                        for (int cc = jj + 1; cc < 32; ++cc) {
                            if (c0 + cc < c1) {
                                const T y = bcast_lane(rw[0][jj], cc);  // L(c0+cc, cj)
#pragma unroll
                                for (int sl = 0; sl < 2; ++sl) {
                                    const int r = c0 + 64 * sl + lane;
                                    const T x = rw[sl][jj];
                                    if (r >= c0 + cc && (upper ? x : y) != T(0))
                                        rw[sl][cc] = __builtin_fma(x, -y, rw[sl][cc]);
                                }
                            }
                        }
                    }
                }
            }
#pragma unroll
            for (int sl = 0; sl < 2; ++sl) {
                const int r = c0 + 64 * sl + lane;
#pragma unroll
                for (int cc = 0; cc < 32; ++cc)
                    if (r < n && c0 + cc < c1 && r >= c0 + cc) S[r + (c0 + cc) * LD] = rw[sl][cc];
            }
            if (lane == 0) *s_fail = f;
        }
        __syncthreads();
        fail = *s_fail;
        if (fail >= 0) {
            // the columns to the right, as the unblocked algorithm leaves them at the stop
            for (int d0 = c1; d0 < n; d0 += 32) left_update(d0, min(n, d0 + 32), fail);
            __syncthreads();
            break;
        }
    }
    return fail;
}

template <typename T>
__global__ __launch_bounds__(PT) void potf2_kernel(int n, T* A, i64 lda, int upper, i64 goff,
                                                   int32_t* info) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* S = reinterpret_cast<T*>(smem_raw);  // lower triangle L(r, c) at S[r + c*LD]
    __shared__ T sinv[16];
    __shared__ int s_flag[2];
    // an earlier block already failed: the reference has thrown, nothing more changes
    if (*info != 0) return;
    const int LD = n + 1, t = threadIdx.x;
    auto load = [&]() {
        if (n == 128) {
            // loads issued 32 at a time before their LDS stores; the whole block is read, the
            // other triangle dropped
            T v[32];
#pragma unroll
            for (int u = 0; u < 32; ++u) {
                const int idx = t + PT * u, i = idx & 127, j = idx >> 7;
                v[u] = (upper ? i <= j : i >= j) ? A[i + (i64)j * lda] : T(0);
            }
#pragma unroll
            for (int u = 0; u < 32; ++u) {
                const int idx = t + PT * u, i = idx & 127, j = idx >> 7;
                if (upper) {
                    if (i <= j) S[j + i * LD] = v[u];
                } else if (i >= j) {
                    S[i + j * LD] = v[u];
                }
            }
        } else {
            for (int idx = t; idx < n * n; idx += PT) {
                const int i = idx % n, j = idx / n;
                if (upper) {
                    if (i <= j) S[j + i * LD] = A[i + (i64)j * lda];
                } else if (i >= j) {
                    S[i + j * LD] = A[i + (i64)j * lda];
                }
            }
        }
    };
    load();
    if (t < 2) s_flag[t] = 0;
    __syncthreads();
    if (!potf2_fast(S, n, LD, sinv, s_flag)) {
        __syncthreads();
        load();
        __syncthreads();
        const int fail = potf2_general(S, n, LD, upper, s_flag);
        if (fail >= 0 && t == 0) atomicCAS(info, 0, (int32_t)(goff + fail + 1));
    }
    __syncthreads();
    for (int idx = t; idx < n * n; idx += PT) {
        const int i = idx % n, j = idx / n;
        if (upper) {
            if (i <= j) A[i + (i64)j * lda] = S[j + i * LD];
        } else if (i >= j) {
            A[i + (i64)j * lda] = S[i + j * LD];
        }
    }
}

// ---------------------------------------------------------------------------------------
// LU without pivoting of an n x n (n <= 128) diagonal block in one workgroup, in LDS:
// lu::Unb (src/lapack_like/factor/LU/Local.hpp:44-61). Per column j: alpha = a(j,j) (exactly
// zero -> SingularMatrixException in the reference: info = goff+j+1 and the block is left as
// it stands), a21 *= 1/alpha (blas::Scal), then Geru(-1): a(i,k) = fma(a(i,j), -a(j,k), a(i,k))
// for every k with a(j,k) != 0, the reference BLAS dger's skip rule.
// ---------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void getf2_nopiv_kernel(int n, T* A, i64 lda, i64 goff,
                                                          int32_t* info) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* S = reinterpret_cast<T*>(smem_raw);  // S[i + j*LD]
    if (*info != 0) return;
    const int LD = n + 1, t = threadIdx.x;
    for (int idx = t; idx < n * n; idx += 256) {
        const int i = idx % n, j = idx / n;
        S[i + j * LD] = A[i + (i64)j * lda];
    }
    __syncthreads();
    int fail = -1;
    for (int j = 0; j < n; ++j) {
        const T alpha = S[j + j * LD];
        if (alpha == T(0)) {
            fail = j;
            break;
        }
        const T inv = T(1) / alpha;
        for (int i = j + 1 + t; i < n; i += 256) S[i + j * LD] = inv * S[i + j * LD];
        __syncthreads();
        const int h = n - (j + 1);
        for (int idx = t; idx < h * h; idx += 256) {
            const int i = j + 1 + idx % h, k = j + 1 + idx / h;
            const T y = S[j + k * LD];
            if (y != T(0)) S[i + k * LD] = __builtin_fma(S[i + j * LD], -y, S[i + k * LD]);
        }
        __syncthreads();
    }
    if (fail >= 0 && t == 0) atomicCAS(info, 0, (int32_t)(goff + fail + 1));
    for (int idx = t; idx < n * n; idx += 256) {
        const int i = idx % n, j = idx / n;
        A[i + (i64)j * lda] = S[i + j * LD];
    }
}

}  // namespace

namespace elx {

template <typename T>
static elx_status_t row_moves_impl(hipStream_t s, const int2* pairs, int npairs, T* A, i64 lda,
                                   i64 r0, i64 rows, i64 c0, i64 c1, i64 c2, i64 c3,
                                   const int32_t* stop) {
    ELX_ARG(npairs <= 256 && rows >= 0);
    const i64 total = std::max<i64>(c1 - c0, 0) + std::max<i64>(c3 - c2, 0);
    if (total <= 0 || npairs <= 0) return ELX_SUCCESS;
    if (c1 < c0) c1 = c0;
    if (c3 < c2) c3 = c2;
    ProfScope prof_(s, kKRowMoves, 2.0 * npairs * (double)total * sizeof(T));
    hipLaunchKernelGGL(row_moves_kernel<T>, dim3(cdiv(total, 4)), dim3(256), 0, s, pairs, npairs,
                       A, lda, r0, rows, c0, c1, c2, c3, stop);
    ELX_HIP(hipGetLastError());
    return ELX_SUCCESS;
}

elx_status_t launch_row_moves_f64(hipStream_t s, const int2* pairs, int npairs, double* A,
                                  i64 lda, i64 r0, i64 rows, i64 c0, i64 c1, i64 c2, i64 c3) {
    return row_moves_impl<double>(s, pairs, npairs, A, lda, r0, rows, c0, c1, c2, c3, nullptr);
}

elx_status_t launch_row_moves(hipStream_t s, const int2* pairs, int npairs, double* A, i64 lda,
                              i64 r0, i64 rows, i64 c0, i64 c1, i64 c2, i64 c3,
                              const int32_t* stop) {
    return row_moves_impl<double>(s, pairs, npairs, A, lda, r0, rows, c0, c1, c2, c3, stop);
}

elx_status_t launch_row_moves(hipStream_t s, const int2* pairs, int npairs, float* A, i64 lda,
                              i64 r0, i64 rows, i64 c0, i64 c1, i64 c2, i64 c3,
                              const int32_t* stop) {
    return row_moves_impl<float>(s, pairs, npairs, A, lda, r0, rows, c0, c1, c2, c3, stop);
}

elx_status_t launch_row_moves_f32_rowmajor(hipStream_t s, const int2* pairs, int npairs,
                                           float* A, i64 lda, i64 r0, i64 rows, i64 c0, i64 c1,
                                           i64 c2, i64 c3) {
    ELX_ARG(npairs <= 256 && rows >= 0);
    if (c1 < c0) c1 = c0;
    if (c3 < c2) c3 = c2;
    const i64 total = (c1 - c0) + (c3 - c2);
    if (total <= 0 || npairs <= 0) return ELX_SUCCESS;
    const i64 slices = cdiv(c1 - c0, 64) + cdiv(c3 - c2, 64);
    ProfScope prof_(s, kKRowMoves, 2.0 * npairs * (double)total * sizeof(float));
    hipLaunchKernelGGL(row_moves_rowmajor_kernel, dim3((unsigned)slices), dim3(512), 0, s, pairs,
                       npairs, A, lda, r0, rows, c0, c1, c2, c3);
    ELX_HIP(hipGetLastError());
    return ELX_SUCCESS;
}

elx_status_t launch_swaps_to_perm(hipStream_t s, const int32_t* dests, i64 nswaps, i64 size,
                                  int32_t* perm, int inverse) {
    if (size <= 0) return ELX_SUCCESS;
    const DeviceInfo& di = device_info();
    const size_t need = sizeof(int32_t) * (size_t)size;
    const size_t dyn_max = (size_t)di.max_lds_per_block - sizeof(int32_t) * kSwapChunk;
    const int in_lds = need <= dyn_max ? 1 : 0;
    static bool attr = false;
    if (!attr) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&swaps_to_perm_kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn_max);
        (void)hipGetLastError();
        attr = true;
    }
    hipLaunchKernelGGL(swaps_to_perm_kernel, dim3(1), dim3(256), in_lds ? need : 0, s, dests,
                       nswaps, size, perm, inverse, in_lds);
    ELX_HIP(hipGetLastError());
    return ELX_SUCCESS;
}

template <typename T>
static elx_status_t gather_rows_impl(hipStream_t s, const int32_t* perm, i64 m, i64 n,
                                     const T* Bin, i64 ldin, T* Bout, i64 ldout) {
    if (m <= 0 || n <= 0) return ELX_SUCCESS;
    ELX_ARG(n <= 65535);
    hipLaunchKernelGGL(gather_rows_kernel<T>, dim3(cdiv(m, 256), (unsigned)n), dim3(256), 0, s,
                       perm, m, n, Bin, ldin, Bout, ldout);
    ELX_HIP(hipGetLastError());
    return ELX_SUCCESS;
}

elx_status_t launch_gather_rows_f64(hipStream_t s, const int32_t* perm, i64 m, i64 n,
                                    const double* Bin, i64 ldin, double* Bout, i64 ldout) {
    return gather_rows_impl<double>(s, perm, m, n, Bin, ldin, Bout, ldout);
}

elx_status_t launch_gather_rows(hipStream_t s, const int32_t* perm, i64 m, i64 n,
                                const double* Bin, i64 ldin, double* Bout, i64 ldout) {
    return gather_rows_impl<double>(s, perm, m, n, Bin, ldin, Bout, ldout);
}

elx_status_t launch_gather_rows(hipStream_t s, const int32_t* perm, i64 m, i64 n,
                                const float* Bin, i64 ldin, float* Bout, i64 ldout) {
    return gather_rows_impl<float>(s, perm, m, n, Bin, ldin, Bout, ldout);
}

elx_status_t launch_potf2_f64(hipStream_t s, int uplo, i64 n, double* A, i64 lda, i64 goff,
                              int32_t* info) {
    if (n <= 0) return ELX_SUCCESS;
    ELX_ARG(n <= 128);
    const size_t lds = sizeof(double) * (size_t)n * (n + 1);
    static bool attr = false;
    if (!attr) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&potf2_kernel<double>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)(sizeof(double) * 128 * 129));
        (void)hipGetLastError();
        attr = true;
    }
    hipLaunchKernelGGL(potf2_kernel<double>, dim3(1), dim3(PT), lds, s, (int)n, A, lda,
                       uplo == kUpper ? 1 : 0, goff, info);
    ELX_HIP(hipGetLastError());
    return ELX_SUCCESS;
}

elx_status_t launch_potf2(hipStream_t s, int uplo, i64 n, double* A, i64 lda, i64 goff,
                          int32_t* info) {
    return launch_potf2_f64(s, uplo, n, A, lda, goff, info);
}

elx_status_t launch_potf2(hipStream_t s, int uplo, i64 n, float* A, i64 lda, i64 goff,
                          int32_t* info) {
    return launch_potf2_f32(s, uplo, n, A, lda, goff, info);
}

template <typename T>
static elx_status_t getf2_nopiv_impl(hipStream_t s, i64 n, T* A, i64 lda, i64 goff,
                                     int32_t* info) {
    if (n <= 0) return ELX_SUCCESS;
    ELX_ARG(n <= 128);
    const size_t lds = sizeof(T) * (size_t)n * (n + 1);
    static bool attr = false;
    if (!attr) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&getf2_nopiv_kernel<T>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)(sizeof(T) * 128 * 129));
        (void)hipGetLastError();
        attr = true;
    }
    hipLaunchKernelGGL(getf2_nopiv_kernel<T>, dim3(1), dim3(256), lds, s, (int)n, A, lda, goff,
                       info);
    ELX_HIP(hipGetLastError());
    return ELX_SUCCESS;
}

elx_status_t launch_getf2_nopiv(hipStream_t s, i64 n, double* A, i64 lda, i64 goff,
                                int32_t* info) {
    return getf2_nopiv_impl<double>(s, n, A, lda, goff, info);
}

elx_status_t launch_getf2_nopiv(hipStream_t s, i64 n, float* A, i64 lda, i64 goff,
                                int32_t* info) {
    return getf2_nopiv_impl<float>(s, n, A, lda, goff, info);
}

elx_status_t launch_potf2_f32(hipStream_t s, int uplo, i64 n, float* A, i64 lda, i64 goff,
                              int32_t* info) {
    if (n <= 0) return ELX_SUCCESS;
    ELX_ARG(n <= 128);
    const size_t lds = sizeof(float) * (size_t)n * (n + 1);
    hipLaunchKernelGGL(potf2_kernel<float>, dim3(1), dim3(PT), lds, s, (int)n, A, lda,
                       uplo == kUpper ? 1 : 0, goff, info);
    ELX_HIP(hipGetLastError());
    return ELX_SUCCESS;
}

}  // namespace elx
