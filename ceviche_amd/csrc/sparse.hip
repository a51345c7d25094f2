// Generic sparse primitives for ceviche's COO interface (entries, indices):
// a deterministic segmented product-sum kernel (SpMV, A^T / A^H products,
// outer-product gathers, SpGEMM numerics and their derivatives), and a dense
// complex128 LU with partial pivoting for small general systems.
//
// The symbolic part (grouping entries by row / column / output position) is
// done once per index set on the host, like the reference's COO->CSR
// conversion (ceviche/utils.py:13-25); every numeric operation runs here.
#include "common.h"

#include <algorithm>
#include <type_traits>

namespace cv {

// out[o(s)] (+)= alpha * sum_{q in [ptr[s], ptr[s+1])} opu(u[iu[q]]) * opv(v[iv[q]])
// with o(s) = oidx ? oidx[s] : s and opu / opv optional conjugation; UNIT:
// segment s is entry s alone, no ptr.  One thread per segment; the sum
// runs in storage order (deterministic).  Bound by the latency of index and
// gather loads that follow each other, so four entries are in flight at a
// time (1.3 million entries in 262144 rows: 52 -> 49 us; as unit segments,
// which need no ptr, 33).
constexpr int kSegBatch = 4;

template <bool UNIT>
__global__ void __launch_bounds__(256)
k_segsum(int64_t n_seg, const int64_t* __restrict__ ptr, const int64_t* __restrict__ iu,
         const int64_t* __restrict__ iv, const cx<double>* __restrict__ u, const cx<double>* __restrict__ v,
         int conj_u, int conj_v, cx<double> alpha, const int64_t* __restrict__ oidx, int accumulate,
         cx<double>* __restrict__ out) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n_seg) return;
    cx<double> acc = czero<double>();
    auto add = [&](cx<double> a, cx<double> b) {
        if (conj_u) a = conj(a);
        if (conj_v) b = conj(b);
        acc = acc + a * b;
    };
    if (UNIT) {
        add(u[iu ? iu[s] : s], v[iv ? iv[s] : s]);
    } else {
        const int64_t end = ptr[s + 1];
        int64_t q = ptr[s];
        for (; q + kSegBatch <= end; q += kSegBatch) {
            int64_t a[kSegBatch], b[kSegBatch];
            cx<double> x[kSegBatch], y[kSegBatch];
#pragma unroll
            for (int e = 0; e < kSegBatch; ++e) {
                a[e] = iu ? iu[q + e] : q + e;
                b[e] = iv ? iv[q + e] : q + e;
            }
#pragma unroll
            for (int e = 0; e < kSegBatch; ++e) {
                x[e] = u[a[e]];
                y[e] = v[b[e]];
            }
#pragma unroll
            for (int e = 0; e < kSegBatch; ++e) add(x[e], y[e]);
        }
        for (; q < end; ++q) add(u[iu ? iu[q] : q], v[iv ? iv[q] : q]);
    }
    const int64_t o = oidx ? oidx[s] : s;
    acc = alpha * acc;
    out[o] = accumulate ? out[o] + acc : acc;
}

// ------------------------------------------------------------- dense LU
// Column-major n x n complex128.  Pivot choice: max |re| + |im| (LAPACK's
// izamax measure), lowest index on ties.
__global__ void __launch_bounds__(256)
k_lu_pivot(int n, cx<double>* __restrict__ A, int k, int32_t* __restrict__ piv, int32_t* __restrict__ info) {
    __shared__ double s_val[256];
    __shared__ int s_idx[256];
    __shared__ int s_p;
    double best = -1.0;
    int bi = n;
    for (int i = k + threadIdx.x; i < n; i += blockDim.x) {
        const cx<double> a = A[(int64_t)k * n + i];
        const double m = fabs(a.re) + fabs(a.im);
        if (m > best || (m == best && i < bi)) {
            best = m;
            bi = i;
        }
    }
    s_val[threadIdx.x] = best;
    s_idx[threadIdx.x] = bi;
    __syncthreads();
    for (int off = blockDim.x / 2; off > 0; off >>= 1) {
        if (threadIdx.x < off) {
            const double ov = s_val[threadIdx.x + off];
            const int oi = s_idx[threadIdx.x + off];
            if (ov > s_val[threadIdx.x] || (ov == s_val[threadIdx.x] && oi < s_idx[threadIdx.x])) {
                s_val[threadIdx.x] = ov;
                s_idx[threadIdx.x] = oi;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        s_p = s_idx[0];
        piv[k] = s_p;
        if (s_val[0] == 0.0 && *info == 0) *info = k + 1;
    }
    __syncthreads();
    const int p = s_p;
    if (p != k) {
        for (int j = threadIdx.x; j < n; j += blockDim.x) {
            const cx<double> t = A[(int64_t)j * n + k];
            A[(int64_t)j * n + k] = A[(int64_t)j * n + p];
            A[(int64_t)j * n + p] = t;
        }
    }
    __syncthreads();
    const cx<double> d = A[(int64_t)k * n + k];
    if (d.re == 0.0 && d.im == 0.0) return;
    const cx<double> inv = cdiv(cone<double>(), d);
    for (int i = k + 1 + threadIdx.x; i < n; i += blockDim.x) A[(int64_t)k * n + i] = A[(int64_t)k * n + i] * inv;
}

// A[i, j] -= A[i, k] A[k, j] for i, j > k (i fastest: coalesced columns)
__global__ void __launch_bounds__(256) k_lu_update(int n, cx<double>* __restrict__ A, int k) {
    const int64_t m = n - k - 1;
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= m * m) return;
    const int i = k + 1 + (int)(e % m);
    const int j = k + 1 + (int)(e / m);
    A[(int64_t)j * n + i] = A[(int64_t)j * n + i] - A[(int64_t)k * n + i] * A[(int64_t)j * n + k];
}

// Blocked factorisation for the last kLuBlockedRows rows and columns (all of a
// matrix of at most that many): a panel of NB columns is factorised by one
// workgroup with its rows in registers, then one launch applies the panel's
// interchanges to all other columns and forms U12 = L11^-1 A12, and one
// subtracts L21 U12.  Column by column through memory (k_lu_pivot, k_lu_update)
// every column cost two launches and three passes over the panel: 12.2 us a
// column at n = 1600, 19.5 ms in all; 3072 rows are what one workgroup's
// registers hold.
constexpr int kLuBlockedRows = 3072;
constexpr int kLuThreads = 1024;

// |re| + |im| (NaN counts as 0)
__device__ __forceinline__ double lu_size(cx<double> a) {
    const double m = fabs(a.re) + fabs(a.im);
    return m >= 0.0 ? m : 0.0;
}

// max of the non-negative values v over lanes, by lane exchanges inside the
// vector unit (an LDS shuffle takes some 100 cycles a step): the lanes of a
// row of 16 (ROW) or the whole wave
template <int CTRL>
__device__ __forceinline__ double lu_dpp_max(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, true);
    return fmax(v, __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo));
}
__device__ __forceinline__ double lu_lane(double v, int lane) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
template <bool ROW>
__device__ __forceinline__ double lu_max(double v) {
    v = lu_dpp_max<0x111>(v);   // row_shr:1
    v = lu_dpp_max<0x112>(v);
    v = lu_dpp_max<0x114>(v);
    v = lu_dpp_max<0x118>(v);
    if (ROW) return lu_lane(v, 15);
    v = lu_dpp_max<0x142>(v);   // row_bcast:15
    v = lu_dpp_max<0x143>(v);   // row_bcast:31
    return lu_lane(v, 63);
}

// lowest row among the lanes of `mask`
__device__ __forceinline__ int lu_min_row(uint64_t mask, int row) {
    int best = __builtin_amdgcn_readlane(row, __builtin_ctzll(mask));
    for (mask &= mask - 1; mask; mask &= mask - 1) best = min(best, __builtin_amdgcn_readlane(row, __builtin_ctzll(mask)));
    return best;
}

// 1 / d by the hardware's estimate of 1 / |d|^2 and two Newton steps (the
// division's 30 operations would be issued by all 16 waves for every column)
__device__ __forceinline__ cx<double> lu_recip(cx<double> d) {
    const double x = d.re * d.re + d.im * d.im;
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    r = __builtin_amdgcn_div_fixup(r, x, 1.0);
    return mk(d.re * r, -d.im * r);
}

// LU with partial pivoting of the m x w panel at P (rows k .. k + m - 1 of the
// matrix, w <= NB columns), thread t holding rows t + q * 1024.  Bound by the
// chain of columns: a pivot search (lane exchanges, then the 16 waves' best
// through LDS), an exchange of two rows through LDS and the rank-1 update in
// registers, two barriers a column.
template <int NB, int RPT>
__global__ void __launch_bounds__(kLuThreads)
k_lu_panel_z(int n, cx<double>* __restrict__ A, int k, int w, int32_t* __restrict__ piv, int32_t* __restrict__ info) {
    __shared__ double s_max[2][kLuThreads / 64];
    __shared__ int s_row[2][kLuThreads / 64];
    __shared__ cx<double> s_piv[2][NB], s_top[2][NB];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int m = n - k;
    cx<double>* P = A + (int64_t)k * n + k;
    cx<double> a[RPT][NB];
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int r = t + q * kLuThreads;
#pragma unroll
        for (int c = 0; c < NB; ++c) a[q][c] = (r < m && c < w) ? P[(int64_t)c * n + r] : czero<double>();
    }
#pragma unroll
    for (int c = 0; c < NB; ++c) {
        if (c < w) {   // uniform
        const int sl = c & 1;
        double best = 0.0;
        int row = c;
#pragma unroll
        for (int q = RPT - 1; q >= 0; --q) {
            const int r = t + q * kLuThreads;
            const double v = r >= c && r < m ? lu_size(a[q][c]) : -1.0;
            if (v >= best) {   // of equal values the lower row
                best = v;
                row = r;
            }
        }
        // a wave without a non-zero candidate proposes row c (not taken unless all are zero)
        const double wmax = lu_max<false>(best);
        const int wrow = wmax == 0.0 ? c : lu_min_row(__ballot(best == wmax), row);
        if (lane == 0) {
            s_max[sl][wave] = wmax;
            s_row[sl][wave] = wrow;
        }
        __syncthreads();
        best = s_max[sl][lane & 15];
        row = s_row[sl][lane & 15];
        const double pmax = lu_max<true>(best);
        const int p = pmax == 0.0 ? c : lu_min_row(__ballot(best == pmax) & 0xffff, row);   // c <= p < m
        if (t == 0) {
            piv[k + c] = k + p;
            if (pmax == 0.0 && *info == 0) *info = k + c + 1;
        }
        // rows c and p change places; the pivot row goes to everyone
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int r = t + q * kLuThreads;
            if (r == p)
#pragma unroll
                for (int j = 0; j < NB; ++j) s_piv[sl][j] = a[q][j];
            if (r == c)
#pragma unroll
                for (int j = 0; j < NB; ++j) s_top[sl][j] = a[q][j];
        }
        __syncthreads();
        const cx<double> d = s_piv[sl][c];   // uniform
        const bool zero = d.re == 0.0 && d.im == 0.0;
        const cx<double> inv = zero ? czero<double>() : lu_recip(d);
        // the pivot row, one entry per lane, broadcast through scalar registers
        // (an LDS read per entry and wave took half of the column's time)
        const cx<double> mine = s_piv[sl][lane & (NB - 1)];
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int r = t + q * kLuThreads;
            if (r == p || r == c) {
#pragma unroll
                for (int j = 0; j < NB; ++j) a[q][j] = r == c ? s_piv[sl][j] : s_top[sl][j];
            }
        }
        if (!zero) {   // a column of zeros stays as it is
            cx<double> l[RPT];
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                l[q] = t + q * kLuThreads > c ? a[q][c] * inv : czero<double>();
                if (t + q * kLuThreads > c) a[q][c] = l[q];
            }
#pragma unroll
            for (int j = c + 1; j < NB; ++j) {
                const cx<double> u = mk(lu_lane(mine.re, j), lu_lane(mine.im, j));
#pragma unroll
                for (int q = 0; q < RPT; ++q) a[q][j] = a[q][j] - l[q] * u;
            }
        }
        }
    }
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        const int r = t + q * kLuThreads;
#pragma unroll
        for (int c = 0; c < NB; ++c)
            if (r < m && c < w) P[(int64_t)c * n + r] = a[q][c];
    }
}

// The panel's interchanges on every column outside it, one thread per column,
// and U12 = L11^-1 A12 on the columns to its right.  The w interchanges touch
// at most 2 w rows; each row's source is found by tracing them backwards, so
// all loads of a column are independent.
template <int NB>
__global__ void __launch_bounds__(64)
k_lu_swap_z(int n, cx<double>* __restrict__ A, int k, int w, const int32_t* __restrict__ piv) {
    __shared__ int s_piv[NB], s_dst[2 * NB], s_src[2 * NB];
    __shared__ cx<double> s_l[NB][NB];   // L11, [column][row]
    const int t = threadIdx.x;
    if (t < w) s_piv[t] = piv[k + t];
    for (int q = t; q < NB * NB; q += 64) {
        const int c = q / NB, r = q % NB;
        s_l[c][r] = (c < w && r < w) ? A[(int64_t)(k + c) * n + k + r] : czero<double>();
    }
    __syncthreads();
    if (t < 2 * NB) {
        const int c = t < NB ? t : t - NB;
        int dst = -1, src = -1;
        if (c < w) {
            dst = t < NB ? k + c : s_piv[c];
            src = dst;
            for (int q = w - 1; q >= 0; --q) src = src == k + q ? s_piv[q] : src == s_piv[q] ? k + q : src;
        }
        s_dst[t] = dst;
        s_src[t] = src;
    }
    __syncthreads();
    int j = blockIdx.x * 64 + t;   // columns outside the panel
    if (j >= n - w) return;
    if (j >= k) j += w;
    cx<double>* col = A + (int64_t)j * n;
    cx<double> top[NB], low[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) {
        top[c] = c < w ? col[s_src[c]] : czero<double>();
        low[c] = c < w ? col[s_src[NB + c]] : czero<double>();
    }
    if (j >= k) {
#pragma unroll
        for (int c = 0; c < NB; ++c) {
#pragma unroll
            for (int r = c + 1; r < NB; ++r) top[r] = top[r] - s_l[c][r] * top[c];   // zeros beyond w
        }
    }
#pragma unroll
    for (int c = 0; c < NB; ++c) {
        if (c < w && s_dst[NB + c] >= k + w) col[s_dst[NB + c]] = low[c];
        if (c < w) col[k + c] = top[c];
    }
}

// A22 -= L21 U12: a lane per row, each of the four waves 16 of a tile's 64
// columns; the rows' multipliers in registers, a column's U12 through scalar
// loads (uniform over the wave; as LDS broadcasts they bound the kernel).
template <int NB>
__global__ void __launch_bounds__(256) k_lu_trail_z(int n, cx<double>* A, int k) {
    const int first = k + NB;
    const int row = first + blockIdx.x * 64 + (threadIdx.x & 63);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col0 = first + blockIdx.y * 64 + 16 * w;
    const int cols = min(16, n - col0);
    cx<double> l[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) l[c] = row < n ? A[(int64_t)(k + c) * n + row] : czero<double>();
    using cu_t = const __attribute__((address_space(4))) double*;
    for (int j = 0; j < cols; ++j) {
        const cu_t u = (cu_t)(A + (int64_t)(col0 + j) * n + k);
        cx<double>* at = A + (int64_t)(col0 + j) * n + row;
        cx<double> v = row < n ? *at : czero<double>();
#pragma unroll
        for (int c = 0; c < NB; ++c) v = v - l[c] * mk(u[2 * c], u[2 * c + 1]);
        if (row < n) *at = v;
    }
}

// Triangular solves with the packed factors (P A = L U), blocks of 64 rows,
// one launch per block: every workgroup subtracts the block solved last from
// its own 64 rows, and the one that holds the next block then solves it.
// KIND 0: L (unit, forward), 1: U (backward), 2: U^T or U^H (forward), 3: L^T
// or L^H (unit, backward).  `blk`: the block solved last (-1 or the number of
// blocks: none yet).
// Bound by the launches and the 64-step chain of a diagonal block.
constexpr int kTri = 64;

template <int KIND>
__global__ void __launch_bounds__(256)
k_lu_tri(int n, const cx<double>* __restrict__ LU, cx<double>* __restrict__ B, int blk, int conjugate) {
    constexpr bool kForward = KIND == 0 || KIND == 2, kTrans = KIND >= 2, kUnit = KIND == 0 || KIND == 3;
    __shared__ cx<double> s_t[kTri][kTri + 1];   // [column][row] of a block (as stored), padded against conflicts
    __shared__ cx<double> s_part[4][kTri];
    __shared__ cx<double> s_y[kTri];
    cx<double>* b = B + (int64_t)blockIdx.x * n;   // right-hand sides along x, which has room for any number
    const int nblk = (n + kTri - 1) / kTri;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int next = kForward ? blk + 1 : blk - 1;
    const int mine = kForward ? next + (int)blockIdx.y : next - (int)blockIdx.y;   // in range by the grid
    const bool solve = blockIdx.y == 0;
    const bool update = blk >= 0 && blk < nblk;
    const int row = mine * kTri + lane;   // the unknown of this lane
    // block (br, bc) of LU as s_t[column][row]
    auto load = [&](int br, int bc) {
        for (int c = w; c < kTri; c += 4) {
            const int r = br * kTri + lane, cc = bc * kTri + c;
            cx<double> v = r < n && cc < n ? LU[(int64_t)cc * n + r] : czero<double>();
            if (conjugate) v.im = -v.im;
            s_t[c][lane] = v;
        }
    };
    cx<double> v = row < n ? b[row] : czero<double>();
    cx<double> diag[kTri / 4];   // the diagonal block of the workgroup that solves, in flight during the update
    if (solve)
#pragma unroll
        for (int q = 0; q < kTri / 4; ++q) {
            const int r = mine * kTri + lane, c = mine * kTri + w + 4 * q;
            diag[q] = r < n && c < n ? LU[(int64_t)c * n + r] : czero<double>();
        }
    if (update) {
        if (threadIdx.x < kTri) s_y[lane] = blk * kTri + lane < n ? b[blk * kTri + lane] : czero<double>();
        if (kTrans) load(blk, mine);
        __syncthreads();
        cx<double> acc = czero<double>();
        for (int q = 0; q < 16; ++q) {
            const int j = 16 * w + q;   // unknown j of the solved block
            cx<double> a;
            if (kTrans) {
                a = s_t[lane][j];
            } else {
                const int c = blk * kTri + j;
                a = row < n && c < n ? LU[(int64_t)c * n + row] : czero<double>();
            }
            acc = acc + a * s_y[j];
        }
        s_part[w][lane] = acc;
        __syncthreads();
        if (w == 0) v = v - (((s_part[0][lane] + s_part[1][lane]) + s_part[2][lane]) + s_part[3][lane]);
    }
    if (!solve) {
        if (w == 0 && row < n) b[row] = v;
        return;
    }
    // after the last read of s_t above (barrier in between)
#pragma unroll
    for (int q = 0; q < kTri / 4; ++q) {
        if (conjugate) diag[q].im = -diag[q].im;
        s_t[w + 4 * q][lane] = diag[q];
    }
    __syncthreads();
    if (w != 0) return;
    cx<double> inv = cone<double>();
    if (!kUnit) inv = row < n ? cdiv(cone<double>(), s_t[lane][lane]) : cone<double>();
#pragma unroll 8
    for (int s = 0; s < kTri; ++s) {
        const int j = kForward ? s : kTri - 1 - s;
        const cx<double> x = kUnit ? v : v * inv;
        const cx<double> xj = mk(lu_lane(x.re, j), lu_lane(x.im, j));
        if (lane == j) v = xj;
        const bool rest = kForward ? lane > j : lane < j;
        if (rest) v = v - (kTrans ? s_t[lane][j] : s_t[j][lane]) * xj;
    }
    if (row < n) b[row] = v;
}

constexpr int kLuPermuteLds = 8192;   // rows whose indices and interchanges fit 64 KiB of LDS

// b = P b (forward: the interchanges in order) or P^T b for n <= kLuPermuteLds:
// the interchanges act on indices in LDS, then one gather.  One workgroup per right-hand side.
__global__ void __launch_bounds__(1024)
k_lu_permute(int n, const int32_t* __restrict__ piv, cx<double>* __restrict__ B, int forward) {
    extern __shared__ int s_idx[];   // n source rows, then the n interchanges
    cx<double>* b = B + (int64_t)blockIdx.x * n;
    int* s_p = s_idx + n;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        s_idx[i] = i;
        s_p[i] = piv[i];
    }
    __syncthreads();
    // one wave, 64 interchanges at a time: each lane traces what ends up in one
    // of the block's rows and in its partner
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x, nblk = (n + 63) / 64;
        for (int k = 0; k < nblk; ++k) {
            const int first = (forward ? k : nblk - 1 - k) * 64, i = first + lane;
            const int p = i < n ? s_p[i] : i;
            int src1 = i, src2 = p;
            for (int q = 0; q < 64; ++q) {
                const int c = forward ? 63 - q : q, x = first + c, y = __builtin_amdgcn_readlane(p, c);
                src1 = src1 == x ? y : src1 == y ? x : src1;
                src2 = src2 == x ? y : src2 == y ? x : src2;
            }
            const int v1 = i < n ? s_idx[src1] : 0, v2 = i < n ? s_idx[src2] : 0;
            __builtin_amdgcn_wave_barrier();
            if (i < n) {
                s_idx[i] = v1;
                s_idx[p] = v2;
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();
    constexpr int kMost = kLuPermuteLds / 1024;
    cx<double> v[kMost];
#pragma unroll
    for (int q = 0; q < kMost; ++q) {
        const int i = threadIdx.x + q * 1024;
        v[q] = i < n ? b[s_idx[i]] : czero<double>();
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kMost; ++q) {
        const int i = threadIdx.x + q * 1024;
        if (i < n) b[i] = v[q];
    }
}

// the same for any n, in memory
__global__ void k_lu_permute_seq(int n, const int32_t* __restrict__ piv, cx<double>* __restrict__ B, int forward) {
    cx<double>* b = B + (int64_t)blockIdx.x * n;
    for (int q = 0; q < n; ++q) {
        const int i = forward ? q : n - 1 - q, p = piv[i];
        const cx<double> t = b[i];
        b[i] = b[p];
        b[p] = t;
    }
}

__global__ void k_zero_i32(int32_t* p) { *p = 0; }

}  // namespace cv

using namespace cv;

namespace cv {

template <bool UNIT>
static int segsum_impl(int64_t n_seg, const int64_t* ptr, const int64_t* iu, const int64_t* iv, const void* u,
                       const void* v, int conj_u, int conj_v, double alpha_re, double alpha_im, const int64_t* oidx,
                       int accumulate, void* out, hipStream_t s) {
    CV_CHECK(n_seg >= 0, "n_seg < 0");
    CV_CHECK((UNIT || ptr) && u && v && out, "null pointer argument");
    if (n_seg == 0) return CV_OK;
    const int64_t nb = (n_seg + 255) / 256;
    CV_CHECK(nb < (1ll << 31), "too many segments");
    k_segsum<UNIT><<<(unsigned)nb, 256, 0, s>>>(n_seg, ptr, iu, iv, (const cx<double>*)u, (const cx<double>*)v, conj_u,
                                                conj_v, mk(alpha_re, alpha_im), oidx, accumulate, (cx<double>*)out);
    CV_LAUNCH_CHECK();
    return CV_OK;
}

}  // namespace cv

extern "C" int cv_segsum(int64_t n_seg, const int64_t* ptr, const int64_t* iu, const int64_t* iv, const void* u,
                         const void* v, int conj_u, int conj_v, double alpha_re, double alpha_im,
                         const int64_t* oidx, int accumulate, void* out, void* stream) {
    return segsum_impl<false>(n_seg, ptr, iu, iv, u, v, conj_u, conj_v, alpha_re, alpha_im, oidx, accumulate, out,
                              as_stream(stream));
}

extern "C" int cv_segsum_unit(int64_t n_seg, const int64_t* iu, const int64_t* iv, const void* u, const void* v,
                              int conj_u, int conj_v, double alpha_re, double alpha_im, const int64_t* oidx,
                              int accumulate, void* out, void* stream) {
    return segsum_impl<true>(n_seg, nullptr, iu, iv, u, v, conj_u, conj_v, alpha_re, alpha_im, oidx, accumulate, out,
                             as_stream(stream));
}

extern "C" int cv_dense_lu(int n, void* A, int32_t* piv, int32_t* info_dev, void* stream) {
    CV_CHECK(n > 0 && A && piv && info_dev, "bad LU arguments");
    hipStream_t s = as_stream(stream);
    k_zero_i32<<<1, 1, 0, s>>>(info_dev);
    cx<double>* Z = (cx<double>*)A;
    int k = 0;
    for (; n - k > kLuBlockedRows; ++k) {
        k_lu_pivot<<<1, 256, 0, s>>>(n, Z, k, piv, info_dev);
        const int64_t m = (int64_t)(n - k - 1) * (n - k - 1);
        k_lu_update<<<(unsigned)((m + 255) / 256), 256, 0, s>>>(n, Z, k);
    }
    auto rest = [&](auto nb) {   // after a panel of nb (or the last w) columns
        constexpr int NB = decltype(nb)::value;
        const int w = std::min(NB, n - k);
        if (n > w) k_lu_swap_z<NB><<<(n - w + 63) / 64, 64, 0, s>>>(n, Z, k, w, piv);
        const int tiles = (n - k - w + 63) / 64;
        if (tiles > 0) k_lu_trail_z<NB><<<dim3(tiles, tiles), 256, 0, s>>>(n, Z, k);
        k += w;
    };
    // A thread holds RPT rows of NB columns in at most 96 of its 128 registers
    using W8 = std::integral_constant<int, 8>;
    using W16 = std::integral_constant<int, 16>;
    while (k < n) {
        const int rows = n - k;
        if (rows > 2 * kLuThreads) {
            k_lu_panel_z<8, 3><<<1, kLuThreads, 0, s>>>(n, Z, k, std::min(8, rows), piv, info_dev);
            rest(W8{});
        } else if (rows > kLuThreads) {
            k_lu_panel_z<8, 2><<<1, kLuThreads, 0, s>>>(n, Z, k, std::min(8, rows), piv, info_dev);
            rest(W8{});
        } else {
            k_lu_panel_z<16, 1><<<1, kLuThreads, 0, s>>>(n, Z, k, std::min(16, rows), piv, info_dev);
            rest(W16{});
        }
    }
    CV_LAUNCH_CHECK();
    return CV_OK;
}

extern "C" int cv_dense_lu_solve(int n, const void* LU, const int32_t* piv, void* B, int nrhs, int trans,
                                 void* stream) {
    CV_CHECK(n > 0 && LU && piv && B && nrhs > 0, "bad solve arguments");
    CV_CHECK(trans >= 0 && trans <= 2, "trans must be 0 (N), 1 (T) or 2 (H)");
    hipStream_t s = as_stream(stream);
    const cx<double>* Z = (const cx<double>*)LU;
    cx<double>* b = (cx<double>*)B;
    const int nblk = (n + kTri - 1) / kTri;
    auto permute = [&](int forward) {
        if (n <= kLuPermuteLds) k_lu_permute<<<nrhs, 1024, 2 * sizeof(int) * (size_t)n, s>>>(n, piv, b, forward);
        else k_lu_permute_seq<<<nrhs, 1, 0, s>>>(n, piv, b, forward);
    };
    // the first launch of a sweep only solves its own block
    auto groups = [&](int left, bool first) { return dim3(nrhs, first ? 1 : left); };
    if (trans == 0) {
        permute(1);
        for (int q = -1; q < nblk - 1; ++q) k_lu_tri<0><<<groups(nblk - 1 - q, q < 0), 256, 0, s>>>(n, Z, b, q, 0);
        for (int q = nblk; q > 0; --q) k_lu_tri<1><<<groups(q, q == nblk), 256, 0, s>>>(n, Z, b, q, 0);
    } else {   // A^T = U^T L^T P: U^T y = b, L^T z = y, x = P^T z
        const int cj = trans == 2;
        for (int q = -1; q < nblk - 1; ++q) k_lu_tri<2><<<groups(nblk - 1 - q, q < 0), 256, 0, s>>>(n, Z, b, q, cj);
        for (int q = nblk; q > 0; --q) k_lu_tri<3><<<groups(q, q == nblk), 256, 0, s>>>(n, Z, b, q, cj);
        permute(0);
    }
    CV_LAUNCH_CHECK();
    return CV_OK;
}
