// FDTD Yee update with UPML integral terms (ceviche/fdtd.py:74-144) and its
// exact discrete adjoint, for float32 / float64 state.
//
// State (18 arrays of nx*ny*nz, C order, z fastest):
//   0..2 H   3..5 D   6..8 ICE   9..11 IH   12..14 ICH   15..17 ID
// E is not stored: E_a = D_a / eps_aa with eps_aa = (eps + roll(eps, 1, a)) / 2
// (utils.py:153-176), formed on the fly from eps.  The PML integrals are only
// touched where their coefficient is non-zero (ICE_a where sigmaH_a != 0, IH_a
// where sigmaH_b sigmaH_c != 0, likewise for D): elsewhere the reference
// multiplies them by an exact zero.
//
// Coefficients (fdtd.py:265-311) are functions of the per-axis sigma profiles
// sigH_a[n_a], sigD_a[n_a] (fdtd.py:224-263) and are formed in-kernel with the
// reference's formula, in the adjoint and the temporally blocked 2D kernels
// separated by axis; interior cells (all sigma zero) use host-computed
// constants.
#include "common.h"

#include <vector>
#include <algorithm>
#include <initializer_list>
#include <type_traits>

namespace cv {

// the constants of coef4 that no cell changes
template <typename R>
struct YeeConst {
    R dt, c0, e0, e2, inv_dt, inv_e0, inv_e2;
};

template <typename R>
struct Fdtd {
    int nx, ny, nz;
    int64_t n;
    R inv_dL;
    double dt, c0, eps0, dL;
    const R* sig;      // sigHx[nx] sigHy[ny] sigHz[nz] sigDx[nx] sigDy[ny] sigDz[nz]
    const R* eps;      // relative permittivity, n
    R* st;             // 18 * n
    // interior coefficients (sigma = 0): m1 and m2 for H and D
    R h1, h2, d1, d2;
    YeeConst<R> yee;
    R cdt, c0dt, half_dt, dL_r;   // c0 dt / dL, c0 dt, dt / (2 eps0), dL
};

template <typename R>
__host__ __device__ __forceinline__ const R* sigH(const Fdtd<R>& f, int a) {
    return f.sig + (a == 0 ? 0 : (a == 1 ? f.nx : f.nx + f.ny));
}
template <typename R>
__host__ __device__ __forceinline__ const R* sigD(const Fdtd<R>& f, int a) {
    return f.sig + (f.nx + f.ny + f.nz) + (a == 0 ? 0 : (a == 1 ? f.nx : f.nx + f.ny));
}

// fdtd.py:272-311 for one component; sa is the component's own-axis sigma,
// sb, sc the other two.  sign = -1 for H (mH2, mH3 negative), +1 for D.
template <typename R>
__host__ __device__ __forceinline__ void coef4(R sa, R sb, R sc, R dt, R c0, R e0, R sign, R& m1, R& m2, R& m3, R& m4) {
    const R m0 = (R(1) / dt + (sb + sc) / R(2) / e0 + sb * sc * dt / R(4) / (e0 * e0));
    m1 = (R(1) / m0 * (R(1) / dt - (sb + sc) / R(2) / e0 - sb * sc * dt / R(4) / (e0 * e0)));
    m2 = sign / m0 * c0;
    m3 = sign / m0 * c0 * dt * sa / e0;
    m4 = R(-1) / m0 * dt * sb * sc / (e0 * e0);
}

__host__ __device__ __forceinline__ int wrapm(int i, int n) { return i == 0 ? n - 1 : i - 1; }
__host__ __device__ __forceinline__ int wrapp(int i, int n) { return i == n - 1 ? 0 : i + 1; }

template <typename R>
__host__ __device__ __forceinline__ int64_t cell(const Fdtd<R>& f, int i, int j, int k) {
    return ((int64_t)i * f.ny + j) * f.nz + k;
}

// (i, j, k) of flat cell c; 32-bit unsigned division when the grid allows it
// (a 64-bit division by a runtime value is a long instruction sequence)
template <typename R>
__host__ __device__ __forceinline__ void decompose(const Fdtd<R>& f, int64_t c, int& i, int& j, int& k) {
    if (f.n <= (int64_t)0xffffffffLL) {
        const uint32_t u = (uint32_t)c, nz = (uint32_t)f.nz, ny = (uint32_t)f.ny;
        const uint32_t ij = u / nz;
        k = (int)(u - ij * nz);
        const uint32_t ii = ij / ny;
        j = (int)(ij - ii * ny);
        i = (int)ii;
    } else {
        const int64_t ij = c / f.nz;
        k = (int)(c - ij * f.nz);
        i = (int)(ij / f.ny);
        j = (int)(ij - (int64_t)i * f.ny);
    }
}

// E_a at (i, j, k) = D_a / ((eps + eps[-e_a]) / 2); D points at the D block (Dx, Dy, Dz)
template <typename R>
__host__ __device__ __forceinline__ R efield(const Fdtd<R>& f, const R* __restrict__ D, int a, int i, int j, int k) {
    const int64_t c = cell(f, i, j, k);
    D += a * f.n;
    int64_t cm;
    if (a == 0) cm = cell(f, wrapm(i, f.nx), j, k);
    else if (a == 1) cm = cell(f, i, wrapm(j, f.ny), k);
    else cm = cell(f, i, j, wrapm(k, f.nz));
    const R eaa = (f.eps[c] + f.eps[cm]) / R(2);
    return (R(1) / eaa) * D[c];
}

// Tangent of E_a = D_a / eps_aa along (dD, d_eps): dD_a / eps_aa -
// D_a d(eps_aa) / eps_aa^2, d(eps_aa) = (d_eps + d_eps[-e_a]) / 2.
template <typename R>
__host__ __device__ __forceinline__ R efield_tangent(const Fdtd<R>& f, const R* __restrict__ D,
                                                     const R* __restrict__ dD, const R* __restrict__ deps, int a,
                                                     int i, int j, int k) {
    const int64_t c = cell(f, i, j, k);
    int64_t cm;
    if (a == 0) cm = cell(f, wrapm(i, f.nx), j, k);
    else if (a == 1) cm = cell(f, i, wrapm(j, f.ny), k);
    else cm = cell(f, i, j, wrapm(k, f.nz));
    const R inv = R(1) / ((f.eps[c] + f.eps[cm]) / R(2));
    const R deaa = (deps[c] + deps[cm]) / R(2);
    return inv * dD[a * f.n + c] - (deaa * inv * inv) * D[a * f.n + c];
}

// The value of the lane above (lane + 1) or below (lane - 1); 0 beyond the wave.
template <int CTRL>
__device__ __forceinline__ float wave_shift(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double wave_shift(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
template <typename R>
__device__ __forceinline__ R lane_above(R v) { return wave_shift<0x130>(v); }   // wave_shl:1
template <typename R>
__device__ __forceinline__ R lane_below(R v) { return wave_shift<0x138>(v); }   // wave_shr:1

// A value that is the same in every lane, kept in scalar registers.
__device__ __forceinline__ float uniform(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double uniform(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// The value of lane s (uniform).
__device__ __forceinline__ float read_lane(float v, int s) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), s));
}
__device__ __forceinline__ double read_lane(double v, int s) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, s);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), s);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// 1 / v: the hardware's estimate (1 ulp), one Newton step and the fix-up of
// zeros, infinities and NaN in float32 (4 operations; the division takes 11)
__device__ __forceinline__ float recip(float v) {
    const float r = __builtin_amdgcn_rcpf(v);
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-v, r, 1.0f), r, r), v, 1.0f);
}
__device__ __forceinline__ double recip(double v) { return 1.0 / v; }

// ========================================= two-phase step kernels
// The per-step kernels (H phase, D phase and their adjoints) give each thread
// V consecutive z cells of one (x, y) line, loaded and stored as one vector:
// they are bound by memory, and a copy with 16-byte lanes reaches 6.2 TB/s
// where one with 4-byte lanes reaches 3.8 (8.3 against 5.6 in the Infinity
// Cache).  Neighbours along z are the next element or the next lane; lanes at
// the end of a line or a wave read that one element from memory.  V divides
// nz and every base pointer is aligned to it (step_width).  At 256^3 float32
// with PML on all faces a step takes 173 + 115 us (H, D phase; 198 + 156 with
// one cell per thread), 40 + 36 B per cell at 3.9 and 5.3 TB/s; the adjoint of
// a step of 131 x 117 x 142 takes 23 + 39 us (57 + 71).
template <typename R, int V>
struct alignas(V * sizeof(R)) Vec {
    R v[V];
    __device__ __forceinline__ R& operator[](int q) { return v[q]; }
    __device__ __forceinline__ const R& operator[](int q) const { return v[q]; }
};

template <typename R, int V>
__device__ __forceinline__ Vec<R, V> ldv(const R* p) {
    return *reinterpret_cast<const Vec<R, V>*>(p);
}
template <typename R, int V>
__device__ __forceinline__ void stv(R* p, const Vec<R, V>& x) {
    *reinterpret_cast<Vec<R, V>*>(p) = x;
}

// Workgroups go round the 8 XCDs in turn: here workgroup b takes block
// b / 8 of the (b mod 8)-th of eight equal ranges, so that the lines beside
// and the slices before and after a block's are in the same L2.  The D phase
// takes 115 us instead of 118 at 256^3 (17.4 instead of 18.9 at 131 x 117 x
// 142), the adjoint's two phases 23 and 39 us instead of 24 and 40; the H
// phase, whose D and eps planes of two slices fill an L2, takes the same in
// either order (173 and 174 us; 23.1 plain and 22.1 in ranges at 131 x 117 x
// 142) and keeps the plain one.
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t blocks) {
    const uint32_t per = blocks / 8, rest = blocks - per * 8, x = b & 7;
    return x * per + min(x, rest) + (b >> 3);
}

// The cells of this thread: line (i, j), z = k0 .. k0 + V - 1.  Threads past
// the end repeat the last group (lane shifts need every lane) and store nothing.
template <typename R, int V>
struct ZGroup {
    int i, j, k0, nz, ny;
    bool live, lo, hi;     // lo / hi: the neighbour below / above is not in the lane beside
    int klo, khi;          // z of the cells below and above the group

    __device__ __forceinline__ ZGroup(const Fdtd<R>& f, uint32_t block) : nz(f.nz), ny(f.ny) {
        const int64_t total = f.n / V;
        int64_t g = (int64_t)block * blockDim.x + threadIdx.x;
        live = g < total;
        if (!live) g = total - 1;
        if (total <= (int64_t)0xffffffffLL) {
            const uint32_t u = (uint32_t)g, ng = (uint32_t)(nz / V), ij = u / ng, ii = ij / (uint32_t)ny;
            k0 = (int)(u - ij * ng) * V;
            i = (int)ii;
            j = (int)(ij - ii * (uint32_t)ny);
        } else {
            const int64_t ng = nz / V, ij = g / ng;
            k0 = (int)(g - ij * ng) * V;
            i = (int)(ij / ny);
            j = (int)(ij - (int64_t)i * ny);
        }
        const int lane = threadIdx.x & 63;
        lo = k0 == 0 || lane == 0;
        hi = k0 + V == nz || lane == 63;
        klo = k0 == 0 ? nz - 1 : k0 - 1;
        khi = k0 + V == nz ? 0 : k0 + V;
    }
    __device__ __forceinline__ int64_t line(int ii, int jj) const { return ((int64_t)ii * ny + jj) * nz; }
    // x one cell up / down along z; edge: the value where the lane beside does not hold it
    __device__ __forceinline__ Vec<R, V> above(const Vec<R, V>& x, R edge) const {
        Vec<R, V> y;
        const R next = lane_above(x[0]);
#pragma unroll
        for (int q = 0; q + 1 < V; ++q) y[q] = x[q + 1];
        y[V - 1] = hi ? (nz == V ? x[0] : edge) : next;
        return y;
    }
    __device__ __forceinline__ Vec<R, V> below(const Vec<R, V>& x, R edge) const {
        Vec<R, V> y;
        const R prev = lane_below(x[V - 1]);
#pragma unroll
        for (int q = V - 1; q > 0; --q) y[q] = x[q - 1];
        y[0] = lo ? (nz == V ? x[V - 1] : edge) : prev;
        return y;
    }
};

// E = D / eps_aa, eps_aa = (eps + eps[-e_a]) / 2
template <typename R, int V>
__device__ __forceinline__ Vec<R, V> e_vec(const Vec<R, V>& d, const Vec<R, V>& e, const Vec<R, V>& em) {
    Vec<R, V> y;
#pragma unroll
    for (int q = 0; q < V; ++q) y[q] = recip((e[q] + em[q]) / R(2)) * d[q];
    return y;
}

__device__ __forceinline__ float fused(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fused(double a, double b, double c) { return __builtin_fma(a, b, c); }

// 1 / v, rounded to nearest like the division (float32: two Newton steps on the
// hardware's estimate round correctly, Markstein 1990; compared with the
// division for every mantissa), and a / d by rd = 1 / d rounded to nearest.
// With divisions instead, a step at 256^3 takes 188 + 121 us.
__device__ __forceinline__ float recip_rn(float v) {
    float r = __builtin_amdgcn_rcpf(v);
    r = fused(fused(-v, r, 1.0f), r, r);
    r = fused(fused(-v, r, 1.0f), r, r);
    return __builtin_amdgcn_div_fixupf(r, v, 1.0f);
}
__device__ __forceinline__ double recip_rn(double v) { return 1.0 / v; }
template <typename R>
__device__ __forceinline__ R quot_rn(R a, R d, R rd) {
#pragma clang fp contract(off)
    R q = a * rd;
    q = fused(fused(-d, q, a), rd, q);
    return fused(fused(-d, q, a), rd, q);
}

// 1 / eps_aa
template <typename R, int V>
__device__ __forceinline__ Vec<R, V> inv_eps(const Vec<R, V>& e, const Vec<R, V>& em) {
    Vec<R, V> y;
#pragma unroll
    for (int q = 0; q < V; ++q) y[q] = recip_rn((e[q] + em[q]) / R(2));
    return y;
}

// PML profile values for the adjoint, b = sigma dt / (2 eps0) and r = 1 / (1 + b) of an axis.
// The coefficients of fdtd.py:272-311 separate into them: for a component
// with own axis a and the others b, c
//   m1 = (1 - b_b - b_c - b_b b_c) r_b r_c,  m2 = +-c0 dt r_b r_c,
//   m3 = 2 b_a m2,  m4 = -4 b_b b_c r_b r_c,
// and m1 = 1, m2 = +-c0 dt where sigma is zero.
template <typename R>
struct Pml1 {
    R b, r;
    __device__ __forceinline__ Pml1() {}
    __device__ __forceinline__ Pml1(R sigma, R half_dt) : b(sigma * half_dt) { r = recip(R(1) + b); }
};
template <typename R, int V>
struct PmlZ {
    R b[V], r[V];
    bool any;
    __device__ __forceinline__ void load(const R* sig, R half_dt) {
        any = false;
#pragma unroll
        for (int q = 0; q < V; ++q) {
            b[q] = sig[q] * half_dt;
            any = any || b[q] != R(0);
        }
    }
    __device__ __forceinline__ void recips() {
#pragma unroll
        for (int q = 0; q < V; ++q) r[q] = recip(R(1) + b[q]);
    }
};

// The axes of component a: its own and the two others' b and r at element q.
template <int A, typename R, int V>
__device__ __forceinline__ void pml_axes(const Pml1<R>& x, const Pml1<R>& y, const PmlZ<R, V>& z, int q, R& ba, R& bb,
                                         R& bc, R& r) {
    ba = A == 0 ? x.b : A == 1 ? y.b : z.b[q];
    bb = A == 0 ? y.b : x.b;
    bc = A == 2 ? y.b : z.b[q];
    r = (A == 0 ? y.r : x.r) * (A == 2 ? y.r : z.r[q]);
}

// One component's step u += curl ch of this thread's cells, with the
// reference's coefficients formed cell by cell (coef4) where a sigma is
// non-zero and i1, i2 (those of sigma = 0) elsewhere; sx, sy, sz the sigmas of
// the axes, sign -1 for H, +1 for D.  ic and iu (at this thread's cells)
// advance where their coefficient is non-zero.
// The roundings are written out (no contraction but the fused products named
// here): a field that a pulse leaves behind is static, its curl cancels and
// what remains of H is rounding, so that any other order of these operations
// gives another H in a few cells (up to 2e-11 of its rms in float64 and 9e-3
// in float32, over runs of 300 steps on grids of 28 to 200 cells a side).
template <int A, typename R, int V>
__device__ __forceinline__ void yee_update(const Fdtd<R>& f, R sign, R i1, R i2, R sx, R sy, const Vec<R, V>& sz,
                                           bool z_any, Vec<R, V>& u, const Vec<R, V>& ch, R* ic, R* iu, bool live) {
#pragma clang fp contract(off)
    const bool has_ic = A == 0 ? sx != R(0) : A == 1 ? sy != R(0) : z_any;
    const bool has_iu = A == 0 ? sy != R(0) && z_any : A == 1 ? sx != R(0) && z_any : sx != R(0) && sy != R(0);
    const YeeConst<R> k = f.yee;
    Vec<R, V> c1, c2;
    if (has_ic) c1 = ldv<R, V>(ic);
    if (has_iu) c2 = ldv<R, V>(iu);
#pragma unroll
    for (int q = 0; q < V; ++q) {
        const R sa = A == 0 ? sx : A == 1 ? sy : sz[q], sb = A == 0 ? sy : sx, sc = A == 2 ? sy : sz[q];
        // coef4, operation by operation
        const R s1 = quot_rn((sb + sc) / R(2), k.e0, k.inv_e0), s2 = quot_rn(sb * sc * k.dt / R(4), k.e2, k.inv_e2);
        const R im0 = recip_rn(k.inv_dt + s1 + s2), m2 = sign * im0 * k.c0;
        const R h = u[q], c = ch[q];
        R v = fused(im0 * (k.inv_dt - s1 - s2), h, m2 * c);
        if (has_ic && sa != R(0)) {
            c1[q] = c1[q] + c;
            v = fused(quot_rn(m2 * k.dt * sa, k.e0, k.inv_e0), c1[q], v);
        }
        if (has_iu && sb != R(0) && sc != R(0)) {
            c2[q] = c2[q] + h;
            v = fused(-im0 * k.dt * sb * sc / k.e2, c2[q], v);
        }
        u[q] = sa == R(0) && sb == R(0) && sc == R(0) ? fused(i2, c, i1 * h) : v;
    }
    if (live && has_ic) stv(ic, c1);
    if (live && has_iu) stv(iu, c2);
}

// the three components
template <typename R, int V>
__device__ __forceinline__ void yee_update3(const Fdtd<R>& f, R sign, R i1, R i2, R sx, R sy, const R* sig_z,
                                            Vec<R, V> (&u)[3], const Vec<R, V> (&ch)[3], R* ic, R* iu, bool live) {
#pragma clang fp contract(off)
    Vec<R, V> sz;
    bool z_any = false;
#pragma unroll
    for (int q = 0; q < V; ++q) {
        sz[q] = sig_z[q];
        z_any = z_any || sz[q] != R(0);
    }
    if (sx != R(0) || sy != R(0) || z_any) {
        yee_update<0>(f, sign, i1, i2, sx, sy, sz, z_any, u[0], ch[0], ic, iu, live);
        yee_update<1>(f, sign, i1, i2, sx, sy, sz, z_any, u[1], ch[1], ic + f.n, iu + f.n, live);
        yee_update<2>(f, sign, i1, i2, sx, sy, sz, z_any, u[2], ch[2], ic + 2 * f.n, iu + 2 * f.n, live);
    } else {
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int q = 0; q < V; ++q) u[a][q] = fused(i2, ch[a][q], i1 * u[a][q]);
    }
}

// ----------------------------------------------------------------- H phase
// H += curl E (fdtd.py:77-101) with E = D / eps_aa formed from D and eps.
template <typename R, int V>
__global__ void __launch_bounds__(256) k_h(Fdtd<R> f, const R* __restrict__ D) {
#pragma clang fp contract(off)
    const ZGroup<R, V> g(f, blockIdx.x);
    const int64_t n = f.n;
    const int i = g.i, j = g.j, ip = wrapp(i, f.nx), jp = wrapp(j, f.ny), im = wrapm(i, f.nx), jm = wrapm(j, f.ny);
    const int64_t l = g.line(i, j), c = l + g.k0, l_jp = g.line(i, jp), l_ip = g.line(ip, j);
    const R *eps = f.eps, *Dx = D, *Dy = D + n, *Dz = D + 2 * n;
    R* H = f.st + c;
    const Vec<R, V> e = ldv<R, V>(eps + c), e_im = ldv<R, V>(eps + g.line(im, j) + g.k0),
                    e_jm = ldv<R, V>(eps + g.line(i, jm) + g.k0), e_jp = ldv<R, V>(eps + l_jp + g.k0),
                    e_jpim = ldv<R, V>(eps + g.line(im, jp) + g.k0), e_ip = ldv<R, V>(eps + l_ip + g.k0),
                    e_ipjm = ldv<R, V>(eps + g.line(ip, jm) + g.k0);
    const Vec<R, V> dx = ldv<R, V>(Dx + c), dy = ldv<R, V>(Dy + c), dz = ldv<R, V>(Dz + c),
                    dx_jp = ldv<R, V>(Dx + l_jp + g.k0), dz_jp = ldv<R, V>(Dz + l_jp + g.k0),
                    dy_ip = ldv<R, V>(Dy + l_ip + g.k0), dz_ip = ldv<R, V>(Dz + l_ip + g.k0);
    Vec<R, V> h[3] = {ldv<R, V>(H), ldv<R, V>(H + n), ldv<R, V>(H + 2 * n)};
    R e_lo = R(0), e_jplo = R(0), e_iplo = R(0), ix_hi = R(0), iy_hi = R(0), dx_hi = R(0), dy_hi = R(0);
    if (g.nz != V) {
        if (g.lo) {
            e_lo = eps[l + g.klo];
            e_jplo = eps[l_jp + g.klo];
            e_iplo = eps[l_ip + g.klo];
        }
        if (g.hi) {
            const R eh = eps[l + g.khi];
            ix_hi = recip_rn((eh + eps[g.line(im, j) + g.khi]) / R(2));
            iy_hi = recip_rn((eh + eps[g.line(i, jm) + g.khi]) / R(2));
            dx_hi = Dx[l + g.khi];
            dy_hi = Dy[l + g.khi];
        }
    }
    const Vec<R, V> ix = inv_eps(e, e_im), iy = inv_eps(e, e_jm), iz = inv_eps(e, g.below(e, e_lo));
    const Vec<R, V> ix_jp = inv_eps(e_jp, e_jpim), iz_jp = inv_eps(e_jp, g.below(e_jp, e_jplo));
    const Vec<R, V> iy_ip = inv_eps(e_ip, e_ipjm), iz_ip = inv_eps(e_ip, g.below(e_ip, e_iplo));
    const Vec<R, V> ix_kp = g.above(ix, ix_hi), iy_kp = g.above(iy, iy_hi), dx_kp = g.above(dx, dx_hi),
                    dy_kp = g.above(dy, dy_hi);
    Vec<R, V> ce[3];   // curl_E, ceviche/derivatives.py:16-22 (forward differences, periodic)
#pragma unroll
    for (int q = 0; q < V; ++q) {
        const R ex = ix[q] * dx[q], ey = iy[q] * dy[q], ez = iz[q] * dz[q];
        ce[0][q] = (fused(iz_jp[q], dz_jp[q], -ez) - fused(iy_kp[q], dy_kp[q], -ey)) * f.inv_dL;
        ce[1][q] = (fused(ix_kp[q], dx_kp[q], -ex) - fused(iz_ip[q], dz_ip[q], -ez)) * f.inv_dL;
        ce[2][q] = (fused(iy_ip[q], dy_ip[q], -ey) - fused(ix_jp[q], dx_jp[q], -ex)) * f.inv_dL;
    }
    yee_update3(f, R(-1), f.h1, f.h2, sigH(f, 0)[i], sigH(f, 1)[j], sigH(f, 2) + g.k0, h, ce, H + 6 * n, H + 9 * n,
                g.live);
    if (!g.live) return;
    stv(H, h[0]);
    stv(H + n, h[1]);
    stv(H + 2 * n, h[2]);
}

// ------------------------------------------------- forward-mode H phase
// H update of cell c of the state f.st with E read through `E(a, i, j, k)`
// (the tangent E of a forward-mode step).
template <typename R, typename EGet>
__host__ __device__ __forceinline__ void h_cell_with(const Fdtd<R>& f, int64_t c, EGet E) {
    int i, j, k;
    decompose(f, c, i, j, k);
    const int64_t n = f.n;
    R* H = f.st;
    R* ICE = f.st + 6 * n;
    R* IH = f.st + 9 * n;
    const int ip = wrapp(i, f.nx), jp = wrapp(j, f.ny), kp = wrapp(k, f.nz);
    const R ex = E(0, i, j, k), ey = E(1, i, j, k), ez = E(2, i, j, k);
    R ce[3];
    // curl_E, ceviche/derivatives.py:16-22 (forward differences, periodic)
    ce[0] = ((E(2, i, jp, k) - ez) - (E(1, i, j, kp) - ey)) * f.inv_dL;
    ce[1] = ((E(0, i, j, kp) - ex) - (E(2, ip, j, k) - ez)) * f.inv_dL;
    ce[2] = ((E(1, ip, j, k) - ey) - (E(0, i, jp, k) - ex)) * f.inv_dL;
    const int pos[3] = {i, j, k};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int ax_b = (a == 0) ? 1 : 0;
        const int ax_c = (a == 2) ? 1 : 2;
        const R sa = sigH(f, a)[pos[a]], sb = sigH(f, ax_b)[pos[ax_b]], sc = sigH(f, ax_c)[pos[ax_c]];
        const int64_t ca = a * n + c;
        const R h = H[ca];
        R hn;
        if (sa == R(0) && sb == R(0) && sc == R(0)) {
            hn = f.h1 * h + f.h2 * ce[a];
        } else {
            R m1, m2, m3, m4;
            coef4<R>(sa, sb, sc, R(f.dt), R(f.c0), R(f.eps0), R(-1), m1, m2, m3, m4);
            hn = m1 * h + m2 * ce[a];
            if (sa != R(0)) {
                const R ice = ICE[ca] + ce[a];
                ICE[ca] = ice;
                hn += m3 * ice;
            }
            if (sb != R(0) && sc != R(0)) {
                const R ih = IH[ca] + h;
                IH[ca] = ih;
                hn += m4 * ih;
            }
        }
        H[ca] = hn;
    }
}

// tangent H update: ft.st is the tangent state, D the primal D of the same step
template <typename R>
__global__ void __launch_bounds__(256) k_h_tangent(Fdtd<R> ft, const R* __restrict__ D, const R* __restrict__ deps) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ft.n) return;
    const R* dD = ft.st + 3 * ft.n;
    h_cell_with(ft, c, [&](int a, int i, int j, int k) { return efield_tangent(ft, D, dD, deps, a, i, j, k); });
}

// ----------------------------------------------------------------- D phase
struct PointSrc {
    int comp;              // 0..2 = Jx, Jy, Jz; -1 none
    int64_t cell;
    double amp;
    const double* amp_dev; // the amplitude in device memory instead, or null
};

// D (read at Din, written at Dout: the same array or two) += curl H + sources
// (fdtd.py:102-132).
template <typename R, int V>
__global__ void __launch_bounds__(256) k_d(Fdtd<R> f, const R* Din, R* Dout, const R* __restrict__ Jx,
                                           const R* __restrict__ Jy, const R* __restrict__ Jz, R jscale, PointSrc ps) {
#pragma clang fp contract(off)
    const ZGroup<R, V> g(f, xcd_block(blockIdx.x, gridDim.x));
    const int64_t n = f.n;
    const int i = g.i, j = g.j;
    const int64_t l = g.line(i, j), c = l + g.k0, c_im = g.line(wrapm(i, f.nx), j) + g.k0,
                  c_jm = g.line(i, wrapm(j, f.ny)) + g.k0;
    const R *Hx = f.st, *Hy = f.st + n, *Hz = f.st + 2 * n;
    const Vec<R, V> hx = ldv<R, V>(Hx + c), hy = ldv<R, V>(Hy + c), hz = ldv<R, V>(Hz + c),
                    hx_jm = ldv<R, V>(Hx + c_jm), hz_jm = ldv<R, V>(Hz + c_jm), hy_im = ldv<R, V>(Hy + c_im),
                    hz_im = ldv<R, V>(Hz + c_im);
    Vec<R, V> d[3] = {ldv<R, V>(Din + c), ldv<R, V>(Din + n + c), ldv<R, V>(Din + 2 * n + c)};
    R hx_lo = R(0), hy_lo = R(0);
    if (g.lo && g.nz != V) {
        hx_lo = Hx[l + g.klo];
        hy_lo = Hy[l + g.klo];
    }
    const Vec<R, V> hx_km = g.below(hx, hx_lo), hy_km = g.below(hy, hy_lo);
    Vec<R, V> ch[3];   // curl_H, ceviche/derivatives.py:24-30 (backward differences, periodic)
#pragma unroll
    for (int q = 0; q < V; ++q) {
        ch[0][q] = ((hz[q] - hz_jm[q]) - (hy[q] - hy_km[q])) * f.inv_dL;
        ch[1][q] = ((hx[q] - hx_km[q]) - (hz[q] - hz_im[q])) * f.inv_dL;
        ch[2][q] = ((hy[q] - hy_im[q]) - (hx[q] - hx_jm[q])) * f.inv_dL;
    }
    R* aux = f.st + c;
    yee_update3(f, R(1), f.d1, f.d2, sigD(f, 0)[i], sigD(f, 1)[j], sigD(f, 2) + g.k0, d, ch, aux + 12 * n,
                aux + 15 * n, g.live);
    if (!g.live) return;
    const R* J[3] = {Jx, Jy, Jz};
    const int64_t at = ps.cell - c;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (J[a])
#pragma unroll
            for (int q = 0; q < V; ++q) d[a][q] = fused(jscale, J[a][c + q], d[a][q]);
        if (ps.comp == a && at >= 0 && at < V) {
            const R amp = R(ps.amp_dev ? *ps.amp_dev : ps.amp);
#pragma unroll
            for (int q = 0; q < V; ++q)
                if (at == q) d[a][q] += amp;
        }
        stv(Dout + a * n + c, d[a]);
    }
}

// ------------------------------------------------------------ probe record
// comp: 0..2 E, 3..5 D, 6..8 H
template <typename R>
__global__ void k_record(Fdtd<R> f, const int32_t* __restrict__ pcomp, const int64_t* __restrict__ pcell,
                         int np, R* __restrict__ out) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    const int comp = pcomp[p];
    const int64_t c = pcell[p];
    R v;
    if (comp < 3) {
        int i, j, k;
        decompose(f, c, i, j, k);
        v = efield(f, f.st + 3 * f.n, comp, i, j, k);
    } else if (comp < 6) {
        v = f.st[(int64_t)comp * f.n + c];
    } else {
        v = f.st[(int64_t)(comp - 6) * f.n + c];
    }
    out[p] = v;
}

// tangent probes: E comps from efield_tangent (primal D of f.st, tangent of
// ft.st), D / H comps straight from the tangent state
template <typename R>
__global__ void k_record_tangent(Fdtd<R> f, Fdtd<R> ft, const R* __restrict__ deps,
                                 const int32_t* __restrict__ pcomp, const int64_t* __restrict__ pcell, int np,
                                 R* __restrict__ out) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    const int comp = pcomp[p];
    const int64_t c = pcell[p];
    R v;
    if (comp < 3) {
        int i, j, k;
        decompose(f, c, i, j, k);
        v = efield_tangent(f, f.st + 3 * f.n, ft.st + 3 * f.n, deps, comp, i, j, k);
    } else if (comp < 6) {
        v = ft.st[(int64_t)comp * f.n + c];
    } else {
        v = ft.st[(int64_t)(comp - 6) * f.n + c];
    }
    out[p] = v;
}

// E = D / eps_aa for all cells (the E fields the reference returns)
template <typename R>
__global__ void __launch_bounds__(256) k_efields(Fdtd<R> f, R* __restrict__ E) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= f.n) return;
    int i, j, k;
    decompose(f, c, i, j, k);
#pragma unroll
    for (int a = 0; a < 3; ++a) E[a * f.n + c] = efield(f, f.st + 3 * f.n, a, i, j, k);
}

// ============================================================== adjoint
// Adjoint state lam (18 arrays, same layout) is the cotangent of the state
// after step t.  With the 1/dL of the curls folded into mu:
//   phase A:  muCH = (n2+n3) lamD + lamICH           (cells c, c+e)
//             T    = lamH + curlE(muCH)
//             lamICE = m3 T + lamICE;  lamIH = m4 T + lamIH;  lamH = m1 T + lamIH
//   phase B:  muCE = m2 T + lamICE                    (cells c, c-e)
//             q    = curlH(muCE)
//             lamID = n4 lamD + lamID; lamICH = n3 lamD + lamICH
//             lamD = n1 lamD + lamID + mE q;   g_mE += D_{t-1} q
// (m*: H coefficients, n*: D coefficients; curl_E^T = curl_H for periodic
// differences, so the adjoint is a time-reversed Yee step.)  T is stored (3
// arrays) only by groups with an H sigma; elsewhere m1 = 1 and lamH is T.

// m2' u + own-sigma integral: mu of component A at element q (cdt = +-c0 dt / dL).
// with_m3: the m3 u term as well (phase A; in phase B it is in the integral).
template <int A, bool WITH_M3, typename R, int V>
__device__ __forceinline__ Vec<R, V> mu_vec(const Fdtd<R>& f, const Pml1<R>& x, const Pml1<R>& y,
                                            const PmlZ<R, V>& z, R cdt, const Vec<R, V>& u, const R* ic) {
    const bool has_ic = A == 0 ? x.b != R(0) : A == 1 ? y.b != R(0) : z.any;
    Vec<R, V> i1, m;
    if (has_ic) i1 = ldv<R, V>(ic);
#pragma unroll
    for (int q = 0; q < V; ++q) {
        R ba, bb, bc, r;
        pml_axes<A>(x, y, z, q, ba, bb, bc, r);
        R w = cdt * r;
        if (WITH_M3) w += w * (R(2) * ba);
        m[q] = w * u[q];
        // the integral is only ever fed where the component's own sigma is non-zero
        if (has_ic && ba != R(0)) m[q] += i1[q] * f.inv_dL;
    }
    return m;
}

// the same for one cell (the neighbour of a group's edge)
template <int A, bool WITH_M3, typename R>
__device__ __forceinline__ R mu_one(const Fdtd<R>& f, R sx, R sy, R sz, R cdt, R u, const R* ic) {
    if (sx == R(0) && sy == R(0) && sz == R(0)) return cdt * u;
    const Pml1<R> x(sx, f.half_dt), y(sy, f.half_dt);
    PmlZ<R, 1> z;
    z.load(&sz, f.half_dt);
    z.recips();
    Vec<R, 1> v;
    v[0] = u;
    return mu_vec<A, WITH_M3, R, 1>(f, x, y, z, cdt, v, ic)[0];
}

template <int A, typename R, int V>
__device__ __forceinline__ void adj_h_update(const Pml1<R>& x, const Pml1<R>& y, const PmlZ<R, V>& z, R c0dt, Vec<R, V>& t,
                                             R* lam_h, R* lam_ic, R* lam_iu, R* T, bool live) {
    const bool has_ic = A == 0 ? x.b != R(0) : A == 1 ? y.b != R(0) : z.any;
    const bool has_iu = A == 0 ? y.b != R(0) && z.any : A == 1 ? x.b != R(0) && z.any : x.b != R(0) && y.b != R(0);
    Vec<R, V> i1, i2, h;
    if (has_ic) i1 = ldv<R, V>(lam_ic);
    if (has_iu) i2 = ldv<R, V>(lam_iu);
#pragma unroll
    for (int q = 0; q < V; ++q) {
        R ba, bb, bc, r;
        pml_axes<A>(x, y, z, q, ba, bb, bc, r);
        const R p = bb * bc;
        R v = ((R(1) - bb - bc - p) * r) * t[q];
        if (has_iu && p != R(0)) {
            i2[q] += (R(-4) * p * r) * t[q];
            v += i2[q];
        }
        if (has_ic && ba != R(0)) i1[q] += (c0dt * r * (R(2) * ba)) * t[q];
        h[q] = v;
    }
    if (!live) return;
    stv(T, t);
    stv(lam_h, h);
    if (has_ic) stv(lam_ic, i1);
    if (has_iu) stv(lam_iu, i2);
}

// Phase A.  g_src (may be null): lam(D_comp) at the source cell, the cotangent
// of the amplitude added at this step.
template <typename R, int V>
__global__ void __launch_bounds__(256) k_adj_a(Fdtd<R> f, R* __restrict__ lam, R* __restrict__ T, int src_comp,
                                               int64_t src_cell, R* __restrict__ g_src) {
    const ZGroup<R, V> g(f, xcd_block(blockIdx.x, gridDim.x));
    const int64_t n = f.n;
    const int i = g.i, j = g.j, ip = wrapp(i, f.nx), jp = wrapp(j, f.ny);
    const int64_t l = g.line(i, j), c = l + g.k0, c_jp = g.line(i, jp) + g.k0, c_ip = g.line(ip, j) + g.k0;
    const R *Lx = lam + 3 * n, *Ly = lam + 4 * n, *Lz = lam + 5 * n;
    const R* ICH = lam + 12 * n;
    const Vec<R, V> dx = ldv<R, V>(Lx + c), dy = ldv<R, V>(Ly + c), dz = ldv<R, V>(Lz + c),
                    dx_jp = ldv<R, V>(Lx + c_jp), dz_jp = ldv<R, V>(Lz + c_jp), dy_ip = ldv<R, V>(Ly + c_ip),
                    dz_ip = ldv<R, V>(Lz + c_ip);
    Vec<R, V> t[3] = {ldv<R, V>(lam + c), ldv<R, V>(lam + n + c), ldv<R, V>(lam + 2 * n + c)};
    if (g_src && g.live && src_cell >= c && src_cell < c + V) g_src[0] = lam[(3 + src_comp) * n + src_cell];
    const R sx = sigD(f, 0)[i], sx_ip = sigD(f, 0)[ip], sy = sigD(f, 1)[j], sy_jp = sigD(f, 1)[jp];
    const R* sz = sigD(f, 2);
    PmlZ<R, V> z;
    z.load(sz + g.k0, f.half_dt);
    Vec<R, V> mx, my, mz, mx_jp, mz_jp, my_ip, mz_ip;
    if (sx != R(0) || sx_ip != R(0) || sy != R(0) || sy_jp != R(0) || z.any) {
        z.recips();
        const Pml1<R> x(sx, f.half_dt), y(sy, f.half_dt), xp(sx_ip, f.half_dt), yp(sy_jp, f.half_dt);
        mx = mu_vec<0, true>(f, x, y, z, f.cdt, dx, ICH + c);
        my = mu_vec<1, true>(f, x, y, z, f.cdt, dy, ICH + n + c);
        mz = mu_vec<2, true>(f, x, y, z, f.cdt, dz, ICH + 2 * n + c);
        mx_jp = mu_vec<0, true>(f, x, yp, z, f.cdt, dx_jp, ICH + c_jp);
        mz_jp = mu_vec<2, true>(f, x, yp, z, f.cdt, dz_jp, ICH + 2 * n + c_jp);
        my_ip = mu_vec<1, true>(f, xp, y, z, f.cdt, dy_ip, ICH + n + c_ip);
        mz_ip = mu_vec<2, true>(f, xp, y, z, f.cdt, dz_ip, ICH + 2 * n + c_ip);
    } else {
#pragma unroll
        for (int q = 0; q < V; ++q) {
            mx[q] = f.cdt * dx[q];
            my[q] = f.cdt * dy[q];
            mz[q] = f.cdt * dz[q];
            mx_jp[q] = f.cdt * dx_jp[q];
            mz_jp[q] = f.cdt * dz_jp[q];
            my_ip[q] = f.cdt * dy_ip[q];
            mz_ip[q] = f.cdt * dz_ip[q];
        }
    }
    R mx_hi = R(0), my_hi = R(0);
    if (g.hi && g.nz != V) {
        const int64_t ch = l + g.khi;
        mx_hi = mu_one<0, true>(f, sx, sy, sz[g.khi], f.cdt, Lx[ch], ICH + ch);
        my_hi = mu_one<1, true>(f, sx, sy, sz[g.khi], f.cdt, Ly[ch], ICH + n + ch);
    }
    const Vec<R, V> mx_kp = g.above(mx, mx_hi), my_kp = g.above(my, my_hi);
#pragma unroll
    for (int q = 0; q < V; ++q) {   // curl_E of muCH (forward differences)
        t[0][q] += (mz_jp[q] - mz[q]) - (my_kp[q] - my[q]);
        t[1][q] += (mx_kp[q] - mx[q]) - (mz_ip[q] - mz[q]);
        t[2][q] += (my_ip[q] - my[q]) - (mx_jp[q] - mx[q]);
    }
    const R hx = sigH(f, 0)[i], hy = sigH(f, 1)[j];
    PmlZ<R, V> hz;
    hz.load(sigH(f, 2) + g.k0, f.half_dt);
    if (hx != R(0) || hy != R(0) || hz.any) {
        hz.recips();
        const Pml1<R> x(hx, f.half_dt), y(hy, f.half_dt);
        const R c0dt = -f.c0dt;
        R* at = lam + c;
        adj_h_update<0>(x, y, hz, c0dt, t[0], at, at + 6 * n, at + 9 * n, T + c, g.live);
        adj_h_update<1>(x, y, hz, c0dt, t[1], at + n, at + 7 * n, at + 10 * n, T + n + c, g.live);
        adj_h_update<2>(x, y, hz, c0dt, t[2], at + 2 * n, at + 8 * n, at + 11 * n, T + 2 * n + c, g.live);
    } else if (g.live) {
#pragma unroll
        for (int a = 0; a < 3; ++a) stv(lam + a * n + c, t[a]);
    }
}

template <int A, typename R, int V>
__device__ __forceinline__ void adj_d_update(const Pml1<R>& x, const Pml1<R>& y, const PmlZ<R, V>& z, R c0dt,
                                             Vec<R, V>& u, R* lam_ic, R* lam_iu, bool live) {
    const bool has_ic = A == 0 ? x.b != R(0) : A == 1 ? y.b != R(0) : z.any;
    const bool has_iu = A == 0 ? y.b != R(0) && z.any : A == 1 ? x.b != R(0) && z.any : x.b != R(0) && y.b != R(0);
    Vec<R, V> i1, i2;
    if (has_ic) i1 = ldv<R, V>(lam_ic);
    if (has_iu) i2 = ldv<R, V>(lam_iu);
#pragma unroll
    for (int q = 0; q < V; ++q) {
        R ba, bb, bc, r;
        pml_axes<A>(x, y, z, q, ba, bb, bc, r);
        const R p = bb * bc;
        R v = ((R(1) - bb - bc - p) * r) * u[q];
        if (has_iu && p != R(0)) {
            i2[q] += (R(-4) * p * r) * u[q];
            v += i2[q];
        }
        if (has_ic && ba != R(0)) i1[q] += (c0dt * r * (R(2) * ba)) * u[q];
        u[q] = v;
    }
    if (live && has_ic) stv(lam_ic, i1);
    if (live && has_iu) stv(lam_iu, i2);
}

// Phase B.
template <typename R, int V>
__global__ void __launch_bounds__(256) k_adj_b(Fdtd<R> f, R* __restrict__ lam, const R* __restrict__ T,
                                               const R* __restrict__ Dprev, R* __restrict__ gmE) {
    const ZGroup<R, V> g(f, xcd_block(blockIdx.x, gridDim.x));
    const int64_t n = f.n;
    const int i = g.i, j = g.j, im = wrapm(i, f.nx), jm = wrapm(j, f.ny);
    const int64_t l = g.line(i, j), c = l + g.k0, c_jm = g.line(i, jm) + g.k0, c_im = g.line(im, j) + g.k0;
    const R* ICE = lam + 6 * n;
    const R sx = sigH(f, 0)[i], sx_im = sigH(f, 0)[im], sy = sigH(f, 1)[j], sy_jm = sigH(f, 1)[jm];
    const R* sz = sigH(f, 2);
    PmlZ<R, V> z;
    z.load(sz + g.k0, f.half_dt);
    // T of a group: the stored one where it has a sigma, lamH elsewhere
    const R* t0 = sx != R(0) || sy != R(0) || z.any ? T : lam;
    const R* tj = sx != R(0) || sy_jm != R(0) || z.any ? T : lam;
    const R* ti = sx_im != R(0) || sy != R(0) || z.any ? T : lam;
    const Vec<R, V> hx = ldv<R, V>(t0 + c), hy = ldv<R, V>(t0 + n + c), hz = ldv<R, V>(t0 + 2 * n + c),
                    hx_jm = ldv<R, V>(tj + c_jm), hz_jm = ldv<R, V>(tj + 2 * n + c_jm),
                    hy_im = ldv<R, V>(ti + n + c_im), hz_im = ldv<R, V>(ti + 2 * n + c_im);
    const Vec<R, V> e = ldv<R, V>(f.eps + c), e_im = ldv<R, V>(f.eps + c_im), e_jm = ldv<R, V>(f.eps + c_jm);
    Vec<R, V> u[3] = {ldv<R, V>(lam + 3 * n + c), ldv<R, V>(lam + 4 * n + c), ldv<R, V>(lam + 5 * n + c)};
    Vec<R, V> dp[3], gm[3];
    if (gmE) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            dp[a] = ldv<R, V>(Dprev + a * n + c);
            gm[a] = ldv<R, V>(gmE + a * n + c);
        }
    }
    const R cdt = -f.cdt;
    Vec<R, V> ux, uy, uz, ux_jm, uz_jm, uy_im, uz_im;
    if (sx != R(0) || sx_im != R(0) || sy != R(0) || sy_jm != R(0) || z.any) {
        z.recips();
        const Pml1<R> x(sx, f.half_dt), y(sy, f.half_dt), xm(sx_im, f.half_dt), ym(sy_jm, f.half_dt);
        ux = mu_vec<0, false>(f, x, y, z, cdt, hx, ICE + c);
        uy = mu_vec<1, false>(f, x, y, z, cdt, hy, ICE + n + c);
        uz = mu_vec<2, false>(f, x, y, z, cdt, hz, ICE + 2 * n + c);
        ux_jm = mu_vec<0, false>(f, x, ym, z, cdt, hx_jm, ICE + c_jm);
        uz_jm = mu_vec<2, false>(f, x, ym, z, cdt, hz_jm, ICE + 2 * n + c_jm);
        uy_im = mu_vec<1, false>(f, xm, y, z, cdt, hy_im, ICE + n + c_im);
        uz_im = mu_vec<2, false>(f, xm, y, z, cdt, hz_im, ICE + 2 * n + c_im);
    } else {
#pragma unroll
        for (int q = 0; q < V; ++q) {
            ux[q] = cdt * hx[q];
            uy[q] = cdt * hy[q];
            uz[q] = cdt * hz[q];
            ux_jm[q] = cdt * hx_jm[q];
            uz_jm[q] = cdt * hz_jm[q];
            uy_im[q] = cdt * hy_im[q];
            uz_im[q] = cdt * hz_im[q];
        }
    }
    R ux_lo = R(0), uy_lo = R(0), e_lo = R(0);
    if (g.lo && g.nz != V) {
        const int64_t cl = l + g.klo;
        const R* tl = sx != R(0) || sy != R(0) || sz[g.klo] != R(0) ? T : lam;
        ux_lo = mu_one<0, false>(f, sx, sy, sz[g.klo], cdt, tl[cl], ICE + cl);
        uy_lo = mu_one<1, false>(f, sx, sy, sz[g.klo], cdt, tl[n + cl], ICE + n + cl);
        e_lo = f.eps[cl];
    }
    const Vec<R, V> ux_km = g.below(ux, ux_lo), uy_km = g.below(uy, uy_lo), e_km = g.below(e, e_lo);
    Vec<R, V> qv[3];   // curl_H of muCE (backward differences)
#pragma unroll
    for (int q = 0; q < V; ++q) {
        qv[0][q] = (uz[q] - uz_jm[q]) - (uy[q] - uy_km[q]);
        qv[1][q] = (ux[q] - ux_km[q]) - (uz[q] - uz_im[q]);
        qv[2][q] = (uy[q] - uy_im[q]) - (ux[q] - ux_jm[q]);
    }
    const R dx = sigD(f, 0)[i], dy = sigD(f, 1)[j];
    PmlZ<R, V> dz;
    dz.load(sigD(f, 2) + g.k0, f.half_dt);
    if (dx != R(0) || dy != R(0) || dz.any) {
        dz.recips();
        const Pml1<R> x(dx, f.half_dt), y(dy, f.half_dt);
        R* at = lam + c;
        adj_d_update<0>(x, y, dz, f.c0dt, u[0], at + 12 * n, at + 15 * n, g.live);
        adj_d_update<1>(x, y, dz, f.c0dt, u[1], at + 13 * n, at + 16 * n, g.live);
        adj_d_update<2>(x, y, dz, f.c0dt, u[2], at + 14 * n, at + 17 * n, g.live);
    }
    if (!g.live) return;
    const Vec<R, V> em[3] = {e_im, e_jm, e_km};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const Vec<R, V> w = e_vec(qv[a], e, em[a]);
#pragma unroll
        for (int q = 0; q < V; ++q) u[a][q] += w[q];
        stv(lam + (3 + a) * n + c, u[a]);
        if (gmE) {
#pragma unroll
            for (int q = 0; q < V; ++q) gm[a][q] += dp[a][q] * qv[a][q];
            stv(gmE + a * n + c, gm[a]);
        }
    }
}

// Probe cotangent injection: lam(comp, cell) += g[p]; for E probes also
// lamD += mE g and g_mE += D_t g.  One thread per probe; atomics make
// repeated (comp, cell) pairs accumulate.
template <typename R>
__global__ void k_inject(Fdtd<R> f, R* __restrict__ lam, const int32_t* __restrict__ pcomp,
                         const int64_t* __restrict__ pcell, int np, const R* __restrict__ g,
                         const R* __restrict__ Dt, R* __restrict__ gmE) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    const int comp = pcomp[p];
    const int64_t c = pcell[p];
    const R gv = g[p];
    if (comp < 3) {
        int i, j, k;
        decompose(f, c, i, j, k);
        int64_t cm;
        if (comp == 0) cm = cell(f, wrapm(i, f.nx), j, k);
        else if (comp == 1) cm = cell(f, i, wrapm(j, f.ny), k);
        else cm = cell(f, i, j, wrapm(k, f.nz));
        const R mE = R(1) / ((f.eps[c] + f.eps[cm]) / R(2));
        atomicAdd(&lam[(3 + comp) * f.n + c], mE * gv);
        if (gmE) atomicAdd(&gmE[comp * f.n + c], Dt[comp * f.n + c] * gv);
    } else if (comp < 6) {
        atomicAdd(&lam[(int64_t)comp * f.n + c], gv);
    } else {
        atomicAdd(&lam[(int64_t)(comp - 6) * f.n + c], gv);
    }
}

// g_eps from g_mE: mE_a = 1/eps_aa, eps_aa = (eps + roll(eps, 1, a))/2
//   g_eps[c] += sum_a 1/2 (g_aa[c] + g_aa[c + e_a]),  g_aa = -mE_a^2 g_mE_a
template <typename R>
__global__ void __launch_bounds__(256) k_eps_grad(Fdtd<R> f, const R* __restrict__ gmE, R* __restrict__ geps) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= f.n) return;
    int i, j, k;
    decompose(f, c, i, j, k);
    auto gaa = [&](int a, int ii, int jj, int kk) -> R {
        const int64_t cc = cell(f, ii, jj, kk);
        int64_t cm;
        if (a == 0) cm = cell(f, wrapm(ii, f.nx), jj, kk);
        else if (a == 1) cm = cell(f, ii, wrapm(jj, f.ny), kk);
        else cm = cell(f, ii, jj, wrapm(kk, f.nz));
        const R mE = R(1) / ((f.eps[cc] + f.eps[cm]) / R(2));
        return -mE * mE * gmE[a * f.n + cc];
    };
    R g = R(0.5) * (gaa(0, i, j, k) + gaa(0, wrapp(i, f.nx), j, k));
    g += R(0.5) * (gaa(1, i, j, k) + gaa(1, i, wrapp(j, f.ny), k));
    g += R(0.5) * (gaa(2, i, j, k) + gaa(2, i, j, wrapp(k, f.nz)));
    geps[c] += g;
}

// Reverse of E = D / eps_aa for a dense cotangent gE[3][n]:
//   gD[a] += mE_a gE[a],  g_mE[a] += D[a] gE[a]
template <typename R>
__global__ void __launch_bounds__(256) k_efields_grad(Fdtd<R> f, const R* __restrict__ gE, R* __restrict__ gD,
                                                      R* __restrict__ gmE) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= f.n) return;
    int i, j, k;
    decompose(f, c, i, j, k);
    const int64_t cm[3] = {cell(f, wrapm(i, f.nx), j, k), cell(f, i, wrapm(j, f.ny), k), cell(f, i, j, wrapm(k, f.nz))};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const R g = gE[a * f.n + c];
        const R mE = R(1) / ((f.eps[c] + f.eps[cm[a]]) / R(2));
        gD[a * f.n + c] += mE * g;
        if (gmE) gmE[a * f.n + c] += f.st[(3 + a) * f.n + c] * g;
    }
}

// ================================================ 2D TM temporal blocking
// Temporally blocked Yee update for nz == 1 with only Hx, Hy, Dz live (TM
// drive: Jz point source, TE fields zero), and its reverse-time adjoint.  One
// workgroup of WV waves owns a region of RR = WV*RPT rows (x) by 64 columns
// (y, contiguous): lane = column, each wave a band of RPT rows, all values of
// a cell in registers.  A neighbour along y is the next lane (DPP wave
// shift), a neighbour along x the next register, and only the rows where two
// waves meet go through LDS (one row of Ez and one of Hy per wave and step).
// TS steps are advanced per launch; after TS steps the cells at least TS away
// from the region edge are exact (the dependency cone of one step is one cell
// on each side, in either direction of time), so the owned tile is the region
// minus a TS-wide halo.  Region loads use periodic indices, which also makes
// small domains exact; what enters at the region's outer edge is zero.
//
// Bound: vector instructions of the region (halo included) on the one
// workgroup a CU holds.  Tiles without PML run a loop of 10 vector operations
// per cell and step, tiles with PML one of 18.  400 x 400 float32 in 16-step
// launches: 18.2 us a launch (0.7 us a step over a prologue of 6.5 us; 25.8
// us with every neighbour through LDS, 30 operations a cell and an amplitude
// load in each step).
struct TmProbes {
    const int32_t* comp;       // 2 Ez, 6 Hx, any other Hy
    const int64_t* cell;       // flat cells
    int n;
};

// The six arrays a TM state is made of.
template <typename R>
struct TmState {
    R *hx, *hy, *dz, *icex, *icey, *idz;
};

template <typename R>
struct TmArgs {
    int nx, ny;
    int tiles_x, tiles_y;      // tile grid
    int t0, nsteps;            // first global step of this launch, steps (<= TS)
    int src_i, src_j;          // source cell, src_i = -1: none
    R inv_dL, dL;
    R cdt;                     // c0 dt / dL
    R half_dt;                 // dt / (2 eps0)
    const R* sig;
    const R* eps;
    TmState<R> in, out;        // distinct buffers
    const double* amp;         // amplitude per global step
    TmProbes probes;
    R* rec;                    // (steps, np), row t - rec_t0
    int rec_t0;
    R* hist;                   // Dz after step t0 + s at hist + s * n, or null
    // adjoint only: in / out hold the cotangent of the state after / before the steps
    const R* dz_hist;          // Dz after step t0 + s at dz_hist + s * n
    const R* dz_before;        // Dz before step t0
    R* gm;                     // accumulated cotangent of 1 / eps_zz
    const R* grec;             // cotangent of rec, row t (global step), or null
    R* gamp;                   // cotangent of the amplitude of global step t, or null
};

__host__ __device__ __forceinline__ int pmod(int a, int n) {
    int r = a % n;
    return r < 0 ? r + n : r;
}

constexpr int kTmConfigs = 12;
constexpr int kTmMaxProbes = 256;
constexpr unsigned short kTmNoProbe = 0xffff;

// Probes inside a tile's region.  tm_probe_slots enters every probe whose cell
// lies in the region (in each of its periodic copies) into s_slot[component][row][column];
// of several probes of one component and cell the last one is entered and
// s_next leads to the one before it.  Returns (uniformly) whether there is any.
template <int RR, int NT>
__device__ __forceinline__ bool tm_probe_slots(const TmProbes& pr, int nx, int ny, int i0, int j0,
                                               unsigned short (*s_slot)[RR][64], unsigned short* s_next, int* s_any) {
    // component, row and column of each probe in the region (kTmNoProbe: none):
    // the search for probes of one cell reads these, 8 at a time (reading comp
    // and cell of 240 probes one after the other took 50 us a launch)
    __shared__ __attribute__((aligned(16))) unsigned short s_key[kTmMaxProbes];
    static_assert(RR <= 64, "6 bits per row");
    if (pr.n == 0) return false;
    if (threadIdx.x == 0) *s_any = 0;
    __syncthreads();
    int pi = 0, pj = 0, kk = 0;
    unsigned key = kTmNoProbe;
    bool mine = false;
    const int p = threadIdx.x;
    static_assert(NT >= kTmMaxProbes, "one thread per probe");
    if (p < pr.n) {
        const int64_t c = pr.cell[p];
        if ((uint64_t)c <= 0xffffffffull) {   // a 64-bit division is a long sequence
            pi = (int)((uint32_t)c / (uint32_t)ny);
            pj = (int)((uint32_t)c - (uint32_t)pi * (uint32_t)ny);
        } else {
            pi = (int)(c / ny);
            pj = (int)(c - (int64_t)pi * ny);
        }
        const int r = pmod(pi - i0, nx), col = pmod(pj - j0, ny), k = pr.comp[p];
        // a cell outside the grid is no tile's; s_slot has three components
        mine = (uint64_t)c < (uint64_t)((int64_t)nx * ny) && r < RR && col < 64;
        kk = k == 2 ? 0 : k == 6 ? 1 : 2;
        if (mine) {
            *s_any = 1;
            key = (unsigned)(kk << 12 | r << 6 | col);
        }
    }
    if (p < kTmMaxProbes) s_key[p] = (unsigned short)key;
    __syncthreads();
    if (!*s_any) return false;   // uniform
    for (int q = threadIdx.x; q < 3 * RR * 64; q += NT) (&s_slot[0][0][0])[q] = kTmNoProbe;
    __syncthreads();
    auto enter = [&] {
        for (int r = pmod(pi - i0, nx); r < RR; r += nx)
            for (int col = pmod(pj - j0, ny); col < 64; col += ny) s_slot[kk][r][col] = (unsigned short)p;
    };
    if (mine) {
        s_next[p] = kTmNoProbe;
        enter();
    }
    __syncthreads();
    const bool other = mine && s_slot[kk][pmod(pi - i0, nx)][pmod(pj - j0, ny)] != p;
    if (!__syncthreads_or(other)) return true;   // one probe per cell: no search
    if (mine) {
        int before = kTmNoProbe;
        bool head = true;
        for (int m = 0; m < pr.n; m += 8) {
            const uint4 v = *reinterpret_cast<const uint4*>(s_key + m);
            const unsigned word[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int h = 0; h < 8; ++h) {
                const bool same = ((word[h / 2] >> (16 * (h & 1))) & 0xffffu) == key;
                if (same && m + h < p) before = m + h;
                if (same && m + h > p) head = false;
            }
        }
        s_next[p] = (unsigned short)before;
        if (head) enter();
    }
    __syncthreads();
    return true;
}

// v modulo n for -n < v < 2 n without a division; tiles reach beyond the grid
// by less than 64 cells, so that holds for every n >= 64.
__device__ __forceinline__ int tm_wrap(int v, int n) {
    if (n < 64) return pmod(v, n);   // uniform
    v += v < 0 ? n : 0;
    return v - (v >= n ? n : 0);
}

// Geometry and coefficients of this thread's cells.  With b = sigma dt / (2
// eps0) the coefficients of fdtd.py:272-311 separate by axis, 1/m0 = dt /
// ((1 + b_b)(1 + b_c)), so two divisions per row and two per column serve
// every cell; where sigma is zero m1 is 1 and m2 is c0 dt exactly.  The 1/dL
// of the curls is folded into m2 and the own sigma's term is factored out:
//   Hx = xa hx + xb (dEz_y + kx icx), xa, xb of the column, kx of the row
//   Hy = ya hy + yb (dEz_x + ky icy), ya, yb of the row, ky of the column
//   Dz = da dz + db dH + dc idz
// with undivided differences dE, dH.  Rows are uniform over the wave and
// kept in scalar registers.
template <typename R, int RPT>
struct TmCells {
    int gi[RPT], gj;
    R shx[RPT], shy, sdx[RPT], sdy;
    R xa, xb, ky, ya[RPT], yb[RPT], kx[RPT];
    R da[RPT], db[RPT], dc[RPT], me[RPT];
    bool pml;   // any sigma of this thread's cells is non-zero

    // base[cell]: the row is uniform over the wave, so the address is a scalar
    // row pointer plus one vector offset for all rows
    template <typename P>
    __device__ __forceinline__ P& at(P* base, int q, int ny) const {
        return (base + (int64_t)gi[q] * ny)[(uint32_t)gj];
    }
    __device__ __forceinline__ bool has_idz(int q) const { return sdx[q] != R(0) && sdy != R(0); }

    // The prologue is paid once per launch by every wave of the CU, so it
    // issues its loads before anything waits, wraps indices without divisions
    // and forms the PML coefficients only where a sigma is non-zero.
    __device__ __forceinline__ void place(const TmArgs<R>& a, int row0, int col) {
        gj = tm_wrap(col, a.ny);
#pragma unroll
        for (int q = 0; q < RPT; ++q) gi[q] = __builtin_amdgcn_readfirstlane(tm_wrap(row0 + q, a.nx));
        // rows through scalar loads (constant address space)
        using csig_t = const __attribute__((address_space(4))) R*;
        const csig_t csig = (csig_t)a.sig;
        shy = a.sig[a.nx + gj];
        sdy = a.sig[2 * a.nx + a.ny + 1 + gj];
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            shx[q] = csig[gi[q]];
            sdx[q] = csig[a.nx + a.ny + 1 + gi[q]];
            me[q] = at(a.eps, q, a.ny);
        }
    }

    __device__ __forceinline__ void init(const TmArgs<R>& a) {
        R cy = R(0), ry = R(1);
        xa = R(1); xb = -a.cdt; ky = R(0);
        pml = shy != R(0) || sdy != R(0);
        if (pml) {
            const R by = shy * a.half_dt;
            cy = sdy * a.half_dt;
            ry = R(1) / (R(1) + cy);
            const R h = R(1) / (R(1) + by);
            xa = (R(1) - by) * h;
            xb = -a.cdt * h;
            ky = R(2) * by * a.dL;
        }
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            R cx_ = R(0), rx = R(1);
            ya[q] = R(1); yb[q] = -a.cdt; kx[q] = R(0);
            if (shx[q] != R(0) || sdx[q] != R(0)) {   // uniform
                pml = true;
                const R bx = shx[q] * a.half_dt;
                cx_ = sdx[q] * a.half_dt;
                rx = R(1) / (R(1) + cx_);
                const R h = R(1) / (R(1) + bx);
                ya[q] = uniform((R(1) - bx) * h);
                yb[q] = uniform(-a.cdt * h);
                kx[q] = uniform(R(2) * bx * a.dL);
            }
            const R r = rx * ry, cc = cx_ * cy;
            da[q] = (R(1) - cx_ - cy - cc) * r;
            db[q] = a.cdt * r;
            dc[q] = R(-4) * cc * r;
            me[q] = recip(me[q]);
        }
    }
};

// Tile of this workgroup: XCD-aware order, consecutive workgroups go to
// different XCDs, so each XCD gets a contiguous run of tiles (halos re-read
// from its own L2).
__device__ __forceinline__ void tm_tile(int tiles_y, int& ti, int& tj) {
    const int nb = gridDim.x;
    int b = blockIdx.x;
    if ((nb & 7) == 0) b = (b & 7) * (nb >> 3) + (b >> 3);
    ti = b / tiles_y;
    tj = b - ti * tiles_y;
}

template <typename R, int WV, int RPT, int TS>
__global__ void __launch_bounds__(64 * WV) k_tm_block(TmArgs<R> a) {
    constexpr int RR = WV * RPT;
    constexpr int NT = 64 * WV;
    constexpr int OX = RR - 2 * TS, OY = 64 - 2 * TS;  // owned tile
    __shared__ R sEz[WV + 1][64];   // Ez of each wave's first row
    __shared__ R sHy[WV + 1][64];   // new Hy of each wave's last row, at [wave + 1]
    __shared__ unsigned short s_slot[3][RR][64];
    __shared__ unsigned short s_next[kTmMaxProbes];
    __shared__ int s_any;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int ti, tj;
    tm_tile(a.tiles_y, ti, tj);
    const int i0 = ti * OX, j0 = tj * OY;
    const int nx = a.nx, ny = a.ny;
    const int64_t n = (int64_t)nx * ny;
    TmCells<R, RPT> g;
    g.place(a, i0 - TS + w * RPT, j0 - TS + lane);
    // Tiles read their halo from `in` and write only their owned cells to
    // `out`: a tile that finishes early never changes what a later tile of
    // the same launch reads.
    R hx[RPT], hy[RPT], dz[RPT], ez[RPT], icx[RPT], icy[RPT], idz[RPT];
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        hx[q] = g.at(a.in.hx, q, ny);
        hy[q] = g.at(a.in.hy, q, ny);
        dz[q] = g.at(a.in.dz, q, ny);
    }
    bool own[RPT], any_own = false;
    const int oj = lane - TS;
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        icx[q] = g.shx[q] != R(0) ? g.at(a.in.icex, q, ny) : R(0);
        icy[q] = g.shy != R(0) ? g.at(a.in.icey, q, ny) : R(0);
        idz[q] = g.has_idz(q) ? g.at(a.in.idz, q, ny) : R(0);
        const int oi = w * RPT + q - TS;
        own[q] = oj >= 0 && oj < OY && j0 + oj < ny && oi >= 0 && oi < OX && i0 + oi < nx;
        any_own = any_own || own[q];
    }
    g.init(a);
#pragma unroll
    for (int q = 0; q < RPT; ++q) ez[q] = g.me[q] * dz[q];
    const bool probes = tm_probe_slots<RR, NT>(a.probes, nx, ny, i0 - TS, j0 - TS, s_slot, s_next, &s_any);
    // (row, component) pairs of this wave that hold a probe of an owned cell
    uint64_t pmask = 0;
    if (probes) {
#pragma unroll
        for (int q = 0; q < RPT; ++q)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                if (!own[q]) s_slot[k][w * RPT + q][lane] = kTmNoProbe;   // this thread's entry only
                if (__ballot(s_slot[k][w * RPT + q][lane] != kTmNoProbe)) pmask |= 1ull << (q * 3 + k);
            }
    }
    // Ez probes: each row's last probe, and the rows with a cell of several
    int last_ez[RPT];
    unsigned several = 0;
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        last_ez[q] = probes ? s_slot[0][w * RPT + q][lane] : kTmNoProbe;
        if (__ballot(last_ez[q] != kTmNoProbe && s_next[last_ez[q] & (kTmMaxProbes - 1)] != kTmNoProbe))
            several |= 1u << q;
    }
    const int src_i = a.src_i, src_j = a.src_j;
    bool src_row = false;   // the source's row is one of this wave's
#pragma unroll
    for (int q = 0; q < RPT; ++q) src_row = src_row || g.gi[q] == src_i;
    // the launch's amplitudes, one per lane: a load inside the time loop would
    // hold up every step of the source's tile
    static_assert(TS <= 64, "one lane per step");
    const R amps = src_row && lane < a.nsteps ? R(a.amp[a.t0 + lane]) : R(0);
    sEz[w][lane] = ez[0];
    if (w == 0) {
        sEz[WV][lane] = R(0);
        sHy[0][lane] = R(0);
    }
    const bool pml = __syncthreads_or(g.pml);

    const R inv = a.inv_dL, cdt = a.cdt;
    auto run = [&](auto with_pml) {
        constexpr bool PML = decltype(with_pml)::value;
        for (int s = 0; s < a.nsteps; ++s) {
            const int t = a.t0 + s;
            // ---- H update: CEx = (Ez[j+1] - Ez)/dL, CEy = -(Ez[i+1] - Ez)/dL
            const R ez_next = sEz[w + 1][lane];
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const R dx = lane_above(ez[q]) - ez[q];
                const R dy = ez[q] - (q + 1 < RPT ? ez[q + 1 < RPT ? q + 1 : q] : ez_next);
                if constexpr (PML) {
                    icx[q] += dx * inv;
                    icy[q] += dy * inv;
                    hx[q] = g.xa * hx[q] + g.xb * (dx + g.kx[q] * icx[q]);
                    hy[q] = g.ya[q] * hy[q] + g.yb[q] * (dy + g.ky * icy[q]);
                } else {
                    hx[q] -= cdt * dx;
                    hy[q] -= cdt * dy;
                }
            }
            sHy[w + 1][lane] = hy[RPT - 1];
            __syncthreads();
            // ---- D update: CHz = (Hy - Hy[i-1])/dL - (Hx - Hx[j-1])/dL
            const R hy_prev = sHy[w][lane];
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const R dh = (hy[q] - (q > 0 ? hy[q > 0 ? q - 1 : 0] : hy_prev)) - (hx[q] - lane_below(hx[q]));
                if constexpr (PML) {
                    idz[q] += dz[q];
                    dz[q] = g.da[q] * dz[q] + g.db[q] * dh;
                    dz[q] += g.dc[q] * idz[q];
                } else {
                    dz[q] += cdt * dh;
                }
            }
            if (src_row) {
                const R amp = read_lane(amps, s);
#pragma unroll
                for (int q = 0; q < RPT; ++q)
                    if (g.gi[q] == src_i && g.gj == src_j) dz[q] += amp;
            }
#pragma unroll
            for (int q = 0; q < RPT; ++q) ez[q] = g.me[q] * dz[q];
            sEz[w][lane] = ez[0];
            if (a.hist && any_own) {
                R* hs = a.hist + (int64_t)s * n;
#pragma unroll
                for (int q = 0; q < RPT; ++q)
                    if (own[q]) g.at(hs, q, ny) = dz[q];
            }
            if (pmask) {
                R* row = a.rec + (int64_t)(t - a.rec_t0) * a.probes.n;
#pragma unroll
                for (int q = 0; q < RPT; ++q)
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        if (!(pmask >> (q * 3 + k) & 1)) continue;
                        const R v = k == 0 ? ez[q] : k == 1 ? hx[q] : hy[q];
                        if (k == 0) {
                            const int last = last_ez[q];
                            if (last != kTmNoProbe) row[last] = v;
                            if (several >> q & 1)
                                for (int p = last != kTmNoProbe ? s_next[last] : last; p != kTmNoProbe; p = s_next[p])
                                    row[p] = v;
                            continue;
                        }
                        for (int p = s_slot[k][w * RPT + q][lane]; p != kTmNoProbe; p = s_next[p]) row[p] = v;
                    }
            }
            __syncthreads();
        }
    };
    if (pml) run(std::true_type{});
    else run(std::false_type{});
    // ---- store the owned tile
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        if (!own[q]) continue;
        g.at(a.out.hx, q, ny) = hx[q];
        g.at(a.out.hy, q, ny) = hy[q];
        g.at(a.out.dz, q, ny) = dz[q];
        if (g.shx[q] != R(0)) g.at(a.out.icex, q, ny) = icx[q];
        if (g.shy != R(0)) g.at(a.out.icey, q, ny) = icy[q];
        if (g.has_idz(q)) g.at(a.out.idz, q, ny) = idz[q];
    }
}

// Reverse-time counterpart of k_tm_block: steps t0 + nsteps - 1 down to t0 of
// the discrete adjoint (k_adj_a / k_adj_b restricted to Hx, Hy, Dz; the TE
// components of a TM run are zero, so their cotangents reach neither eps nor
// the amplitude).  Per step: the cotangents of that step's probes are added,
// the amplitude's cotangent is read, then
//   muCH = n2 lamD;  T = lamH + curlE(muCH);  lamICE += m3 T;  lamH = m1 T
//   muCE = m2 T + lamICE;  q = curlH(muCE)   (muCH and muCE divided by dL)
//   lamID += n4 lamD;  lamD = n1 lamD + lamID + mE q;  g_mE += D_{t-1} q.
// D_{t-1} of the owned cells comes from the history that k_tm_block wrote.
// 26 us per 16 steps at 400 x 400 float32; the whole gradient of a 2000-step
// run takes 8.2 ms (126 ms with one-step launches of the general kernels and
// a copy of D between them).
template <typename R, int WV, int RPT, int TS>
__global__ void __launch_bounds__(64 * WV) k_tm_adjoint(TmArgs<R> a) {
    constexpr int RR = WV * RPT;
    constexpr int NT = 64 * WV;
    constexpr int OX = RR - 2 * TS, OY = 64 - 2 * TS;
    __shared__ R sMz[WV + 1][64];   // muCHz of each wave's first row
    __shared__ R sUy[WV + 1][64];   // muCEy of each wave's last row, at [wave + 1]
    __shared__ unsigned short s_slot[3][RR][64];
    __shared__ unsigned short s_next[kTmMaxProbes];
    __shared__ int s_any;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int ti, tj;
    tm_tile(a.tiles_y, ti, tj);
    const int i0 = ti * OX, j0 = tj * OY;
    const int nx = a.nx, ny = a.ny;
    const int64_t n = (int64_t)nx * ny;
    TmCells<R, RPT> g;
    g.place(a, i0 - TS + w * RPT, j0 - TS + lane);
    R hx[RPT], hy[RPT], dz[RPT], icx[RPT], icy[RPT], idz[RPT], gm[RPT], dn[RPT];
    bool own[RPT], any_own = false;
    const int oj = lane - TS;
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        hx[q] = g.at(a.in.hx, q, ny);
        hy[q] = g.at(a.in.hy, q, ny);
        dz[q] = g.at(a.in.dz, q, ny);
        const int oi = w * RPT + q - TS;
        own[q] = oj >= 0 && oj < OY && j0 + oj < ny && oi >= 0 && oi < OX && i0 + oi < nx;
        any_own = any_own || own[q];
        gm[q] = own[q] ? g.at(a.gm, q, ny) : R(0);
        dn[q] = own[q] ? g.at(a.dz_hist + (int64_t)(a.nsteps - 1) * n, q, ny) : R(0);   // Dz after the last step
    }
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        icx[q] = g.shx[q] != R(0) ? g.at(a.in.icex, q, ny) : R(0);
        icy[q] = g.shy != R(0) ? g.at(a.in.icey, q, ny) : R(0);
        idz[q] = g.has_idz(q) ? g.at(a.in.idz, q, ny) : R(0);
    }
    g.init(a);
    // cotangents enter in the halo as well, so every cell of the region keeps its slot
    const bool probes =
        a.grec && tm_probe_slots<RR, NT>(a.probes, nx, ny, i0 - TS, j0 - TS, s_slot, s_next, &s_any);
    uint64_t pmask = 0;
    if (probes) {
#pragma unroll
        for (int q = 0; q < RPT; ++q)
#pragma unroll
            for (int k = 0; k < 3; ++k)
                if (__ballot(s_slot[k][w * RPT + q][lane] != kTmNoProbe)) pmask |= 1ull << (q * 3 + k);
    }
    const int src_i = a.gamp ? a.src_i : -1, src_j = a.src_j;
    bool src_row = false;
#pragma unroll
    for (int q = 0; q < RPT; ++q) src_row = src_row || g.gi[q] == src_i;
    if (w == 0) {
        sMz[WV][lane] = R(0);
        sUy[0][lane] = R(0);
    }
    const bool pml = __syncthreads_or(g.pml);

    const R inv = a.inv_dL, cdt = a.cdt;
    auto run = [&](auto with_pml) {
        constexpr bool PML = decltype(with_pml)::value;
        // Ez-probe cotangent of each row's cell (its last probe), loaded a step ahead
        R pre[RPT];
        auto fetch = [&](int t) {
            const R* row = a.grec + (int64_t)t * a.probes.n;
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                if (!(pmask >> (3 * q) & 1)) continue;
                const int p = s_slot[0][w * RPT + q][lane];
                pre[q] = p != kTmNoProbe ? row[p] : R(0);
            }
        };
        auto inject = [&](int t) {
            const R* row = a.grec + (int64_t)t * a.probes.n;
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                if (pmask >> (3 * q) & 1) {
                    const int head = s_slot[0][w * RPT + q][lane];
                    R v = pre[q];
                    if (head != kTmNoProbe)
                        for (int p = s_next[head]; p != kTmNoProbe; p = s_next[p]) v += row[p];
                    dz[q] += g.me[q] * v;
                    gm[q] += dn[q] * v;
                }
                if (pmask >> (3 * q + 1) & 1)
                    for (int p = s_slot[1][w * RPT + q][lane]; p != kTmNoProbe; p = s_next[p]) hx[q] += row[p];
                if (pmask >> (3 * q + 2) & 1)
                    for (int p = s_slot[2][w * RPT + q][lane]; p != kTmNoProbe; p = s_next[p]) hy[q] += row[p];
            }
        };
        R dp[RPT];   // Dz before the step, loaded while the step before it runs
        auto load_dp = [&](int s) {
            if (!any_own) return;
            const R* hs = s > 0 ? a.dz_hist + (int64_t)(s - 1) * n : a.dz_before;
#pragma unroll
            for (int q = 0; q < RPT; ++q) dp[q] = own[q] ? g.at(hs, q, ny) : R(0);
        };
        if (pmask) fetch(a.t0 + a.nsteps - 1);
        load_dp(a.nsteps - 1);
        for (int s = a.nsteps - 1; s >= 0; --s) {
            const int t = a.t0 + s;
            if (pmask) {
                inject(t);
                if (s > 0) fetch(t - 1);
            }
            if (src_row) {
#pragma unroll
                for (int q = 0; q < RPT; ++q)
                    if (own[q] && g.gi[q] == src_i && g.gj == src_j) a.gamp[t] = dz[q];
            }
            R mz[RPT];
#pragma unroll
            for (int q = 0; q < RPT; ++q) mz[q] = (PML ? g.db[q] : cdt) * dz[q];
            sMz[w][lane] = mz[0];
            __syncthreads();
            const R mz_next = sMz[w + 1][lane];
            R ux[RPT], uy[RPT];
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const R tx = hx[q] + (lane_above(mz[q]) - mz[q]);
                const R ty = hy[q] + (mz[q] - (q + 1 < RPT ? mz[q + 1 < RPT ? q + 1 : q] : mz_next));
                if constexpr (PML) {
                    const R bx = g.xb * tx, by = g.yb[q] * ty;
                    icx[q] += g.kx[q] * bx;
                    icy[q] += g.ky * by;
                    ux[q] = bx + icx[q] * inv;
                    uy[q] = by + icy[q] * inv;
                    hx[q] = g.xa * tx;
                    hy[q] = g.ya[q] * ty;
                } else {
                    ux[q] = -cdt * tx;
                    uy[q] = -cdt * ty;
                    hx[q] = tx;
                    hy[q] = ty;
                }
            }
            sUy[w + 1][lane] = uy[RPT - 1];
            __syncthreads();
            const R uy_prev = sUy[w][lane];
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const R c = (uy[q] - (q > 0 ? uy[q > 0 ? q - 1 : 0] : uy_prev)) - (ux[q] - lane_below(ux[q]));
                if constexpr (PML) {
                    idz[q] += g.dc[q] * dz[q];
                    dz[q] = g.da[q] * dz[q] + idz[q] + g.me[q] * c;
                } else {
                    dz[q] += g.me[q] * c;
                }
                if (any_own) {
                    gm[q] += dp[q] * c;
                    dn[q] = dp[q];
                }
            }
            if (s > 0) load_dp(s - 1);
        }
    };
    if (pml) run(std::true_type{});
    else run(std::false_type{});
#pragma unroll
    for (int q = 0; q < RPT; ++q) {
        if (!own[q]) continue;
        g.at(a.out.hx, q, ny) = hx[q];
        g.at(a.out.hy, q, ny) = hy[q];
        g.at(a.out.dz, q, ny) = dz[q];
        if (g.shx[q] != R(0)) g.at(a.out.icex, q, ny) = icx[q];
        if (g.shy != R(0)) g.at(a.out.icey, q, ny) = icy[q];
        if (g.has_idz(q)) g.at(a.out.idz, q, ny) = idz[q];
        g.at(a.gm, q, ny) = gm[q];
    }
}

// TM arrays of an 18-array state, and of a packed buffer of the six arrays.
template <typename R>
static TmState<R> tm_of_state(R* st, int64_t n) {
    return TmState<R>{st, st + n, st + 5 * n, st + 6 * n, st + 7 * n, st + 17 * n};
}
template <typename R>
static TmState<R> tm_of_packed(R* p, int64_t n) {
    return TmState<R>{p, p + n, p + 2 * n, p + 3 * n, p + 4 * n, p + 5 * n};
}

// out = in for the values a TM run reads or writes: the fields everywhere, an
// integral where its sigma is non-zero (the rest of `out` keeps its values).
template <typename R>
__global__ void __launch_bounds__(256) k_tm_copy(TmArgs<R> a) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= (int64_t)a.nx * a.ny) return;
    const int i = (int)(c / a.ny), j = (int)(c - (int64_t)i * a.ny);
    a.out.hx[c] = a.in.hx[c];
    a.out.hy[c] = a.in.hy[c];
    a.out.dz[c] = a.in.dz[c];
    if (a.sig[i] != R(0)) a.out.icex[c] = a.in.icex[c];
    if (a.sig[a.nx + j] != R(0)) a.out.icey[c] = a.in.icey[c];
    if (a.sig[a.nx + a.ny + 1 + i] != R(0) && a.sig[2 * a.nx + a.ny + 1 + j] != R(0)) a.out.idz[c] = a.in.idz[c];
}

template <typename R>
static TmArgs<R> tm_args(const Fdtd<R>& f) {
    TmArgs<R> a = {};
    a.nx = f.nx;
    a.ny = f.ny;
    a.src_i = -1;
    a.inv_dL = R(1.0 / f.dL);
    a.dL = f.dL_r;
    a.cdt = f.cdt;
    a.half_dt = f.half_dt;
    a.sig = f.sig;
    a.eps = f.eps;
    return a;
}

template <typename R>
static void tm_source(TmArgs<R>& a, int64_t cell) {
    a.src_i = cell >= 0 ? (int)(cell / a.ny) : -1;
    a.src_j = cell >= 0 ? (int)(cell % a.ny) : -1;
}

template <typename R>
static void tm_copy(TmArgs<R> a, TmState<R> in, TmState<R> out, hipStream_t s) {
    a.in = in;
    a.out = out;
    k_tm_copy<R><<<(unsigned)(((int64_t)a.nx * a.ny + 255) / 256), 256, 0, s>>>(a);
}

// One launch sequence of a TM run over steps [a.t0, a.t0 + n_steps) from `in`:
// the launches alternate between the buffers w0 and w1 (`in` may be one of
// them) and the last one writes `out`, which must not be the buffer it reads
// (null: the next of w0 and w1).  reverse: the adjoint steps, last step first, `in` the
// cotangent after the steps; a.dz_hist and a.hist start at step a.t0.
template <typename R, int WV, int RPT, int TS>
static void launch_tm(TmArgs<R> a, TmState<R> in, TmState<R> out, TmState<R> w0, TmState<R> w1, int n_steps,
                      bool reverse, hipStream_t s) {
    static_assert(WV * RPT > 2 * TS && 64 > 2 * TS, "the owned tile must not be empty");
    constexpr int OX = WV * RPT - 2 * TS, OY = 64 - 2 * TS;
    a.tiles_x = (a.nx + OX - 1) / OX;
    a.tiles_y = (a.ny + OY - 1) / OY;
    const int64_t n = (int64_t)a.nx * a.ny;
    const int nblocks = a.tiles_x * a.tiles_y;
    const int t0 = a.t0;
    R* hist = a.hist;
    const R* dz_hist = a.dz_hist;
    const R* dz_before = a.dz_before;
    TmState<R> cur = in;
    for (int done = 0; done < n_steps; done += TS) {
        a.nsteps = std::min(TS, n_steps - done);
        const int first = reverse ? n_steps - done - a.nsteps : done;
        a.t0 = t0 + first;
        a.hist = hist ? hist + (int64_t)first * n : nullptr;
        a.dz_hist = dz_hist ? dz_hist + (int64_t)first * n : nullptr;
        a.dz_before = first > 0 && dz_hist ? dz_hist + (int64_t)(first - 1) * n : dz_before;
        a.in = cur;
        a.out = done + TS >= n_steps && out.hx ? out : (cur.hx == w0.hx ? w1 : w0);
        if (reverse) k_tm_adjoint<R, WV, RPT, TS><<<nblocks, 64 * WV, 0, s>>>(a);
        else k_tm_block<R, WV, RPT, TS><<<nblocks, 64 * WV, 0, s>>>(a);
        cur = a.out;
    }
}

template <typename R>
static int dispatch_tm(int cfg, const TmArgs<R>& a, TmState<R> in, TmState<R> out, TmState<R> w0, TmState<R> w1,
                       int n_steps, bool reverse, hipStream_t s) {
    switch (cfg) {
        case 0: launch_tm<R, 4, 4, 2>(a, in, out, w0, w1, n_steps, reverse, s); break;
        case 1: launch_tm<R, 4, 4, 4>(a, in, out, w0, w1, n_steps, reverse, s); break;
        case 2: launch_tm<R, 4, 8, 4>(a, in, out, w0, w1, n_steps, reverse, s); break;
        case 3: launch_tm<R, 4, 8, 8>(a, in, out, w0, w1, n_steps, reverse, s); break;
        case 4: launch_tm<R, 4, 16, 8>(a, in, out, w0, w1, n_steps, reverse, s); break;
        case 5: launch_tm<R, 4, 16, 4>(a, in, out, w0, w1, n_steps, reverse, s); break;
        case 6: launch_tm<R, 8, 4, 8>(a, in, out, w0, w1, n_steps, reverse, s); break;
        case 7: launch_tm<R, 16, 4, 16>(a, in, out, w0, w1, n_steps, reverse, s); break;
        case 8: launch_tm<R, 16, 2, 8>(a, in, out, w0, w1, n_steps, reverse, s); break;
        case 9: launch_tm<R, 16, 4, 8>(a, in, out, w0, w1, n_steps, reverse, s); break;
        case 10: launch_tm<R, 8, 4, 4>(a, in, out, w0, w1, n_steps, reverse, s); break;
        case 11: launch_tm<R, 16, 2, 4>(a, in, out, w0, w1, n_steps, reverse, s); break;
        default: CV_CHECK(false, "unknown TM tile configuration %d", cfg);
    }
    return CV_OK;
}

// ================================================ fused single-pass 3D step
// One kernel per step: the thread of cell c recomputes the new H at c and at
// its three backward neighbours (c - e_x, c - e_y, c - e_z) from the OLD state
// A, then forms the new D at c, writing H, D and the PML integrals of c to the
// NEW state B (ping-pong, so no cell reads a value another thread has already
// advanced).  DRAM traffic is one read of H, D, eps and one write of H, D per
// cell-step; the neighbour values come from cache.
template <typename R>
__host__ __device__ __forceinline__ R h_comp(const Fdtd<R>& f, const R* __restrict__ A, int a, int i, int j, int k,
                                             R& ice_out, R& ih_out) {
    const int64_t n = f.n;
    const R* D = A + 3 * n;
    const int ip = wrapp(i, f.nx), jp = wrapp(j, f.ny), kp = wrapp(k, f.nz);
    R ce;
    if (a == 0)
        ce = ((efield(f, D, 2, i, jp, k) - efield(f, D, 2, i, j, k)) -
              (efield(f, D, 1, i, j, kp) - efield(f, D, 1, i, j, k))) * f.inv_dL;
    else if (a == 1)
        ce = ((efield(f, D, 0, i, j, kp) - efield(f, D, 0, i, j, k)) -
              (efield(f, D, 2, ip, j, k) - efield(f, D, 2, i, j, k))) * f.inv_dL;
    else
        ce = ((efield(f, D, 1, ip, j, k) - efield(f, D, 1, i, j, k)) -
              (efield(f, D, 0, i, jp, k) - efield(f, D, 0, i, j, k))) * f.inv_dL;
    const int pos[3] = {i, j, k};
    const int ax_b = (a == 0) ? 1 : 0;
    const int ax_c = (a == 2) ? 1 : 2;
    const R sa = sigH(f, a)[pos[a]], sb = sigH(f, ax_b)[pos[ax_b]], sc = sigH(f, ax_c)[pos[ax_c]];
    const int64_t ca = a * n + cell(f, i, j, k);
    const R h = A[ca];
    if (sa == R(0) && sb == R(0) && sc == R(0)) return f.h1 * h + f.h2 * ce;
    R m1, m2, m3, m4;
    coef4<R>(sa, sb, sc, R(f.dt), R(f.c0), R(f.eps0), R(-1), m1, m2, m3, m4);
    R hn = m1 * h + m2 * ce;
    if (sa != R(0)) {
        ice_out = A[6 * n + ca] + ce;
        hn += m3 * ice_out;
    }
    if (sb != R(0) && sc != R(0)) {
        ih_out = A[9 * n + ca] + h;
        hn += m4 * ih_out;
    }
    return hn;
}

template <typename R>
__host__ __device__ __forceinline__ void fused_cell(const Fdtd<R>& f, const R* __restrict__ A, R* __restrict__ B,
                                                    PointSrc ps, int64_t c) {
    int i, j, k;
    decompose(f, c, i, j, k);
    const int64_t n = f.n;
    const int im = wrapm(i, f.nx), jm = wrapm(j, f.ny), km = wrapm(k, f.nz);
    R h[3], ice[3], ih[3];
    for (int a = 0; a < 3; ++a) {
        ice[a] = R(0);
        ih[a] = R(0);
        h[a] = h_comp(f, A, a, i, j, k, ice[a], ih[a]);
    }
    R dummy0, dummy1;
    // backward neighbours' new H components used by curl_H at c
    const R hz_jm = h_comp(f, A, 2, i, jm, k, dummy0, dummy1);
    const R hy_km = h_comp(f, A, 1, i, j, km, dummy0, dummy1);
    const R hx_km = h_comp(f, A, 0, i, j, km, dummy0, dummy1);
    const R hz_im = h_comp(f, A, 2, im, j, k, dummy0, dummy1);
    const R hy_im = h_comp(f, A, 1, im, j, k, dummy0, dummy1);
    const R hx_jm = h_comp(f, A, 0, i, jm, k, dummy0, dummy1);
    R ch[3];
    ch[0] = ((h[2] - hz_jm) - (h[1] - hy_km)) * f.inv_dL;
    ch[1] = ((h[0] - hx_km) - (h[2] - hz_im)) * f.inv_dL;
    ch[2] = ((h[1] - hy_im) - (h[0] - hx_jm)) * f.inv_dL;
    const int pos[3] = {i, j, k};
    for (int a = 0; a < 3; ++a) {
        const int64_t ca = a * n + c;
        B[ca] = h[a];
        const int ax_b = (a == 0) ? 1 : 0;
        const int ax_c = (a == 2) ? 1 : 2;
        {
            const R sa = sigH(f, a)[pos[a]], sb = sigH(f, ax_b)[pos[ax_b]], sc = sigH(f, ax_c)[pos[ax_c]];
            if (sa != R(0)) B[6 * n + ca] = ice[a];
            if (sb != R(0) && sc != R(0)) B[9 * n + ca] = ih[a];
        }
        const R sa = sigD(f, a)[pos[a]], sb = sigD(f, ax_b)[pos[ax_b]], sc = sigD(f, ax_c)[pos[ax_c]];
        const R d = A[3 * n + ca];
        R dn;
        if (sa == R(0) && sb == R(0) && sc == R(0)) {
            dn = f.d1 * d + f.d2 * ch[a];
        } else {
            R m1, m2, m3, m4;
            coef4<R>(sa, sb, sc, R(f.dt), R(f.c0), R(f.eps0), R(1), m1, m2, m3, m4);
            dn = m1 * d + m2 * ch[a];
            if (sa != R(0)) {
                const R ich = A[12 * n + ca] + ch[a];
                B[12 * n + ca] = ich;
                dn += m3 * ich;
            }
            if (sb != R(0) && sc != R(0)) {
                const R idv = A[15 * n + ca] + d;
                B[15 * n + ca] = idv;
                dn += m4 * idv;
            }
        }
        if (ps.comp == a && ps.cell == c) dn += R(ps.amp);
        B[3 * n + ca] = dn;
    }
}

template <typename R>
__global__ void __launch_bounds__(256) k_fused(Fdtd<R> f, const R* __restrict__ A, R* __restrict__ B, PointSrc ps,
                                               const double* __restrict__ amp_dev, int t) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= f.n) return;
    if (ps.comp >= 0) ps.amp = amp_dev[t];
    fused_cell(f, A, B, ps, c);
}

// =================================== x-marching single-pass 3D step
// One workgroup (16 / kMRpt waves) owns a region of 16 rows (y) x 64 lanes
// (z) of (y, z) columns and marches along x over a chunk of slices; each
// thread keeps kMRpt cells of the region (consecutive rows, its lane) in
// registers:
// per slice i it forms E(i+1) from the loads of D(i+1) and eps, the new H(i)
// from E(i) (own cell, and the y+1 / z+1 neighbours through LDS) and E(i+1),
// then the new D(i) from H(i) (own, and y-1 / z-1 through LDS) and H(i-1),
// which it carried from the previous slice.  H is valid on region rows 0..14
// and lanes 0..62, D on rows 1..14 and lanes 1..62: the owned 14 x 62 cells.
// Reads come from the old state A only and writes go to B (ping-pong), so
// workgroup order does not matter; a chunk starts by recomputing H(i0-1).
// DRAM traffic per cell-step: H, D, eps read and H, D written (52 B in
// float32) plus the 1 / 14 and 1 / 62 halo fractions.  The update and its
// coefficients (coef4) are those of k_h and k_d; which products are fused is
// left to the compiler here, so single roundings differ.
constexpr int kMRows = 16, kMLanes = 64;
constexpr int kMOwnY = kMRows - 2, kMOwnZ = kMLanes - 2;

template <typename R, int kMRpt>
__global__ void __launch_bounds__(64 * kMRows / kMRpt) k_march(Fdtd<R> f, const R* __restrict__ A, R* __restrict__ B,
                                                             PointSrc ps, const double* __restrict__ amp_dev, int t,
                                                             int tiles_y, int tiles_z, int chunk) {
    __shared__ R sE[3][kMRows][kMLanes];
    __shared__ R sH[3][kMRows][kMLanes];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int b = blockIdx.x;
    const int tz = b % tiles_z;
    b /= tiles_z;
    const int ty = b % tiles_y;
    const int chk = b / tiles_y;
    const int i0 = chk * chunk;
    const int i1 = min(f.nx, i0 + chunk);
    if (i0 >= i1) return;   // uniform over the workgroup
    if (ps.comp >= 0) ps.amp = amp_dev[t];
    const int64_t n = f.n;
    const int ny = f.ny, nz = f.nz;
    const R* Dx = A + 3 * n;
    const R* Dy = A + 4 * n;
    const R* Dz = A + 5 * n;
    // region coordinates of this thread's cells
    const int zz = tz * kMOwnZ - 1 + lane;            // unwrapped z
    const int k = pmod(zz, nz);
    const int km = wrapm(k, nz);
    int j[kMRpt], jm[kMRpt];
    bool own[kMRpt];
    const bool own_z = lane >= 1 && lane <= kMLanes - 2 && zz < nz;
#pragma unroll
    for (int q = 0; q < kMRpt; ++q) {
        const int r = w * kMRpt + q;
        const int yy = ty * kMOwnY - 1 + r;
        j[q] = pmod(yy, ny);
        jm[q] = wrapm(j[q], ny);
        own[q] = own_z && r >= 1 && r <= kMRows - 2 && yy < ny;
    }
    const R sHy_k = sigH(f, 2)[k], sDz_k = sigD(f, 2)[k];
    R sHy_j[kMRpt], sDy_j[kMRpt];
#pragma unroll
    for (int q = 0; q < kMRpt; ++q) {
        sHy_j[q] = sigH(f, 1)[j[q]];
        sDy_j[q] = sigD(f, 1)[j[q]];
    }
    auto cidx = [&](int xi, int q) -> int64_t { return ((int64_t)xi * ny + j[q]) * nz + k; };

    // raw loads of slice xi (D and the four eps values E needs), issued
    // early so that they are in flight during the previous slice's work
    struct Raw {
        R d[kMRpt][3];
        R e0[kMRpt], ex[kMRpt], ey[kMRpt], ez[kMRpt];
    };
    auto load_raw = [&](int xi, Raw& rw) {
        const int xm = wrapm(xi, f.nx);
#pragma unroll
        for (int q = 0; q < kMRpt; ++q) {
            const int64_t c = cidx(xi, q);
            rw.e0[q] = f.eps[c];
            rw.ex[q] = f.eps[((int64_t)xm * ny + j[q]) * nz + k];
            rw.ey[q] = f.eps[((int64_t)xi * ny + jm[q]) * nz + k];
            rw.ez[q] = f.eps[((int64_t)xi * ny + j[q]) * nz + km];
            rw.d[q][0] = Dx[c];
            rw.d[q][1] = Dy[c];
            rw.d[q][2] = Dz[c];
        }
    };
    auto to_E = [&](const Raw& rw, R (&e)[kMRpt][3]) {
#pragma unroll
        for (int q = 0; q < kMRpt; ++q) {
            const R ea = (rw.e0[q] + rw.ex[q]) / R(2);
            const R eb = (rw.e0[q] + rw.ey[q]) / R(2);
            const R eg = (rw.e0[q] + rw.ez[q]) / R(2);
            e[q][0] = (R(1) / ea) * rw.d[q][0];
            e[q][1] = (R(1) / eb) * rw.d[q][1];
            e[q][2] = (R(1) / eg) * rw.d[q][2];
        }
    };
    auto load_H = [&](int xi, R (&h)[kMRpt][3]) {
#pragma unroll
        for (int q = 0; q < kMRpt; ++q) {
            const int64_t c = cidx(xi, q);
#pragma unroll
            for (int a = 0; a < 3; ++a) h[q][a] = A[a * n + c];
        }
    };
    // new H of slice xi at this thread's cells; eC = E(xi) (also in sE),
    // eN = E(xi+1), hO = old H(xi)
    auto h_new = [&](int xi, const R (&eC)[kMRpt][3], const R (&eN)[kMRpt][3], const R (&hO)[kMRpt][3],
                     R (&h)[kMRpt][3], bool store) {
        const R sHx = sigH(f, 0)[xi];
#pragma unroll
        for (int q = 0; q < kMRpt; ++q) {
            const int r = w * kMRpt + q;
            const int rp = min(r + 1, kMRows - 1), lp = min(lane + 1, kMLanes - 1);
            R ce[3];
            ce[0] = ((sE[2][rp][lane] - eC[q][2]) - (sE[1][r][lp] - eC[q][1])) * f.inv_dL;
            ce[1] = ((sE[0][r][lp] - eC[q][0]) - (eN[q][2] - eC[q][2])) * f.inv_dL;
            ce[2] = ((eN[q][1] - eC[q][1]) - (sE[0][rp][lane] - eC[q][0])) * f.inv_dL;
            const int64_t c = cidx(xi, q);
            const R sg[3] = {sHx, sHy_j[q], sHy_k};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const int ax_b = (a == 0) ? 1 : 0;
                const int ax_c = (a == 2) ? 1 : 2;
                const R sa = sg[a], sb = sg[ax_b], sc = sg[ax_c];
                const int64_t ca = a * n + c;
                const R hv = hO[q][a];
                R hn;
                if (sa == R(0) && sb == R(0) && sc == R(0)) {
                    hn = f.h1 * hv + f.h2 * ce[a];
                } else {
                    R m1, m2, m3, m4;
                    coef4<R>(sa, sb, sc, R(f.dt), R(f.c0), R(f.eps0), R(-1), m1, m2, m3, m4);
                    hn = m1 * hv + m2 * ce[a];
                    if (sa != R(0)) {
                        const R ice = A[6 * n + ca] + ce[a];
                        if (store && own[q]) B[6 * n + ca] = ice;
                        hn += m3 * ice;
                    }
                    if (sb != R(0) && sc != R(0)) {
                        const R ih = A[9 * n + ca] + hv;
                        if (store && own[q]) B[9 * n + ca] = ih;
                        hn += m4 * ih;
                    }
                }
                h[q][a] = hn;
                if (store && own[q]) B[ca] = hn;
            }
        }
    };

    Raw rwA, rwB;
    R eC[kMRpt][3], eN[kMRpt][3], dC[kMRpt][3], hP[kMRpt][3], hC[kMRpt][3], hO[kMRpt][3], hON[kMRpt][3];
    // H(i0 - 1) from E(i0 - 1), E(i0) and old H(i0 - 1)
    const int xprev = wrapm(i0, f.nx);
    load_raw(xprev, rwA);
    load_raw(i0, rwB);
    load_H(xprev, hO);
    to_E(rwA, eC);
    to_E(rwB, eN);
#pragma unroll
    for (int q = 0; q < kMRpt; ++q)
#pragma unroll
        for (int a = 0; a < 3; ++a) sE[a][w * kMRpt + q][lane] = eC[q][a];
    load_raw(wrapp(i0, f.nx), rwA);     // slice i0 + 1 in flight
    __syncthreads();
    h_new(xprev, eC, eN, hO, hP, false);
    load_H(i0, hO);                     // old H(i0) in flight
#pragma unroll
    for (int q = 0; q < kMRpt; ++q)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            eC[q][a] = eN[q][a];
            dC[q][a] = rwB.d[q][a];
        }
    for (int xi = i0; xi < i1; ++xi) {
        __syncthreads();   // every read of sE / sH of the previous slice is done
#pragma unroll
        for (int q = 0; q < kMRpt; ++q)
#pragma unroll
            for (int a = 0; a < 3; ++a) sE[a][w * kMRpt + q][lane] = eC[q][a];
        to_E(rwA, eN);                      // E(xi + 1), loaded one slice ago
        R dN[kMRpt][3];
#pragma unroll
        for (int q = 0; q < kMRpt; ++q)
#pragma unroll
            for (int a = 0; a < 3; ++a) dN[q][a] = rwA.d[q][a];
        const int xn2 = wrapp(wrapp(xi, f.nx), f.nx);
        if (xi + 1 < i1) {
            load_raw(xn2, rwA);             // slice xi + 2 in flight
            load_H(wrapp(xi, f.nx), hON);   // old H(xi + 1) in flight
        }
        __syncthreads();
        h_new(xi, eC, eN, hO, hC, true);
#pragma unroll
        for (int q = 0; q < kMRpt; ++q)
#pragma unroll
            for (int a = 0; a < 3; ++a) sH[a][w * kMRpt + q][lane] = hC[q][a];
        __syncthreads();
        const R sDx = sigD(f, 0)[xi];
#pragma unroll
        for (int q = 0; q < kMRpt; ++q) {
            const int r = w * kMRpt + q;
            const int rm = max(r - 1, 0), lm = max(lane - 1, 0);
            R ch[3];
            ch[0] = ((hC[q][2] - sH[2][rm][lane]) - (hC[q][1] - sH[1][r][lm])) * f.inv_dL;
            ch[1] = ((hC[q][0] - sH[0][r][lm]) - (hC[q][2] - hP[q][2])) * f.inv_dL;
            ch[2] = ((hC[q][1] - hP[q][1]) - (hC[q][0] - sH[0][rm][lane])) * f.inv_dL;
            const int64_t c = cidx(xi, q);
            const R sg[3] = {sDx, sDy_j[q], sDz_k};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const int ax_b = (a == 0) ? 1 : 0;
                const int ax_c = (a == 2) ? 1 : 2;
                const R sa = sg[a], sb = sg[ax_b], sc = sg[ax_c];
                const int64_t ca = a * n + c;
                const R dv = dC[q][a];
                R dn;
                if (sa == R(0) && sb == R(0) && sc == R(0)) {
                    dn = f.d1 * dv + f.d2 * ch[a];
                } else {
                    R m1, m2, m3, m4;
                    coef4<R>(sa, sb, sc, R(f.dt), R(f.c0), R(f.eps0), R(1), m1, m2, m3, m4);
                    dn = m1 * dv + m2 * ch[a];
                    if (sa != R(0)) {
                        const R ich = A[12 * n + ca] + ch[a];
                        if (own[q]) B[12 * n + ca] = ich;
                        dn += m3 * ich;
                    }
                    if (sb != R(0) && sc != R(0)) {
                        const R idv = A[15 * n + ca] + dv;
                        if (own[q]) B[15 * n + ca] = idv;
                        dn += m4 * idv;
                    }
                }
                if (ps.comp == a && ps.cell == c) dn += R(ps.amp);
                if (own[q]) B[3 * n + ca] = dn;
            }
        }
#pragma unroll
        for (int q = 0; q < kMRpt; ++q)
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                hP[q][a] = hC[q][a];
                eC[q][a] = eN[q][a];
                dC[q][a] = dN[q][a];
                hO[q][a] = hON[q][a];
            }
    }
}

// ==================================== slab-marching single-pass 3D step
// A workgroup of nz threads (one z line each, nz a multiple of 64 up to 256)
// owns a band of TJ whole (y, z) rows and marches along x over a chunk of
// slices, so z needs no halo and y one row on each side.  Per slice xi it
// holds E(xi) and E(xi+1) of rows -1..TJ (E = D / eps_aa formed once from D
// and eps of the band), forms the new H(xi) of rows -1..TJ-1 (row -1 only
// Hx, Hz, the y-1 values the D update needs), then the new D(xi) of the band
// from H(xi) and the H(xi-1) carried from the previous slice.  The z+1
// neighbours of E and the z-1 neighbours of H go through LDS.  All reads come
// from the old state A and all writes go to B (ping-pong), so neighbouring
// bands may recompute each other's halo rows in any order; a chunk starts by
// recomputing H(i0-1).  HBM traffic per cell-step: H, D, eps read, H, D
// written (52 B in float32, plus the PML integrals inside the PML); the halo
// rows are re-read by the neighbouring band on the same XCD (consecutive
// bands of a chunk are mapped to one XCD).  The update and its coefficients
// (coef4) are those of k_h and k_d; which products are fused is left to the
// compiler here, so single roundings differ.
constexpr int kSlabMaxNz = 256;

// Load / store at a 32-bit byte offset through a raw buffer resource over
// one slice of one array (base and size uniform, in scalar registers; one
// vector register per address).  An offset outside the slice reads 0 and
// drops the store.  Resource word 3 = 0x00020000, the gfx9 raw-buffer format.
template <typename R>
__device__ __forceinline__ R ld_at(const R* base, uint32_t byte_off, uint32_t bytes) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)bytes, 0x00020000);
    if constexpr (sizeof(R) == 4)
        return __builtin_bit_cast(R, __builtin_amdgcn_raw_buffer_load_b32(r, (int)byte_off, 0, 0));
    else
        return __builtin_bit_cast(R, __builtin_amdgcn_raw_buffer_load_b64(r, (int)byte_off, 0, 0));
}
template <typename R>
__device__ __forceinline__ void st_at(R* base, uint32_t byte_off, uint32_t bytes, R v) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)bytes, 0x00020000);
    if constexpr (sizeof(R) == 4)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, (int)byte_off, 0, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0)), v),
                                              r, (int)byte_off, 0, 0);
}

template <typename R, int TJ>
__global__ void __launch_bounds__(kSlabMaxNz) k_slab(Fdtd<R> f, const R* __restrict__ A, R* __restrict__ B,
                                                     const R* __restrict__ sig, const R* __restrict__ epsv,
                                                     PointSrc ps, const double* __restrict__ amp_dev, int t,
                                                     int tiles_y, int chunk, int map_bands) {
    __shared__ R sE[2][TJ + 1][kSlabMaxNz];   // Ex of rows 0..TJ-1 at [0][r], Ey of rows -1..TJ-1 at [1][r+1]
    __shared__ R sH[2][TJ][kSlabMaxNz];       // new Hx, Hy of rows 0..TJ-1
    // Workgroup b runs on XCD b % 8; consecutive bands of a chunk go to one
    // XCD in consecutive dispatch order, so halo rows are re-read from the
    // same L2.  map_bands: when the bands split evenly over the 8 XCDs, XCD x
    // takes bands [x T/8, (x+1) T/8) of every chunk (T = bands), which
    // spreads the x-PML chunks over all XCDs; otherwise XCD x takes a range
    // of whole chunks.
    const int b = blockIdx.x;
    int ty, ch;
    if (!map_bands) {   // XCD x takes a contiguous range of whole chunks
        const int nb = gridDim.x;
        const int l = ((nb & 7) == 0) ? (b & 7) * (nb >> 3) + (b >> 3) : b;
        ty = l % tiles_y;
        ch = l / tiles_y;
    } else if ((tiles_y & 7) == 0) {
        const int per = tiles_y >> 3, j = b >> 3;
        ty = (b & 7) * per + j % per;
        ch = j / per;
    } else {
        ty = b % tiles_y;
        ch = b / tiles_y;
    }
    const int i0 = ch * chunk;
    const int i1 = min(f.nx, i0 + chunk);
    if (i0 >= i1) return;   // uniform over the workgroup
    const int64_t n = f.n;
    const int nx = f.nx, ny = f.ny, nz = f.nz;
    const int64_t plane = (int64_t)ny * nz;
    const uint32_t sbytes = (uint32_t)(plane * (int64_t)sizeof(R));   // bytes of one slice
    // the point source as (slice, offset in the slice); slice -1 = none
    int src_x = -1;
    uint32_t src_off = 0;
    R src_amp = R(0);
    if (ps.comp >= 0) {
        src_x = (int)(ps.cell / plane);
        src_off = (uint32_t)(ps.cell - (int64_t)src_x * plane) * (uint32_t)sizeof(R);
        src_amp = R(amp_dev[t]);
    }
    // sigma with workgroup-uniform indices through scalar loads (constant
    // address space), which a vector-memory wait does not wait for
    using csig_t = const __attribute__((address_space(4))) R*;
    const csig_t csig = (csig_t)sig;
    const int k = threadIdx.x;
    const int kp = (k + 1 == nz) ? 0 : k + 1;
    const int km = (k == 0) ? nz - 1 : k - 1;
    // byte offsets in a slice of rows -2..TJ of the band (wrapped) at index r + 2
    uint32_t off[TJ + 3], offm[TJ + 3];
#pragma unroll
    for (int q = 0; q < TJ + 3; ++q) {
        const uint32_t row = (uint32_t)pmod(ty * TJ + q - 2, ny) * (uint32_t)nz;
        off[q] = (row + (uint32_t)k) * (uint32_t)sizeof(R);
        offm[q] = (row + (uint32_t)km) * (uint32_t)sizeof(R);
    }
    R sHyj[TJ + 1], sDyj[TJ];   // sigma_y of rows -1..TJ-1 (H) and 0..TJ-1 (D)
#pragma unroll
    for (int q = 0; q < TJ + 1; ++q) sHyj[q] = csig[nx + pmod(ty * TJ + q - 1, ny)];
#pragma unroll
    for (int q = 0; q < TJ; ++q) sDyj[q] = csig[nx + ny + nz + nx + ty * TJ + q];
    const R sHzk = sig[nx + ny + k], sDzk = sig[2 * (nx + ny) + nz + k];

    // D of rows -1..TJ (Dy of row TJ is not needed), eps of rows -2..TJ, eps at
    // z-1 of rows -1..TJ, all of slice xi
    struct Raw {
        R d[3][TJ + 2];
        R e[TJ + 3];
        R ek[TJ + 2];
    };
    auto load_raw = [&](int xi, Raw& rw) {
        const R* ep = epsv + (int64_t)xi * plane;
        const R* dp = A + 3 * n + (int64_t)xi * plane;
#pragma unroll
        for (int q = 0; q < TJ + 3; ++q) rw.e[q] = ld_at(ep, off[q], sbytes);
#pragma unroll
        for (int q = 0; q < TJ + 2; ++q) {
            rw.ek[q] = ld_at(ep, offm[q + 1], sbytes);
            rw.d[0][q] = ld_at(dp, off[q + 1], sbytes);
            if (q < TJ + 1) rw.d[1][q] = ld_at(dp + n, off[q + 1], sbytes);
            rw.d[2][q] = ld_at(dp + 2 * n, off[q + 1], sbytes);
        }
    };
    // eps of the previous slice, rows -1..TJ, for eps_xx
    auto to_E = [&](const Raw& rw, const R (&ep)[TJ + 2], R (&e)[3][TJ + 2]) {
#pragma unroll
        for (int q = 0; q < TJ + 2; ++q) {
            const R e0 = rw.e[q + 1];
            const R exx = (e0 + ep[q]) / R(2);
            const R eyy = (e0 + rw.e[q]) / R(2);
            const R ezz = (e0 + rw.ek[q]) / R(2);
            e[0][q] = (R(1) / exx) * rw.d[0][q];
            e[1][q] = (q < TJ + 1) ? (R(1) / eyy) * rw.d[1][q] : R(0);
            e[2][q] = (R(1) / ezz) * rw.d[2][q];
        }
    };
    // old H of rows -1..TJ-1 (Hy of row -1 is not needed)
    auto load_H = [&](int xi, R (&h)[3][TJ + 1]) {
        const R* hp = A + (int64_t)xi * plane;
#pragma unroll
        for (int q = 0; q < TJ + 1; ++q) {
            h[0][q] = ld_at(hp, off[q + 1], sbytes);
            h[1][q] = (q > 0) ? ld_at(hp + n, off[q + 1], sbytes) : R(0);
            h[2][q] = ld_at(hp + 2 * n, off[q + 1], sbytes);
        }
    };
    auto put_E = [&](const R (&e)[3][TJ + 2]) {
#pragma unroll
        for (int q = 0; q < TJ + 1; ++q) {
            if (q < TJ) sE[0][q][k] = e[0][q + 1];
            sE[1][q][k] = e[1][q];
        }
    };
    // PML integrals the general H update of slice xi reads (ICE where the
    // component's own sigma is non-zero, IH where both others are), all
    // issued together; an integral that is not needed gets an offset past
    // the slice (reads 0, no memory access).
    auto h_aux_load = [&](int xi, R (&ice)[3][TJ + 1], R (&ih)[3][TJ + 1]) {
        const R* ap = A + (int64_t)xi * plane;
        const R sHx = csig[xi];
#pragma unroll
        for (int q = 0; q < TJ + 1; ++q) {
            const R sg[3] = {sHx, sHyj[q], sHzk};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const R sa = sg[a], sb = sg[(a == 0) ? 1 : 0], sc = sg[(a == 2) ? 1 : 2];
                ice[a][q] = ld_at(ap + (6 + a) * n, sa != R(0) ? off[q + 1] : sbytes, sbytes);
                ih[a][q] = ld_at(ap + (9 + a) * n, (sb != R(0) && sc != R(0)) ? off[q + 1] : sbytes, sbytes);
            }
        }
    };
    // new H of slice xi, rows -1..TJ-1 (index r + 1), from E(xi) = eC (z+1
    // values in sE), E(xi+1) = eN, the old H and the integrals of
    // h_aux_load; `store` writes the band's rows and their PML integrals to
    // B.  Components: row -1 Hx, Hz only, or (hyz_only) Hy, Hz of rows
    // 0..TJ-1.
    auto h_new = [&](int xi, const R (&eC)[3][TJ + 2], const R (&eN)[3][TJ + 2], const R (&hO)[3][TJ + 1],
                     const R (&ice0)[3][TJ + 1], const R (&ih0)[3][TJ + 1], R (&h)[3][TJ + 1], bool store,
                     bool hyz_only) {
        R* bp = B + (int64_t)xi * plane;
        const R sHx = csig[xi];
#pragma unroll
        for (int q = 0; q < TJ + 1; ++q) {
            const int r = q - 1;
            const R ex = eC[0][q], ey = eC[1][q], ez = eC[2][q];
            R ce[3];
            // curl_E, ceviche/derivatives.py:16-22 (forward differences, periodic)
            ce[0] = ((eC[2][q + 1] - ez) - (sE[1][q][kp] - ey)) * f.inv_dL;
            ce[1] = (r >= 0) ? ((sE[0][r < 0 ? 0 : r][kp] - ex) - (eN[2][q] - ez)) * f.inv_dL : R(0);
            ce[2] = ((eN[1][q] - ey) - (eC[0][q + 1] - ex)) * f.inv_dL;
            const uint32_t o = off[q + 1];
            const R sg[3] = {sHx, sHyj[q], sHzk};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                if ((r < 0 && a == 1) || (hyz_only && (r < 0 || a == 0))) {
                    h[a][q] = R(0);
                    continue;
                }
                const int ax_b = (a == 0) ? 1 : 0;
                const int ax_c = (a == 2) ? 1 : 2;
                const R sa = sg[a], sb = sg[ax_b], sc = sg[ax_c];
                const int64_t ca = a * n;
                const R hv = hO[a][q];
                R hn;
                if (sa == R(0) && sb == R(0) && sc == R(0)) {
                    hn = f.h1 * hv + f.h2 * ce[a];
                } else {
                    R m1, m2, m3, m4;
                    coef4<R>(sa, sb, sc, R(f.dt), R(f.c0), R(f.eps0), R(-1), m1, m2, m3, m4);
                    hn = m1 * hv + m2 * ce[a];
                    if (sa != R(0)) {
                        const R ice = ice0[a][q] + ce[a];
                        if (store && r >= 0) st_at(bp + 6 * n + ca, o, sbytes, ice);
                        hn += m3 * ice;
                    }
                    if (sb != R(0) && sc != R(0)) {
                        const R ih = ih0[a][q] + hv;
                        if (store && r >= 0) st_at(bp + 9 * n + ca, o, sbytes, ih);
                        hn += m4 * ih;
                    }
                }
                h[a][q] = hn;
                if (store && r >= 0) st_at(bp + ca, o, sbytes, hn);
            }
        }
    };

    // Fast path: a slice outside the x PML in a band whose rows are outside
    // the y PML.  There the only live PML integrals are those of the z axis
    // (ICE of Hz, ICH of Dz, on z-PML lanes), their values are prefetched a
    // slice ahead with the other loads (lanes outside the z PML pass an
    // offset past the slice: no memory access), and the coefficients depend
    // on the lane only: coef4(0, 0, s_z) for the x and y components and
    // coef4(s_z, 0, 0) for z, the same calls with the same arguments as the
    // general update, which the remaining slices use.
    bool band_ypml = false;
#pragma unroll
    for (int q = 0; q < TJ + 1; ++q) band_ypml |= sHyj[q] != R(0);
#pragma unroll
    for (int q = 0; q < TJ; ++q) band_ypml |= sDyj[q] != R(0);
    R cHxy1 = f.h1, cHxy2 = f.h2, cHz1 = f.h1, cHz2 = f.h2, cHz3 = R(0);
    R cDxy1 = f.d1, cDxy2 = f.d2, cDz1 = f.d1, cDz2 = f.d2, cDz3 = R(0);
    if (sHzk != R(0)) {
        R m4;
        coef4<R>(R(0), R(0), sHzk, R(f.dt), R(f.c0), R(f.eps0), R(-1), cHxy1, cHxy2, cHz3, m4);
        coef4<R>(sHzk, R(0), R(0), R(f.dt), R(f.c0), R(f.eps0), R(-1), cHz1, cHz2, cHz3, m4);
    }
    if (sDzk != R(0)) {
        R m4;
        coef4<R>(R(0), R(0), sDzk, R(f.dt), R(f.c0), R(f.eps0), R(1), cDxy1, cDxy2, cDz3, m4);
        coef4<R>(sDzk, R(0), R(0), R(f.dt), R(f.c0), R(f.eps0), R(1), cDz1, cDz2, cDz3, m4);
    }
    // ICE of Hz (rows -1..TJ-1) and ICH of Dz (rows 0..TJ-1) of slice xi
    auto load_zaux = [&](int xi, R (&ice)[TJ + 1], R (&ich)[TJ]) {
        const R* ap = A + (int64_t)xi * plane;
#pragma unroll
        for (int q = 0; q < TJ + 1; ++q) ice[q] = ld_at(ap + 8 * n, sHzk != R(0) ? off[q + 1] : sbytes, sbytes);
#pragma unroll
        for (int q = 0; q < TJ; ++q) ich[q] = ld_at(ap + 14 * n, sDzk != R(0) ? off[q + 2] : sbytes, sbytes);
    };
    // new H of slice xi on the fast path (same rows and components as h_new)
    auto h_fast = [&](int xi, const R (&eC)[3][TJ + 2], const R (&eN)[3][TJ + 2], const R (&hO)[3][TJ + 1],
                      const R (&ice)[TJ + 1], R (&h)[3][TJ + 1]) {
        R* bp = B + (int64_t)xi * plane;
#pragma unroll
        for (int q = 0; q < TJ + 1; ++q) {
            const int r = q - 1;
            const R ex = eC[0][q], ey = eC[1][q], ez = eC[2][q];
            const uint32_t o = off[q + 1];
            const R ce0 = ((eC[2][q + 1] - ez) - (sE[1][q][kp] - ey)) * f.inv_dL;
            const R ce2 = ((eN[1][q] - ey) - (eC[0][q + 1] - ex)) * f.inv_dL;
            h[0][q] = cHxy1 * hO[0][q] + cHxy2 * ce0;
            if (r >= 0) {
                const R ce1 = ((sE[0][r < 0 ? 0 : r][kp] - ex) - (eN[2][q] - ez)) * f.inv_dL;
                h[1][q] = cHxy1 * hO[1][q] + cHxy2 * ce1;
            } else {
                h[1][q] = R(0);
            }
            R hz = cHz1 * hO[2][q] + cHz2 * ce2;
            if (sHzk != R(0)) {
                const R ice_n = ice[q] + ce2;
                if (r >= 0) st_at(bp + 8 * n, o, sbytes, ice_n);
                hz += cHz3 * ice_n;
            }
            h[2][q] = hz;
            if (r >= 0) {
                st_at(bp, o, sbytes, h[0][q]);
                st_at(bp + n, o, sbytes, h[1][q]);
                st_at(bp + 2 * n, o, sbytes, hz);
            }
        }
    };
    R zIce[TJ + 1], zIch[TJ];        // z-PML integrals of slice xi (fast path)

    R eP[TJ + 2];                    // eps of the slice before the one last loaded, rows -1..TJ
    R eC[3][TJ + 2], eN[3][TJ + 2];  // E(xi), E(xi+1)
    R dC[3][TJ], dN[3][TJ];          // old D(xi), D(xi+1) of the band
    R hC[3][TJ + 1];                 // new H(xi)
    R hPy[TJ], hPz[TJ];              // new Hy, Hz of H(xi-1), rows 0..TJ-1
    R hO[3][TJ + 1];                 // old H(xi)
    Raw rw;
    const int xm1 = wrapm(i0, nx), xm2 = wrapm(xm1, nx);
    {
        const R* ep = epsv + (int64_t)xm2 * plane;
#pragma unroll
        for (int q = 0; q < TJ + 2; ++q) eP[q] = ld_at(ep, off[q + 1], sbytes);
    }
    // H(i0-1) from E(i0-1), E(i0) and the old H(i0-1)
    load_raw(xm1, rw);
    to_E(rw, eP, eC);
#pragma unroll
    for (int q = 0; q < TJ + 2; ++q) eP[q] = rw.e[q + 1];
    load_raw(i0, rw);
    to_E(rw, eP, eN);
#pragma unroll
    for (int q = 0; q < TJ + 2; ++q) eP[q] = rw.e[q + 1];
#pragma unroll
    for (int q = 0; q < TJ; ++q)
#pragma unroll
        for (int a = 0; a < 3; ++a) dC[a][q] = rw.d[a][q + 1];
    load_H(xm1, hO);
    put_E(eC);
    {
        R ice[3][TJ + 1], ih[3][TJ + 1];
        h_aux_load(xm1, ice, ih);
        __syncthreads();
        h_new(xm1, eC, eN, hO, ice, ih, hC, false, true);
    }
#pragma unroll
    for (int q = 0; q < TJ; ++q) {
        hPy[q] = hC[1][q + 1];
        hPz[q] = hC[2][q + 1];
    }
    // E(i0), E(i0+1), old H(i0)
    load_raw(wrapp(i0, nx), rw);
    load_H(i0, hO);
#pragma unroll
    for (int q = 0; q < TJ + 2; ++q)
#pragma unroll
        for (int a = 0; a < 3; ++a) eC[a][q] = eN[a][q];
    to_E(rw, eP, eN);
#pragma unroll
    for (int q = 0; q < TJ + 2; ++q) eP[q] = rw.e[q + 1];
#pragma unroll
    for (int q = 0; q < TJ; ++q)
#pragma unroll
        for (int a = 0; a < 3; ++a) dN[a][q] = rw.d[a][q + 1];
    load_zaux(i0, zIce, zIch);
    __syncthreads();   // every read of sE holding E(i0-1) is done
    put_E(eC);
    __syncthreads();

    for (int xi = i0; xi < i1; ++xi) {
        const bool more = xi + 1 < i1;   // uniform
        const bool fast = !band_ypml && csig[xi] == R(0) && csig[nx + ny + nz + xi] == R(0);   // uniform
        R zIceN[TJ + 1], zIchN[TJ];
        if (more) load_zaux(wrapp(xi, nx), zIceN, zIchN);    // issued before the slice xi + 2 loads
        R ice[3][TJ + 1], ih[3][TJ + 1];
        if (!fast) h_aux_load(xi, ice, ih);                  // likewise
        if (more) load_raw(wrapp(wrapp(xi, nx), nx), rw);   // slice xi + 2 in flight
        if (fast) h_fast(xi, eC, eN, hO, zIce, hC);
        else h_new(xi, eC, eN, hO, ice, ih, hC, true, false);
#pragma unroll
        for (int q = 0; q < TJ; ++q) {
            sH[0][q][k] = hC[0][q + 1];
            sH[1][q][k] = hC[1][q + 1];
        }
        if (more) load_H(wrapp(xi, nx), hO);   // old H(xi + 1) in flight
        __syncthreads();
        const int64_t p = (int64_t)xi * plane;
        R* bp = B + p;
        const R* ap = A + p;
        const R sDx = csig[nx + ny + nz + xi];
        R ich0[3][TJ], id0[3][TJ];   // PML integrals of the general D update, loaded together
        if (!fast) {
#pragma unroll
            for (int q = 0; q < TJ; ++q) {
                const R sg[3] = {sDx, sDyj[q], sDzk};
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const R sa = sg[a], sb = sg[(a == 0) ? 1 : 0], sc = sg[(a == 2) ? 1 : 2];
                    ich0[a][q] = ld_at(ap + (12 + a) * n, sa != R(0) ? off[q + 2] : sbytes, sbytes);
                    id0[a][q] = ld_at(ap + (15 + a) * n, (sb != R(0) && sc != R(0)) ? off[q + 2] : sbytes, sbytes);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < TJ; ++q) {
            const int qh = q + 1;   // index of row q in hC
            R ch[3];
            // curl_H, ceviche/derivatives.py:24-30 (backward differences, periodic)
            ch[0] = ((hC[2][qh] - hC[2][qh - 1]) - (hC[1][qh] - sH[1][q][km])) * f.inv_dL;
            ch[1] = ((hC[0][qh] - sH[0][q][km]) - (hC[2][qh] - hPz[q])) * f.inv_dL;
            ch[2] = ((hC[1][qh] - hPy[q]) - (hC[0][qh] - hC[0][qh - 1])) * f.inv_dL;
            const uint32_t o = off[q + 2];
            if (fast) {
                R dn[3];
                dn[0] = cDxy1 * dC[0][q] + cDxy2 * ch[0];
                dn[1] = cDxy1 * dC[1][q] + cDxy2 * ch[1];
                dn[2] = cDz1 * dC[2][q] + cDz2 * ch[2];
                if (sDzk != R(0)) {
                    const R ich = zIch[q] + ch[2];
                    st_at(bp + 14 * n, o, sbytes, ich);
                    dn[2] += cDz3 * ich;
                }
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    if (ps.comp == a && xi == src_x && o == src_off) dn[a] += src_amp;
                    st_at(bp + 3 * n + a * n, o, sbytes, dn[a]);
                }
                continue;
            }
            const R sg[3] = {sDx, sDyj[q], sDzk};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const int ax_b = (a == 0) ? 1 : 0;
                const int ax_c = (a == 2) ? 1 : 2;
                const R sa = sg[a], sb = sg[ax_b], sc = sg[ax_c];
                const int64_t ca = a * n;
                const R dv = dC[a][q];
                R dn;
                if (sa == R(0) && sb == R(0) && sc == R(0)) {
                    dn = f.d1 * dv + f.d2 * ch[a];
                } else {
                    R m1, m2, m3, m4;
                    coef4<R>(sa, sb, sc, R(f.dt), R(f.c0), R(f.eps0), R(1), m1, m2, m3, m4);
                    dn = m1 * dv + m2 * ch[a];
                    if (sa != R(0)) {
                        const R ich = ich0[a][q] + ch[a];
                        st_at(bp + 12 * n + ca, o, sbytes, ich);
                        dn += m3 * ich;
                    }
                    if (sb != R(0) && sc != R(0)) {
                        const R idv = id0[a][q] + dv;
                        st_at(bp + 15 * n + ca, o, sbytes, idv);
                        dn += m4 * idv;
                    }
                }
                if (ps.comp == a && xi == src_x && o == src_off) dn += src_amp;
                st_at(bp + 3 * n + ca, o, sbytes, dn);
            }
        }
        if (more) {
#pragma unroll
            for (int q = 0; q < TJ; ++q) {
                hPy[q] = hC[1][q + 1];
                hPz[q] = hC[2][q + 1];
            }
#pragma unroll
            for (int q = 0; q < TJ + 2; ++q)
#pragma unroll
                for (int a = 0; a < 3; ++a) eC[a][q] = eN[a][q];
#pragma unroll
            for (int q = 0; q < TJ; ++q)
#pragma unroll
                for (int a = 0; a < 3; ++a) dC[a][q] = dN[a][q];
            to_E(rw, eP, eN);   // E(xi + 2)
#pragma unroll
            for (int q = 0; q < TJ + 2; ++q) eP[q] = rw.e[q + 1];
#pragma unroll
            for (int q = 0; q < TJ; ++q)
#pragma unroll
                for (int a = 0; a < 3; ++a) dN[a][q] = rw.d[a][q + 1];
#pragma unroll
            for (int q = 0; q < TJ + 1; ++q) zIce[q] = zIceN[q];
#pragma unroll
            for (int q = 0; q < TJ; ++q) zIch[q] = zIchN[q];
            put_E(eC);
            __syncthreads();
        }
    }
}

// slab kernel applicability and launch shape: nz a multiple of 64 up to
// kSlabMaxNz; bands of 2 rows when ny is even, else 1 (4-row bands hold
// more registers: fewer waves, slower at 256^3, and float64 spills); chunks
// of 8 slices (the fastest of 8, 16, 32, 64 measured at 256^3), or the
// tuning override (g_slab_target then sets the chunk from a target
// workgroup count)
static int g_slab_rows = 0, g_slab_chunk = 0, g_slab_target = 0, g_slab_map = 0;

static bool slab_shape(int nx, int ny, int nz, int elem, int& tj, int& chunk, int& nb) {
    if (nz % 64 != 0 || nz > kSlabMaxNz) return false;
    if ((int64_t)ny * nz * elem >= ((int64_t)1 << 32)) return false;   // byte offsets in a slice fit 32 bits
    tj = (ny % 2 == 0) ? 2 : 1;
    if (g_slab_rows > 0 && ny % g_slab_rows == 0) tj = g_slab_rows;
    const int tiles_y = ny / tj;
    int nch = (nx + 7) / 8;
    if (g_slab_target > 0) nch = std::max(1, std::min((g_slab_target + tiles_y - 1) / tiles_y, nx / 8));
    chunk = (nx + nch - 1) / nch;
    if (g_slab_chunk > 0) chunk = std::min(nx, g_slab_chunk);
    nch = (nx + chunk - 1) / chunk;
    nb = tiles_y * nch;
    return true;
}

template <typename R>
static void launch_slab(const Fdtd<R>& f, const R* A, R* B, PointSrc ps, const double* amp_dev, int t, int tj,
                        int chunk, int nb, hipStream_t s) {
    const int tiles_y = f.ny / tj;
    if (tj == 4) k_slab<R, 4><<<nb, f.nz, 0, s>>>(f, A, B, f.sig, f.eps, ps, amp_dev, t, tiles_y, chunk, g_slab_map);
    else if (tj == 2) k_slab<R, 2><<<nb, f.nz, 0, s>>>(f, A, B, f.sig, f.eps, ps, amp_dev, t, tiles_y, chunk, g_slab_map);
    else k_slab<R, 1><<<nb, f.nz, 0, s>>>(f, A, B, f.sig, f.eps, ps, amp_dev, t, tiles_y, chunk, g_slab_map);
}

}  // namespace cv

// Launch-shape override of the slab-marching 3D step (band rows 1, 2 or 4,
// slices per chunk, target workgroup count; 0 keeps the automatic choice;
// map_bands 1 gives each XCD a range of bands of every chunk, 0 a range of
// whole chunks), process-wide, for tuning sweeps.
extern "C" int cv_fdtd_slab_tuning(int band_rows, int chunk, int target_workgroups, int map_bands) {
    CV_CHECK(band_rows == 0 || band_rows == 1 || band_rows == 2 || band_rows == 4, "band rows must be 0, 1, 2 or 4");
    CV_CHECK(chunk >= 0 && target_workgroups >= 0, "chunk and target must be >= 0");
    cv::g_slab_rows = band_rows;
    cv::g_slab_chunk = chunk;
    cv::g_slab_target = target_workgroups;
    cv::g_slab_map = map_bands ? 1 : 0;
    return CV_OK;
}

namespace cv {

// ------------------------------------------------------------ host glue
template <typename R>
static int make_fdtd(const cv_fdtd_desc* d, const void* sig, const void* eps, void* state, Fdtd<R>& f) {
    CV_CHECK(d && sig && eps && state, "null pointer argument");
    CV_CHECK(d->nx > 0 && d->ny > 0 && d->nz > 0, "empty grid");
    f.nx = d->nx;
    f.ny = d->ny;
    f.nz = d->nz;
    f.n = (int64_t)d->nx * d->ny * d->nz;
    f.inv_dL = R(1.0 / d->dL);
    f.dt = d->dt;
    f.c0 = d->c0;
    f.eps0 = d->eps0;
    f.dL = d->dL;
    f.cdt = R(d->c0 * d->dt / d->dL);
    f.c0dt = R(d->c0 * d->dt);
    f.half_dt = R(d->dt / (2.0 * d->eps0));
    f.dL_r = R(d->dL);
    YeeConst<R>& y = f.yee;
    y.dt = R(d->dt);
    y.c0 = R(d->c0);
    y.e0 = R(d->eps0);
    y.e2 = y.e0 * y.e0;
    y.inv_dt = R(1) / y.dt;
    y.inv_e0 = R(1) / y.e0;
    y.inv_e2 = R(1) / y.e2;
    f.sig = (const R*)sig;
    f.eps = (const R*)eps;
    f.st = (R*)state;
    // interior coefficients with the reference formula at sigma = 0, in R
    const R dt = R(d->dt), c0 = R(d->c0), e0 = R(d->eps0);
    const R m0 = (R(1) / dt + (R(0) + R(0)) / R(2) / e0 + R(0) * R(0) * dt / R(4) / (e0 * e0));
    f.h1 = (R(1) / m0 * (R(1) / dt - (R(0) + R(0)) / R(2) / e0 - R(0) * R(0) * dt / R(4) / (e0 * e0)));
    f.h2 = R(-1) / m0 * c0;
    f.d1 = f.h1;
    f.d2 = R(1) / m0 * c0;
    return CV_OK;
}

// Cells per thread of the two-phase kernels: 16 bytes (4 float32 or 2 float64)
// where nz and every array allow aligned vectors, else the widest that does.
template <typename R>
static int step_width(const Fdtd<R>& f, std::initializer_list<const void*> arrays) {
    int v = 16 / (int)sizeof(R);
    uintptr_t bits = 0;
    for (const void* p : arrays) bits |= (uintptr_t)p;
    while (v > 1 && (f.nz % v != 0 || bits % (v * sizeof(R)) != 0)) v >>= 1;
    return v;
}

static inline unsigned int nblk(int64_t n) { return (unsigned int)((n + 255) / 256); }

}  // namespace cv

using namespace cv;

namespace cv {

template <typename R>
static void launch_h(const Fdtd<R>& f, const R* D, hipStream_t s) {
    const int v = step_width(f, {f.st, D, f.eps});
    if constexpr (sizeof(R) == 4)
        if (v == 4) {
            k_h<R, 4><<<nblk(f.n / 4), 256, 0, s>>>(f, D);
            return;
        }
    if (v == 2) k_h<R, 2><<<nblk(f.n / 2), 256, 0, s>>>(f, D);
    else k_h<R, 1><<<nblk(f.n), 256, 0, s>>>(f, D);
}

template <typename R>
static void launch_d(const Fdtd<R>& f, const R* Din, R* Dout, const R* Jx, const R* Jy, const R* Jz, R jscale,
                     PointSrc ps, hipStream_t s) {
    const int v = step_width(f, {f.st, Din, Dout});
    if constexpr (sizeof(R) == 4)
        if (v == 4) {
            k_d<R, 4><<<nblk(f.n / 4), 256, 0, s>>>(f, Din, Dout, Jx, Jy, Jz, jscale, ps);
            return;
        }
    if (v == 2) k_d<R, 2><<<nblk(f.n / 2), 256, 0, s>>>(f, Din, Dout, Jx, Jy, Jz, jscale, ps);
    else k_d<R, 1><<<nblk(f.n), 256, 0, s>>>(f, Din, Dout, Jx, Jy, Jz, jscale, ps);
}

template <typename R>
static void launch_adjoint(const Fdtd<R>& f, R* lam, R* T, const R* Dprev, R* gmE, int src_comp, int64_t src_cell,
                           R* g_src, hipStream_t s) {
    const int v = step_width(f, {lam, T, Dprev, gmE, f.eps});
    if constexpr (sizeof(R) == 4)
        if (v == 4) {
            k_adj_a<R, 4><<<nblk(f.n / 4), 256, 0, s>>>(f, lam, T, src_comp, src_cell, g_src);
            k_adj_b<R, 4><<<nblk(f.n / 4), 256, 0, s>>>(f, lam, T, Dprev, gmE);
            return;
        }
    if (v == 2) {
        k_adj_a<R, 2><<<nblk(f.n / 2), 256, 0, s>>>(f, lam, T, src_comp, src_cell, g_src);
        k_adj_b<R, 2><<<nblk(f.n / 2), 256, 0, s>>>(f, lam, T, Dprev, gmE);
    } else {
        k_adj_a<R, 1><<<nblk(f.n), 256, 0, s>>>(f, lam, T, src_comp, src_cell, g_src);
        k_adj_b<R, 1><<<nblk(f.n), 256, 0, s>>>(f, lam, T, Dprev, gmE);
    }
}

template <typename R>
static int step_impl(const cv_fdtd_desc* d, const void* sig, const void* eps, void* state, const void* Jx,
                     const void* Jy, const void* Jz, double jscale, int src_comp, int64_t src_cell, const double* amp,
                     int n_steps, const int32_t* probe_comp, const int64_t* probe_cell, int n_probes, void* rec,
                     hipStream_t s) {
    Fdtd<R> f;
    int rc = make_fdtd<R>(d, sig, eps, state, f);
    if (rc) return rc;
    CV_CHECK(src_comp < 0 || (src_cell >= 0 && src_cell < f.n), "source cell out of range");
    R* D = f.st + 3 * f.n;
    for (int t = 0; t < n_steps; ++t) {
        const PointSrc ps{src_comp, src_cell, (src_comp >= 0 && amp) ? amp[t] : 0.0, nullptr};
        launch_h(f, D, s);
        launch_d(f, D, D, (const R*)Jx, (const R*)Jy, (const R*)Jz, R(jscale), ps, s);
        if (n_probes > 0)
            k_record<R><<<(n_probes + 63) / 64, 64, 0, s>>>(f, probe_comp, probe_cell, n_probes,
                                                            (R*)rec + (int64_t)t * n_probes);
    }
    CV_LAUNCH_CHECK();
    return CV_OK;
}

template <typename R>
static int step_history_impl(const cv_fdtd_desc* d, const void* sig, const void* eps, void* state, void* D_hist,
                             int src_comp, int64_t src_cell, const double* amp_dev, int n_steps, hipStream_t s) {
    Fdtd<R> f;
    int rc = make_fdtd<R>(d, sig, eps, state, f);
    if (rc) return rc;
    CV_CHECK(src_comp < 0 || (src_cell >= 0 && src_cell < f.n), "source cell out of range");
    R* D = (R*)D_hist;
    CV_HIP(hipMemcpyAsync(D, f.st + 3 * f.n, sizeof(R) * 3 * f.n, hipMemcpyDeviceToDevice, s));
    for (int t = 0; t < n_steps; ++t, D += 3 * f.n) {
        const PointSrc ps{src_comp, src_cell, 0.0, src_comp >= 0 ? amp_dev + t : nullptr};
        launch_h(f, D, s);
        launch_d<R>(f, D, D + 3 * f.n, nullptr, nullptr, nullptr, R(1), ps, s);
    }
    CV_LAUNCH_CHECK();
    return CV_OK;
}

}  // namespace cv

extern "C" int cv_fdtd_step(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps, void* state,
                            const void* Jx, const void* Jy, const void* Jz, double jscale, int src_comp,
                            int64_t src_cell, const double* amp, int n_steps, const int32_t* probe_comp,
                            const int64_t* probe_cell, int n_probes, void* rec, void* stream) {
    hipStream_t s = as_stream(stream);
    CV_CHECK(n_steps >= 0, "n_steps < 0");
    CV_CHECK(src_comp >= -1 && src_comp < 3, "src_comp must be -1 (none) or 0..2");
    CV_CHECK(n_probes == 0 || (probe_comp && probe_cell && rec), "probes need comp, cell and rec buffers");
    if (dtype == CV_F32)
        return step_impl<float>(d, sig, eps, state, Jx, Jy, Jz, jscale, src_comp, src_cell, amp, n_steps, probe_comp,
                                probe_cell, n_probes, rec, s);
    if (dtype == CV_F64)
        return step_impl<double>(d, sig, eps, state, Jx, Jy, Jz, jscale, src_comp, src_cell, amp, n_steps, probe_comp,
                                 probe_cell, n_probes, rec, s);
    CV_CHECK(false, "unknown dtype %d", dtype);
}

extern "C" int cv_fdtd_step_history(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps, void* state,
                                    void* D_hist, int src_comp, int64_t src_cell, const double* amp_dev, int n_steps,
                                    void* stream) {
    hipStream_t s = as_stream(stream);
    CV_CHECK(D_hist, "null history buffer");
    CV_CHECK(n_steps >= 0, "n_steps < 0");
    CV_CHECK(src_comp >= -1 && src_comp < 3, "src_comp must be -1 (none) or 0..2");
    CV_CHECK(src_comp < 0 || amp_dev, "a source needs its amplitude array");
    if (dtype == CV_F32)
        return step_history_impl<float>(d, sig, eps, state, D_hist, src_comp, src_cell, amp_dev, n_steps, s);
    if (dtype == CV_F64)
        return step_history_impl<double>(d, sig, eps, state, D_hist, src_comp, src_cell, amp_dev, n_steps, s);
    CV_CHECK(false, "unknown dtype %d", dtype);
}

template <typename R>
static int step_tangent_impl(const cv_fdtd_desc* d, const void* sig, const void* eps, void* state, void* tstate,
                             const void* deps, const void* Jx, const void* Jy, const void* Jz, const void* dJx,
                             const void* dJy, const void* dJz, double jscale, int src_comp, int64_t src_cell,
                             const double* amp, const double* damp, int n_steps, const int32_t* probe_comp,
                             const int64_t* probe_cell, int n_probes, void* rec, void* trec, hipStream_t s) {
    Fdtd<R> f, ft;
    int rc = make_fdtd<R>(d, sig, eps, state, f);
    if (rc) return rc;
    rc = make_fdtd<R>(d, sig, eps, tstate, ft);
    if (rc) return rc;
    CV_CHECK(src_comp < 0 || (src_cell >= 0 && src_cell < f.n), "source cell out of range");
    const R* D = f.st + 3 * f.n;
    for (int t = 0; t < n_steps; ++t) {
        PointSrc ps{src_comp, src_cell, (src_comp >= 0 && amp) ? amp[t] : 0.0, nullptr};
        PointSrc pt{src_comp, src_cell, (src_comp >= 0 && damp) ? damp[t] : 0.0, nullptr};
        launch_h(f, D, s);
        k_h_tangent<R><<<nblk(f.n), 256, 0, s>>>(ft, D, (const R*)deps);   // primal D still at step t
        R* dD = ft.st + 3 * ft.n;
        launch_d(f, D, f.st + 3 * f.n, (const R*)Jx, (const R*)Jy, (const R*)Jz, R(jscale), ps, s);
        launch_d(ft, dD, dD, (const R*)dJx, (const R*)dJy, (const R*)dJz, R(jscale), pt, s);
        if (n_probes > 0) {
            if (rec)
                k_record<R><<<(n_probes + 63) / 64, 64, 0, s>>>(f, probe_comp, probe_cell, n_probes,
                                                                (R*)rec + (int64_t)t * n_probes);
            k_record_tangent<R><<<(n_probes + 63) / 64, 64, 0, s>>>(f, ft, (const R*)deps, probe_comp, probe_cell,
                                                                    n_probes, (R*)trec + (int64_t)t * n_probes);
        }
    }
    CV_LAUNCH_CHECK();
    return CV_OK;
}

extern "C" int cv_fdtd_step_tangent(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps,
                                    void* state, void* tstate, const void* d_eps, const void* Jx, const void* Jy,
                                    const void* Jz, const void* dJx, const void* dJy, const void* dJz,
                                    double jscale, int src_comp, int64_t src_cell, const double* amp,
                                    const double* d_amp, int n_steps, const int32_t* probe_comp,
                                    const int64_t* probe_cell, int n_probes, void* rec, void* trec, void* stream) {
    CV_CHECK(n_steps >= 0, "n_steps < 0");
    CV_CHECK(state && tstate && d_eps && state != tstate, "null or aliased state / tangent buffers");
    CV_CHECK(src_comp >= -1 && src_comp < 3, "src_comp must be -1 (none) or 0..2");
    CV_CHECK(n_probes == 0 || (probe_comp && probe_cell && trec), "probes need comp, cell and trec buffers");
    hipStream_t s = as_stream(stream);
    if (dtype == CV_F32)
        return step_tangent_impl<float>(d, sig, eps, state, tstate, d_eps, Jx, Jy, Jz, dJx, dJy, dJz, jscale,
                                        src_comp, src_cell, amp, d_amp, n_steps, probe_comp, probe_cell, n_probes,
                                        rec, trec, s);
    if (dtype == CV_F64)
        return step_tangent_impl<double>(d, sig, eps, state, tstate, d_eps, Jx, Jy, Jz, dJx, dJy, dJz, jscale,
                                         src_comp, src_cell, amp, d_amp, n_steps, probe_comp, probe_cell, n_probes,
                                         rec, trec, s);
    CV_CHECK(false, "unknown dtype %d", dtype);
}

template <typename R>
__global__ void __launch_bounds__(256) k_efields_tangent(Fdtd<R> f, const R* __restrict__ dD,
                                                         const R* __restrict__ deps, R* __restrict__ dE) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= f.n) return;
    int i, j, k;
    decompose(f, c, i, j, k);
#pragma unroll
    for (int a = 0; a < 3; ++a) dE[a * f.n + c] = efield_tangent(f, f.st + 3 * f.n, dD, deps, a, i, j, k);
}

extern "C" int cv_fdtd_efields_tangent(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps,
                                       const void* state, const void* tstate, const void* d_eps, void* dE,
                                       void* stream) {
    CV_CHECK(state && tstate && d_eps && dE, "null pointer argument");
    hipStream_t s = as_stream(stream);
    if (dtype == CV_F32) {
        Fdtd<float> f;
        int rc = make_fdtd<float>(d, sig, eps, const_cast<void*>(state), f);
        if (rc) return rc;
        k_efields_tangent<float><<<nblk(f.n), 256, 0, s>>>(f, (const float*)tstate + 3 * f.n, (const float*)d_eps,
                                                           (float*)dE);
    } else if (dtype == CV_F64) {
        Fdtd<double> f;
        int rc = make_fdtd<double>(d, sig, eps, const_cast<void*>(state), f);
        if (rc) return rc;
        k_efields_tangent<double><<<nblk(f.n), 256, 0, s>>>(f, (const double*)tstate + 3 * f.n,
                                                            (const double*)d_eps, (double*)dE);
    } else {
        CV_CHECK(false, "unknown dtype %d", dtype);
    }
    CV_LAUNCH_CHECK();
    return CV_OK;
}

extern "C" int cv_fdtd_efields(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps,
                               const void* state, void* E, void* stream) {
    hipStream_t s = as_stream(stream);
    CV_CHECK(E, "null E");
    if (dtype == CV_F32) {
        Fdtd<float> f;
        int rc = make_fdtd<float>(d, sig, eps, (void*)state, f);
        if (rc) return rc;
        k_efields<float><<<nblk(f.n), 256, 0, s>>>(f, (float*)E);
    } else if (dtype == CV_F64) {
        Fdtd<double> f;
        int rc = make_fdtd<double>(d, sig, eps, (void*)state, f);
        if (rc) return rc;
        k_efields<double><<<nblk(f.n), 256, 0, s>>>(f, (double*)E);
    } else {
        CV_CHECK(false, "unknown dtype %d", dtype);
    }
    CV_LAUNCH_CHECK();
    return CV_OK;
}

namespace cv {

// n_steps adjoint steps, last first; D_hist: D before step t at D_hist + t * 3 n
template <typename R>
static int adjoint_impl(const cv_fdtd_desc* d, const void* sig, const void* eps, void* lam_, void* tmp,
                        const void* D_prev, const void* D_after, int64_t D_stride, void* g_mE,
                        const int32_t* probe_comp, const int64_t* probe_cell, int n_probes, const void* g_probe,
                        int src_comp, int64_t src_cell, void* g_src, int n_steps, hipStream_t s) {
    Fdtd<R> f;
    int rc = make_fdtd<R>(d, sig, eps, lam_, f);
    if (rc) return rc;
    R* lam = (R*)lam_;
    CV_CHECK(!g_src || (src_comp >= 0 && src_comp < 3 && src_cell >= 0 && src_cell < f.n),
             "source gradient requested for an invalid source (%d, %lld)", src_comp, (long long)src_cell);
    for (int t = n_steps - 1; t >= 0; --t) {
        if (n_probes > 0 && g_probe)
            k_inject<R><<<(n_probes + 255) / 256, 256, 0, s>>>(f, lam, probe_comp, probe_cell, n_probes,
                                                               (const R*)g_probe + (int64_t)t * n_probes,
                                                               (const R*)D_after + t * D_stride, (R*)g_mE);
        launch_adjoint(f, lam, (R*)tmp, (const R*)D_prev + t * D_stride, (R*)g_mE, src_comp, src_cell,
                       g_src ? (R*)g_src + t : nullptr, s);
    }
    CV_LAUNCH_CHECK();
    return CV_OK;
}

}  // namespace cv

extern "C" int cv_fdtd_adjoint_step(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps,
                                    void* lam, void* tmp, const void* D_prev, void* g_mE, const int32_t* probe_comp,
                                    const int64_t* probe_cell, int n_probes, const void* g_probe,
                                    const void* D_t, int src_comp, int64_t src_cell, void* g_src, void* stream) {
    hipStream_t s = as_stream(stream);
    CV_CHECK(lam && tmp, "null adjoint buffers");
    if (dtype == CV_F32)
        return adjoint_impl<float>(d, sig, eps, lam, tmp, D_prev, D_t, 0, g_mE, probe_comp, probe_cell, n_probes,
                                   g_probe, src_comp, src_cell, g_src, 1, s);
    if (dtype == CV_F64)
        return adjoint_impl<double>(d, sig, eps, lam, tmp, D_prev, D_t, 0, g_mE, probe_comp, probe_cell, n_probes,
                                    g_probe, src_comp, src_cell, g_src, 1, s);
    CV_CHECK(false, "unknown dtype %d", dtype);
}

extern "C" int cv_fdtd_adjoint_steps(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps, void* lam,
                                     void* tmp, const void* D_hist, void* g_mE, const int32_t* probe_comp,
                                     const int64_t* probe_cell, int n_probes, const void* g_rec, int src_comp,
                                     int64_t src_cell, void* g_amp, int n_steps, void* stream) {
    hipStream_t s = as_stream(stream);
    CV_CHECK(d && lam && tmp && D_hist && g_mE, "null adjoint buffers");
    CV_CHECK(n_steps >= 0, "n_steps < 0");
    CV_CHECK(n_probes == 0 || !g_rec || (probe_comp && probe_cell), "probes need comp and cell buffers");
    const int64_t n3 = 3 * (int64_t)d->nx * d->ny * d->nz;
    if (dtype == CV_F32)
        return adjoint_impl<float>(d, sig, eps, lam, tmp, D_hist, (const float*)D_hist + n3, n3, g_mE, probe_comp,
                                   probe_cell, n_probes, g_rec, src_comp, src_cell, g_amp, n_steps, s);
    if (dtype == CV_F64)
        return adjoint_impl<double>(d, sig, eps, lam, tmp, D_hist, (const double*)D_hist + n3, n3, g_mE, probe_comp,
                                    probe_cell, n_probes, g_rec, src_comp, src_cell, g_amp, n_steps, s);
    CV_CHECK(false, "unknown dtype %d", dtype);
}

extern "C" int cv_fdtd_eps_grad(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps,
                                const void* g_mE, void* g_eps, void* stream) {
    hipStream_t s = as_stream(stream);
    CV_CHECK(g_mE && g_eps, "null gradient buffers");
    if (dtype == CV_F32) {
        Fdtd<float> f;
        int rc = make_fdtd<float>(d, sig, eps, (void*)g_mE, f);
        if (rc) return rc;
        k_eps_grad<float><<<nblk(f.n), 256, 0, s>>>(f, (const float*)g_mE, (float*)g_eps);
    } else if (dtype == CV_F64) {
        Fdtd<double> f;
        int rc = make_fdtd<double>(d, sig, eps, (void*)g_mE, f);
        if (rc) return rc;
        k_eps_grad<double><<<nblk(f.n), 256, 0, s>>>(f, (const double*)g_mE, (double*)g_eps);
    } else {
        CV_CHECK(false, "unknown dtype %d", dtype);
    }
    CV_LAUNCH_CHECK();
    return CV_OK;
}

extern "C" int cv_fdtd_efields_grad(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps,
                                    const void* state, const void* gE, void* gD, void* g_mE, void* stream) {
    hipStream_t s = as_stream(stream);
    CV_CHECK(gE && gD, "null gradient buffers");
    if (dtype == CV_F32) {
        Fdtd<float> f;
        int rc = make_fdtd<float>(d, sig, eps, (void*)state, f);
        if (rc) return rc;
        k_efields_grad<float><<<nblk(f.n), 256, 0, s>>>(f, (const float*)gE, (float*)gD, (float*)g_mE);
    } else if (dtype == CV_F64) {
        Fdtd<double> f;
        int rc = make_fdtd<double>(d, sig, eps, (void*)state, f);
        if (rc) return rc;
        k_efields_grad<double><<<nblk(f.n), 256, 0, s>>>(f, (const double*)gE, (double*)gD, (double*)g_mE);
    } else {
        CV_CHECK(false, "unknown dtype %d", dtype);
    }
    CV_LAUNCH_CHECK();
    return CV_OK;
}

extern "C" int cv_fdtd_tm_configs(int* rpt, int* ts, int* waves, int max_n) {
    static const int R_[kTmConfigs] = {4, 4, 8, 8, 16, 16, 4, 4, 2, 4, 4, 2};
    static const int T_[kTmConfigs] = {2, 4, 4, 8, 8, 4, 8, 16, 8, 8, 4, 4};
    static const int W_[kTmConfigs] = {4, 4, 4, 4, 4, 4, 8, 16, 16, 16, 8, 16};
    for (int i = 0; i < kTmConfigs && i < max_n; ++i) {
        if (rpt) rpt[i] = R_[i];
        if (ts) ts[i] = T_[i];
        if (waves) waves[i] = W_[i];
    }
    return kTmConfigs;
}

namespace cv {

template <typename R>
static int run_tm_impl(const cv_fdtd_desc* d, const void* sig, const void* eps, void* state, void* state_alt,
                       int64_t src_cell, const double* amp_dev, int t0, int n_steps, TmProbes probes, void* rec,
                       int rec_t0, int config, hipStream_t s) {
    Fdtd<R> f;
    int rc = make_fdtd<R>(d, sig, eps, state, f);
    if (rc) return rc;
    CV_CHECK(src_cell < f.n, "source cell out of range");
    if (n_steps <= 0) return CV_OK;
    TmArgs<R> a = tm_args(f);
    tm_source(a, src_cell);
    a.amp = amp_dev;
    a.probes = probes;
    a.rec = (R*)rec;
    a.rec_t0 = rec_t0;
    a.t0 = t0;
    const TmState<R> A = tm_of_state(f.st, f.n), B = tm_of_state((R*)state_alt, f.n);
    int ts[kTmConfigs];
    cv_fdtd_tm_configs(nullptr, ts, nullptr, kTmConfigs);
    // the last launch may not write the buffer it reads: an odd number of
    // launches ends in the other one and is copied back
    const bool odd = ((n_steps + ts[config] - 1) / ts[config]) % 2 != 0;
    rc = dispatch_tm<R>(config, a, A, odd ? B : A, A, B, n_steps, false, s);
    if (rc) return rc;
    if (odd) tm_copy(a, B, A, s);
    return CV_OK;
}

template <typename R>
static int run_tm_checkpoints_impl(const cv_fdtd_desc* d, const void* sig, const void* eps, void* state, void* work,
                                   void* checkpoints, int checkpoint_every, int64_t src_cell, const double* amp_dev,
                                   int n_steps, TmProbes probes, void* rec, int config, hipStream_t s) {
    Fdtd<R> f;
    int rc = make_fdtd<R>(d, sig, eps, state, f);
    if (rc) return rc;
    CV_CHECK(src_cell < f.n, "source cell out of range");
    if (n_steps <= 0) return CV_OK;
    TmArgs<R> a = tm_args(f);
    tm_source(a, src_cell);
    a.amp = amp_dev;
    a.probes = probes;
    a.rec = (R*)rec;
    const TmState<R> A = tm_of_state(f.st, f.n);
    const TmState<R> w0 = tm_of_packed((R*)work, f.n), w1 = tm_of_packed((R*)work + 6 * f.n, f.n);
    auto ck = [&](int k) { return tm_of_packed((R*)checkpoints + (int64_t)k * 6 * f.n, f.n); };
    // a segment's last launch writes the next checkpoint, the run's last one the state
    tm_copy(a, A, ck(0), s);
    for (int k = 0, t = 0; t < n_steps; ++k, t += checkpoint_every) {
        const int m = std::min(checkpoint_every, n_steps - t);
        a.t0 = t;
        rc = dispatch_tm<R>(config, a, ck(k), t + m < n_steps ? ck(k + 1) : A, w0, w1, m, false, s);
        if (rc) return rc;
    }
    return CV_OK;
}

template <typename R>
static int tm_adjoint_impl(const cv_fdtd_desc* d, const void* sig, const void* eps, const void* checkpoints,
                           int checkpoint_every, int64_t src_cell, const double* amp_dev, int n_steps, void* work,
                           void* dz_hist, void* lam, void* g_mEz, TmProbes probes, const void* g_rec, void* g_amp,
                           int config, hipStream_t s) {
    Fdtd<R> f;
    int rc = make_fdtd<R>(d, sig, eps, lam, f);
    if (rc) return rc;
    CV_CHECK(src_cell < f.n, "source cell out of range");
    const int64_t n = f.n;
    const TmState<R> w0 = tm_of_packed((R*)work, n), w1 = tm_of_packed((R*)work + 6 * n, n);
    const TmState<R> l0 = tm_of_packed((R*)lam, n), l1 = tm_of_packed((R*)lam + 6 * n, n);
    R* hist = (R*)dz_hist;
    const int nseg = n_steps > 0 ? (n_steps + checkpoint_every - 1) / checkpoint_every : 0;
    TmState<R> cur = l0;
    // The adjoint holds about 1.4 times the forward kernel's registers.  In
    // float64, 16 waves of more than two rows a thread do not fit 128 of them
    // (20 us a step with three rows, spilling, against 9.8 us with two, at
    // 1211 x 901), so those shapes take the two-row one.
    const int adj = sizeof(R) == 8 && (config == 7 || config == 9) ? 8 : config;
    for (int k = nseg - 1; k >= 0; --k) {
        const int t = k * checkpoint_every, m = std::min(checkpoint_every, n_steps - t);
        const TmState<R> start = tm_of_packed((R*)checkpoints + (int64_t)k * 6 * n, n);
        // the segment again, with Dz after each of its steps
        TmArgs<R> a = tm_args(f);
        a.t0 = t;
        tm_source(a, src_cell);
        a.amp = amp_dev;
        a.hist = hist;
        rc = dispatch_tm<R>(config, a, start, TmState<R>{}, w0, w1, m, false, s);
        if (rc) return rc;
        TmArgs<R> b = tm_args(f);
        b.t0 = t;
        tm_source(b, src_cell);
        b.probes = probes;
        b.grec = (const R*)g_rec;
        b.gamp = (R*)g_amp;
        b.gm = (R*)g_mEz;
        b.dz_hist = hist;
        b.dz_before = start.dz;
        const TmState<R> other = cur.hx == l0.hx ? l1 : l0;
        int ts[kTmConfigs];
        cv_fdtd_tm_configs(nullptr, ts, nullptr, kTmConfigs);
        const bool odd = ((m + ts[adj] - 1) / ts[adj]) % 2 != 0;
        const TmState<R> end = odd ? other : cur;
        rc = dispatch_tm<R>(adj, b, cur, end, l0, l1, m, true, s);
        if (rc) return rc;
        cur = end;
    }
    if (cur.hx != l0.hx) tm_copy(tm_args(f), cur, l0, s);
    return CV_OK;
}

static int tm_checks(const cv_fdtd_desc* d, int n_steps, const int32_t* probe_comp, const int64_t* probe_cell,
                     int n_probes, int64_t src_cell, const double* amp_dev, int config) {
    CV_CHECK(d && d->nz == 1, "the TM kernel needs nz == 1");
    CV_CHECK(n_probes >= 0 && n_probes <= kTmMaxProbes, "the TM kernel records at most %d probes", kTmMaxProbes);
    CV_CHECK(n_steps >= 0, "bad step range");
    CV_CHECK(n_probes == 0 || (probe_comp && probe_cell), "probes need comp and cell buffers");
    CV_CHECK(src_cell < 0 || amp_dev, "a source needs its amplitude array");
    CV_CHECK(config >= 0 && config < kTmConfigs,
             "unknown TM tile configuration %d", config);
    return CV_OK;
}

}  // namespace cv

extern "C" int cv_fdtd_run_tm(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps, void* state,
                              void* state_alt, int64_t src_cell, const double* amp_dev, int t0, int n_steps,
                              const int32_t* probe_comp, const int64_t* probe_cell, int n_probes, void* rec,
                              int rec_t0, int config, void* stream) {
    hipStream_t s = as_stream(stream);
    CV_CHECK(state && state_alt && state != state_alt, "two distinct state buffers are needed");
    CV_CHECK(t0 >= 0, "bad step range");
    CV_CHECK(n_probes == 0 || rec, "probes need a record buffer");
    int rc = tm_checks(d, n_steps, probe_comp, probe_cell, n_probes, src_cell, amp_dev, config);
    if (rc) return rc;
    const TmProbes pr{probe_comp, probe_cell, n_probes};
    if (dtype == CV_F32)
        rc = run_tm_impl<float>(d, sig, eps, state, state_alt, src_cell, amp_dev, t0, n_steps, pr, rec, rec_t0, config,
                                s);
    else if (dtype == CV_F64)
        rc = run_tm_impl<double>(d, sig, eps, state, state_alt, src_cell, amp_dev, t0, n_steps, pr, rec, rec_t0, config,
                                 s);
    else
        CV_CHECK(false, "unknown dtype %d", dtype);
    if (rc) return rc;
    CV_LAUNCH_CHECK();
    return CV_OK;
}

extern "C" int cv_fdtd_run_tm_checkpoints(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps,
                                          void* state, void* work, void* checkpoints, int checkpoint_every,
                                          int64_t src_cell, const double* amp_dev, int n_steps,
                                          const int32_t* probe_comp, const int64_t* probe_cell, int n_probes, void* rec,
                                          int config, void* stream) {
    hipStream_t s = as_stream(stream);
    CV_CHECK(state && work && checkpoints, "null pointer argument");
    CV_CHECK(checkpoint_every > 0, "checkpoint_every must be positive");
    CV_CHECK(n_probes == 0 || rec, "probes need a record buffer");
    int rc = tm_checks(d, n_steps, probe_comp, probe_cell, n_probes, src_cell, amp_dev, config);
    if (rc) return rc;
    const TmProbes pr{probe_comp, probe_cell, n_probes};
    if (dtype == CV_F32)
        rc = run_tm_checkpoints_impl<float>(d, sig, eps, state, work, checkpoints, checkpoint_every, src_cell, amp_dev,
                                            n_steps, pr, rec, config, s);
    else if (dtype == CV_F64)
        rc = run_tm_checkpoints_impl<double>(d, sig, eps, state, work, checkpoints, checkpoint_every, src_cell, amp_dev,
                                             n_steps, pr, rec, config, s);
    else
        CV_CHECK(false, "unknown dtype %d", dtype);
    if (rc) return rc;
    CV_LAUNCH_CHECK();
    return CV_OK;
}

extern "C" int cv_fdtd_tm_adjoint(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps,
                                  const void* checkpoints, int checkpoint_every, int64_t src_cell,
                                  const double* amp_dev, int n_steps, void* work, void* dz_hist, void* lam,
                                  void* g_mEz, const int32_t* probe_comp, const int64_t* probe_cell, int n_probes,
                                  const void* g_rec, void* g_amp, int config, void* stream) {
    hipStream_t s = as_stream(stream);
    CV_CHECK(checkpoints && work && dz_hist && lam && g_mEz, "null pointer argument");
    CV_CHECK(checkpoint_every > 0, "checkpoint_every must be positive");
    int rc = tm_checks(d, n_steps, probe_comp, probe_cell, n_probes, src_cell, amp_dev, config);
    if (rc) return rc;
    const TmProbes pr{probe_comp, probe_cell, n_probes};
    if (dtype == CV_F32)
        rc = tm_adjoint_impl<float>(d, sig, eps, checkpoints, checkpoint_every, src_cell, amp_dev, n_steps, work,
                                    dz_hist, lam, g_mEz, pr, g_rec, g_amp, config, s);
    else if (dtype == CV_F64)
        rc = tm_adjoint_impl<double>(d, sig, eps, checkpoints, checkpoint_every, src_cell, amp_dev, n_steps, work,
                                     dz_hist, lam, g_mEz, pr, g_rec, g_amp, config, s);
    else
        CV_CHECK(false, "unknown dtype %d", dtype);
    if (rc) return rc;
    CV_LAUNCH_CHECK();
    return CV_OK;
}

extern "C" int cv_fdtd_run_fused(int dtype, const cv_fdtd_desc* d, const void* sig, const void* eps, void* state_a,
                                 void* state_b, int comp, int64_t src_cell, const double* amp_dev, int t0,
                                 int n_steps, const int32_t* probe_comp, const int64_t* probe_cell, int n_probes,
                                 void* rec, int rec_t0, void* stream) {
    hipStream_t s = as_stream(stream);
    CV_CHECK(state_a && state_b && state_a != state_b, "two distinct state buffers are needed");
    CV_CHECK(comp >= -1 && comp < 3, "comp must be -1 (none) or 0..2");
    CV_CHECK(comp < 0 || amp_dev, "a source needs its amplitude array");
    CV_CHECK(n_probes == 0 || (probe_comp && probe_cell && rec), "probes need comp, cell and rec buffers");
    if (dtype == CV_F32) {
        Fdtd<float> f;
        int rc = make_fdtd<float>(d, sig, eps, state_a, f);
        if (rc) return rc;
        CV_CHECK(comp < 0 || (src_cell >= 0 && src_cell < f.n), "source cell out of range");
        float* A = (float*)state_a;
        float* B = (float*)state_b;
        for (int t = 0; t < n_steps; ++t) {
            PointSrc ps{comp, src_cell, 0.0, nullptr};
            int tj, chunk_s, nb_s;
            if (f.nz > 1 && slab_shape(f.nx, f.ny, f.nz, 4, tj, chunk_s, nb_s)) {
                launch_slab<float>(f, A, B, ps, amp_dev, t0 + t, tj, chunk_s, nb_s, s);
            } else if (f.nz > 1) {
                const int ty = (f.ny + kMOwnY - 1) / kMOwnY, tz = (f.nz + kMOwnZ - 1) / kMOwnZ;
                const int nch = std::max(1, std::min(f.nx / 4 > 0 ? f.nx / 4 : 1, (2048 + ty * tz - 1) / (ty * tz)));
                const int chunk = (f.nx + nch - 1) / nch;
                const int nb = ty * tz * ((f.nx + chunk - 1) / chunk);
                k_march<float, 1><<<nb, 64 * kMRows, 0, s>>>(f, A, B, ps, amp_dev, t0 + t, ty, tz, chunk);
            } else {
                k_fused<float><<<nblk(f.n), 256, 0, s>>>(f, A, B, ps, amp_dev, t0 + t);
            }
            if (n_probes > 0) {
                Fdtd<float> g = f;
                g.st = B;
                k_record<float><<<(n_probes + 63) / 64, 64, 0, s>>>(g, probe_comp, probe_cell, n_probes,
                                                                    (float*)rec + (int64_t)(t0 + t - rec_t0) * n_probes);
            }
            float* tmp = A;
            A = B;
            B = tmp;
        }
    } else if (dtype == CV_F64) {
        Fdtd<double> f;
        int rc = make_fdtd<double>(d, sig, eps, state_a, f);
        if (rc) return rc;
        CV_CHECK(comp < 0 || (src_cell >= 0 && src_cell < f.n), "source cell out of range");
        double* A = (double*)state_a;
        double* B = (double*)state_b;
        for (int t = 0; t < n_steps; ++t) {
            PointSrc ps{comp, src_cell, 0.0, nullptr};
            int tj, chunk_s, nb_s;
            if (f.nz > 1 && slab_shape(f.nx, f.ny, f.nz, 8, tj, chunk_s, nb_s)) {
                launch_slab<double>(f, A, B, ps, amp_dev, t0 + t, tj, chunk_s, nb_s, s);
            } else if (f.nz > 1) {
                const int ty = (f.ny + kMOwnY - 1) / kMOwnY, tz = (f.nz + kMOwnZ - 1) / kMOwnZ;
                const int nch = std::max(1, std::min(f.nx / 4 > 0 ? f.nx / 4 : 1, (2048 + ty * tz - 1) / (ty * tz)));
                const int chunk = (f.nx + nch - 1) / nch;
                const int nb = ty * tz * ((f.nx + chunk - 1) / chunk);
                k_march<double, 1><<<nb, 64 * kMRows, 0, s>>>(f, A, B, ps, amp_dev, t0 + t, ty, tz, chunk);
            } else {
                k_fused<double><<<nblk(f.n), 256, 0, s>>>(f, A, B, ps, amp_dev, t0 + t);
            }
            if (n_probes > 0) {
                Fdtd<double> g = f;
                g.st = B;
                k_record<double><<<(n_probes + 63) / 64, 64, 0, s>>>(g, probe_comp, probe_cell, n_probes,
                                                                     (double*)rec + (int64_t)(t0 + t - rec_t0) * n_probes);
            }
            double* tmp = A;
            A = B;
            B = tmp;
        }
    } else {
        CV_CHECK(false, "unknown dtype %d", dtype);
    }
    CV_LAUNCH_CHECK();
    return CV_OK;
}
