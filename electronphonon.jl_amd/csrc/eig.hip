// Batched Hermitian eigensolve for small matrices (n <= 32), one wavefront or a part of one per matrix.
//
// Replaces the reference's eigen_batched / eigvals_batched (src/wannier_to_bloch_batched.jl:30-65,
// CUDA method ext/ElectronPhononCUDAExt.jl:80-115): ascending eigenvalues, orthonormal eigenvectors,
// no degeneracy gauge fixing (the reference's batched path applies none either). The per-k path's
// degenerate-band gauge fixing (solve_eigen_el!, src/diagonalize.jl:47-85) is a separate kernel at the end
// of this file, applied to the eigenpairs afterwards.
//
// Method (FP32, all in LDS and registers; 8, 16 or 32 lanes of a wave a matrix, so up to 8 matrices a wave):
//   1. Householder reduction of the Hermitian matrix to tridiagonal form, one reflector per column;
//      the reflector vectors are kept in the zeroed part of the matrix for the back-transform.
//   2. Diagonal phase scaling turns the complex tridiagonal into a real symmetric one.
//   3. Implicit QL with Wilkinson-type shifts on (d, e) (the published EISPACK imtql2 scheme): every lane
//      of a matrix runs the scalar recurrence on d and e in LDS, the rotations are applied to the rows of Z
//      in parallel (lane = row).
//   4. Eigenvectors V = H_0 ... H_{n-3} D Z, one column per lane.
// Bound by the chain of a rotation (hypot, two quotients, the recurrence) and by the instructions around it: 110592
// matrices of n = 16 in 1.65 ms; with a matrix a wave, d and e in its lanes and the library's hypot and divisions, 4.5.
// A second kernel refines in FP64 against the FP64 matrix: a full Rayleigh-Ritz step in the basis of
// the FP32 eigenvectors (FP64 orthonormalisation, projection, parallel Jacobi), which gives FP64-grade
// eigenvalues and orthonormal vectors also for exactly and nearly degenerate bands.
#include "common.hpp"

#include <mutex>

namespace ephip {

struct c32 {
    float re, im;
};
struct c64u {  // a caller's element, aligned to its parts
    double re, im;
};
struct alignas(16) c64 {  // one in LDS, moved by 16-byte accesses
    double re, im;
};

template <class TIn>
__device__ __forceinline__ c32 load_c32(const TIn *p, int64_t i) {
    return c32{static_cast<float>(p[i].re), static_cast<float>(p[i].im)};
}

// W lanes a matrix, 64 / W matrices a wave. LDS per matrix: A (n*n c32) | Z (n columns of n f32, pitch n | 1) | v, w, ec
// (n c32 each) | d and e (n c32), padded so that the matrices of a wave start W banks apart.
__host__ __device__ constexpr int heev_zpitch(int n) { return n | 1; }
__host__ __device__ constexpr int heev_lds_floats(int n, int W) {
    const int f = 2 * n * n + n * heev_zpitch(n) + (n & 1) + 8 * n;
    return f + (W - f % 64 + 64) % 64;
}

template <int W>
__device__ __forceinline__ float lanes_sum(float v) {
#pragma unroll
    for (int off = W / 2; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

template <class TIn, int W, bool VEC>
__global__ __launch_bounds__(256) void heev_c32_kernel(int n, int64_t nb, const TIn *__restrict__ H,
                                                       c32 *__restrict__ U, float *__restrict__ E,
                                                       int *__restrict__ info) {
// every contraction is written out: the vectors' phases come from rounding, so every form rounds alike
#pragma clang fp contract(off)
    auto fma = [](float x, float y, float z) { return __builtin_fmaf(x, y, z); };
    extern __shared__ float lds[];
    const int lane = threadIdx.x & (W - 1);
    const int64_t slot = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / W;
    const bool active = slot < nb;
    if (!__any(active)) return;  // whole wave exits together; no workgroup barriers below
    const int64_t b = active ? slot : nb - 1;  // lanes without a matrix work along on the last one, and write nothing
    c32 *A = reinterpret_cast<c32 *>(lds + (threadIdx.x / W) * heev_lds_floats(n, W));
    const int nn = n * n, zp = heev_zpitch(n);
    float *Z = reinterpret_cast<float *>(A + nn);
    c32 *Vh = reinterpret_cast<c32 *>(Z + n * zp + (n & 1));
    c32 *Wh = Vh + n;
    c32 *EC = Wh + n;
    c32 *DE = EC + n;  // d_i, e_i
    const TIn *Hb = H + b * nn;

    // 1. Hermitian matrix from the upper triangle ('U' convention)
    for (int j = 0; j < n; j++)
        if (lane <= j) {
            c32 v = load_c32(Hb, lane + (int64_t)n * j);
            if (lane == j) v.im = 0.f;
            A[lane + n * j] = v;
            if (lane < j) A[j + n * lane] = c32{v.re, -v.im};
        }
    wave_lds_sync();

    for (int j = 0; j + 2 < n; j++) {
        const int m = n - j - 1;
        c32 x{0.f, 0.f};
        if (lane < m) x = A[(j + 1 + lane) + n * j];
        const float xn2 = lanes_sum<W>(fma(x.im, x.im, x.re * x.re));
        const bool reflects = xn2 != 0.f;
        const float xn = sqrtf(xn2);
        const c32 x0 = A[(j + 1) + n * j];
        const float ax0 = hypotf(x0.re, x0.im);
        const float p0r = ax0 > 0.f ? x0.re / ax0 : 1.f, p0i = ax0 > 0.f ? x0.im / ax0 : 0.f;
        const c32 alpha{-p0r * xn, -p0i * xn};
        c32 v = x;
        if (lane == 0) {
            v.re = fma(p0r, xn, x.re);
            v.im = fma(p0i, xn, x.im);
        }
        const float vn = sqrtf(lanes_sum<W>(fma(v.re, v.re, v.im * v.im)));
        v.re /= vn;
        v.im /= vn;
        if (lane < m && reflects) {
            Vh[lane] = v;
            A[(j + 1 + lane) + n * j] = v;
        }
        wave_lds_sync();
        // p = A22 v
        c32 p{0.f, 0.f};
        if (lane < m) {
            for (int k = 0; k < m; k++) {
                const c32 a = A[(j + 1 + lane) + n * (j + 1 + k)];
                const c32 vk = Vh[k];
                p.re += fma(a.re, vk.re, -(a.im * vk.im));
                p.im += fma(a.im, vk.re, a.re * vk.im);
            }
        }
        const float K = lanes_sum<W>(fma(v.im, p.im, v.re * p.re));  // Re(v^H p), zero on idle lanes
        const c32 w{fma(-v.re, K, p.re), fma(-v.im, K, p.im)};
        if (lane < m) Wh[lane] = w;
        wave_lds_sync();
        // A22 -= 2 (v w^H + w v^H)
        if (lane < m && reflects)
            for (int c = 0; c < m; c++) {
                const c32 vc = Vh[c], wc = Wh[c];
                c32 &a = A[(j + 1 + lane) + n * (j + 1 + c)];
                a.re = fma(-2.f, fma(v.re, wc.re, v.im * wc.im) + fma(w.re, vc.re, w.im * vc.im), a.re);
                a.im = fma(-2.f, fma(v.im, wc.re, -(v.re * wc.im)) + fma(w.im, vc.re, -(w.re * vc.im)), a.im);
            }
        if (lane == 0) EC[j] = reflects ? alpha : c32{0.f, 0.f};
        wave_lds_sync();
    }
    if (n >= 2 && lane == 0) EC[n - 2] = A[(n - 1) + n * (n - 2)];
    wave_lds_sync();

    // 2. real tridiagonal: d, e, and the phase tau_i of lane i
    float tr = 1.f, ti = 0.f;
    if (lane < n) {
        float ae = 0.f;
        c32 f{1.f, 0.f};
        if (lane + 1 < n) {
            const c32 ec = EC[lane];
            ae = hypotf(ec.re, ec.im);
            if (ae > 0.f) f = c32{ec.re / ae, ec.im / ae};
            Wh[lane] = f;
        }
        DE[lane] = c32{A[lane + n * lane].re, ae};
    }
    wave_lds_sync();
    {
        float cr = 1.f, ci = 0.f;
        for (int jj = 0; jj + 1 < n; jj++) {
            const c32 f = Wh[jj];
            if (DE[jj].im > 0.f) {
                const float nr = fma(cr, f.re, -(ci * f.im)), ni = fma(cr, f.im, ci * f.re);
                cr = nr;
                ci = ni;
            }
            if (lane == jj + 1) {
                tr = cr;
                ti = ci;
            }
        }
    }
    if (VEC && lane < n)
        for (int c = 0; c < n; c++) Z[lane + zp * c] = (lane == c) ? 1.f : 0.f;
    wave_lds_sync();

    // 3. implicit QL; the matrices of a wave sweep together. d and e of the next rotation and its column of Z are
    // loaded a rotation ahead.
    int fail = 0, l = 0, iter = 0;
    const float eps = 1.1920929e-07f;
    const int row = lane < n ? lane : n - 1;
    float *const Zr = Z + row;
    while (true) {
        const bool last = lane >= n - 1;
        const c32 own = DE[row];
        const bool splits = last || fabsf(own.im) <= eps * (fabsf(own.re) + fabsf(DE[row + !last].re));
        const uint32_t cut = (uint32_t)(__ballot(splits) >> (threadIdx.x & 63 & ~(W - 1)));
        // bit k of cut: e_k is negligible, from k = n - 1 on it is set; the first block of more than one row
        const int l0 = l + __builtin_ctz(~(cut >> l) | (1u << min(n - l, 31)));
        if (l0 > l) iter = 0;
        l = l0;
        if (l >= n - 1) break;
        if (iter++ == 60) {
            fail = 1;
            break;
        }
        const int m = l + __builtin_ctz(cut >> l);
        const c32 dl = DE[l], dm = DE[m];
        c32 de = DE[m - 1];
        float zf = 0.f, zi = 0.f;
        if (VEC) {
            zf = Zr[zp * m];
            zi = Zr[zp * (m - 1)];
        }
        float g = (DE[l + 1].re - dl.re) / (2.f * dl.im);
        g = dm.re - dl.re + dl.im / (g + copysignf(hypotf(g, 1.f), g));
        float s = 1.f, c = 1.f, p = 0.f, d1 = dm.re;
        c32 *pd = DE + m - 1;
        float *pz = Zr + zp * (m - 1);
        while (true) {
            const bool end = pd == DE + l;
            const c32 next = pd[end ? 0 : -1];
            float zn = 0.f;
            if (VEC) zn = pz[end ? 0 : -zp];
            const float f = s * de.im, bb = c * de.im;
            float r, y;
            if (fminf(fabsf(f), fabsf(g)) > 0x1p-60f && fmaxf(fabsf(f), fabsf(g)) < 0x1p60f) {
                // nothing has to be scaled: r by the hardware's square root, about an ulp from hypotf's, and f / r and
                // g / r for that r by Newton's iteration and Markstein's correction from one reciprocal
                r = __builtin_amdgcn_sqrtf(fma(f, f, g * g));
                y = __builtin_amdgcn_rcpf(r);
                y = fma(fma(-r, y, 1.f), y, y);
                s = f * y;
                c = g * y;
                s = fma(fma(-r, s, f), y, s);
                c = fma(fma(-r, c, g), y, c);
                s = fma(fma(-r, s, f), y, s);
                c = fma(fma(-r, c, g), y, c);
            } else {
                r = hypotf(f, g);
                if (r == 0.f) {
                    pd[1] = c32{d1 - p, 0.f};
                    DE[m].im = 0.f;
                    if (VEC) pz[zp] = zf;
                    break;
                }
                s = f / r;
                c = g / r;
            }
            const float gd = d1 - p;
            const float t = fma(bb, 2.f * c, (de.re - gd) * s);
            p = s * t;
            g = fma(c, t, -bb);
            pd[1] = c32{fma(s, t, gd), r};
            if (VEC) {
                pz[zp] = fma(c, zf, s * zi);
                zf = fma(c, zi, -(s * zf));
            }
            if (end) {
                pd[0] = c32{de.re - p, g};
                DE[m].im = 0.f;
                if (VEC) pz[0] = zf;
                break;
            }
            d1 = de.re;
            de = next;
            zi = zn;
            pd--;
            pz -= zp;
        }
    }
    wave_lds_sync();

    // ascending order: lane i's eigenvalue goes to position rank_i (stable for ties)
    const float d = DE[row].re;
    int rank = 0;
    for (int k = 0; k < n; k++) {
        const float dk = DE[k].re;
        rank += (dk < d || (dk == d && k < lane)) ? 1 : 0;
    }
    if (active && lane < n) E[b * n + rank] = d;
    if (active && info && lane == 0) info[b] = fail;
    if constexpr (!VEC) return;

    // 4. eigenvectors: lane = column of Y = D Z, in registers, then the reflectors
    if (lane < n) Wh[lane] = c32{tr, ti};
    wave_lds_sync();
    c32 Y[W];
#pragma unroll
    for (int r = 0; r < W; r++)
        if (r < n) {
            const float z = Z[r + zp * row];
            const c32 t = Wh[r];
            Y[r] = c32{t.re * z, t.im * z};
        }
    for (int j = n - 3; j >= 0; j--) {
        float sr = 0.f, si = 0.f;
#pragma unroll
        for (int r = 1; r < W; r++)
            if (r > j && r < n) {
                const c32 vi = A[r + n * j];
                sr += fma(vi.re, Y[r].re, vi.im * Y[r].im);
                si += fma(vi.re, Y[r].im, -(vi.im * Y[r].re));
            }
#pragma unroll
        for (int r = 1; r < W; r++)
            if (r > j && r < n) {
                const c32 vi = A[r + n * j];
                Y[r].re = fma(-2.f, fma(sr, vi.re, -(si * vi.im)), Y[r].re);
                Y[r].im = fma(-2.f, fma(si, vi.re, sr * vi.im), Y[r].im);
            }
    }
    wave_lds_sync();
    if (lane < n)
#pragma unroll
        for (int r = 0; r < W; r++)
            if (r < n) A[r + n * rank] = Y[r];
    wave_lds_sync();
    if (!active) return;
    c32 *Ub = U + b * nn;
    for (int e = lane; e < nn; e += W) Ub[e] = A[e];
}

// ---------------------------------------------------------------------------------------------
// FP64 refinement, one, two or four matrices per wave, in the basis of the FP32 eigenvectors:
//   1. Q = V orthonormalised in FP64 by two Loewdin steps Q <- Q (3/2 I - 1/2 Q^H Q)
//      (V is orthonormal to ~1e-6, two steps reach ~1e-23);
//   2. M = Q^H H Q is unitarily similar to H and nearly diagonal (off-diagonal ~ FP32 residual);
//   3. cyclic Jacobi sweeps on M in FP64, the n/2 disjoint rotations of a round-robin round applied
//      in parallel, accumulated into Q. Convergence is quadratic from a nearly diagonal start, and exact or
//      close eigenvalue pairs need no special handling (a degenerate pair gets a well-defined 45-degree
//      rotation).
// Eigenvalues are diag(M) sorted ascending, eigenvectors the matching columns of Q (rounded to FP32).
// LDS per matrix: Q and M (n columns of c64, column pitch ld = n | 1); M holds Q^H Q and H before. The odd pitch
// spreads the 16-byte column-strided accesses (lane = column) over the banks; with ld = n = 16 every lane of such an
// access fell on the same banks. Its accesses bound the kernel, then the FP64 arithmetic; 16-byte alignment halves their
// cycles (an 8-byte aligned element goes as two 8-byte accesses with a stride of 16).
// 110592 matrices of n = 16: 2.9 ms; one lane a row working through the rotations of one matrix took 15.4.
// ---------------------------------------------------------------------------------------------
__host__ __device__ constexpr int refine_ld(int n) { return n | 1; }
__host__ __device__ constexpr int refine_lds_doubles(int n) { return 4 * n * refine_ld(n); }

__device__ __forceinline__ double rdl64(double v, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}

// Products with the contraction written out: the vectors' phases come from rounding, so every form of these kernels
// rounds alike.
__device__ __forceinline__ c64 cmul(c64 a, c64 b) {
    return c64{__builtin_fma(a.re, b.re, -(a.im * b.im)), __builtin_fma(a.re, b.im, a.im * b.re)};
}
__device__ __forceinline__ c64 cmul_swapped(c64 a, c64 b) {  // a * b as cmul(b, a) rounds it
    return c64{__builtin_fma(a.re, b.re, -(a.im * b.im)), __builtin_fma(a.im, b.re, a.re * b.im)};
}
__device__ __forceinline__ c64 cmulc(c64 a, c64 b) {  // conj(a) * b
    return c64{__builtin_fma(a.re, b.re, a.im * b.im), __builtin_fma(a.re, b.im, -(a.im * b.re))};
}
__device__ __forceinline__ c64 cadd(c64 a, c64 b) { return c64{a.re + b.re, a.im + b.im}; }

// e / n for e < 2048, n <= 32 by a multiplication: an integer division by a run-time n costs twenty instructions
struct SmallDiv {
    int n;
    unsigned magic;
    __device__ explicit SmallDiv(int n_) : n(n_), magic(65536u / n_ + 1u) {}
    __device__ int div(int e) const { return (int)(((unsigned)e * magic) >> 16); }
    __device__ int mod(int e) const { return e - div(e) * n; }
};

// n x n matrices in LDS with column pitch ld (element (r, j) at r + ld*j), W lanes a matrix (l = lane of W). A lane
// forms tiles of 2 x 2 entries, so an operand read serves two of them, and keeps them in registers: out may be A or B.
// The sum over k of an entry runs in order. NT * W >= the ceil(n/2)^2 tiles.
// out = alpha * A B + beta * C (OP == 0) or A^H B (OP == 1); C is read before out is written
template <int OP, int NT, int W>
__device__ __forceinline__ void lds_gemm(int n, int ld, const c64 *A, const c64 *B, c64 *out, double alpha, double beta,
                                         const c64 *C, int l) {
    const int T = (n + 1) >> 1;
    const SmallDiv byT(T);
    c64 acc[NT][2][2];
    int r[NT][2], j[NT][2];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int e = min(l + t * W, T * T - 1);  // the lanes left over repeat the last tile
        const int tj = byT.div(e), tr = e - T * tj;
        r[t][0] = 2 * tr;
        r[t][1] = min(2 * tr + 1, n - 1);  // an odd n's repeated row or column writes the same value again
        j[t][0] = 2 * tj;
        j[t][1] = min(2 * tj + 1, n - 1);
#pragma unroll
        for (int x = 0; x < 4; x++) acc[t][x >> 1][x & 1] = c64{0.0, 0.0};
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
        for (int k = 0; k < n; k++) {
            c64 a[2], b[2];
#pragma unroll
            for (int x = 0; x < 2; x++) {
                a[x] = OP ? A[k + ld * r[t][x]] : A[r[t][x] + ld * k];
                b[x] = B[k + ld * j[t][x]];
            }
#pragma unroll
            for (int x = 0; x < 4; x++)
                acc[t][x >> 1][x & 1] =
                    cadd(acc[t][x >> 1][x & 1], OP ? cmulc(a[x >> 1], b[x & 1]) : cmul_swapped(a[x >> 1], b[x & 1]));
        }
    if constexpr (OP == 0) {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int x = 0; x < 4; x++) {
                c64 &v = acc[t][x >> 1][x & 1];
                v = c64{alpha * v.re, alpha * v.im};
                if (beta != 0.0) {
                    const c64 c = C[r[t][x >> 1] + ld * j[t][x & 1]];
                    v = c64{v.re + beta * c.re, v.im + beta * c.im};
                }
            }
    }
    wave_lds_sync();
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int x = 0; x < 4; x++) out[r[t][x >> 1] + ld * j[t][x & 1]] = acc[t][x >> 1][x & 1];
    wave_lds_sync();
}

// Parallel cyclic Jacobi on the n x n Hermitian M (LDS, column pitch ldm, n <= 32): the n/2 disjoint
// rotations of a round-robin round are applied in parallel and accumulated into the n columns of Q (qrows x n, column
// pitch ldq, qrows <= 64). A wave works on G matrices, 64 / G lanes each (active: this lane's group has one). Each
// rotation has its own lanes: all of them form it from M, which costs no more than one lane's forming it and needs no
// table in LDS, then they share its rows of M and Q, then its columns of M. Stops
// when the strict upper triangle's Frobenius norm (the part the rotations remove; rounding leaves M Hermitian only
// to a few ulps, and unitary rotations cannot remove that anti-Hermitian residue) is <= tol/sqrt(2) x the
// Frobenius norm, or after 12 sweeps. A pivot below 1e-20 of its diagonal scale is left alone: rotating it
// would only shrink it further, towards the subnormal range where its phase can no longer be normalised
// and the rotation stops being unitary. The norms are summed in the order of one matrix a wave for any G.
template <int G>
__device__ void wave_jacobi(int n, c64 *M, int ldm, c64 *Q, int ldq, int qrows, int lane, double tol, bool active) {
    constexpr int W = 64 / G, CH = 4;
    const int l = lane & (W - 1);
    const int nn = n * n;
    const int N = n + (n & 1);
    const int npairs = N / 2;
    const int L = W / npairs;  // lanes of a rotation
    const int pair = l / L, sub = l - pair * L;
    const SmallDiv byn(n);
    for (int sweep = 0; sweep < 12; sweep++) {
        double off, tot;
        {
            double offs[G], tots[G];
#pragma unroll
            for (int v = 0; v < G; v++) {
                offs[v] = tots[v] = 0.0;
                for (int e = l + W * v; e < nn; e += 64) {
                    const int c = byn.div(e), r = e - n * c;
                    const c64 me = M[r + ldm * c];
                    const double a2 = me.re * me.re + me.im * me.im;
                    tots[v] += a2;
                    if (r < c) offs[v] += 2.0 * a2;
                }
            }
#pragma unroll
            for (int h = G / 2; h >= 1; h >>= 1)
#pragma unroll
                for (int v = 0; v < h; v++) {
                    offs[v] += offs[v + h];
                    tots[v] += tots[v + h];
                }
            off = offs[0];
            tot = tots[0];
        }
#pragma unroll
        for (int x = W / 2; x >= 1; x >>= 1) {
            off += __shfl_xor(off, x, 64);
            tot += __shfl_xor(tot, x, 64);
        }
        if (off <= tol * tol * tot) active = false;
        if (!__any(active)) break;
        for (int rd = 0; rd < N - 1; rd++) {
            int a, c;
            if (pair == 0) {
                a = N - 1;
                c = rd;
            } else {  // (rd + pair) and (rd - pair) modulo N - 1
                a = rd + pair;
                c = rd - pair;
                if (a >= N - 1) a -= N - 1;
                if (c < 0) c += N - 1;
            }
            const int p = min(a, c), q = max(a, c);
            const bool rotates = active && pair < npairs && q < n;  // q == n: the dummy partner of an odd n
            // G = diag(1, e^{-i phi}) [[cs, sn], [-sn, cs]] on (p, q); its upper row is real
            c64 gpp{1.0, 0.0}, gpq{0.0, 0.0}, gqp{0.0, 0.0}, gqq{1.0, 0.0};
            if (rotates) {
                const c64 mpq = M[p + ldm * q];
                const double mpp = M[p + ldm * p].re, mqq = M[q + ldm * q].re;
                const double amp = hypot(mpq.re, mpq.im);
                const double scale = fabs(mpp) + fabs(mqq);
                if (amp > 1e-20 * scale && amp > 1e-280) {
                    const double er = mpq.re / amp, ei = mpq.im / amp;
                    const double tau = (mqq - mpp) / (2.0 * amp);
                    const double t = (tau >= 0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
                    const double cs = 1.0 / sqrt(1.0 + t * t), sn = t * cs;
                    gpp.re = cs;
                    gpq.re = sn;
                    gqp = c64{-sn * er, sn * ei};
                    gqq = c64{cs * er, -cs * ei};
                }
            }
            wave_lds_sync();
            if (rotates) {  // M <- M G, Q <- Q G, CH rows at once
                const int rows = n + qrows;
                for (int i = sub; i < rows; i += CH * L) {
                    c64 *xp[CH], *xq[CH], vp[CH], vq[CH];
#pragma unroll
                    for (int u = 0; u < CH; u++) {
                        const int r = i + u * L < rows ? i + u * L : i;  // past the end: the first one's values again
                        c64 *X = r < n ? M + r : Q + (r - n);
                        const int ldx = r < n ? ldm : ldq;
                        xp[u] = X + ldx * p;
                        xq[u] = X + ldx * q;
                        vp[u] = *xp[u];
                        vq[u] = *xq[u];
                    }
#pragma unroll
                    for (int u = 0; u < CH; u++) {
                        *xp[u] = cadd(cmul(vp[u], gpp), cmul(vq[u], gqp));
                        *xq[u] = cadd(cmul(vp[u], gpq), cmul(vq[u], gqq));
                    }
                }
            }
            wave_lds_sync();
            if (rotates) {  // M <- G^H M
                for (int i = sub; i < n; i += CH * L) {
                    c64 *xp[CH], *xq[CH], vp[CH], vq[CH];
#pragma unroll
                    for (int u = 0; u < CH; u++) {
                        const int col = i + u * L < n ? i + u * L : i;
                        xp[u] = M + p + ldm * col;
                        xq[u] = M + q + ldm * col;
                        vp[u] = *xp[u];
                        vq[u] = *xq[u];
                    }
#pragma unroll
                    for (int u = 0; u < CH; u++) {
                        *xp[u] = cadd(cmulc(gpp, vp[u]), cmulc(gqp, vq[u]));
                        *xq[u] = cadd(cmulc(gpq, vp[u]), cmulc(gqq, vq[u]));
                    }
                }
            }
            wave_lds_sync();
        }
    }
}

template <int G, int NT>
__global__ __launch_bounds__(256) void heev_refine_kernel(int n, int64_t nb, const c64u *__restrict__ H,
                                                          c32 *__restrict__ U, double *__restrict__ E64,
                                                          double tol) {
    extern __shared__ double lds64[];
    constexpr int W = 64 / G;
    const int lane = threadIdx.x & 63, l = lane & (W - 1);
    const int64_t slot = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / W;
    const int nn = n * n, ld = refine_ld(n), nl = n * ld;
    const bool active = slot < nb;
    if (!__any(active)) return;
    const int64_t b = active ? slot : nb - 1;  // lanes without a matrix compute along on the last one, and write nothing
    const SmallDiv byn(n);
    c64 *Q = reinterpret_cast<c64 *>(lds64) + (threadIdx.x / W) * 2 * nl;
    c64 *M = Q + nl;
    for (int e = l; e < nn; e += W) {
        const int j = byn.div(e), i = e - n * j;
        const c32 u = U[b * nn + e];
        Q[i + ld * j] = c64{u.re, u.im};
    }
    wave_lds_sync();
    // 1. two Loewdin steps: M = Q^H Q, Q = 3/2 Q - 1/2 Q M
    for (int it = 0; it < 2; it++) {
        lds_gemm<1, NT, W>(n, ld, Q, Q, M, 0.0, 0.0, nullptr, l);
        lds_gemm<0, NT, W>(n, ld, Q, M, Q, -0.5, 1.5, Q, l);
    }
    // 2. M = Q^H (H Q), H where M goes
    for (int e = l; e < nn; e += W) {
        const int j = byn.div(e), i = e - n * j;
        const c64u hu = (i <= j) ? H[b * nn + i + (int64_t)n * j] : H[b * nn + j + (int64_t)n * i];
        c64 h{hu.re, hu.im};
        if (i > j) h.im = -h.im;
        if (i == j) h.im = 0.0;
        M[i + ld * j] = h;
    }
    wave_lds_sync();
    lds_gemm<0, NT, W>(n, ld, M, Q, M, 1.0, 0.0, nullptr, l);
    lds_gemm<1, NT, W>(n, ld, Q, M, M, 0.0, 0.0, nullptr, l);
    // 3. parallel cyclic Jacobi
    wave_jacobi<G>(n, M, ld, Q, ld, n, lane, tol, active);
    if (!active) return;
    // 4. ascending order; the rank of a column goes beside its eigenvalue
    if (l < n) {
        const double d = M[l + ld * l].re;
        int rank = 0;
        for (int k = 0; k < n; k++) {
            const double dk = M[k + ld * k].re;
            rank += (dk < d || (dk == d && k < l)) ? 1 : 0;
        }
        E64[b * n + rank] = d;
        M[l + ld * l].im = rank;
    }
    wave_lds_sync();
    for (int e = l; e < nn; e += W) {
        const int j = byn.div(e), r = e - n * j;
        const c64 v = Q[r + ld * j];
        U[b * nn + r + (int64_t)n * (int)M[j + ld * j].im] = c32{static_cast<float>(v.re), static_cast<float>(v.im)};
    }
}


// ---------------------------------------------------------------------------------------------
// Degenerate-band gauge fixing of the reference's per-k eigensolve (solve_eigen_el!,
// src/diagonalize.jl:47-85), one wave per matrix, after the eigenpairs are known. Bands are grouped as
// the reference groups them: a group starts at band a and runs while |E_i - E_a| <= cutoff. In each group
// of m > 1 bands the fixed Hermitian perturbation P (src/diagonalize.jl:11-18; the matrix of EPW's
// hamwan2bloch) is projected, M = U_g^H P U_g, M is diagonalised by the FP64 Jacobi and U_g <- U_g V with
// the columns in ascending order of M's eigenvalues. The gauge inside each group is then fixed by H and P
// alone (up to one phase per column), whatever gauge the solver returned. Matrices without a pair closer
// than the cutoff are not touched. LDS (one wave per workgroup): U_g | W = P U_g | M (n*n c64 each),
// ranks.
// ---------------------------------------------------------------------------------------------
__host__ __device__ constexpr int gauge_lds_bytes(int n) { return 3 * n * n * 16 + 4 * n; }

__device__ __forceinline__ c64 degeneracy_perturbation(int r, int c) {  // P[r, c], 0-based row r, column c
    return c64{0.25644832 + 0.005 * (double)(r + c + 2), 0.0125 * (double)(r - c)};
}

__device__ void gauge_fix_group(int n, int a, int m, c32 *__restrict__ Ub, c64 *Ug, c64 *W, c64 *M,
                                int *rank_s, int lane) {
    for (int t = lane; t < n * m; t += 64) {
        const c32 u = Ub[t % n + n * (a + t / n)];
        Ug[t] = c64{u.re, u.im};
    }
    wave_lds_sync();
    for (int t = lane; t < n * m; t += 64) {  // W = P U_g
        const int r = t % n, c = t / n;
        c64 acc{0.0, 0.0};
        for (int k = 0; k < n; k++) acc = cadd(acc, cmul_swapped(degeneracy_perturbation(r, k), Ug[k + n * c]));
        W[t] = acc;
    }
    wave_lds_sync();
    for (int t = lane; t < m * m; t += 64) {  // M = U_g^H W, upper triangle, mirrored: exactly Hermitian
        const int i = t % m, j = t / m;
        if (i > j) continue;
        c64 acc{0.0, 0.0};
        for (int r = 0; r < n; r++) acc = cadd(acc, cmulc(Ug[r + n * i], W[r + n * j]));
        if (i == j) acc.im = 0.0;
        M[t] = acc;
        M[j + m * i] = c64{acc.re, -acc.im};
    }
    wave_lds_sync();
    wave_jacobi<1>(m, M, m, Ug, n, n, lane, 1e-15, true);
    const double d = lane < m ? M[lane + m * lane].re : 0.0;
    int rank = 0;
    for (int k = 0; k < m; k++) {
        const double dk = rdl64(d, k);
        rank += (dk < d || (dk == d && k < lane)) ? 1 : 0;
    }
    if (lane < m) rank_s[lane] = rank;
    wave_lds_sync();
    for (int t = lane; t < n * m; t += 64) {
        const int r = t % n, c = t / n;
        Ub[r + n * (a + rank_s[c])] = c32{static_cast<float>(Ug[t].re), static_cast<float>(Ug[t].im)};
    }
    wave_lds_sync();
}

__global__ __launch_bounds__(64) void degenerate_gauge_kernel(int n, int64_t nb, const double *__restrict__ E64,
                                                              c32 *__restrict__ U, double cutoff) {
    extern __shared__ double lds64[];
    const int lane = threadIdx.x;
    const int64_t b = blockIdx.x;
    const double e = lane < n ? E64[b * n + lane] : 0.0;
    bool any = false;  // is_degenerate: some neighbouring pair closer than the cutoff
    for (int i = 0; i + 1 < n && !any; i++) any = fabs(rdl64(e, i + 1) - rdl64(e, i)) < cutoff;
    if (!any) return;
    c64 *Ug = reinterpret_cast<c64 *>(lds64);
    c64 *W = Ug + n * n;
    c64 *M = W + n * n;
    int *rank_s = reinterpret_cast<int *>(M + n * n);
    c32 *Ub = U + b * n * n;
    double first = rdl64(e, 0);
    int a = 0;
    for (int i = 0; i + 1 < n; i++) {  // wave-uniform walk over the ascending eigenvalues
        const double next = rdl64(e, i + 1);
        int last;
        if (fabs(first - next) > cutoff)
            last = i;
        else if (i == n - 2)
            last = i + 1;
        else
            continue;
        if (last > a) gauge_fix_group(n, a, last - a + 1, Ub, Ug, W, M, rank_s, lane);
        first = next;
        a = i + 1;
    }
}

}  // namespace ephip

using namespace ephip;

// Waves per workgroup. The LDS decides how many matrices share a CU: of the workgroups of 1, 2 and 4 waves that its
// 160 KiB hold, the larger ones where they hold as many waves.
static int eig_waves_per_block(size_t lds_per_wave) {
    int best = 1;
    for (int w : {2, 4}) {
        const size_t cu = 160 * 1024;
        if (w * lds_per_wave <= 64 * 1024 && cu / (w * lds_per_wave) * w >= cu / (best * lds_per_wave) * best) best = w;
    }
    return best;
}

template <int G, int NT>
static void refine_launch(int n, int64_t nb, const void *H64, void *U, double *E64, double tol, void *stream) {
    const size_t lds_wave = G * sizeof(double) * refine_lds_doubles(n);
    const int wpb = eig_waves_per_block(lds_wave);
    heev_refine_kernel<G, NT><<<(unsigned)((nb + G * wpb - 1) / (G * wpb)), 64 * wpb, wpb * lds_wave, as_stream(stream)>>>(
        n, nb, static_cast<const c64u *>(H64), static_cast<c32 *>(U), E64, tol);
}

static int heev_launch_check(int n, int64_t nb) {
    EPHIP_REQUIRE(n >= 1 && n <= 32, "heev: n=%d outside 1..32 (one wavefront per matrix)", n);
    EPHIP_REQUIRE(nb >= 0, "heev: negative batch");
    EPHIP_REQUIRE((nb + 3) / 4 <= 0x7fffffffLL, "heev: batch too large");
    return EPHIP_OK;
}

template <int W>
static void heev_launch(int n, int64_t nb, const void *H, int h_is_c64, void *U, float *E, int *info, void *stream) {
    const int per = 64 / W;
    const size_t lds_wave = per * sizeof(float) * heev_lds_floats(n, W);
    const int wpb = eig_waves_per_block(lds_wave);
    const unsigned grid = (unsigned)((nb + per * wpb - 1) / (per * wpb));
    hipStream_t s = as_stream(stream);
    auto go = [&](auto kernel, auto h) {
        kernel<<<grid, 64 * wpb, wpb * lds_wave, s>>>(n, nb, h, static_cast<c32 *>(U), E, info);
    };
    if (h_is_c64) {
        const c64u *h = static_cast<const c64u *>(H);
        U ? go(heev_c32_kernel<c64u, W, true>, h) : go(heev_c32_kernel<c64u, W, false>, h);
    } else {
        const c32 *h = static_cast<const c32 *>(H);
        U ? go(heev_c32_kernel<c32, W, true>, h) : go(heev_c32_kernel<c32, W, false>, h);
    }
}

extern "C" int ephip_heev_c32(int32_t n, int64_t nb, const void *H, int32_t h_is_c64, void *U, float *E,
                              int32_t *info, void *stream) {
    int st = heev_launch_check(n, nb);
    if (st) return st;
    if (nb == 0) return EPHIP_OK;
    EPHIP_REQUIRE(H && E, "heev: null device pointer");
    // as few lanes as hold a row each: 27000 matrices of n = 16 in 444 us with 16 lanes, 583 with 32; 30000 of n = 8 in
    // 69 us with 8, 113 with 16; the small batches, bound by one matrix's chain, are no slower (500: 125 and 142, 42, 44)
    if (n <= 8)
        heev_launch<8>(n, nb, H, h_is_c64, U, E, info, stream);
    else if (n <= 16)
        heev_launch<16>(n, nb, H, h_is_c64, U, E, info, stream);
    else
        heev_launch<32>(n, nb, H, h_is_c64, U, E, info, stream);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_heev_refine(int32_t n, int64_t nb, const void *H64, void *U, const float *E32, double *E64,
                                 double tol, void *stream) {
    int st = heev_launch_check(n, nb);
    if (st) return st;
    if (nb == 0) return EPHIP_OK;
    EPHIP_REQUIRE(H64 && U && E64, "heev_refine: null device pointer");
    EPHIP_REQUIRE(tol >= 0.0, "heev_refine: negative tolerance");
    (void)E32;
    const double t = tol > 0.0 ? tol : 1e-15;
    // Matrices a wave. Two share the forming of the rotations, which every lane of a wave waits for: 27000 of n = 16 in
    // 744 us for 1137, 13824 of n = 12 in 271 for 463. While one a wave leaves SIMDs idle (a matrix each, 256 CUs), it
    // is the quicker: 500 of n = 16 in 58 us for 72. Four up to n = 8, where they still fill the lanes, win from the
    // smallest batch on: 500 of n = 8 in 29 us for 30, 30000 in 139 for 292 (two) and 595 (one). Above n = 16 the LDS
    // holds too few matrices to pair them.
    if (n > 16)
        refine_launch<1, 4>(n, nb, H64, U, E64, t, stream);
    else if (n <= 8)
        refine_launch<4, 1>(n, nb, H64, U, E64, t, stream);
    else if (nb > 1024)
        refine_launch<2, 2>(n, nb, H64, U, E64, t, stream);
    else
        refine_launch<1, 1>(n, nb, H64, U, E64, t, stream);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_degenerate_gauge_fix(int32_t n, int64_t nb, const double *E64, void *U, double cutoff,
                                          void *stream) {
    int st = heev_launch_check(n, nb);
    if (st) return st;
    EPHIP_REQUIRE(cutoff >= 0.0, "degenerate_gauge_fix: negative cutoff");
    EPHIP_REQUIRE(nb <= 0x7fffffffLL, "degenerate_gauge_fix: batch too large");
    if (nb == 0) return EPHIP_OK;
    EPHIP_REQUIRE(E64 && U, "degenerate_gauge_fix: null device pointer");
    degenerate_gauge_kernel<<<(unsigned)nb, 64, gauge_lds_bytes(n), as_stream(stream)>>>(
        n, nb, E64, static_cast<c32 *>(U), cutoff);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

// eigen_batched / eigvals_batched with the FP64 accuracy of the reference's zheev: the FP32 wave solve
// followed by the FP64 refinement, as one entry each. Per matrix, eigvals_batched keeps the FP32
// eigenvectors (8 n^2 bytes) and eigenvalues (4 n bytes) in the caller's workspace: the refinement needs
// the vectors even when only values are returned.
static int64_t eigvals_work_bytes_per_matrix(int n) { return 8LL * n * n + 4LL * n; }

static int eigen_refined_run(int32_t n, int64_t nb, const void *H64, double *E64, void *U, float *E32, int32_t *info,
                             void *stream) {
    int st = ephip_heev_c32(n, nb, H64, 1, U, E32, info, stream);
    if (st) return st;
    return ephip_heev_refine(n, nb, H64, U, E32, E64, 0.0, stream);
}

extern "C" int ephip_eigen_batched(int32_t n, int64_t nb, const void *H64, double *E64, void *U, float *work,
                                   int32_t *info, void *stream) {
    int st = heev_launch_check(n, nb);
    if (st) return st;
    if (nb == 0) return EPHIP_OK;
    EPHIP_REQUIRE(H64 && E64 && U && work, "eigen_batched: null device pointer");
    return eigen_refined_run(n, nb, H64, E64, U, work, info, stream);
}

extern "C" int ephip_eigvals_batched(int32_t n, int64_t nb, const void *H64, double *E64, void *work, int32_t *info,
                                     void *stream) {
    int st = heev_launch_check(n, nb);
    if (st) return st;
    if (nb == 0) return EPHIP_OK;
    EPHIP_REQUIRE(H64 && E64 && work, "eigvals_batched: null device pointer");
    char *w = static_cast<char *>(work);
    return eigen_refined_run(n, nb, H64, E64, w, reinterpret_cast<float *>(w + 8LL * n * n * nb), info, stream);
}

// ---------------------------------------------------------------------------------------------
// Allocation-free eigenvalue entry: the workspace of ephip_eigvals_batched (FP32 eigenvectors, then FP32
// eigenvalues) lives in a file-scope device array instead of a caller buffer. Each GPU the library runs
// on holds its own copy until the process ends; its address on a device is looked up once, with that
// device current, and kept. Calls that overlap on one GPU share the array and race.
// ---------------------------------------------------------------------------------------------
namespace ephip {

constexpr size_t EIG_SCRATCH_BYTES = size_t(16) << 20;  // 16 MiB per GPU
constexpr int EIG_SCRATCH_DEVICES = 64;

static __device__ __align__(256) char scratch[EIG_SCRATCH_BYTES];

static std::mutex g_scratch_mu;
static void *g_scratch_ptr[EIG_SCRATCH_DEVICES];

// Device address of this GPU's scratch array (the host-side name is not a device address).
static int scratch_address(void **out) {
    int dev = -1;
    EPHIP_TRY_HIP(hipGetDevice(&dev));
    EPHIP_REQUIRE(dev >= 0 && dev < EIG_SCRATCH_DEVICES, "eigvals_batched_noalloc: device %d outside 0..%d", dev,
                  EIG_SCRATCH_DEVICES - 1);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        EPHIP_TRY_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        EPHIP_REQUIRE(p != nullptr, "eigvals_batched_noalloc: no device address for the scratch array");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return EPHIP_OK;
}

}  // namespace ephip

extern "C" int ephip_eigvals_batched_noalloc(int32_t n, int64_t nb, const void *H64, double *E64, int32_t *info,
                                             void *stream) {
    int st = heev_launch_check(n, nb);
    if (st) return st;
    if (nb == 0) return EPHIP_OK;
    const int64_t per = eigvals_work_bytes_per_matrix(n);
    const int64_t cap = (int64_t)(EIG_SCRATCH_BYTES / (size_t)per);
    EPHIP_REQUIRE(nb <= cap,
                  "eigvals_batched_noalloc: %lld matrices of n=%d need %lld bytes of workspace; the %zu-byte scratch "
                  "holds %lld (call in chunks, or use ephip_eigvals_batched with a caller workspace)",
                  (long long)nb, n, (long long)(nb * per), EIG_SCRATCH_BYTES, (long long)cap);
    EPHIP_REQUIRE(H64 && E64, "eigvals_batched_noalloc: null device pointer");
    void *w = nullptr;
    st = scratch_address(&w);
    if (st) return st;
    char *wc = static_cast<char *>(w);
    // every entry of the workspace is written by the FP32 solve before the refinement reads it: no clearing
    return eigen_refined_run(n, nb, H64, E64, wc, reinterpret_cast<float *>(wc + 8LL * n * n * nb), info, stream);
}
