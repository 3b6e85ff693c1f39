// The outer-q loop by per-axis partial sums (csrc/staged.hip's counterpart for run_eph_over_q_and_k,
// src/calculator/run_eph_over_q_and_k.jl:526-610), for a tile of q at once:
//   * RR->Rq: the phase sum over Rp at up to 16 q (staged_rq_fourier_kernel) and the phonon-mode rotation
//     (staged_rq_modes_kernel), written with the tile's q side by side, rows (i, j, nu, q) per Re;
//   * Rq->kq: stage 1 and the k-side projection over those rows as for RR->kR (ephip_gridopt_stage1_planes,
//     ephip_staged_project with columns g = i + nw (nu + nm q)), where the phase sums over Re cost 8 nw^2 nm nr flops
//     per (k, q);
//   * the k+q-window rotation and g2 of every (k, q) of the tile (staged_rq_rotate_kernel).
// 16 q, 5735 k, 16 orbitals, 12 modes, 7^3 boxes: 11.5 ms with the phase sums at every k, 1.33 here (0.71 RR->Rq, 0.61
// stages 1 to 3, 0.07 window rotation).
#include "common.hpp"

namespace ephip {

constexpr int RQ_COLS = 16;   // q of one Fourier launch: the columns of a 16x16x4 MFMA

// Phases e^{2 pi i R_r . x_j} of nq <= 16 points, [r][16], zero for j >= nq and for r past nr (up to a multiple of 4).
__global__ void staged_rq_phases_kernel(int nr, const int *__restrict__ irvec, int nq, const double *__restrict__ xq,
                                        float2 *__restrict__ out) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x, r = e / RQ_COLS, j = e % RQ_COLS;
    if (r >= (nr + 3) / 4 * 4) return;
    float c = 0.f, s = 0.f;
    if (r < nr && j < nq)
        cis2pi(irvec[3 * r] * xq[3 * j] + irvec[3 * r + 1] * xq[3 * j + 1] + irvec[3 * r + 2] * xq[3 * j + 2], c, s);
    out[e] = make_float2(c, s);
}

// out[j][d] = sum_r op[d, r] e_j(r) for up to 16 columns j: the columns on the MFMA's rows, 16 operator rows d on its
// columns, four r per step; a lane's operator value is its own B operand, so nothing goes through LDS and a wave
// streams 128 rows d (two neighbours per lane and load when VEC). The operator is read once for the 16 q:
// 2.9 GB (16 orbitals, 12 modes, 7^3 x 7^3) in 0.65 ms, 4.5 TB/s, where the 64-column tiles of the general kernel, 48
// columns idle, took 2.02. Bound by HBM.
template <bool VEC>
__global__ __launch_bounds__(256) void staged_rq_fourier_kernel(int64_t nd, int nr, const cplx<float> *__restrict__ op,
                                                                int64_t ldop, const float2 *__restrict__ ph, int nq,
                                                                cplx<float> *__restrict__ out, int64_t ldout) {
    constexpr int NB = 4;  // pairs of 16-row blocks per wave
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, il = lane & 15, kq = lane >> 4;
    const int64_t d0 = ((int64_t)blockIdx.x * 4 + wave) * 32 * NB;
    if (d0 >= nd) return;  // whole wave
    // this lane's two rows of block pair b
    int64_t da[NB], db[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int64_t x = d0 + 32 * b + 2 * il;
        da[b] = min(x, nd - (VEC ? 2 : 1));
        db[b] = VEC ? da[b] + 1 : min(x + 1, nd - 1);
    }
    f32x4 re[2 * NB], im[2 * NB];
#pragma unroll
    for (int b = 0; b < 2 * NB; b++) re[b] = im[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto load = [&](int r0, float4 (&v)[NB], float2 &p) {
        const int r = r0 + kq;
        p = ph[r * RQ_COLS + il];  // zero past nr
        const cplx<float> *o = op + ldop * min(r, nr - 1);
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if constexpr (VEC) {
                v[b] = *reinterpret_cast<const float4 *>(o + da[b]);
            } else {
                const cplx<float> x = o[da[b]], y = o[db[b]];
                v[b] = make_float4(x.re, x.im, y.re, y.im);
            }
        }
    };
    float4 v[NB], w[NB];
    float2 p, pn;
    load(0, v, p);
    for (int r0 = 0; r0 < nr; r0 += 4) {
        if (r0 + 4 < nr) load(r0 + 4, w, pn);  // the next step's loads in flight during the products
#pragma unroll
        for (int b = 0; b < NB; b++) {
            re[2 * b] = __builtin_amdgcn_mfma_f32_16x16x4f32(p.x, v[b].x, re[2 * b], 0, 0, 0);
            im[2 * b] = __builtin_amdgcn_mfma_f32_16x16x4f32(p.x, v[b].y, im[2 * b], 0, 0, 0);
            re[2 * b + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(p.x, v[b].z, re[2 * b + 1], 0, 0, 0);
            im[2 * b + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(p.x, v[b].w, im[2 * b + 1], 0, 0, 0);
        }
#pragma unroll
        for (int b = 0; b < NB; b++) {
            re[2 * b] = __builtin_amdgcn_mfma_f32_16x16x4f32(-p.y, v[b].y, re[2 * b], 0, 0, 0);
            im[2 * b] = __builtin_amdgcn_mfma_f32_16x16x4f32(p.y, v[b].x, im[2 * b], 0, 0, 0);
            re[2 * b + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(-p.y, v[b].w, re[2 * b + 1], 0, 0, 0);
            im[2 * b + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(p.y, v[b].z, im[2 * b + 1], 0, 0, 0);
        }
#pragma unroll
        for (int b = 0; b < NB; b++) v[b] = w[b];
        p = pn;
    }
    // a lane holds columns j = 4 (lane / 16) + x of its rows
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int64_t d = d0 + 32 * b + 2 * il;
#pragma unroll
        for (int x = 0; x < 4; x++) {
            const int j = 4 * kq + x;
            if (j >= nq) continue;
            cplx<float> *o = out + ldout * j + d;
            if (VEC) {
                if (d < nd)
                    *reinterpret_cast<float4 *>(o) = make_float4(re[2 * b][x], im[2 * b][x], re[2 * b + 1][x], im[2 * b + 1][x]);
            } else {
                if (d < nd) o[0] = cplx<float>{re[2 * b][x], im[2 * b][x]};
                if (d + 1 < nd) o[1] = cplx<float>{re[2 * b + 1][x], im[2 * b + 1][x]};
            }
        }
    }
}

// Phonon-mode rotation of the tile: out[(nbasis (nu' + nm q)) + b + ldout Re] = sum_nu g_q[b + nbasis (nu + nm Re)]
// u_q[nu, nu'] (g_q at g + ldg q). One thread per (b, Re, q) holds its nm values (NMT >= nm registers, or reads them again
// per nu' when NMT = 0); u_q in LDS.
template <int NMT>
__global__ __launch_bounds__(256) void staged_rq_modes_kernel(int nbasis, int nm, int nre, const cplx<float> *__restrict__ g,
                                                              int64_t ldg, const cplx<float> *__restrict__ uph,
                                                              cplx<float> *__restrict__ out, int64_t ldout) {
    extern __shared__ float2 rq_u[];  // [nu'][nu]
    const int q = blockIdx.y;
    for (int e = threadIdx.x; e < nm * nm; e += blockDim.x) {
        const cplx<float> v = uph[(int64_t)nm * nm * q + e];
        rq_u[e] = make_float2(v.re, v.im);
    }
    __syncthreads();
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)nbasis * nre) return;
    const int64_t b = e % nbasis, re = e / nbasis;
    const cplx<float> *src = g + ldg * q + b + (int64_t)nbasis * nm * re;
    cplx<float> *dst = out + ldout * re + (int64_t)nbasis * nm * q + b;
    float xr[NMT > 0 ? NMT : 1], xi[NMT > 0 ? NMT : 1];
    if constexpr (NMT > 0) {
#pragma unroll
        for (int n = 0; n < NMT; n++) {
            const cplx<float> v = src[(int64_t)nbasis * min(n, nm - 1)];
            xr[n] = v.re;
            xi[n] = v.im;
        }
    }
    for (int n2 = 0; n2 < nm; n2++) {
        const float2 *u = rq_u + n2 * nm;
        float sr = 0.f, si = 0.f;
        auto add = [&](int n, float ar, float ai) {
            const float2 w = u[n];
            sr = fmaf(ar, w.x, sr);
            sr = fmaf(-ai, w.y, sr);
            si = fmaf(ar, w.y, si);
            si = fmaf(ai, w.x, si);
        };
        if constexpr (NMT > 0) {
#pragma unroll
            for (int n = 0; n < NMT; n++)
                if (n < nm) add(n, xr[n], xi[n]);  // uniform
        } else {
            for (int n = 0; n < nm; n++) {
                const cplx<float> v = src[(int64_t)nbasis * n];
                add(n, v.re, v.im);
            }
        }
        dst[(int64_t)nbasis * n2] = cplx<float>{sr, si};
    }
}

// k+q window and g2: for the k of a batch (positions k0 .. k0 + nk - 1 of the surviving list, states ks) and every q of
// the tile, t[n, m, nu] = sum_i conj(U_kq[i, m]) A_u[i + nw (nu + nm q)], u the unit of band n of k; g2 = |t|^2 / (2 omega),
// slot [m + nbw (n + nbw nu)] of row (q, k) as ephip_eph_rotate_rqkq_g2, zeros outside the windows. One thread per
// (k, q, nu), nu fastest: a unit's operator is read once, in whole lines. ikq[q ldk + k]: the grid index of k+q.
__global__ __launch_bounds__(256) void staged_rq_rotate_kernel(
    int nw, int nm, int nbw, int nq, int64_t k0, int nk, const int64_t *__restrict__ ks, const double *__restrict__ xk,
    const double *__restrict__ xq, int n1, int n2, int n3, const int *__restrict__ kus, const cplx<float> *__restrict__ A,
    int64_t lda, const cplx<float> *__restrict__ U, const int64_t *__restrict__ bmin, const int64_t *__restrict__ bmax,
    const double *__restrict__ omega, int64_t ldk, int64_t *__restrict__ ikq, float *__restrict__ g2,
    float2 *__restrict__ ep) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)nk * nq * nm) return;
    const int nu = (int)(e % nm), q = (int)(e / nm % nq);
    const int64_t k = k0 + e / ((int64_t)nm * nq), s = ks[k];
    auto red = [](double x, int n) {
        const int c = (int)rint(x * n) % n;
        return c < 0 ? c + n : c;
    };
    const int64_t kq = ((int64_t)red(xk[3 * s] + xq[3 * q], n1) * n2 + red(xk[3 * s + 1] + xq[3 * q + 1], n2)) * n3 +
                       red(xk[3 * s + 2] + xq[3 * q + 2], n3);
    const int64_t row = ldk * q + k;
    if (nu == 0) ikq[row] = kq;
    const int u0 = kus[k] - kus[k0], nbk = min(kus[k + 1] - kus[k], nbw);
    const int64_t b0 = bmin[kq];
    const int nbq = b0 > 0 ? min((int)(bmax[kq] - b0 + 1), nbw) : 0;
    const cplx<float> *uq = U + (int64_t)nw * nw * kq + (b0 > 0 ? nw * (b0 - 1) : 0);
    const float w2 = 2.f * static_cast<float>(omega[(int64_t)nm * q + nu]);
    const int64_t o = (row * nm + nu) * nbw * nbw;
    for (int n = 0; n < nbw; n++) {
        const cplx<float> *a = A + (int64_t)(u0 + min(n, nbk - 1)) * lda + (int64_t)nw * (nu + (int64_t)nm * q);
        for (int m0 = 0; m0 < nbw; m0 += 2) {
            float tr[2] = {0.f, 0.f}, ti[2] = {0.f, 0.f};
            if (n < nbk && m0 < nbq) {
                const int mb = m0 + 1 < nbq ? nw : 0;  // the second band, or the first again
                for (int i = 0; i < nw; i++) {
                    const cplx<float> v = a[i];
#pragma unroll
                    for (int x = 0; x < 2; x++) {
                        const cplx<float> w = uq[nw * m0 + x * mb + i];
                        tr[x] = fmaf(w.re, v.re, tr[x]);
                        tr[x] = fmaf(w.im, v.im, tr[x]);
                        ti[x] = fmaf(w.re, v.im, ti[x]);
                        ti[x] = fmaf(-w.im, v.re, ti[x]);
                    }
                }
                if (!mb) tr[1] = ti[1] = 0.f;
            }
#pragma unroll
            for (int x = 0; x < 2; x++)
                if (m0 + x < nbw) {
                    const bool in = n < nbk && m0 + x < nbq;
                    g2[o + nbw * n + m0 + x] = in ? (tr[x] * tr[x] + ti[x] * ti[x]) / w2 : 0.f;
                    if (ep) ep[o + nbw * n + m0 + x] = make_float2(tr[x], ti[x]);
                }
        }
    }
}

}  // namespace ephip

using namespace ephip;

extern "C" int ephip_staged_rr_to_rq(int64_t nbasis, int32_t nm, int32_t nre, int32_t nrp, const void *op, int64_t ldop,
                                     const int32_t *irvec, int32_t nq, const double *xq, const void *uph, void *phases,
                                     void *work, int64_t ldwork, void *out, int64_t ldout, void *stream) {
    EPHIP_REQUIRE(nbasis >= 1 && nbasis <= 1024 && nm >= 1 && nm <= 48 && nre >= 1 && nrp >= 1 && nq >= 0 && nq <= 65535,
                  "staged_rr_to_rq: bad sizes");
    const int64_t nd = nbasis * nm * nre;
    EPHIP_REQUIRE(ldop >= nd && ldwork >= nd && ldout >= nbasis * nm * nq, "staged_rr_to_rq: leading dimension too small");
    if (nq == 0) return EPHIP_OK;
    EPHIP_REQUIRE(op && irvec && xq && uph && phases && work && out, "staged_rr_to_rq: null device pointer");
    hipStream_t st = as_stream(stream);
    auto o = static_cast<const cplx<float> *>(op);
    auto w = static_cast<cplx<float> *>(work);
    const int rows = (nrp + 3) / 4 * 4 * RQ_COLS;
    // two neighbouring rows per load: 16-byte aligned when the operand's columns and the outputs' are
    const bool vec = (ldop & 1) == 0 && (ldwork & 1) == 0 && (nd & 1) == 0 && (reinterpret_cast<uintptr_t>(op) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(work) & 15) == 0;
    for (int j = 0; j < nq; j += RQ_COLS) {
        const int m = min(RQ_COLS, nq - j);
        auto ph = static_cast<float2 *>(phases) + (int64_t)(j / RQ_COLS) * rows;
        staged_rq_phases_kernel<<<(rows + 255) / 256, 256, 0, st>>>(nrp, irvec, m, xq + 3 * j, ph);
        EPHIP_LAUNCHED();
        (vec ? staged_rq_fourier_kernel<true> : staged_rq_fourier_kernel<false>)<<<(unsigned)((nd + 511) / 512), 256, 0, st>>>(
            nd, nrp, o, ldop, ph, m, w + ldwork * j, ldwork);
        EPHIP_LAUNCHED();
    }
    using K = decltype(&staged_rq_modes_kernel<3>);
    const K k = nm <= 3 ? staged_rq_modes_kernel<3> : nm <= 6 ? staged_rq_modes_kernel<6> : nm <= 9 ? staged_rq_modes_kernel<9>
              : nm <= 12 ? staged_rq_modes_kernel<12> : nm <= 18 ? staged_rq_modes_kernel<18> : staged_rq_modes_kernel<0>;
    k<<<dim3((unsigned)((nbasis * nre + 255) / 256), (unsigned)nq), 256, sizeof(float2) * nm * nm, st>>>(
        (int)nbasis, nm, nre, w, ldwork, static_cast<const cplx<float> *>(uph), static_cast<cplx<float> *>(out), ldout);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_staged_rq_rotate(int32_t nw, int32_t nm, int32_t nbw, int32_t nq, int64_t k0, int32_t nk,
                                      const int64_t *ks, const double *xk, const double *xq, const int32_t *ngrid,
                                      const int32_t *kus, const void *A, int64_t lda, const void *U, const int64_t *bmin,
                                      const int64_t *bmax, const double *omega, int64_t ldk, int64_t *ikq, float *g2,
                                      void *ep, void *stream) {
    EPHIP_REQUIRE(nw >= 1 && nm >= 1 && nbw >= 1 && nbw <= nw && nq >= 0 && nk >= 0 && k0 >= 0 && ldk >= k0 + nk,
                  "staged_rq_rotate: bad sizes");
    EPHIP_REQUIRE(ngrid && ngrid[0] > 0 && ngrid[1] > 0 && ngrid[2] > 0 &&
                      (int64_t)ngrid[0] * ngrid[1] * ngrid[2] < 0x7fffffffLL,
                  "staged_rq_rotate: bad grid");
    EPHIP_REQUIRE(lda >= (int64_t)nw * nm * nq, "staged_rq_rotate: lda too small");
    const int64_t n = (int64_t)nk * nq * nm;
    if (n == 0) return EPHIP_OK;
    EPHIP_REQUIRE(n <= MAX_THREADS_X, "staged_rq_rotate: too many (k, q, mode)");
    EPHIP_REQUIRE(ks && xk && xq && kus && A && U && bmin && bmax && omega && ikq && g2, "staged_rq_rotate: null device pointer");
    staged_rq_rotate_kernel<<<(unsigned)((n + 255) / 256), 256, 0, as_stream(stream)>>>(
        nw, nm, nbw, nq, k0, nk, ks, xk, xq, ngrid[0], ngrid[1], ngrid[2], kus, static_cast<const cplx<float> *>(A), lda,
        static_cast<const cplx<float> *>(U), bmin, bmax, omega, ldk, ikq, g2, static_cast<float2 *>(ep));
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}
