// RR->kR stages 2 and 3 with the k-side projection for boxes that span -h .. h along axes 2 and 3, at most 16
// Wannier functions: the per-axis sums of src/wannier/GridOpt.jl:73-139 with the window projection of
// src/calculator/run_eph_over_k_and_kq.jl:657-659, as gridopt.hip and staged.hip, in the lane-private form below.
//
// A lane is one (operator column g, orbital j) and keeps it from the first load to the projection. With
//   sum_b e[b] B[b] = B[h] + sum_p (cos_p S_p + i sin_p D_p),  S_p = B[h+p] + B[h-p],  D_p = B[h+p] - B[h-p],
// the real and the imaginary part of a stage are the same real matrix (1, cos_p, sin_p) applied to
// (B[h].re, S.re, -D.im) and (B[h].im, S.im, D.re): N steps each, half of the complex product's work. A 4x4x1 FP32
// MFMA whose A operand is broadcast from one block to all sixteen (cbsz 4, abid the step) is just that for the 64
// lanes of a wave, y[row] += M[row][step] x[step] with x and y in the lane's own registers and one register of M for
// all steps: stage 2 takes four lines of the plane at a time, stage 3 four units of a line. The product with U_k
// and the sum over j (a reduce-scatter by lane swaps, then row rotations) run on the VALU beside them; only the
// tables go through LDS.
#include "lanes.hpp"

namespace ephip {

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
constexpr int LP_PLANES = 8, LP_LINES = 256, LP_WIN = 128;

struct LpArgs {
    const cplx<float> *op1[LP_PLANES];
    int l0[LP_PLANES], l1[LP_PLANES];
    int nw;
    int64_t ngcol, nd;
    int lb0;
    const int *ustart;   // first unit of each line of the batch, one more for the end
    const float *c2, *c3;  // (1, cos, sin) of each line along axis 2 and of each unit along axis 3
    const cplx<float> *ucol;
    cplx<float> *A;
    int64_t lda;
};

// JL lanes take j (nw padded to 4, 8 or 16), the other 64 / JL the columns of a wave; gridDim.y runs over the k1
// planes, gridDim.z splits a plane's lines where the operator has few columns.
template <int N, int JL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(N == 7 ? 2 : 3))) void lane_project_kernel(LpArgs a) {
    constexpr int CL = 64 / JL;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = lane / CL, p = blockIdx.y;
    const int64_t g = ((int64_t)blockIdx.x * 4 + wave) * CL + lane % CL;
    const bool dv = g < a.ngcol && j < a.nw;
    const cplx<float> *o = a.op1[p] + (dv ? g % a.nw + a.nw * (j + (int64_t)a.nw * (g / a.nw)) : 0);
    float xr[N][N], xi[N][N];
#pragma unroll
    for (int c = 0; c < N; c++) {
        float br[N], bi[N];
#pragma unroll
        for (int b = 0; b < N; b++) {
            const cplx<float> v = o[a.nd * (b + N * c)];  // lanes without a row read row 0
            br[b] = dv ? v.re : 0.f;
            bi[b] = dv ? v.im : 0.f;
        }
        lp_fold<N>(xr[c], xi[c], br, bi);
    }
    const int nl = a.l1[p] - a.l0[p];
    const int la = a.l0[p] - a.lb0 + (int)((int64_t)nl * blockIdx.z / gridDim.z);
    const int lz = a.l0[p] - a.lb0 + (int)((int64_t)nl * (blockIdx.z + 1) / gridDim.z);
    if (la >= lz) return;
    // Stores go through a buffer descriptor whose range check drops the lanes that hold no sum, and the tables through
    // LDS: loads in this loop, or a branch around the stores, would make every wait a wait for the stores too.
    const int64_t g0 = ((int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(wave)) * CL;
    const int urow = (lane & 15) < CL && g0 + (lane & 15) < a.ngcol ? lane >> 4 : 4;
    const int off = (int)(8 * ((int64_t)(lane >> 4) * a.lda + (lane & 15)));
    __shared__ float c2s[LP_LINES * LP_STEPS], c3s[(LP_WIN + 4) * LP_STEPS];
    __shared__ cplx<float> us[(LP_WIN + 4) * JL];
    __shared__ int lu[LP_LINES + 1];  // first unit of each line
    const int row = lane & 3, step = (lane >> 2) & (LP_STEPS - 1);
    const int uend = __builtin_amdgcn_readfirstlane(a.ustart[lz]);
    for (int e = threadIdx.x; e <= lz - la; e += 256) lu[e] = a.ustart[la + e];
    for (int e = threadIdx.x; e < (lz - la) * LP_STEPS; e += 256) c2s[e] = a.c2[(int64_t)la * LP_STEPS + e];
    int u = __builtin_amdgcn_readfirstlane(a.ustart[la]), w0 = 0;
    float m3 = 0.f;
    cplx<float> w{0.f, 0.f};
    const auto window = [&]() {  // the tables of the next LP_WIN units from u on
        __syncthreads();
        w0 = u;
        const int n = min(LP_WIN, uend - u);
        for (int e = threadIdx.x; e < n * LP_STEPS; e += 256) c3s[e] = a.c3[(int64_t)u * LP_STEPS + e];
        for (int e = threadIdx.x; e < n * JL; e += 256) us[e] = a.ucol[(int64_t)u * JL + e];
        __syncthreads();
    };
    const auto fetch = [&](int v) {  // four units; rows past the window or the last unit are never used
        m3 = c3s[(v - w0 + row) * LP_STEPS + step];
        w = us[(v - w0 + row) * JL + j];
    };
    window();
    fetch(u);
    for (int l = la; l < lz; l += 4) {
        const float m2 = c2s[LP_STEPS * (min(l + row, lz - 1) - la) + step];
        f32x4 tr[N], ti[N];  // stage 2 of four lines, before the fold over c
#pragma unroll
        for (int c = 0; c < N; c++) lp_apply<N>(tr[c], ti[c], m2, xr[c], xi[c]);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if (l + r >= lz) break;
            const int ue = __builtin_amdgcn_readfirstlane(lu[l - la + r + 1]);
            if (u >= ue) continue;
            float br[N], bi[N], zr[N], zi[N];
#pragma unroll
            for (int c = 0; c < N; c++) {
                br[c] = tr[c][r];
                bi[c] = ti[c][r];
            }
            lp_fold<N>(zr, zi, br, bi);
            while (u < ue) {
                const int next = min(u + 4, ue);
                if (next > w0 + LP_WIN) {  // the same for all waves: they run through the same units
                    window();
                    fetch(u);
                }
                const float m = m3;
                const cplx<float> uw = w;
                fetch(next);
                f32x4 gr, gi;
                lp_apply<N>(gr, gi, m, zr, zi);
                float vr[4], vi[4];
                lp_times<0>(vr[0], vi[0], uw.re, uw.im, gr[0], gi[0]);
                lp_times<1>(vr[1], vi[1], uw.re, uw.im, gr[1], gi[1]);
                lp_times<2>(vr[2], vi[2], uw.re, uw.im, gr[2], gi[2]);
                lp_times<3>(vr[3], vi[3], uw.re, uw.im, gr[3], gi[3]);
                const float sr = lp_reduce<JL>(vr), si = lp_reduce<JL>(vi);
                const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(a.A + g0 + (int64_t)u * a.lda, 0, 0x7fffffff, 0x00020000);
                __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(sr), __float_as_uint(si)}, rsrc,
                                                      urow < next - u ? off : -1, 0, 0);
                u = next;
            }
        }
    }
}

// Tables of a batch (k0 <= k < k1, lines l0 <= l < l1): first unit of each line, (1, cos, sin) of every line along
// axis 2 and of every unit along axis 3, the U column of every unit padded to jl.
__global__ __launch_bounds__(256) void lane_tables_kernel(int nw, int jl, int h, const double *__restrict__ xk,
                                                          int64_t k0, int64_t k1, int l0, int l1,
                                                          const int *__restrict__ line_start, int nunits,
                                                          const int *__restrict__ kus, const int *__restrict__ ukpos,
                                                          const int64_t *__restrict__ ustate,
                                                          const int *__restrict__ uband,
                                                          const cplx<float> *__restrict__ U, int *__restrict__ ustart,
                                                          float *__restrict__ c2, float *__restrict__ c3,
                                                          cplx<float> *__restrict__ ucol) {
    const int64_t n_u = (int64_t)nunits * jl, n_3 = (int64_t)nunits * LP_STEPS;
    const int64_t n_2 = (int64_t)(l1 - l0) * LP_STEPS;
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < n_u) {
        const int64_t u = e / jl, j = e % jl;
        ucol[e] = j < nw ? U[(int64_t)nw * nw * ustate[u] + j + (int64_t)nw * uband[u]] : cplx<float>{0.f, 0.f};
        return;
    }
    e -= n_u;
    if (e < n_3 + n_2) {
        const bool unit = e < n_3;
        const int64_t f = unit ? e : e - n_3, at = f / LP_STEPS;
        const int s = (int)(f % LP_STEPS);
        const int64_t k = unit ? ukpos[kus[k0] + at] : max((int64_t)line_start[l0 + at], k0);
        float cr = 0.f, ci = 0.f;
        if (s <= 2 * h) cis2pi(xk[3 * k + (unit ? 2 : 1)] * (double)(s <= h ? s : s - h), cr, ci);
        (unit ? c3 : c2)[f] = s <= h ? cr : ci;
        return;
    }
    e -= n_3 + n_2;
    if (e <= l1 - l0) {
        const int64_t k = min(max((int64_t)line_start[l0 + e], k0), k1);
        ustart[e] = kus[k] - kus[k0];
    }
}

}  // namespace ephip

using namespace ephip;

extern "C" int ephip_lane_tables(int32_t nw, int32_t jl, int32_t np, const double *xk, int64_t k0, int64_t k1,
                                 int32_t l0, int32_t l1, const int32_t *line_start, int32_t nunits,
                                 const int32_t *kus, const int32_t *ukpos, const int64_t *ustate,
                                 const int32_t *uband, const void *U, int32_t *ustart, float *c2, float *c3,
                                 void *ucol, void *stream) {
    EPHIP_REQUIRE(nw >= 1 && nw <= jl && (jl == 4 || jl == 8 || jl == 16), "lane_tables: nw=%d, jl=%d", nw, jl);
    EPHIP_REQUIRE((np == 3 || np == 5 || np == 7) && k0 >= 0 && k1 >= k0 && l0 >= 0 && l1 >= l0 && nunits >= 0,
                  "lane_tables: bad sizes");
    if (k1 == k0 || l1 == l0) return EPHIP_OK;
    EPHIP_REQUIRE(xk && line_start && kus && ukpos && ustate && uband && U && ustart && c2 && c3 && ucol,
                  "lane_tables: null pointer");
    const int64_t n = (int64_t)nunits * (jl + LP_STEPS) + (int64_t)(l1 - l0) * LP_STEPS + (l1 - l0) + 1;
    lane_tables_kernel<<<(unsigned)((n + 255) / 256), 256, 0, as_stream(stream)>>>(
        nw, jl, np / 2, xk, k0, k1, l0, l1, line_start, nunits, kus, ukpos, ustate, uband,
        static_cast<const cplx<float> *>(U), ustart, c2, c3, static_cast<cplx<float> *>(ucol));
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

template <int N>
static void lane_project_launch(const LpArgs &a, int jl, dim3 grid, hipStream_t st) {
    if (jl == 4)
        lane_project_kernel<N, 4><<<grid, 256, 0, st>>>(a);
    else if (jl == 8)
        lane_project_kernel<N, 8><<<grid, 256, 0, st>>>(a);
    else
        lane_project_kernel<N, 16><<<grid, 256, 0, st>>>(a);
}

extern "C" int ephip_lane_project(int32_t nw, int32_t jl, int64_t ngcol, int32_t np, int32_t nplanes,
                                  const void *const *op1, const int32_t *l0, const int32_t *l1, int32_t lb0,
                                  const int32_t *ustart, const float *c2, const float *c3, const void *ucol, void *A,
                                  int64_t lda, void *stream) {
    EPHIP_REQUIRE(nw >= 1 && nw <= jl && (jl == 4 || jl == 8 || jl == 16), "lane_project: nw=%d, jl=%d", nw, jl);
    EPHIP_REQUIRE(np == 3 || np == 5 || np == 7, "lane_project: box face np x np with np 3, 5 or 7 (got %d)", np);
    EPHIP_REQUIRE(nplanes >= 1 && nplanes <= LP_PLANES, "lane_project: %d planes (1..%d)", nplanes, LP_PLANES);
    EPHIP_REQUIRE(ngcol >= 0 && ngcol % nw == 0 && lb0 >= 0 && lda >= ngcol,
                  "lane_project: bad sizes (columns a multiple of nw, lda >= columns)");
    if (ngcol == 0) return EPHIP_OK;
    EPHIP_REQUIRE(op1 && l0 && l1 && ustart && c2 && c3 && ucol && A, "lane_project: null pointer");
    LpArgs a{};
    int lines = 0;
    for (int p = 0; p < nplanes; p++) {
        EPHIP_REQUIRE(op1[p] && l0[p] >= lb0 && l1[p] >= l0[p], "lane_project: bad plane %d", p);
        a.op1[p] = static_cast<const cplx<float> *>(op1[p]);
        a.l0[p] = l0[p];
        a.l1[p] = l1[p];
        lines = max(lines, l1[p] - l0[p]);
    }
    if (lines == 0) return EPHIP_OK;
    a.nw = nw;
    a.ngcol = ngcol;
    a.nd = ngcol * nw;
    a.lb0 = lb0;
    a.ustart = ustart;
    a.c2 = c2;
    a.c3 = c3;
    a.ucol = static_cast<const cplx<float> *>(ucol);
    a.A = static_cast<cplx<float> *>(A);
    a.lda = lda;
    const int64_t cols = 4 * (64 / jl), gx = (ngcol + cols - 1) / cols;
    EPHIP_REQUIRE(gx <= 0x7fffffffLL && 32 * lda < 0x7fffffffLL, "lane_project: too many columns");
    // parts of a plane's lines: enough workgroups for four waves a SIMD, at least two groups of four lines each
    int64_t z = (1024 + gx * nplanes - 1) / (gx * nplanes);
    z = max(min(z, (int64_t)(lines + 7) / 8), (int64_t)(lines + LP_LINES - 1) / LP_LINES);
    const dim3 grid((unsigned)gx, (unsigned)nplanes, (unsigned)z);
    (np == 3 ? lane_project_launch<3> : np == 5 ? lane_project_launch<5> : lane_project_launch<7>)(a, jl, grid,
                                                                                                  as_stream(stream));
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}
