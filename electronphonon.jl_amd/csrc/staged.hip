// Staged ("GridOpt") outer-k transforms for every model shape: any number of Wannier functions up to 32, any
// number of phonon modes and window bands. The per-axis partial sums of src/wannier/GridOpt.jl:73-139 and of
// src/wannier/batched_gridopt_interpolator.jl, as in gridopt.hip, whose kernels are laid out for 8 or 16
// Wannier functions; here the work is split over what every shape has enough of:
//   * RR->kR with the k-side projection: 16 operator columns per workgroup, four j per wave on FP32 MFMAs, one
//     launch for all k1 planes of a batch;
//   * kR->kq with the rotations and g2: one thread per pair of (kept q, window band) slots of one q line.
#include "lanes.hpp"

namespace ephip {

// (sr, si) += (ar + i ai)(br + i bi), four FMAs
__device__ __forceinline__ void st_cmac(float &sr, float &si, float ar, float ai, float br, float bi) {
    sr = fmaf(ar, br, sr);
    sr = fmaf(-ai, bi, sr);
    si = fmaf(ar, bi, si);
    si = fmaf(ai, br, si);
}

// Boxes that span -h .. h along an axis (N = 2h + 1) are summed in pairs of opposite offsets:
//   sum_b e[b] B[b] = B[h] + sum_j (cos_j S_j + i sin_j D_j),  S_j = B[h+j] + B[h-j],  D_j = B[h+j] - B[h-j],
// S_j kept at h + j and D_j at h - j: four FMAs per pair where two complex multiply-adds take eight.
template <int N>
__device__ __forceinline__ void st_fold(float (&vr)[N], float (&vi)[N]) {
    constexpr int H = N / 2;
#pragma unroll
    for (int j = 1; j <= H; j++) {
        const float pr = vr[H + j], pi = vi[H + j], mr = vr[H - j], mi = vi[H - j];
        vr[H + j] = pr + mr;
        vi[H + j] = pi + mi;
        vr[H - j] = pr - mr;
        vi[H - j] = pi - mi;
    }
}

// The sum from folded (SYM) or plain values; e holds the N phases, of which SYM reads those of positive offsets.
template <int N, bool SYM>
__device__ __forceinline__ void st_sum(float &sr, float &si, const float2 *e, const float (&vr)[N],
                                       const float (&vi)[N]) {
    if constexpr (SYM) {
        constexpr int H = N / 2;
        sr = vr[H];
        si = vi[H];
#pragma unroll
        for (int j = 1; j <= H; j++) {
            const float c = e[H + j].x, s = e[H + j].y;
            sr = fmaf(c, vr[H + j], sr);
            sr = fmaf(-s, vi[H - j], sr);
            si = fmaf(c, vi[H + j], si);
            si = fmaf(s, vr[H - j], si);
        }
    } else {
        sr = si = 0.f;
#pragma unroll
        for (int b = 0; b < N; b++) st_cmac(sr, si, e[b].x, e[b].y, vr[b], vi[b]);
    }
}

// ---------------------------------------------------------------------------------------------
// RR->kR stages 2 and 3 with the k-side projection. op1 of a k1 plane: rows d = i + nw (j + nw rest), face
// (b, c) padded to N x N (ephip_gridopt_stage1_planes, nb = 1). Along a (k1, k2) line
//   A[(k, n)][g] = sum_{j, c} U_k[j, n] e^{2 pi i k3 (r3min + c)} op2[(j, c)][g],  g = i + nw rest,
// with op2 = sum_b e^{2 pi i k2 (r2min + b)} op1: a workgroup takes 16 consecutive g and all j, four j per wave
// (nw padded to a multiple of 4, so 4, 8, 12 .. orbitals run 1, 2, 3 .. waves and idle rows are at most 3), the
// line's units 16 at a time on the rows of a 16x16x4 MFMA. Each lane's op2 is its own B operand; the complex
// product takes four real MFMAs in four independent accumulators. The waves' partial tiles meet in LDS.
// gridDim.y runs over the k1 planes and gridDim.z splits a plane's lines, which keeps small operators (a few
// thousand g) from leaving the chip idle: at 8 orbitals, 6 modes, 5^3 boxes, k 8^3 the eight planes took 248 us in
// eight launches of 188 workgroups (the VALU form of gridopt.hip) and take 58 us in one. The direct phase sums and
// their projection took about 2.6 ms at 12 orbitals, 9 modes, 5^3 (1242 k) and 9.6 ms at 16 orbitals, 12 modes
// (4096 k, split-BF16); here 0.64 and 2.8 ms. Bound by the latency of a line's tables and of the two barriers.
// ---------------------------------------------------------------------------------------------
constexpr int SP_PLANES = 8, SP_KLINE = 64, SP_PAIRS = 128;
struct SpPlanes {
    const cplx<float> *op1[SP_PLANES];
    int l0[SP_PLANES], l1[SP_PLANES];
};

template <int N, bool SYM>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(N <= 7 ? 3 : 2))) void staged_project_kernel(
    int nw, int64_t ngcol, SpPlanes pl, int64_t k0, int64_t k1, int lb0, const int *__restrict__ line_start,
    const int *__restrict__ kus, const int *__restrict__ ukpos, const cplx<float> *__restrict__ ucol,
    const cplx<float> *__restrict__ ph2g, const cplx<float> *__restrict__ ph3g, int max_pairs,
    cplx<float> *__restrict__ A, int64_t lda) {
    extern __shared__ float2 sp_lds[];
    const int nwave = blockDim.x >> 6, nwp = 4 * nwave, bd = blockDim.x;
    float2 *ph2 = sp_lds;                               // [2][N]
    float2 *ph3 = ph2 + 2 * N;                          // [2][SP_KLINE N]
    float2 *uc = ph3 + 2 * SP_KLINE * N;                // [2][max_pairs nwp]: U_k[j, n] of the line's units
    int *pk = reinterpret_cast<int *>(uc + 2 * max_pairs * nwp);  // [2][max_pairs]: unit -> its k on the line
    f32x4 *red = reinterpret_cast<f32x4 *>(pk + 2 * max_pairs);   // [2][2][nwave][64] (offset a multiple of 16)
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int j = t >> 4;
    const int64_t g = (int64_t)blockIdx.x * 16 + (t & 15);
    const bool gv = g < ngcol, dv = gv && j < nw;
    const int p = blockIdx.y;
    const cplx<float> *op1 = pl.op1[p];
    const int64_t nd = ngcol * nw;
    const int64_t row = dv ? g % nw + nw * (j + (int64_t)nw * (g / nw)) : 0;
    float vr[N][N], vi[N][N];
#pragma unroll
    for (int c = 0; c < N; c++)
#pragma unroll
        for (int b = 0; b < N; b++) {
            const cplx<float> v = dv ? op1[row + nd * (b + N * c)] : cplx<float>{0.f, 0.f};
            vr[c][b] = v.re;
            vi[c][b] = v.im;
        }
    if constexpr (SYM) {
#pragma unroll
        for (int c = 0; c < N; c++) st_fold<N>(vr[c], vi[c]);  // over b, for the stage-2 sums
    }
    const int nl = pl.l1[p] - pl.l0[p];
    const int la = pl.l0[p] + (int)((int64_t)nl * blockIdx.z / gridDim.z);
    const int lz = pl.l0[p] + (int)((int64_t)nl * (blockIdx.z + 1) / gridDim.z);
    const int ku0 = kus[k0];
    int lb = 0, tb = 0;  // line buffer, tile buffer
    for (int l = la; l < lz; l++) {
        const int64_t kb = max((int64_t)line_start[l], k0), ke = min((int64_t)line_start[l + 1], k1);
        const int nkl = (int)(ke - kb);  // uniform, at most SP_KLINE (the caller's line pieces)
        if (nkl <= 0) continue;
        const int u0 = kus[kb] - ku0, npl = min(kus[ke] - kus[kb], max_pairs);
        float2 *ucl = uc + lb * max_pairs * nwp;
        for (int e = t; e < N; e += bd) {
            const cplx<float> v = ph2g[(int64_t)(l - lb0) * N + e];
            ph2[lb * N + e] = make_float2(v.re, v.im);
        }
        for (int e = t; e < nkl * N; e += bd) {
            const cplx<float> v = ph3g[(kb - k0) * N + e];
            ph3[lb * SP_KLINE * N + e] = make_float2(v.re, v.im);
        }
        for (int e = t; e < npl * nwp; e += bd) {
            const int q = e / nwp, jj = e % nwp;
            cplx<float> v{0.f, 0.f};
            if (jj < nw) v = ucol[(int64_t)(u0 + q) * nw + jj];
            ucl[e] = make_float2(v.re, v.im);
        }
        for (int e = t; e < npl; e += bd) pk[lb * max_pairs + e] = (int)(ukpos[ku0 + u0 + e] - kb);
        __syncthreads();  // this line's tables staged (the other buffers were last read before it)
        float o2r[N], o2i[N];
#pragma unroll
        for (int c = 0; c < N; c++) st_sum<N, SYM>(o2r[c], o2i[c], ph2 + lb * N, vr[c], vi[c]);
        for (int p0 = 0; p0 < npl; p0 += 16) {
            // A operand: row = unit p0 + lane % 16 (zero past the line's units), column j
            const int q = p0 + (lane & 15);
            int kk = 0;
            float ur = 0.f, ui = 0.f;
            if (q < npl) {
                kk = pk[lb * max_pairs + q];
                const float2 w = ucl[q * nwp + j];
                ur = w.x;
                ui = w.y;
            }
            f32x4 prr = {0.f, 0.f, 0.f, 0.f}, pii = prr, pri = prr, pir = prr;
#pragma unroll
            for (int c = 0; c < N; c++) {
                const float2 e = ph3[lb * SP_KLINE * N + kk * N + c];
                const float wr = ur * e.x - ui * e.y, wi = ur * e.y + ui * e.x;
                prr = __builtin_amdgcn_mfma_f32_16x16x4f32(wr, o2r[c], prr, 0, 0, 0);
                pii = __builtin_amdgcn_mfma_f32_16x16x4f32(wi, o2i[c], pii, 0, 0, 0);
                pri = __builtin_amdgcn_mfma_f32_16x16x4f32(wr, o2i[c], pri, 0, 0, 0);
                pir = __builtin_amdgcn_mfma_f32_16x16x4f32(wi, o2r[c], pir, 0, 0, 0);
            }
            const f32x4 xr = prr - pii, xi = pri + pir;
            // a lane holds units 4 (lane / 16) + r, column g = lane % 16
            if (nwave == 1) {  // uniform
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int q2 = p0 + 4 * (lane >> 4) + r;
                    if (gv && q2 < npl) A[(int64_t)(u0 + q2) * lda + g] = cplx<float>{xr[r], xi[r]};
                }
                continue;
            }
            f32x4 *rd = red + (size_t)tb * 2 * nwave * 64;
            rd[wave * 64 + lane] = xr;
            rd[(nwave + wave) * 64 + lane] = xi;
            __syncthreads();
            for (int e = t; e < 256; e += bd) {
                const int row_u = e >> 4, src = (e & 15) + 16 * (row_u >> 2), r = row_u & 3;
                const float *rf = reinterpret_cast<const float *>(rd);
                float sr = 0.f, si = 0.f;
                for (int w = 0; w < nwave; w++) {
                    sr += rf[(w * 64 + src) * 4 + r];
                    si += rf[((nwave + w) * 64 + src) * 4 + r];
                }
                const int64_t go = (int64_t)blockIdx.x * 16 + (e & 15);
                if (go < ngcol && p0 + row_u < npl) A[(int64_t)(u0 + p0 + row_u) * lda + go] = cplx<float>{sr, si};
            }
            tb ^= 1;
        }
        lb ^= 1;
    }
}

__host__ inline size_t sp_lds_bytes(int n, int nwave, int max_pairs) {
    return sizeof(float2) * (2 * (size_t)n + 2 * (size_t)SP_KLINE * n + 2 * (size_t)max_pairs * 4 * nwave) +
           sizeof(int) * 2 * (size_t)max_pairs + sizeof(f32x4) * 4 * (size_t)nwave * 64;
}

// ---------------------------------------------------------------------------------------------
// kR->kq over Rp for the q of a uniform grid with the k+q-window and phonon rotations and g2. One workgroup per
// (unit, q1). Every kept q of the slab, in line (q2) order, makes ceil(window bands / NB) entries of NB bands; a
// thread takes NQ consecutive entries of one line, so the sum over i in t = sum_i conj(U_kq[i, m]) g[i] stays in
// the thread (no cross-lane reduction) and one read of the line's stage-2 sums from LDS serves all of them. tb
// threads hold a segment's entries; nug such groups take one mode each, so a pass covers nug modes: stage 1
// (B1[b, c] = sum_a e1 A) and stage 2 (B2[line][row][c] = sum_b e2 B1) by all threads through LDS, stage 3
// (g = sum_c e3 B2) and the product with U in registers, t[entry][nu] into LDS. At the end the phonon rotation,
// with u_ph of a batch of columns staged in LDS where B1 and B2 were (read by column once, in full lines: read by
// each (band, mode) from memory it took most of the kernel's time).
// Against the direct sums and the rotation kernel (g(k, q) stored and read back), ms: 4 orbitals, 3 modes, 7^3 boxes,
// q 24^3, 2794 units 17.5 -> 1.0; 12 orbitals, 9 modes, 5^3, q 18 x 15 x 12, 1260 units 3.7 -> 1.0; 16 orbitals, 12
// modes, 5 window bands, 5^3, q 8^3, 10505 units 19.0 (split-BF16) -> 8.6. Bound by the chain of latencies and
// barriers of a workgroup whose slab is small: waves wait 55% of their time, the VALU is 58% busy (4 orbitals).
// Kept q are taken in segments: at most NQ tb entries and lines together and at most ls non-empty lines (the size
// of B2); a line may be cut. The pitch of a line in B2 is 16 bytes over a multiple of 16, so the lines that the
// lanes of a wave read lie in different banks.
// ---------------------------------------------------------------------------------------------
constexpr int SQ_LINES = 64, SQ_CPL = 4, SQ_COLS = 64 * SQ_CPL;

struct SqArgs {
    int nw, nm, nbw, n1, dense, s1, s2, s3, m1, m2, m3, tb, nug, ls, split;
    const float2 *e1, *e2, *e3;              // phases of q1 [m1][n1], q2 [m2][NE], q3 [m3][NE]
    unsigned mg_rows, mg_nm, mg_nm2, mg_rn;  // floor(e / d) = umulhi(e, ceil(2^32 / d)) for e < 2^16
    const int *rmap;
    const cplx<float> *A;
    int64_t lda;
    int ldr;
    const int *line_off, *col_index, *ikq;
    int64_t cs;
    const cplx<float> *U;
    const int64_t *bmin, *bmax;
    const cplx<float> *uph;
    const double *omega;
    float *g2;
    float2 *ep;
};

__host__ inline unsigned sq_magic(int d) { return d == 1 ? 0u : (unsigned)(((1ull << 32) + d - 1) / d); }
__device__ __forceinline__ int sq_div(int e, unsigned magic) {  // magic 0: divisor 1
    return magic ? (int)__umulhi((unsigned)e, magic) : e;
}

// LDS carve-up, in float2: ph2 | ph3 | t | B1 | B2 (u_ph of a batch in the end); then ints
template <int N>
__host__ __device__ inline int sq_line_pitch(int gc) { return gc * ((N + 1) & ~1) + 2; }
template <int N>
__host__ __device__ inline int sq_b_floats2(const SqArgs &a) {  // B1 and B2, at least one column of u_ph
    const int gc = a.nug * a.nw, b = N * N * gc + (N * N * gc & 1) + a.ls * sq_line_pitch<N>(gc);
    const int one = a.nm * (((a.nm + 1) & ~1) + 2);
    return b > one ? b : one;
}
template <int N>
__host__ __device__ inline size_t sq_lds_bytes(const SqArgs &a, int nq, int nb) {
    const int ne = (N + 1) & ~1, tt = nq * nb * a.tb * (((a.nm + 1) & ~1) + 2);
    return sizeof(float2) * ((size_t)(a.m2 + a.m3) * ne + (size_t)tt + (size_t)sq_b_floats2<N>(a)) +
           sizeof(int) * (2 * (SQ_LINES + 1) + SQ_LINES + 4 * SQ_COLS + (size_t)nq * a.tb + 5);
}

template <int N, bool SYM, int NWT, int NQ, int NB>
__global__ __launch_bounds__(512) void staged_kq_kernel(SqArgs a) {
    constexpr int NE = (N + 1) & ~1, H = N / 2;
    extern __shared__ float4 sq_lds[];
    const int t = threadIdx.x, bd = blockDim.x, lane = t & 63, wave = t >> 6;
    const int nw = a.nw, nm = a.nm, m2 = a.m2, m3 = a.m3;
    const int tb = a.tb, grp = t / tb, ts = t - grp * tb;  // mode group, thread in the group
    const int gc = a.nug * nw, pitch = sq_line_pitch<N>(gc);
    const int tp = ((nm + 1) & ~1) + 2;  // pitch of t and u_ph rows: 16-byte aligned, spread over the banks
    float2 *ph2 = reinterpret_cast<float2 *>(sq_lds), *ph3 = ph2 + m2 * NE;
    float2 *tq = ph3 + m3 * NE;                       // [NQ tb][NB][tp]
    float2 *B1 = tq + (size_t)NQ * NB * tb * tp;
    float2 *B2 = B1 + N * N * gc + (N * N * gc & 1);  // 16-byte aligned
    int *lsl = reinterpret_cast<int *>(B1 + sq_b_floats2<N>(a));  // [lines + 1] first entry of each line
    int *ltk = lsl + SQ_LINES + 1;     // [lines + 1] first task of each line
    int *lq2 = ltk + SQ_LINES + 1;     // [lines] q2
    int *cent = lq2 + SQ_LINES;        // [SQ_COLS] first entry of a column
    int *cmeta = cent + SQ_COLS;       // [SQ_COLS] window bands | first band << 8 | q3 << 16
    int *ckq = cmeta + SQ_COLS;        // [SQ_COLS] k+q state
    int *ciq = ckq + SQ_COLS;          // [SQ_COLS] q
    int *stab = ciq + SQ_COLS;         // [NQ tb] entry -> column | band group << 16 | line << 24, or -1
    int *seg = stab + NQ * tb;         // columns, lines, tasks of the segment
    // the m1 workgroups of a unit read the same operator: runs of (unit, q1) pairs go to one XCD (workgroups are
    // dealt to the 8 XCDs in turn), whose L2 then serves them
    const int64_t T = (int64_t)gridDim.x * gridDim.y, L = blockIdx.x + (int64_t)gridDim.x * blockIdx.y;
    const int64_t xc = L & 7, base = T >> 3, rem = T & 7, id = xc * base + (xc < rem ? xc : rem) + (L >> 3);
    const int u = (int)(id / gridDim.x), q1 = (int)(id - (int64_t)u * gridDim.x);
    const int *lo_u = a.line_off + (int64_t)u * (a.m1 * m2 + 1) + q1 * m2;
    const int64_t row0 = (int64_t)u * a.cs;
    const cplx<float> *au = a.A + (int64_t)u * a.lda;
    int c0 = lo_u[0];
    const int c_end = lo_u[m2];
    if (c0 >= c_end) return;  // uniform
    const int rows = gc, items = N * N * rows, last_row = nm * nw - 1;
    // stage 1 of the modes from nu0 on, by the threads w0 .. bd - 1 (rows past the last mode repeat it, unused)
    const float2 *e1 = a.e1 + q1 * a.n1;
    auto stage1 = [&](int nu0, int w0) {
        const int r0 = nu0 * nw, step_t = bd - w0;
        if (SYM || a.dense) {  // n1 = N: S1 items per thread with their loads in flight together
            constexpr int S1 = N <= 5 ? 4 : 3;
            float2 ph[N];
#pragma unroll
            for (int x = 0; x < N; x++) ph[x] = e1[x];  // uniform
            for (int e0 = t - w0; e0 < items; e0 += S1 * step_t) {
                float vr[S1][N], vi[S1][N];
#pragma unroll
                for (int y = 0; y < S1; y++) {
                    const int e = min(e0 + y * step_t, items - 1);
                    const int bc = sq_div(e, a.mg_rows), r = min(r0 + e - bc * rows, last_row);
                    const int c = bc / N, b = bc - N * c;
                    if (a.dense) {
                        unsigned o = (unsigned)((a.s2 * b + a.s3 * c) * a.ldr + r);
                        const unsigned step = (unsigned)(a.s1 * a.ldr);
#pragma unroll
                        for (int x = 0; x < N; x++) {
                            const cplx<float> v = au[o];
                            o += step;
                            vr[y][x] = v.re;
                            vi[y][x] = v.im;
                        }
                    } else {
#pragma unroll
                        for (int x = 0; x < N; x++) {
                            const int ir = a.rmap[b + 8 * (x + N * c)];
                            const cplx<float> v = au[(unsigned)(a.ldr * max(ir, 0) + r)];
                            vr[y][x] = ir >= 0 ? v.re : 0.f;
                            vi[y][x] = ir >= 0 ? v.im : 0.f;
                        }
                    }
                }
#pragma unroll
                for (int y = 0; y < S1; y++) {
                    float sr, si;
                    if constexpr (SYM) st_fold<N>(vr[y], vi[y]);
                    st_sum<N, SYM>(sr, si, ph, vr[y], vi[y]);
                    if (e0 + y * step_t < items) B1[e0 + y * step_t] = make_float2(sr, si);
                }
            }
        } else {
            for (int e = t - w0; e < items; e += step_t) {
                const int bc = sq_div(e, a.mg_rows), r = min(r0 + e - bc * rows, last_row), c = bc / N, b = bc - N * c;
                float sr = 0.f, si = 0.f;
                for (int x = 0; x < a.n1; x++) {
                    const int ir = a.rmap[b + 8 * (x + a.n1 * c)];
                    cplx<float> v = au[(unsigned)(a.ldr * max(ir, 0) + r)];
                    if (ir < 0) v = cplx<float>{0.f, 0.f};
                    const float2 p = e1[x];
                    st_cmac(sr, si, p.x, p.y, v.re, v.im);
                }
                B1[e] = make_float2(sr, si);
            }
        }
    };
    for (int e = t; e < (m2 + m3) * NE; e += bd) ph2[e] = e < m2 * NE ? a.e2[e] : a.e3[e - m2 * NE];
    while (true) {  // segments (uniform)
        if (wave == 0) {
            // ---- the segment's columns, entries, lines and tasks, by one wave (SQ_CPL consecutive columns per
            // lane), while the others run stage 1 of the first modes
            int kq[SQ_CPL], iq[SQ_CPL], nb[SQ_CPL], mlo[SQ_CPL], ng[SQ_CPL], q2[SQ_CPL], v[SQ_CPL];
#pragma unroll
            for (int x = 0; x < SQ_CPL; x++) {
                const int64_t r = row0 + min(c0 + SQ_CPL * lane + x, c_end - 1);
                kq[x] = a.ikq[r];
                iq[x] = a.col_index[r];
            }
#pragma unroll
            for (int x = 0; x < SQ_CPL; x++) {
                const int b0 = (int)a.bmin[kq[x]], b1 = (int)a.bmax[kq[x]];
                nb[x] = b0 > 0 ? min(b1 - b0 + 1, a.nbw) : 0;
                mlo[x] = b0 > 0 ? b0 - 1 : 0;
                ng[x] = (nb[x] + NB - 1) / NB;
                q2[x] = iq[x] / m3;  // q1 m2 + q2
            }
            const int before = __shfl_up(q2[SQ_CPL - 1], 1, 64);
            int pre = 0;  // inclusive prefix over the columns of (entries | lines << 16)
#pragma unroll
            for (int x = 0; x < SQ_CPL; x++) {
                const int last = x ? q2[x - 1] : before;
                const bool ok = c0 + SQ_CPL * lane + x < c_end;
                pre += ok ? ng[x] | ((lane == 0 && x == 0) || last != q2[x] ? 1 << 16 : 0) : 0;
                v[x] = pre;
            }
            int tot = pre;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int o = __shfl_up(tot, off, 64);
                if (lane >= off) tot += o;
            }
            // a column is taken while entries + lines <= NQ tb (so tasks <= tb) and lines <= ls: a prefix of them, and
            // at least one (sq_choose)
            int taken = 0, end = 0;
            bool in[SQ_CPL];
#pragma unroll
            for (int x = 0; x < SQ_CPL; x++) {
                v[x] += tot - pre;
                const int ne = v[x] & 0xffff, nl = v[x] >> 16, kk = SQ_CPL * lane + x;
                in[x] = c0 + kk < c_end && ne + (NQ > 1 ? nl : 0) <= NQ * tb && nl <= a.ls;
                taken += in[x] ? 1 : 0;
                if (in[x]) {
                    end = v[x];
                    const int last = x ? q2[x - 1] : before;
                    if (kk == 0 || last != q2[x]) {
                        lsl[nl - 1] = ne - ng[x];
                        lq2[nl - 1] = q2[x] - q1 * m2;
                    }
                    ckq[kk] = kq[x];
                    ciq[kk] = iq[x];
                    cmeta[kk] = nb[x] | (mlo[x] << 8) | ((iq[x] - q2[x] * m3) << 16);
                }
            }
            for (int e = lane; e < NQ * tb; e += 64) stab[e] = -1;
            const int ncol = (int)wave_sum((float)taken);  // at most SQ_COLS: exact
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) end = max(end, __shfl_xor(end, off, 64));  // both parts grow
            const int nlin = end >> 16;
            if (lane == 0) lsl[nlin] = end & 0xffff;
            wave_lds_sync();
            const int mine = lane < nlin ? (lsl[lane + 1] - lsl[lane] + NQ - 1) / NQ : 0;  // tasks of a line
            int p = mine;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int o = __shfl_up(p, off, 64);
                if (lane >= off) p += o;
            }
            ltk[lane] = p - mine;
            if (lane == 63) seg[2] = p;
            if (lane == 0) {
                seg[0] = ncol;
                seg[1] = nlin;
            }
            wave_lds_sync();
#pragma unroll
            for (int x = 0; x < SQ_CPL; x++) {
                if (!in[x]) continue;
                const int l = (v[x] >> 16) - 1, kk = SQ_CPL * lane + x;
                const int e = NQ * ltk[l] + (v[x] & 0xffff) - ng[x] - lsl[l];
                cent[kk] = e;
                for (int m = 0; m < ng[x]; m++) stab[e + m] = kk | (m << 16) | (l << 24);
            }
            if (bd == 64) stage1(0, 0);
        } else {
            stage1(0, 64);
        }
        __syncthreads();  // tables of the segment, phases, B1 of the first modes
        const int ncol = seg[0], nlin = seg[1], ntask = seg[2];
        // ---- this thread's NQ entries of NB bands
        const bool act = ts < ntask && grp < a.nug;
        float ur[NQ * NB][NWT], ui[NQ * NB][NWT];
        float2 e3[NQ][SYM ? H + 1 : N];
        int line = 0;
#pragma unroll
        for (int x = 0; x < NQ; x++) {
            const int s0 = act ? stab[NQ * ts] : -1;  // the first entry of a task is always there
            const int sx = act ? stab[NQ * ts + x] : -1;
            const int kk = (sx >= 0 ? sx : max(s0, 0)) & 0xffff, meta = cmeta[kk];
            if (x == 0) line = s0 >= 0 ? (s0 >> 24) & 0xff : 0;
            const int mg = sx >= 0 ? ((sx >> 16) & 0xff) * NB : 0, left = sx >= 0 ? (meta & 0xff) - mg : 0;
            const cplx<float> *uk = a.U + (int64_t)nw * nw * ckq[kk] + nw * (((meta >> 8) & 0xff) + mg);
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int i = 0; i < NWT; i++) {
                    cplx<float> w{0.f, 0.f};
                    if (i < nw && b < left) w = uk[nw * b + i];
                    ur[x * NB + b][i] = w.re;
                    ui[x * NB + b][i] = w.im;
                }
            const float2 *pq = ph3 + ((meta >> 16) & 0xff) * NE;
            if constexpr (SYM) {
#pragma unroll
                for (int j = 1; j <= H; j++) e3[x][j] = pq[H + j];
            } else {
#pragma unroll
                for (int c = 0; c < N; c++) e3[x][c] = pq[c];
            }
        }
        const float4 *b2l = reinterpret_cast<const float4 *>(B2 + line * pitch + grp * nw * NE);
        float2 *tl = tq + (size_t)NQ * NB * ts * tp + grp;
        // ---- the modes, nug at a time
        for (int nu0 = 0; nu0 < nm; nu0 += a.nug) {
            if (nu0) {
                stage1(nu0, 0);
                __syncthreads();  // B1 written; every thread is past the last round's reads of B2
            }
            for (int e = t; e < N * rows * a.split; e += bd) {  // stage 2: one (row, c), every split-th line
                const int part = sq_div(e, a.mg_rn), f = e - part * (N * rows), r = f / N, c = f - N * r;
                float vr[N], vi[N];
#pragma unroll
                for (int b = 0; b < N; b++) {
                    const float2 v = B1[(b + N * c) * rows + r];
                    vr[b] = v.x;
                    vi[b] = v.y;
                    if constexpr (SYM) {  // folded over c for stage 3 (linear, so ahead of the sum over b)
                        const float2 w = B1[(b + N * (N - 1 - c)) * rows + r];
                        const float sg = c > H ? 1.f : c < H ? -1.f : 0.f;  // S_j = v + w, D_j = w - v
                        vr[b] = c < H ? w.x - vr[b] : fmaf(sg, w.x, vr[b]);
                        vi[b] = c < H ? w.y - vi[b] : fmaf(sg, w.y, vi[b]);
                    }
                }
                if constexpr (SYM) st_fold<N>(vr, vi);
                float2 *o = B2 + r * NE + c;
                for (int l = part; l < nlin; l += a.split) {
                    float sr, si;
                    st_sum<N, SYM>(sr, si, ph2 + lq2[l] * NE, vr, vi);
                    o[l * pitch] = make_float2(sr, si);
                }
            }
            __syncthreads();  // B2 of this segment's lines
            if (act && nu0 + grp < nm) {
                float tr[NQ * NB], ti[NQ * NB];
#pragma unroll
                for (int x = 0; x < NQ * NB; x++) tr[x] = ti[x] = 0.f;
#pragma unroll
                for (int i = 0; i < NWT; i++) {
                    if (i < nw) {  // uniform
                        float vr[NE], vi[NE];
#pragma unroll
                        for (int h = 0; h < NE / 2; h++) {
                            const float4 v = b2l[i * (NE / 2) + h];
                            vr[2 * h] = v.x;
                            vi[2 * h] = v.y;
                            vr[2 * h + 1] = v.z;
                            vi[2 * h + 1] = v.w;
                        }
#pragma unroll
                        for (int x = 0; x < NQ; x++) {
                            float gr, gi;
                            if constexpr (SYM) {
                                gr = vr[H];
                                gi = vi[H];
#pragma unroll
                                for (int j = 1; j <= H; j++) {
                                    gr = fmaf(e3[x][j].x, vr[H + j], gr);
                                    gr = fmaf(-e3[x][j].y, vi[H - j], gr);
                                    gi = fmaf(e3[x][j].x, vi[H + j], gi);
                                    gi = fmaf(e3[x][j].y, vr[H - j], gi);
                                }
                            } else {
                                gr = gi = 0.f;
#pragma unroll
                                for (int c = 0; c < N; c++) st_cmac(gr, gi, e3[x][c].x, e3[x][c].y, vr[c], vi[c]);
                            }
#pragma unroll
                            for (int b = 0; b < NB; b++) {
                                const int y = x * NB + b;
                                tr[y] = fmaf(ur[y][i], gr, tr[y]);
                                tr[y] = fmaf(ui[y][i], gi, tr[y]);
                                ti[y] = fmaf(ur[y][i], gi, ti[y]);
                                ti[y] = fmaf(-ui[y][i], gr, ti[y]);
                            }
                        }
                    }
                }
#pragma unroll
                for (int x = 0; x < NQ * NB; x++) tl[x * tp + nu0] = make_float2(tr[x], ti[x]);
            }
        }
        __syncthreads();  // t of the segment; B1 and B2 no longer read
        // ---- phonon rotation and g2, a batch of columns at a time
        float2 *ub = B1;  // [column][n2][tp]
        const int nm2 = nm * nm, per = max(1, sq_b_floats2<N>(a) / (nm * tp));
        for (int k0 = 0; k0 < ncol; k0 += per) {
            const int nc = min(per, ncol - k0);
            if (nm & 1) {
                for (int e0 = t; e0 < nc * nm2; e0 += 4 * bd) {
                    float2 v[4];
                    int o[4];
#pragma unroll
                    for (int y = 0; y < 4; y++) {
                        const int e = min(e0 + y * bd, nc * nm2 - 1), kk = sq_div(e, a.mg_nm2), f = e - kk * nm2;
                        const int n2 = sq_div(f, a.mg_nm);
                        v[y] = reinterpret_cast<const float2 *>(a.uph)[(int64_t)nm2 * ciq[k0 + kk] + f];
                        o[y] = (kk * nm + n2) * tp + f - n2 * nm;
                    }
#pragma unroll
                    for (int y = 0; y < 4; y++)
                        if (e0 + y * bd < nc * nm2) ub[o[y]] = v[y];
                }
            } else {  // two modes per load (even offsets)
                const int h2 = nm2 / 2;
                for (int e0 = t; e0 < nc * h2; e0 += 4 * bd) {
                    float4 v[4];
                    int o[4];
#pragma unroll
                    for (int y = 0; y < 4; y++) {
                        const int e = min(e0 + y * bd, nc * h2 - 1), kk = sq_div(2 * e, a.mg_nm2), f = 2 * e - kk * nm2;
                        const int n2 = sq_div(f, a.mg_nm);
                        v[y] = reinterpret_cast<const float4 *>(a.uph)[(int64_t)h2 * ciq[k0 + kk] + (f >> 1)];
                        o[y] = (kk * nm + n2) * tp + f - n2 * nm;
                    }
#pragma unroll
                    for (int y = 0; y < 4; y++)
                        if (e0 + y * bd < nc * h2) *reinterpret_cast<float4 *>(ub + o[y]) = v[y];
                }
            }
            __syncthreads();
            // entries of the batch's columns (those of a line's unfilled last task are -1), all their bands
            const int ea = cent[k0], ez = k0 + nc < ncol ? cent[k0 + nc] : NQ * ntask;
            for (int e = t; e < (ez - ea) * NB * nm; e += bd) {
                const int eb = sq_div(e, a.mg_nm), n2 = e - eb * nm, en = ea + eb / NB, b = eb % NB;
                const int sx = stab[en];
                if (sx < 0) continue;
                const int kk = sx & 0xffff, m = ((sx >> 16) & 0xff) * NB + b;
                if (m >= (cmeta[kk] & 0xff)) continue;
                const float2 *tv = tq + (en * NB + b) * tp, *uv = ub + ((kk - k0) * nm + n2) * tp;
                float er = 0.f, ei = 0.f;
                int n = 0;
                for (; n + 1 < nm; n += 2) {
                    const float4 x = *reinterpret_cast<const float4 *>(tv + n), y = *reinterpret_cast<const float4 *>(uv + n);
                    st_cmac(er, ei, x.x, x.y, y.x, y.y);
                    st_cmac(er, ei, x.z, x.w, y.z, y.w);
                }
                if (n < nm) st_cmac(er, ei, tv[n].x, tv[n].y, uv[n].x, uv[n].y);
                const int64_t row = row0 + c0 + kk;
                const float w2 = 2.f * static_cast<float>(a.omega[(int64_t)nm * ciq[kk] + n2]);
                const int64_t oi = (row * a.nbw + m) * nm + n2;
                a.g2[oi] = (er * er + ei * ei) / w2;
                if (a.ep) a.ep[oi] = make_float2(er, ei);
            }
            __syncthreads();  // the batch's u_ph no longer read
        }
        // zeros past the k+q window
        for (int m = 1; m < a.nbw; m++)
            for (int e = t; e < ncol * nm; e += bd) {
                const int kk = sq_div(e, a.mg_nm), n2 = e - kk * nm;
                if (m < (cmeta[kk] & 0xff)) continue;
                const int64_t oi = ((row0 + c0 + kk) * a.nbw + m) * nm + n2;
                a.g2[oi] = 0.f;
                if (a.ep) a.ep[oi] = make_float2(0.f, 0.f);
            }
        c0 += ncol;
        if (c0 >= c_end) break;
        __syncthreads();  // the segment's tables no longer read
    }
}

// The same in the lane-private form of lanes.hpp (nw <= 16, nm <= 16, boxes that span -h .. h): a lane is one
// (mode, i), a wave 64 / JL modes. Stage 1 ends in the lane's registers; stage 2 forms four q2 lines at a time and
// stage 3 four entries (kept q, window band) of a line, both as 4x4x1 MFMAs; the product with U and the sum over i run
// on the VALU and leave t in LDS for the phonon rotation. The tables of the slab are laid down once; U columns and
// stage-3 rows are staged for at most LQ_ENT entries of the four lines, in equal parts.
// ms, staged_kq_kernel -> this: 16 orbitals, 12 modes, 5^3 boxes, 5 window bands, q 8^3, 10505 units 8.7 -> 5.0 (5.9 with
// parts of 64 and the row of u_ph read as it was used; 5.5 at four waves a SIMD, which spill); 12 orbitals, 9 modes,
// q 18 x 15 x 12, 1260 units 1.09 -> 0.82. Whole passes: 12, 12, 5^3, q 16^3, 3 bands 12.3 -> 4.5; 10, 15, q 20^3
// 5.6 -> 2.7; 12, 12, 7^3, q 12^3 3.56 -> 3.25. Waves wait for the staging and its barriers 54% of their time; VALU
// 46% busy, MFMAs 9% (5 window bands; 42%, 53%, 13% at 12 orbitals).
constexpr int LQ_ENT = 96, LQ_TP = 18, LQ_SLAB = 4096;  // LQ_SLAB: words of the tables of a slab

__host__ inline size_t lq_lds_bytes(const SqArgs &a, int jl) {
    return sizeof(float) * LP_STEPS * (size_t)(a.m2 + a.m3 + LQ_ENT + 4) +
           sizeof(float2) * (size_t)(LQ_ENT + 4) * (jl + LQ_TP) + sizeof(int) * ((4 + (size_t)a.nbw) * a.m2 * a.m3 + a.m2 + 2);
}

template <int N, int JL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(N == 7 ? 2 : N == 5 ? 3 : 4))) void lane_kq_kernel(
    SqArgs a) {
    constexpr int NE = (N + 1) & ~1, H = N / 2, CL = 64 / JL;
    extern __shared__ float4 sq_lds[];
    const int nw = a.nw, nm = a.nm, m2 = a.m2, m3 = a.m3, slab = m2 * m3;
    float2 *tq = reinterpret_cast<float2 *>(sq_lds);         // [LQ_ENT + 4][LQ_TP]
    float2 *us = tq + (LQ_ENT + 4) * LQ_TP;                  // [LQ_ENT + 4][JL]: conj U_kq
    float *c2t = reinterpret_cast<float *>(us + (LQ_ENT + 4) * JL), *c3t = c2t + LP_STEPS * m2;
    float *c3e = c3t + LP_STEPS * m3;                        // [LQ_ENT + 4]: stage-3 row of an entry
    int *skq = reinterpret_cast<int *>(c3e + LP_STEPS * (LQ_ENT + 4));  // k+q state of a kept q
    int *siq = skq + slab, *smeta = siq + slab;              // q; window bands | first band << 8 | q3 << 16
    int *eoff = smeta + slab;                                // [slab + 1] first entry of a kept q
    int *slo = eoff + slab + 1;                              // [m2 + 1] first kept q of a line
    int *ent = slo + m2 + 1;                                 // [slab nbw] entry -> kept q | band << 16
    const int t = threadIdx.x, bd = blockDim.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    // runs of (unit, q1) pairs go to one XCD, as in staged_kq_kernel
    const int64_t T = (int64_t)gridDim.x * gridDim.y, L = blockIdx.x + (int64_t)gridDim.x * blockIdx.y;
    const int64_t xc = L & 7, base = T >> 3, rem = T & 7, id = xc * base + (xc < rem ? xc : rem) + (L >> 3);
    const int u = (int)(id / gridDim.x), q1 = (int)(id - (int64_t)u * gridDim.x);
    const int *lo_u = a.line_off + (int64_t)u * (a.m1 * m2 + 1) + q1 * m2;
    const int sb = lo_u[0], n = lo_u[m2] - sb;
    if (n <= 0) return;  // uniform; n <= slab
    const int64_t row0 = (int64_t)u * a.cs + sb;
    for (int kk = t; kk < n; kk += bd) {
        const int kq = a.ikq[row0 + kk], iq = a.col_index[row0 + kk];
        const int b0 = (int)a.bmin[kq], b1 = (int)a.bmax[kq];
        skq[kk] = kq;
        siq[kk] = iq;
        smeta[kk] = (b0 > 0 ? min(b1 - b0 + 1, a.nbw) | ((b0 - 1) << 8) : 0) | ((iq % m3) << 16);
    }
    for (int l = t; l <= m2; l += bd) slo[l] = lo_u[l] - sb;
    for (int e = t; e < LP_STEPS * (m2 + m3); e += bd) {  // (1, cos, sin) of the q2 and q3
        const int f = e / LP_STEPS, s = e % LP_STEPS;
        const float2 *ph = f < m2 ? a.e2 + f * NE : a.e3 + (f - m2) * NE;
        c2t[e] = s == 0 ? 1.f : s <= H ? ph[H + s].x : s <= 2 * H ? ph[s].y : 0.f;
    }
    __syncthreads();
    if (wave == 0) {
        int run = 0;
        for (int k0 = 0; k0 < n; k0 += 64) {
            const int v = k0 + lane < n ? smeta[k0 + lane] & 0xff : 0;
            int p = v;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int o = __shfl_up(p, off, 64);
                if (lane >= off) p += o;
            }
            if (k0 + lane < n) eoff[k0 + lane] = run + p - v;
            for (int m = 0; m < v; m++) ent[run + p - v + m] = (k0 + lane) | (m << 16);
            run += __builtin_amdgcn_readlane(p, 63);
        }
        if (lane == 0) eoff[n] = run;
    }
    const int j = lane / CL, nu = wave * CL + lane % CL;
    const bool ok = j < nw && nu < nm;
    const int r0 = ok ? j + nw * nu : 0;
    const cplx<float> *au = a.A + (int64_t)u * a.lda;
    const float2 *e1 = a.e1 + q1 * a.n1;
    float xr[N][N], xi[N][N];
#pragma unroll
    for (int c = 0; c < N; c++) {
        float br[N], bi[N];
#pragma unroll
        for (int b = 0; b < N; b++) br[b] = bi[b] = 0.f;
#pragma unroll
        for (int x = 0; x < N; x++)
#pragma unroll
            for (int b = 0; b < N; b++) {  // absent R: column 0 loaded, zero used
                const int ir = a.rmap[b + 8 * (x + N * c)];  // uniform; the N entries are contiguous
                const cplx<float> v = au[(int64_t)a.ldr * max(ir, 0) + r0];
                const float kr = ir >= 0 ? v.re : 0.f, ki = ir >= 0 ? v.im : 0.f;
                st_cmac(br[b], bi[b], e1[x].x, e1[x].y, kr, ki);
            }
#pragma unroll
        for (int b = 0; b < N; b++) {
            br[b] = ok ? br[b] : 0.f;
            bi[b] = ok ? bi[b] : 0.f;
        }
        lp_fold<N>(xr[c], xi[c], br, bi);
        __builtin_amdgcn_sched_barrier(0);  // one c's loads in flight: all of them would spill
    }
    __syncthreads();  // eoff, ent
    const int row = lane & 3, step = (lane >> 2) & (LP_STEPS - 1);
    float2 *tl = tq + (lane >> 4) * LQ_TP + wave * CL + (lane & (CL - 1));
    for (int l = 0; l < m2; l += 4) {
        const int ka = __builtin_amdgcn_readfirstlane(slo[l]), kz = __builtin_amdgcn_readfirstlane(slo[min(l + 4, m2)]);
        if (ka == kz) continue;  // uniform
        const int ea = __builtin_amdgcn_readfirstlane(eoff[ka]), ez = __builtin_amdgcn_readfirstlane(eoff[kz]);
        const float mc2 = c2t[LP_STEPS * min(l + row, m2 - 1) + step];
        f32x4 tr[N], ti[N];  // stage 2 of four lines, before the fold over c
#pragma unroll
        for (int c = 0; c < N; c++) lp_apply<N>(tr[c], ti[c], mc2, xr[c], xi[c]);
        // the entries of the four lines in equal parts of at most LQ_ENT
        const int parts = (ez - ea + LQ_ENT - 1) / LQ_ENT, part = (ez - ea + parts - 1) / parts;
        for (int cb = ea; cb < ez; cb += part) {
            const int ce = min(cb + part, ez);
            __syncthreads();  // the last entries' tables no longer read
            for (int e0 = t; e0 < (ce - cb) * JL; e0 += 4 * bd) {  // four loads in flight
                cplx<float> v[4];
#pragma unroll
                for (int y = 0; y < 4; y++) {
                    const int e = min(e0 + y * bd, (ce - cb) * JL - 1), s = ent[cb + e / JL], kk = s & 0xffff, jj = min(e % JL, nw - 1);
                    v[y] = a.U[(int64_t)nw * nw * skq[kk] + jj + nw * (((smeta[kk] >> 8) & 0xff) + (s >> 16))];
                }
#pragma unroll
                for (int y = 0; y < 4; y++) {
                    const int e = e0 + y * bd;
                    if (e < (ce - cb) * JL) us[e] = e % JL < nw ? make_float2(v[y].re, -v[y].im) : make_float2(0.f, 0.f);
                }
            }
            for (int e = t; e < (ce - cb) * LP_STEPS; e += bd)
                c3e[e] = c3t[LP_STEPS * (smeta[ent[cb + e / LP_STEPS] & 0xffff] >> 16) + e % LP_STEPS];
            __syncthreads();
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (l + r >= m2) break;
                const int es = max(cb, __builtin_amdgcn_readfirstlane(eoff[slo[l + r]]));
                const int ee = min(ce, __builtin_amdgcn_readfirstlane(eoff[slo[l + r + 1]]));
                if (es >= ee) continue;
                float br[N], bi[N], zr[N], zi[N];
#pragma unroll
                for (int c = 0; c < N; c++) {
                    br[c] = tr[c][r];
                    bi[c] = ti[c][r];
                }
                lp_fold<N>(zr, zi, br, bi);
                float m = c3e[(es - cb + row) * LP_STEPS + step];
                float2 w = us[(es - cb + row) * JL + j];
                for (int e = es - cb; e < ee - cb; e += 4) {
                    const float mm = m;
                    const float2 ww = w;
                    const int nx = min(e + 4, LQ_ENT);  // rows past the line are formed and written, then written over
                    m = c3e[(nx + row) * LP_STEPS + step];
                    w = us[(nx + row) * JL + j];
                    f32x4 gr, gi;
                    lp_apply<N>(gr, gi, mm, zr, zi);
                    float vr[4], vi[4];
                    lp_times<0>(vr[0], vi[0], ww.x, ww.y, gr[0], gi[0]);
                    lp_times<1>(vr[1], vi[1], ww.x, ww.y, gr[1], gi[1]);
                    lp_times<2>(vr[2], vi[2], ww.x, ww.y, gr[2], gi[2]);
                    lp_times<3>(vr[3], vi[3], ww.x, ww.y, gr[3], gi[3]);
                    tl[e * LQ_TP] = make_float2(lp_reduce<JL>(vr), lp_reduce<JL>(vi));
                }
            }
            __syncthreads();  // t of the entries
            for (int e = t; e < (ce - cb) * nm; e += bd) {
                const int x = sq_div(e, a.mg_nm), n2 = e - x * nm, s = ent[cb + x], kk = s & 0xffff;
                const int64_t col = (int64_t)nm * siq[kk] + n2;
                const float2 *uv = reinterpret_cast<const float2 *>(a.uph) + col * nm;
                const float w2 = 2.f * static_cast<float>(a.omega[col]);
                const float2 *tv = tq + x * LQ_TP;
                float er = 0.f, ei = 0.f;
                for (int y0 = 0; y0 < nm; y0 += 12) {  // the row of u_ph, its loads in flight together
                    float4 p[6];
#pragma unroll
                    for (int y = 0; y < 6; y++) {
                        const int k = y0 + 2 * y;
                        if (k >= nm) break;
                        if (nm & 1) {  // t of the mode past the last is zero
                            const float2 f = uv[k], g = uv[min(k + 1, nm - 1)];
                            p[y] = make_float4(f.x, f.y, g.x, g.y);
                        } else {
                            p[y] = *reinterpret_cast<const float4 *>(uv + k);
                        }
                    }
#pragma unroll
                    for (int y = 0; y < 6; y++) {
                        const int k = y0 + 2 * y;
                        if (k >= nm) break;
                        const float4 q = *reinterpret_cast<const float4 *>(tv + k);
                        st_cmac(er, ei, q.x, q.y, p[y].x, p[y].y);
                        st_cmac(er, ei, q.z, q.w, p[y].z, p[y].w);
                    }
                }
                const int64_t oi = ((row0 + kk) * a.nbw + (s >> 16)) * nm + n2;
                a.g2[oi] = (er * er + ei * ei) / w2;
                if (a.ep) a.ep[oi] = make_float2(er, ei);
            }
        }
        for (int m = 0; m < a.nbw; m++)  // zeros past the k+q window
            for (int e = t; e < (kz - ka) * nm; e += bd) {
                const int x = sq_div(e, a.mg_nm), n2 = e - x * nm;
                if (m < (smeta[ka + x] & 0xff)) continue;
                const int64_t oi = ((row0 + ka + x) * a.nbw + m) * nm + n2;
                a.g2[oi] = 0.f;
                if (a.ep) a.ep[oi] = make_float2(0.f, 0.f);
            }
    }
}

// e^{2 pi i (x / m) (pmin + b)} for x < m, b < n (zero for n <= b < ne)
__global__ void staged_phases_kernel(int m, int n, int ne, int pmin, float2 *__restrict__ out) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= m * ne) return;
    float c = 0.f, s = 0.f;
    if (e % ne < n) cis2pi((double)(e / ne) / m * (double)(pmin + e % ne), c, s);
    out[e] = make_float2(c, s);
}

}  // namespace ephip

using namespace ephip;

extern "C" int ephip_staged_phases(int32_t m, int32_t n, int32_t ne, int32_t pmin, void *out, void *stream) {
    EPHIP_REQUIRE(m >= 1 && n >= 1 && ne >= n && (int64_t)m * ne < ((int64_t)1 << 31), "staged_phases: bad sizes");
    EPHIP_REQUIRE(out, "staged_phases: null device pointer");
    staged_phases_kernel<<<(unsigned)(((int64_t)m * ne + 255) / 256), 256, 0, as_stream(stream)>>>(
        m, n, ne, pmin, static_cast<float2 *>(out));
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_staged_project(int32_t nw, int64_t ngcol, int32_t np, int32_t r2min, int32_t nplanes,
                                    const void *const *op1, const int32_t *l0, const int32_t *l1, int64_t k0,
                                    int64_t k1, int32_t lb0, const int32_t *line_start, int32_t max_line_units,
                                    const int32_t *kus, const int32_t *ukpos, const void *ucol, const void *ph2,
                                    const void *ph3, void *A, int64_t lda, void *stream) {
    EPHIP_REQUIRE(nw >= 1 && nw <= 32, "staged_project: nw=%d outside 1..32", nw);
    EPHIP_REQUIRE(np >= 3 && np <= 8, "staged_project: padded box face np x np with 3 <= np <= 8 (got %d)", np);
    EPHIP_REQUIRE(nplanes >= 1 && nplanes <= SP_PLANES, "staged_project: %d planes (1..%d)", nplanes, SP_PLANES);
    EPHIP_REQUIRE(ngcol >= 0 && ngcol % nw == 0 && k0 >= 0 && k1 >= k0 && lb0 >= 0 && lda >= ngcol,
                  "staged_project: bad sizes (columns a multiple of nw, lda >= columns)");
    EPHIP_REQUIRE(max_line_units >= 1 && max_line_units <= SP_PAIRS,
                  "staged_project: lines (or line pieces) of at most %d k and %d units (got %d units)", SP_KLINE,
                  SP_PAIRS, max_line_units);
    if (ngcol == 0 || k1 == k0) return EPHIP_OK;
    EPHIP_REQUIRE(op1 && l0 && l1 && line_start && kus && ukpos && ucol && ph2 && ph3 && A,
                  "staged_project: null pointer");
    SpPlanes pl{};
    int lines = 0;
    for (int p = 0; p < nplanes; p++) {
        EPHIP_REQUIRE(op1[p] && l0[p] >= lb0 && l1[p] >= l0[p], "staged_project: bad plane %d", p);
        pl.op1[p] = static_cast<const cplx<float> *>(op1[p]);
        pl.l0[p] = l0[p];
        pl.l1[p] = l1[p];
        lines = max(lines, l1[p] - l0[p]);
    }
    if (lines == 0) return EPHIP_OK;
    const int64_t gx = (ngcol + 15) / 16;
    EPHIP_REQUIRE(gx <= 0x7fffffffLL, "staged_project: too many columns");
    const int nwave = (nw + 3) / 4;
    // parts of a plane's lines: enough workgroups for about 16 waves per CU, at least two lines each
    int64_t z = (4096 + gx * nplanes * nwave - 1) / (gx * nplanes * nwave);
    z = max((int64_t)1, min(z, (int64_t)(lines + 1) / 2));
    using K = decltype(&staged_project_kernel<3, false>);
    static const K kern[6] = {staged_project_kernel<3, false>, staged_project_kernel<4, false>,
                              staged_project_kernel<5, false>, staged_project_kernel<6, false>,
                              staged_project_kernel<7, false>, staged_project_kernel<8, false>};
    static const K kern_sym[3] = {staged_project_kernel<3, true>, staged_project_kernel<5, true>,
                                  staged_project_kernel<7, true>};
    const bool sym = (np & 1) && r2min == -(np / 2);
    const K k = sym ? kern_sym[(np - 3) / 2] : kern[np - 3];
    const int max_pairs = (max_line_units + 1) & ~1;  // even: the partial tiles stay 16-byte aligned
    const size_t lds = sp_lds_bytes(np, nwave, max_pairs);
    if (lds > 64 * 1024)
        EPHIP_TRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    k<<<dim3((unsigned)gx, (unsigned)nplanes, (unsigned)z), 64 * nwave, lds, as_stream(stream)>>>(
        nw, ngcol, pl, k0, k1, lb0, line_start, kus, ukpos, static_cast<const cplx<float> *>(ucol),
        static_cast<const cplx<float> *>(ph2), static_cast<const cplx<float> *>(ph3), max_pairs,
        static_cast<cplx<float> *>(A), lda);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

// Form by the mean window width w (bands per kept q): two kept q per thread while most windows hold one band
// (a band's g is then formed for itself), else one kept q with up to 2 or 4 of its bands, which share g.
struct SqForm {
    int nq, nb;      // kept q of a thread, bands of each
    double entries;  // expected entries of one (unit, q1) slab
};
static SqForm sq_form(int nw, double cols, double width) {
    if (width < 1.4) return SqForm{2, 1, cols * width};
    if (width < 1.9 || nw > 16) return SqForm{1, 2, cols * (0.5 + 0.5 * width)};
    return SqForm{1, 4, cols * (width < 3.0 ? 1.05 : 0.3 + 0.25 * width)};
}

// The workgroup: a.tb, a.nug, a.ls and a.split; false if none fits.
template <int N>
static bool sq_choose(SqArgs &a, const SqForm f) {
    const size_t cu_lds = 160 * 1024, most = 152 * 1024;
    // threads of a group: NQ entries each; room for the entries and lines of most slabs (a slab past it takes a
    // second segment, which repeats stages 1 and 2)
    const double want = fmin(1024.0, (1.15 * f.entries + (f.nq > 1 ? a.m2 : 0.0)) / f.nq);
    // never fewer than the entries of one kept q with nbw bands take, and its line (17 threads of two for 32 bands)
    const int tb_min = max(16, ((a.nbw + f.nb - 1) / f.nb + (f.nq > 1) + f.nq - 1) / f.nq);
    const int tb_want = max((tb_min + 7) & ~7, min(128, (int)(want / 8 + 1) * 8));
    // (group size, mode groups): a workgroup is a chain of latencies, about a quarter of it per pass over nug modes,
    // so the number of workgroups a CU holds (LDS; registers: U takes 2 NQ NB nw of them) over that length counts.
    // Measured, ms per pass: 4 orbitals, 3 modes, 7^3 boxes, q 24^3: 1.38 at 6 workgroups and 3 passes, 1.77 at 4 and
    // 1 pass; 12 orbitals, 9 modes, 5^3: 2.38, 1.96, 1.90, 2.2 at 6, 4, 3, 2 workgroups and 9, 5, 3, 2 passes;
    // 16 orbitals, 12 modes, 5 window bands: 13.8, 11.8, 17.1 at 2, 2, 1 workgroups and 6, 4, 3 passes.
    double best = -1.0;
    SqArgs c = a;
    const int nwt = a.nw <= 4 ? 4 : a.nw <= 8 ? 8 : a.nw <= 12 ? 12 : a.nw <= 16 ? 16 : 32;
    const int simd_waves = max(1, min(4, 512 / (2 * f.nq * f.nb * nwt + 72)));
    for (int tb = tb_want; tb >= tb_min; tb -= 16)
        for (int nug = 1; nug <= min(a.nm, 512 / tb); nug++) {
            a.tb = tb;
            a.nug = nug;
            a.ls = min(a.m2, SQ_LINES);
            while (sq_lds_bytes<N>(a, f.nq, f.nb) > cu_lds / 2 && a.ls > 8) a.ls--;
            while (sq_lds_bytes<N>(a, f.nq, f.nb) > most && a.ls > 1) a.ls--;
            const size_t lds = sq_lds_bytes<N>(a, f.nq, f.nb);
            if (lds > most || N * N * nug * a.nw >= 65536) continue;
            const int rounds = (a.nm + nug - 1) / nug, waves = (tb * nug + 63) / 64;
            const int blocks = min((int)(cu_lds / lds), simd_waves / ((waves + 3) / 4) * (waves < 4 ? 4 / waves : 1));
            const double s = blocks / (1.0 + 0.25 * rounds) * tb / tb_want * (waves == 1 ? 0.8 : 1.0);
            if (s > best) best = s, c = a;
        }
    if (best <= 0.0) return false;
    a = c;
    const int bd = (a.tb * a.nug + 63) & ~63, rows = a.nug * a.nw;
    // stage 2: (row, c) items split over the lines so that the threads have equal shares
    a.split = 1;
    best = 0.0;
    for (int s = 1; s <= 8; s++) {
        const int items = N * rows * s, rounds = (items + bd - 1) / bd;
        const double use = (double)items / ((double)rounds * bd) / (1.0 + 0.05 * s);
        if (use > best && items < 65536) {
            best = use;
            a.split = s;
        }
    }
    return true;
}

template <int N, bool SYM, int NQ, int NB>
static int staged_kq_launch_form(SqArgs a, int nunits, const SqForm f, hipStream_t st) {
    EPHIP_REQUIRE(sq_choose<N>(a, f), "staged_kq: nw=%d nm=%d nbw=%d do not fit a workgroup", a.nw, a.nm, a.nbw);
    const int bd = (a.tb * a.nug + 63) & ~63, rows = a.nug * a.nw;
    a.mg_rows = sq_magic(rows);
    a.mg_rn = sq_magic(N * rows);
    a.mg_nm = sq_magic(a.nm);
    a.mg_nm2 = sq_magic(a.nm * a.nm);
    const size_t lds = sq_lds_bytes<N>(a, NQ, NB);
    using K = decltype(&staged_kq_kernel<N, SYM, 4, NQ, NB>);
    const K k = a.nw <= 4 ? staged_kq_kernel<N, SYM, 4, NQ, NB> : a.nw <= 8 ? staged_kq_kernel<N, SYM, 8, NQ, NB>
              : a.nw <= 12 ? staged_kq_kernel<N, SYM, 12, NQ, NB> : a.nw <= 16 ? staged_kq_kernel<N, SYM, 16, NQ, NB>
                                                                               : staged_kq_kernel<N, SYM, 32, NQ, NB>;
    if (lds > 64 * 1024)
        EPHIP_TRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    k<<<dim3((unsigned)a.m1, (unsigned)nunits), bd, lds, st>>>(a);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

template <int N>
static int lane_kq_launch(SqArgs a, int nunits, hipStream_t st) {
    a.mg_nm = sq_magic(a.nm);
    lane_kq_kernel<N, 16><<<dim3((unsigned)a.m1, (unsigned)nunits), 64 * ((a.nm + 3) / 4), lq_lds_bytes(a, 16), st>>>(a);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

template <int N, bool SYM>
static int staged_kq_launch(const SqArgs &a, int nunits, double cols, double width, hipStream_t st) {
    const SqForm f = sq_form(a.nw, cols, width);
    if (f.nq == 2) return staged_kq_launch_form<N, SYM, 2, 1>(a, nunits, f, st);
    if (f.nb == 2) return staged_kq_launch_form<N, SYM, 1, 2>(a, nunits, f, st);
    return staged_kq_launch_form<N, SYM, 1, 4>(a, nunits, f, st);
}

extern "C" int ephip_staged_kq_group(int32_t nw, int32_t nm, int32_t nbw, int32_t np, int32_t m2, int32_t m3,
                                     double cols_hint, double width_hint, int32_t *group) {
    EPHIP_REQUIRE(nw >= 1 && nw <= 32 && nm >= 1 && nm <= 48 && nbw >= 1 && nbw <= nw && np >= 3 && np <= 8 && m2 >= 1 &&
                      m2 <= SQ_LINES && m3 >= 1 && m3 <= 64 && group,
                  "staged_kq_group: bad sizes");
    SqArgs a{};
    a.nw = nw, a.nm = nm, a.nbw = nbw, a.m2 = m2, a.m3 = m3;
    const SqForm f = sq_form(nw, cols_hint, width_hint);
    const bool ok = np == 3   ? sq_choose<3>(a, f)
                    : np == 4 ? sq_choose<4>(a, f)
                    : np == 5 ? sq_choose<5>(a, f)
                    : np == 6 ? sq_choose<6>(a, f)
                    : np == 7 ? sq_choose<7>(a, f)
                              : sq_choose<8>(a, f);
    EPHIP_REQUIRE(ok, "staged_kq: nw=%d nm=%d nbw=%d do not fit a workgroup", nw, nm, nbw);
    const int g[5] = {f.nq, f.nb, a.tb, a.nug, a.ls};
    for (int i = 0; i < 5; i++) group[i] = g[i];
    return EPHIP_OK;
}

extern "C" int ephip_staged_kq(int32_t nw, int32_t nm, int32_t nbw, int32_t nunits, int32_t n1, int32_t np,
                               int32_t p1min, int32_t p2min, int32_t p3min, const int32_t *rmap, const int32_t *qgrid,
                               const void *e1, const void *e2, const void *e3, const void *A, int64_t lda, int64_t ldr, const int32_t *line_off,
                               const int32_t *col_index, const int32_t *ikq, int64_t cs, const void *U,
                               const int64_t *bmin, const int64_t *bmax, const void *uph, const double *omega,
                               const int32_t *dense_strides, double cols_hint, double width_hint, float *g2, void *ep,
                               void *stream) {
    EPHIP_REQUIRE(nw >= 1 && nw <= 32 && nm >= 1 && nm <= 48, "staged_kq: nw=%d (1..32), nm=%d (1..48)", nw, nm);
    EPHIP_REQUIRE(nbw >= 1 && nbw <= nw, "staged_kq: nbw=%d outside 1..nw", nbw);
    EPHIP_REQUIRE(n1 >= 1 && n1 <= 32 && np >= 3 && np <= 8, "staged_kq: Rp box n1=%d (<= 32), np=%d (3..8)", n1, np);
    EPHIP_REQUIRE(qgrid && qgrid[0] >= 1 && qgrid[1] >= 1 && qgrid[2] >= 1 && qgrid[0] <= 65535 &&
                      qgrid[1] <= SQ_LINES && qgrid[2] <= 64,
                  "staged_kq: q grid n1 n2 n3 with n1 <= 65535 and n2, n3 <= 64");
    EPHIP_REQUIRE(nunits >= 0 && nunits <= 65535 && ldr >= (int64_t)nw * nm && lda >= ldr &&
                      lda < ((int64_t)1 << 31) && cs >= 0,
                  "staged_kq: bad sizes");
    if (nunits == 0) return EPHIP_OK;
    EPHIP_REQUIRE(rmap && e1 && e2 && e3 && A && line_off && col_index && ikq && U && bmin && bmax && uph && omega && g2,
                  "staged_kq: null device pointer");
    SqArgs a{};
    a.nw = nw, a.nm = nm, a.nbw = nbw, a.n1 = n1;
    a.dense = dense_strides != nullptr && n1 == np;
    if (a.dense) {
        a.s1 = dense_strides[0], a.s2 = dense_strides[1], a.s3 = dense_strides[2];
        EPHIP_REQUIRE(a.s1 >= 0 && a.s2 >= 0 && a.s3 >= 0 &&
                          (int64_t)(a.s1 + (int64_t)a.s2 + a.s3) * (np - 1) < ((int64_t)1 << 31),
                      "staged_kq: bad dense-box strides");
    }
    a.m1 = qgrid[0], a.m2 = qgrid[1], a.m3 = qgrid[2];
    a.e1 = static_cast<const float2 *>(e1), a.e2 = static_cast<const float2 *>(e2);
    a.e3 = static_cast<const float2 *>(e3);
    a.rmap = rmap, a.A = static_cast<const cplx<float> *>(A), a.lda = lda, a.ldr = (int)ldr;
    a.line_off = line_off, a.col_index = col_index, a.ikq = ikq, a.cs = cs;
    a.U = static_cast<const cplx<float> *>(U), a.bmin = bmin, a.bmax = bmax;
    a.uph = static_cast<const cplx<float> *>(uph), a.omega = omega, a.g2 = g2, a.ep = static_cast<float2 *>(ep);
    const bool sym = (np & 1) && n1 == np && p1min == -(np / 2) && p2min == -(np / 2) && p3min == -(np / 2);
    hipStream_t st = as_stream(stream);
    // One lane per (mode, i): from 9 modes on, where a workgroup has three waves or four. With one or two the tables of a
    // slab, read in turn, take too long: whole passes of 9 orbitals, 3 modes 0.52 -> 0.83 ms, 10, 6 (7^3 boxes) 1.33 ->
    // 1.35; and at 8 lanes per mode 8, 6 84 -> 91 us. Slabs whose tables pass LQ_SLAB words (16 KB) would leave two
    // workgroups a CU.
    if (sym && nw > 8 && nw <= 16 && nm > 8 && nm <= 16 && (4 + nbw) * a.m2 * a.m3 <= LQ_SLAB) {
        if (np == 3) return lane_kq_launch<3>(a, nunits, st);
        if (np == 5) return lane_kq_launch<5>(a, nunits, st);
        return lane_kq_launch<7>(a, nunits, st);
    }
    if (sym) {
        if (np == 3) return staged_kq_launch<3, true>(a, nunits, cols_hint, width_hint, st);
        if (np == 5) return staged_kq_launch<5, true>(a, nunits, cols_hint, width_hint, st);
        return staged_kq_launch<7, true>(a, nunits, cols_hint, width_hint, st);
    }
    switch (np) {
        case 3: return staged_kq_launch<3, false>(a, nunits, cols_hint, width_hint, st);
        case 4: return staged_kq_launch<4, false>(a, nunits, cols_hint, width_hint, st);
        case 5: return staged_kq_launch<5, false>(a, nunits, cols_hint, width_hint, st);
        case 6: return staged_kq_launch<6, false>(a, nunits, cols_hint, width_hint, st);
        case 7: return staged_kq_launch<7, false>(a, nunits, cols_hint, width_hint, st);
        default: return staged_kq_launch<8, false>(a, nunits, cols_hint, width_hint, st);
    }
}
