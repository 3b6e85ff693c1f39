// Boltzmann transport on the outer-k payload (FP64): scattering increments, the scattering-out rates
// and scattering-in matrix, band velocities, and the sparse product of the iterative solver.
//
// bte_scattering_increments restates src/boltzmann/bte_scattering_core.jl:33-84 (occupation
// conventions 1..6, vanishing-delta guards) with the smeared delta of src/common/smearing.jl;
// the accumulation follows the device kernel ext/ElectronPhononCUDAExt.jl:323-372 /
// bte_window_accumulate! (src/boltzmann/boltzmann_calculator.jl:336-372): atomic S_out, plain S_in.
// S_in is stored in the outer-k loop's own sparse layout: row (unit u, kept column c, k+q band slot m).
#include <algorithm>

#include "common.hpp"

namespace ephip {

__device__ __forceinline__ double occ_fd(double e, double T) { return 1.0 / (exp(e / T) + 1.0); }
__device__ __forceinline__ double occ_fd_deriv(double e, double T) {
    return -1.0 / (2.0 + exp(e / T) + exp(-e / T)) / T;
}
__device__ __forceinline__ double occ_boson(double e, double T) { return e == 0.0 ? 0.0 : 1.0 / expm1(e / T); }
__device__ __forceinline__ double smear(int method, double eta, double x) {
    if (method == 1) return (1.0 / sqrt(M_PI)) / eta * exp(-(x / eta) * (x / eta));
    return (eta / M_PI) / (x * x + eta * eta);
}

__device__ void bte_increments(int method, double ek, double ekq, double wq, double g2, double wtq, double mu,
                               double T, int smearing, double eta, double &so, double &si) {
    const double d1 = smear(smearing, eta, ek - ekq + wq);
    const double d2 = smear(smearing, eta, ek - ekq - wq);
    so = 0.0;
    si = 0.0;
    if (d1 == 0.0 && d2 == 0.0) return;
    const double nq = occ_boson(wq, T), fk = occ_fd(ek - mu, T), fkq = occ_fd(ekq - mu, T);
    double f1o, f2o, f1i, f2i;
    if (method == 1) {
        f1o = nq + fkq; f2o = nq + 1 - fkq;
        f1i = nq + fk;  f2i = nq + 1 - fk;
    } else if (method == 2) {
        const double preo = fkq * (1 - fkq) / (fk * (1 - fk));
        f1o = preo * (nq + 1 - fk); f2o = preo * (nq + fk);
        const double prei = fk * (1 - fk) / (fkq * (1 - fkq));
        f1i = prei * (nq + 1 - fkq); f2i = prei * (nq + fkq);
    } else if (method == 3) {
        const double preo = (1 - fkq) / (1 - fk);
        f1o = preo * nq; f2o = preo * (nq + 1);
        const double prei = (1 - fk) / (1 - fkq);
        f1i = prei * nq; f2i = prei * (nq + 1);
    } else if (method == 4) {
        const double preo = fkq / fk;
        f1o = preo * (nq + 1); f2o = preo * nq;
        const double prei = fk / fkq;
        f1i = prei * (nq + 1); f2i = prei * nq;
    } else if (method == 5) {
        const double dk = occ_fd_deriv(ek - mu, T), dkq = occ_fd_deriv(ekq - mu, T);
        f1o = sqrt(nq * (nq + 1) * dkq / dk); f2o = f1o;
        f1i = sqrt(nq * (nq + 1) * dk / dkq); f2i = f1i;
    } else {
        const double no = occ_boson(ekq - ek, T);
        f1o = no + fkq; f2o = -(no + fkq);
        const double ni = occ_boson(ek - ekq, T);
        f1i = ni + fk; f2i = -(ni + fk);
    }
    const double pref = 2.0 * M_PI * wtq * g2;
    so = ((d1 == 0.0 ? 0.0 : d1 * f1o) + (d2 == 0.0 ? 0.0 : d2 * f2o)) * pref;
    si = ((d2 == 0.0 ? 0.0 : d2 * f1i) + (d1 == 0.0 ? 0.0 : d1 * f2i)) * pref;
}

// in: (n x 8) rows {ek, ekq, wq, g2, wtq, mu, T, eta}; out: (n x 2) {s_out, s_in}
__global__ void bte_increments_kernel(int64_t n, int method, int smearing, const double *__restrict__ in,
                                      double *__restrict__ out) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const double *r = in + 8 * e;
    double so, si;
    bte_increments(method, r[0], r[1], r[2], r[3], r[4], r[5], r[6], smearing, r[7], so, si);
    out[2 * e] = so;
    out[2 * e + 1] = si;
}

// One thread per (unit u, kept column c, k+q slot m). i = unit_state_index[u] (initial state);
// f = state_offset[ikq] + m (final state); energies e_state[i], e_state[f]; modes below w_cut skipped.
// S_out[i + nstates*iT] += sum_nu s_out (atomic). S_in is compacted: the unit's kept columns are
// rows rowptr[u] .. rowptr[u] + count[u] - 1, S_in[(row*nbw + m)*nT + iT] = sum_nu s_in, and
// row_code[row] = first final state | (number of k+q window slots << 27) of the row.
__global__ void bte_accumulate_kernel(int nunits, int64_t cs, int nbw, int nm, const int *__restrict__ count,
                                      const int *__restrict__ col_index, const int *__restrict__ ikq,
                                      const float *__restrict__ g2, const int64_t *__restrict__ unit_state_index,
                                      const int64_t *__restrict__ state_offset, const int64_t *__restrict__ bmin,
                                      const int64_t *__restrict__ bmax, const double *__restrict__ e_state,
                                      const double *__restrict__ omega, double wtq, int nT,
                                      const double *__restrict__ mus, const double *__restrict__ Ts,
                                      const double *__restrict__ etas, int method, int smearing, double w_cut,
                                      int64_t nstates, const int64_t *__restrict__ rowptr, double *__restrict__ S_out,
                                      double *__restrict__ S_in, uint32_t *__restrict__ row_code) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int u = blockIdx.y;
    if (u >= nunits || e >= cs * nbw) return;
    const int64_t c = e / nbw;
    const int m = (int)(e % nbw);
    if (c >= count[u]) return;
    const int64_t row = (int64_t)u * cs + c;      // payload row
    const int64_t orow = rowptr[u] + c;           // compacted output row
    const int64_t kq = ikq[row];
    const int nbkq = bmin[kq] > 0 ? min((int)(bmax[kq] - bmin[kq] + 1), nbw) : 0;
    if (m == 0) row_code[orow] = (uint32_t)state_offset[kq] | ((uint32_t)nbkq << 27);
    double *sin_row = S_in + (orow * nbw + m) * nT;
    if (m >= nbkq) {
        for (int t = 0; t < nT; t++) sin_row[t] = 0.0;
        return;
    }
    const int64_t i = unit_state_index[u];
    const int64_t f = state_offset[kq] + m;
    const double ek = e_state[i], ekq = e_state[f];
    const int iq = col_index[row];
    const float *gr = g2 + row * nbw * nm + (int64_t)m * nm;
    for (int t = 0; t < nT; t++) {
        double so = 0.0, si = 0.0;
        for (int nu = 0; nu < nm; nu++) {
            const double w = omega[(int64_t)nm * iq + nu];
            if (w < w_cut) continue;
            double a, b;
            bte_increments(method, ek, ekq, w, (double)gr[nu], wtq, mus[t], Ts[t], smearing, etas[t], a, b);
            so += a;
            si += b;
        }
        atomicAdd(&S_out[i + nstates * t], so);
        sin_row[t] = si;
    }
}

// ---------------------------------------------------------------------------------------------
// The same sums with everything that does not depend on the (state, mode) pair taken out of the inner loop:
//   tab_q: phonon frequency and, per temperature, occupation of every (mode, q), q fastest (lanes hold
//          neighbouring q): omega[nu][q], then n (method 5: sqrt(n (n + 1))) [t][nu][q];
//   tab_s: per temperature and state, the Fermi function (method 5: its energy derivative) [t][state].
// What is left per (state pair, mode) is the two smeared deltas, shared by temperatures of one width, and a few
// multiplications: 2 FP64 exponentials where the per-term form takes 10 per temperature. S_out is summed over the
// wave before its atomic (where every (kept q, band) of a unit added to the same address).
// ---------------------------------------------------------------------------------------------
__global__ void bte_tables_kernel(int nq, int nm, const double *__restrict__ omega, int64_t nstates,
                                  const double *__restrict__ e_state, int nT, const double *__restrict__ mus,
                                  const double *__restrict__ Ts, int method, double *__restrict__ tab_q,
                                  double *__restrict__ tab_s) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, nmq = (int64_t)nm * nq;
    if (e < nmq) {
        const int64_t nu = e / nq, q = e % nq;
        const double w = omega[nm * q + nu];
        tab_q[e] = w;
        for (int t = 0; t < nT; t++) {
            const double n = occ_boson(w, Ts[t]);
            tab_q[(1 + t) * nmq + e] = method == 5 ? sqrt(n * (n + 1)) : n;
        }
    } else if (e < nmq + nT * nstates) {
        const int64_t f = e - nmq, t = f / nstates, i = f % nstates;
        const double x = e_state[i] - mus[t];
        tab_s[f] = method == 5 ? occ_fd_deriv(x, Ts[t]) : occ_fd(x, Ts[t]);
    }
}

// Factors of the increments that the modes of one (initial, final) state pair share, at one temperature.
template <int METHOD>
struct BtePair {
    double a, b, c, d;
    __device__ void set(double si, double sf, double ek, double ekq, double T) {
        if constexpr (METHOD == 1) {
            a = si;
            b = sf;
        } else if constexpr (METHOD == 2) {
            const double gi = si * (1 - si), gf = sf * (1 - sf);
            a = si;
            b = sf;
            c = gf / gi;
            d = gi / gf;
        } else if constexpr (METHOD == 3) {
            c = (1 - sf) / (1 - si);
            d = (1 - si) / (1 - sf);
        } else if constexpr (METHOD == 4) {
            c = sf / si;
            d = si / sf;
        } else if constexpr (METHOD == 5) {
            c = sqrt(sf / si);
            d = sqrt(si / sf);
        } else {
            c = occ_boson(ekq - ek, T) + sf;
            d = occ_boson(ek - ekq, T) + si;
        }
    }
    // n: the mode's occupation factor; so = d1 f1o + d2 f2o, si = d2 f1i + d1 f2i (vanishing deltas left out, and g2 where
    // both vanish, whatever the factors and g2 are)
    __device__ void add(double n, double d1, double d2, double pref, double &so, double &si) const {
        double f1o, f2o, f1i, f2i;
        if constexpr (METHOD == 1) {
            f1o = n + b, f2o = n + 1 - b, f1i = n + a, f2i = n + 1 - a;
        } else if constexpr (METHOD == 2) {
            f1o = c * (n + 1 - a), f2o = c * (n + a), f1i = d * (n + 1 - b), f2i = d * (n + b);
        } else if constexpr (METHOD == 3) {
            f1o = c * n, f2o = c * (n + 1), f1i = d * n, f2i = d * (n + 1);
        } else if constexpr (METHOD == 4) {
            f1o = c * (n + 1), f2o = c * n, f1i = d * (n + 1), f2i = d * n;
        } else if constexpr (METHOD == 5) {
            f1o = f2o = n * c, f1i = f2i = n * d;
        } else {
            f1o = c, f2o = -c, f1i = d, f2i = -d;
        }
        const double pg = d1 == 0.0 && d2 == 0.0 ? 0.0 : pref;
        so += ((d1 == 0.0 ? 0.0 : d1 * f1o) + (d2 == 0.0 ? 0.0 : d2 * f2o)) * pg;
        si += ((d2 == 0.0 ? 0.0 : d2 * f1i) + (d1 == 0.0 ? 0.0 : d1 * f2i)) * pg;
    }
};

// The kept (q, window band) pairs of 256 columns are listed in LDS, so that lanes hold pairs: taken column by column
// the few second bands cost every wave that has one a whole pass (measured 1.33 against 0.80 ms, 3.07M rows of 12
// modes at 3 temperatures, and 0.38 since the units come first in the grid; the per-term form took 7.65 ms). Bound by the
// FP64 exponentials.
template <int METHOD, int NT>  // NT temperatures per pass
__global__ __launch_bounds__(256) void bte_accumulate_tab_kernel(
    int nunits, int64_t cs, int nbw, int nm, int nq, const int *__restrict__ count, const int *__restrict__ col_index,
    const int *__restrict__ ikq, const float *__restrict__ g2, const int64_t *__restrict__ unit_state_index,
    const int64_t *__restrict__ state_offset, const int64_t *__restrict__ bmin, const int64_t *__restrict__ bmax,
    const double *__restrict__ e_state, const double *__restrict__ tab_q, const double *__restrict__ tab_s, double wtq,
    int nT, const double *__restrict__ Ts, const double *__restrict__ etas, int smearing, double w_cut,
    int64_t nstates, const int64_t *__restrict__ rowptr, double *__restrict__ S_out, double *__restrict__ S_in,
    uint32_t *__restrict__ row_code, int quad) {
    __shared__ int ciq[256], cf0[256], wsum[4];
    extern __shared__ uint16_t list[];  // [256 nbw] column | band << 8
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t c0 = units_first_tile() * 256;
    const int u = blockIdx.x, cnt = count[u];
    if (c0 >= cnt) return;  // uniform
    const int64_t i = unit_state_index[u], row0 = (int64_t)u * cs + c0, orow0 = rowptr[u] + c0;
    int nb = 0;
    if (c0 + t < cnt) {
        const int64_t kq = ikq[row0 + t];
        nb = bmin[kq] > 0 ? min((int)(bmax[kq] - bmin[kq] + 1), nbw) : 0;
        ciq[t] = col_index[row0 + t];
        cf0[t] = (int)state_offset[kq];
        row_code[orow0 + t] = (uint32_t)cf0[t] | ((uint32_t)nb << 27);
        for (int m = nb; m < nbw; m++)
            for (int x = 0; x < nT; x++) S_in[((orow0 + t) * nbw + m) * nT + x] = 0.0;
    }
    int pre = nb;  // inclusive prefix
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(pre, off, 64);
        if (lane >= off) pre += o;
    }
    if (lane == 63) wsum[wave] = pre;
    __syncthreads();
    int npair = 0;
    for (int w = 0; w < 4; w++) {
        if (w == wave) pre += npair;
        npair += wsum[w];
    }
    for (int m = 0; m < nb; m++) list[pre - nb + m] = (uint16_t)(t | (m << 8));
    __syncthreads();
    const double ek = e_state[i], pre2 = 2.0 * M_PI * wtq;
    const int64_t nmq = (int64_t)nm * nq;
    for (int t0 = 0; t0 < nT; t0 += NT) {
        double tot[NT];
        double eta[NT], ie[NT], nrm[NT];  // width, its inverse, prefactor of the delta
#pragma unroll
        for (int x = 0; x < NT; x++) {
            tot[x] = 0.0;
            eta[x] = etas[min(t0 + x, nT - 1)];
            ie[x] = 1.0 / eta[x];
            nrm[x] = smearing == 1 ? (1.0 / sqrt(M_PI)) / eta[x] : eta[x] / M_PI;
        }
        for (int e = t; e < npair; e += 256) {
            const int col = list[e] & 255, m = list[e] >> 8, iq = ciq[col];
            const int64_t f = cf0[col] + m;
            const double ekq = e_state[f], x0 = ek - ekq;
            double so[NT], si[NT];
            BtePair<METHOD> pr[NT];
#pragma unroll
            for (int x = 0; x < NT; x++) {
                const int tt = min(t0 + x, nT - 1);
                so[x] = si[x] = 0.0;
                pr[x].set(tab_s[tt * nstates + i], tab_s[tt * nstates + f], ek, ekq, Ts[tt]);
            }
            const float *gr = g2 + ((row0 + col) * nbw + m) * nm;
            for (int nu0 = 0; nu0 < nm; nu0 += 4) {  // four modes' loads in flight together
                double w[4], n[4][NT];
                float g[4];
                if (quad) {  // nm a multiple of 4 and g2 16-byte aligned
                    const float4 v = *reinterpret_cast<const float4 *>(gr + nu0);
                    g[0] = v.x, g[1] = v.y, g[2] = v.z, g[3] = v.w;
                } else {
#pragma unroll
                    for (int y = 0; y < 4; y++) g[y] = gr[min(nu0 + y, nm - 1)];
                }
#pragma unroll
                for (int y = 0; y < 4; y++) {
                    const int64_t at = (int64_t)min(nu0 + y, nm - 1) * nq + iq;
                    w[y] = tab_q[at];
#pragma unroll
                    for (int x = 0; x < NT; x++) n[y][x] = tab_q[(1 + min(t0 + x, nT - 1)) * nmq + at];
                }
#pragma unroll
                for (int y = 0; y < 4; y++) {
                    const bool in = nu0 + y < nm && !(w[y] < w_cut);  // else both deltas zero: nothing added
                    const double pref = pre2 * (double)g[y];
                    double d1 = 0.0, d2 = 0.0;
#pragma unroll
                    for (int x = 0; x < NT; x++) {
                        if (x == 0 || eta[x] != eta[x - 1]) {  // uniform: one width for all temperatures as a rule
                            const double a = x0 + w[y], b = x0 - w[y];
                            if (smearing == 1) {
                                d1 = nrm[x] * exp(-(a * ie[x]) * (a * ie[x]));
                                d2 = nrm[x] * exp(-(b * ie[x]) * (b * ie[x]));
                            } else {
                                d1 = nrm[x] / (a * a + eta[x] * eta[x]);
                                d2 = nrm[x] / (b * b + eta[x] * eta[x]);
                            }
                            if (!in) d1 = d2 = 0.0;
                        }
                        pr[x].add(n[y][x], d1, d2, pref, so[x], si[x]);
                    }
                }
            }
#pragma unroll
            for (int x = 0; x < NT; x++)
                if (t0 + x < nT) {
                    S_in[((orow0 + col) * nbw + m) * nT + t0 + x] = si[x];
                    tot[x] += so[x];
                }
        }
#pragma unroll
        for (int x = 0; x < NT; x++)
            if (t0 + x < nT) {
                const double v = wave_sum(tot[x]);
                if (lane == 0) atomicAdd(&S_out[i + nstates * (t0 + x)], v);
            }
    }
}

// bte_window_accumulate! with the reference's arguments (ext/ElectronPhononCUDAExt.jl:323-372, generic
// src/boltzmann/boltzmann_calculator.jl:336-372): one thread per (m, n, j) of a q batch. i = imap_i[n]
// (outer state, 1-based, 0 = outside the window), f = imap_f[m + ld_f (ikqs[j] - 1)] (inner state); per
// temperature the increments of every mode with w >= w_cut are summed; S_out[(i - 1) + ld_so iT] gets an
// atomic add, S_in[(i - i0 - 1) + ld_si1 ((f - 1) + ld_si2 iT)] the plain write (each (i, f) hit once).
// g2vals (nbkq, nbk, nm, nq) and w (nm, nq) in R (float or double); everything else FP64 / int64.
template <typename R>
__global__ void bte_window_accumulate_kernel(double *__restrict__ S_out, int64_t ld_so, double *__restrict__ S_in,
                                             int64_t ld_si1, int64_t ld_si2, const R *__restrict__ g2vals,
                                             const R *__restrict__ wq, const int64_t *__restrict__ imap_i,
                                             const int64_t *__restrict__ imap_f, int64_t ld_f, int64_t nk_f,
                                             const int64_t *__restrict__ ikqs, const double *__restrict__ e_i,
                                             const double *__restrict__ e_f, const double *__restrict__ wf, int nT,
                                             const double *__restrict__ mus, const double *__restrict__ Ts,
                                             const double *__restrict__ etas, int method, int smearing, double w_cut,
                                             int nbkq, int nbk, int nm, int64_t nq, int64_t i0,
                                             uint32_t *__restrict__ dropped) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (int64_t)nbkq * nbk * nq) return;
    const int m = (int)(e % nbkq);
    const int n = (int)((e / nbkq) % nbk);
    const int64_t j = e / ((int64_t)nbkq * nbk);
    const int64_t i = imap_i[n];
    if (i <= 0) return;
    const int64_t kq = ikqs[j];
    if (kq < 1 || kq > nk_f || i - i0 < 1 || i - i0 > ld_si1) {
        if (dropped) atomicAdd(dropped, 1u);
        return;
    }
    const int64_t f = imap_f[m + ld_f * (kq - 1)];
    if (f <= 0) return;
    if (f > ld_si2) {
        if (dropped) atomicAdd(dropped, 1u);
        return;
    }
    const double ek = e_i[i - 1], ekq = e_f[f - 1], wtq = wf[f - 1];
    const R *gr = g2vals + m + (int64_t)nbkq * (n + (int64_t)nbk * nm * j);
    const int64_t nbb = (int64_t)nbkq * nbk;
    for (int t = 0; t < nT; t++) {
        double so = 0.0, si = 0.0;
        for (int nu = 0; nu < nm; nu++) {
            const double w = (double)wq[nu + (int64_t)nm * j];
            if (w < w_cut) continue;
            double a, b;
            bte_increments(method, ek, ekq, w, (double)gr[nbb * nu], wtq, mus[t], Ts[t], smearing, etas[t], a, b);
            so += a;
            si += b;
        }
        atomicAdd(&S_out[(i - 1) + ld_so * t], so);
        S_in[(i - i0 - 1) + ld_si1 * ((f - 1) + ld_si2 * t)] = si;
    }
}

// Diagonal band velocities: v[s][a] = Re(u^H dH_a u) for state s = (k = state_k[s], band = state_band[s]);
// dH: per state-k column, 3 operators of nw*nw (c64), column index state_col[s].
__global__ void band_velocity_kernel(int nw, int64_t nstates, const int64_t *__restrict__ state_col,
                                     const int *__restrict__ state_band, const int64_t *__restrict__ state_k,
                                     const double2 *__restrict__ dH, int64_t ld_dh,
                                     const float2 *__restrict__ U, double *__restrict__ v) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nstates * 3) return;
    const int64_t s = e / 3;
    const int a = (int)(e % 3);
    const double2 *M = dH + ld_dh * state_col[s] + (int64_t)a * nw * nw;
    const float2 *u = U + (int64_t)nw * nw * state_k[s] + (int64_t)nw * state_band[s];
    double acc = 0.0;
    for (int j = 0; j < nw; j++) {
        double wr = 0.0, wi = 0.0;
        for (int i = 0; i < nw; i++) {
            const double2 mij = M[i + (int64_t)nw * j];
            const float2 ui = u[i];
            // conj(u_i) M_ij
            wr += ui.x * mij.x + ui.y * mij.y;
            wi += ui.x * mij.y - ui.y * mij.x;
        }
        const float2 uj = u[j];
        acc += wr * uj.x - wi * uj.y;
    }
    v[3 * s + a] = acc;
}

// Full rotated operator of one (direction a, k) per workgroup, FP64 (U promoted from complex64):
// out[m + nw n] = (U_k^H M_a(k) U_k)[m, n], plus the Berry-connection term i (e_m - e_n) rbar[m, n] when the
// energies and rbar are given. U_k, M_a(k) and T = M_a U_k sit in LDS (nw <= 32: 3 x 16 KB); each thread
// forms whole entries of T, then of out, in the same order for every k.
constexpr int VEL_NW_MAX = 32;
__global__ void __launch_bounds__(256) el_velocity_full_kernel(int nw, const double2 *__restrict__ M, int64_t ld_m,
                                                               const float2 *__restrict__ U,
                                                               const double *__restrict__ E,
                                                               const double2 *__restrict__ rbar, int64_t ld_r,
                                                               double2 *__restrict__ out, int64_t ld_out) {
    __shared__ double2 us[VEL_NW_MAX * VEL_NW_MAX], ms[VEL_NW_MAX * VEL_NW_MAX], ts[VEL_NW_MAX * VEL_NW_MAX];
    const int a = (int)(blockIdx.x % 3);
    const int64_t k = blockIdx.x / 3;
    const int n2 = nw * nw;
    const double2 *mk = M + ld_m * k + (int64_t)a * n2;
    const float2 *uk = U + (int64_t)n2 * k;
    for (int e = threadIdx.x; e < n2; e += blockDim.x) {
        const float2 v = uk[e];
        us[e] = make_double2(v.x, v.y);
        ms[e] = mk[e];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < n2; e += blockDim.x) {  // T[i, n] = sum_j M[i, j] U[j, n]
        const int i = e % nw, n = e / nw;
        double re = 0.0, im = 0.0;
        for (int j = 0; j < nw; j++) {
            const double2 x = ms[i + nw * j], y = us[j + nw * n];
            re += x.x * y.x - x.y * y.y;
            im += x.x * y.y + x.y * y.x;
        }
        ts[e] = make_double2(re, im);
    }
    __syncthreads();
    double2 *ok = out + ld_out * k + (int64_t)a * n2;
    for (int e = threadIdx.x; e < n2; e += blockDim.x) {  // out[m, n] = sum_i conj(U[i, m]) T[i, n]
        const int m = e % nw, n = e / nw;
        double re = 0.0, im = 0.0;
        for (int i = 0; i < nw; i++) {
            const double2 x = us[i + nw * m], y = ts[i + nw * n];
            re += x.x * y.x + x.y * y.y;
            im += x.x * y.y - x.y * y.x;
        }
        if (rbar) {  // + i (e_m - e_n) rbar[m, n]
            const double de = E[(int64_t)nw * k + m] - E[(int64_t)nw * k + n];
            const double2 r = rbar[ld_r * k + (int64_t)a * n2 + e];
            re -= de * r.y;
            im += de * r.x;
        }
        ok[e] = make_double2(re, im);
    }
}

// y[i, :] = sum over the unit's rows and k+q slots S_in[row, m, iT] x[f, :] (3 components), one
// wavefront per unit (i = unit_state_index[u]); lanes take consecutive rows, f = first state of the
// row's code + m for m below the row's slot count.
__global__ void __launch_bounds__(256) bte_spmv_kernel(int nunits, int nbw, int nT, int iT,
                                                      const int64_t *__restrict__ rowptr,
                                                      const uint32_t *__restrict__ row_code,
                                                      const int64_t *__restrict__ unit_state_index,
                                                      const double *__restrict__ S_in,
                                                      const double *__restrict__ x, double *__restrict__ y) {
    const int lane = threadIdx.x & 63;
    const int u = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6);
    if (u >= nunits) return;  // whole wavefront exits together
    const int64_t r0 = rowptr[u], r1 = rowptr[u + 1];
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    for (int64_t row = r0 + lane; row < r1; row += 64) {
        const uint32_t code = row_code[row];
        const int f0 = (int)(code & 0x7ffffffu), nb = (int)(code >> 27);
        const double *sr = S_in + row * nbw * nT + iT;
        for (int m = 0; m < nb; m++) {
            const double sv = sr[(int64_t)m * nT];
            const double *xf = x + 3 * (int64_t)(f0 + m);
            a0 += sv * xf[0];
            a1 += sv * xf[1];
            a2 += sv * xf[2];
        }
    }
    a0 = wave_sum(a0);
    a1 = wave_sum(a1);
    a2 = wave_sum(a2);
    if (lane == 0) {
        double *yi = y + 3 * unit_state_index[u];
        yi[0] = a0;
        yi[1] = a1;
        yi[2] = a2;
    }
}

// One iteration's vector work: df <- mixing (y / inv_tau + rhs) + (1 - mixing) df (nothing if y is null), and the nine
// sums over states of df_a v_b, a block's in part[9 block ..]; then one block adds these, scales them and compares with
// the previous ones. Bound by the launches at the few thousand states of a window, by HBM at millions. It takes 100 us
// off an iteration of 2158 states: 15 launches, a 3 x 2158 x 3 matrix product of 64 us among them, and 2 copies before.
constexpr int BTE_STEP_BLOCKS = 256;

__device__ __forceinline__ void block_sum9(double (&a)[9], double (*red)[9]) {  // 4 waves; the sums end in red[0]
    for (int c = 0; c < 9; c++) {
        const double v = wave_sum(a[c]);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][c] = v;
    }
    __syncthreads();
    if (threadIdx.x < 9) red[0][threadIdx.x] += red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
    __syncthreads();
}

__global__ void __launch_bounds__(256) bte_step_kernel(int64_t n, const double *__restrict__ y,
                                                      const double *__restrict__ inv_tau,
                                                      const double *__restrict__ rhs, double mixing,
                                                      double *__restrict__ df, const double *__restrict__ vs,
                                                      double *__restrict__ part) {
    __shared__ double red[4][9];
    double a[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        double f[3];
        for (int c = 0; c < 3; c++) {
            f[c] = df[3 * i + c];
            if (y) {
                f[c] = (y[3 * i + c] / inv_tau[i] + rhs[3 * i + c]) * mixing + f[c] * (1.0 - mixing);
                df[3 * i + c] = f[c];
            }
        }
        for (int c = 0; c < 9; c++) a[c] += f[c / 3] * vs[3 * i + c % 3];
    }
    block_sum9(a, red);
    if (threadIdx.x < 9) part[9 * blockIdx.x + threadIdx.x] = red[0][threadIdx.x];
}

// out[0..8] = scale * sums, out[9] = |out - old| / |out| (Frobenius; 0 without old). old may not be out.
__global__ void __launch_bounds__(256) bte_step_sum_kernel(int nblocks, const double *__restrict__ part, double scale,
                                                          const double *__restrict__ old, double *__restrict__ out) {
    __shared__ double red[4][9];
    double a[9];
    for (int c = 0; c < 9; c++) a[c] = (int)threadIdx.x < nblocks ? part[9 * threadIdx.x + c] : 0.0;
    block_sum9(a, red);
    if (threadIdx.x != 0) return;
    double d2 = 0.0, s2 = 0.0;
    for (int c = 0; c < 9; c++) {
        const double v = scale * red[0][c];
        out[c] = v;
        s2 += v * v;
        if (old) d2 += (v - old[c]) * (v - old[c]);
    }
    out[9] = old ? sqrt(d2) / sqrt(s2) : 0.0;
}

}  // namespace ephip

using namespace ephip;

static inline unsigned nbk(int64_t n, int bs = 256) { return (unsigned)((n + bs - 1) / bs); }

extern "C" int ephip_bte_increments(int64_t n, int32_t method, int32_t smearing, const double *in, double *out,
                                    void *stream) {
    EPHIP_REQUIRE(method >= 1 && method <= 6, "bte_increments: method %d outside 1..6", method);
    EPHIP_REQUIRE(smearing == 1 || smearing == 2, "bte_increments: smearing must be 1 (Gaussian) or 2 (Lorentzian)");
    if (n <= 0) return EPHIP_OK;
    EPHIP_REQUIRE(in && out, "bte_increments: null device pointer");
    bte_increments_kernel<<<nbk(n), 256, 0, as_stream(stream)>>>(n, method, smearing, in, out);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_bte_accumulate_units(int32_t nunits, int64_t cs, int32_t nbw, int32_t nm, const int32_t *count,
                                          const int32_t *col_index, const int32_t *ikq, const float *g2,
                                          const int64_t *unit_state_index, const int64_t *state_offset,
                                          const int64_t *bmin, const int64_t *bmax, const double *e_state,
                                          const double *omega, double wtq, int32_t nT, const double *mus,
                                          const double *Ts, const double *etas, int32_t method, int32_t smearing,
                                          double w_cut, int64_t nstates, const int64_t *rowptr, double *S_out,
                                          double *S_in, uint32_t *row_code, void *stream) {
    EPHIP_REQUIRE(nunits >= 0 && nunits <= 65535 && cs >= 0 && nbw >= 1 && nbw <= 31 && nm >= 1 && nT >= 1,
                  "bte_accumulate_units: bad sizes");
    EPHIP_REQUIRE(nstates < (1LL << 27), "bte_accumulate_units: %lld states exceed the row code range",
                  (long long)nstates);
    EPHIP_REQUIRE(method >= 1 && method <= 6 && (smearing == 1 || smearing == 2),
                  "bte_accumulate_units: bad method/smearing");
    if (nunits == 0 || cs == 0) return EPHIP_OK;
    EPHIP_REQUIRE(count && col_index && ikq && g2 && unit_state_index && state_offset && bmin && bmax && e_state &&
                      omega && mus && Ts && etas && rowptr && S_out && S_in && row_code,
                  "bte_accumulate_units: null device pointer");
    dim3 g(nbk(cs * nbw), (unsigned)nunits);
    bte_accumulate_kernel<<<g, 256, 0, as_stream(stream)>>>(nunits, cs, nbw, nm, count, col_index, ikq, g2,
                                                            unit_state_index, state_offset, bmin, bmax, e_state, omega,
                                                            wtq, nT, mus, Ts, etas, method, smearing, w_cut, nstates,
                                                            rowptr, S_out, S_in, row_code);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_bte_tables(int32_t nq, int32_t nm, const double *omega, int64_t nstates, const double *e_state,
                                int32_t nT, const double *mus, const double *Ts, int32_t method, double *tab_q,
                                double *tab_s, void *stream) {
    EPHIP_REQUIRE(nq >= 0 && nm >= 1 && nstates >= 0 && nT >= 1, "bte_tables: bad sizes");
    EPHIP_REQUIRE(method >= 1 && method <= 6, "bte_tables: method %d outside 1..6", method);
    const int64_t n = (int64_t)nm * nq + nT * nstates;
    if (n == 0) return EPHIP_OK;
    EPHIP_REQUIRE(n <= MAX_THREADS_X, "bte_tables: too many entries");
    EPHIP_REQUIRE(omega && e_state && mus && Ts && tab_q && tab_s, "bte_tables: null device pointer");
    bte_tables_kernel<<<nbk(n), 256, 0, as_stream(stream)>>>(nq, nm, omega, nstates, e_state, nT, mus, Ts, method, tab_q,
                                                            tab_s);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_bte_accumulate_tables(int32_t nunits, int64_t cs, int32_t nbw, int32_t nm, int32_t nq,
                                           const int32_t *count, const int32_t *col_index, const int32_t *ikq,
                                           const float *g2, const int64_t *unit_state_index,
                                           const int64_t *state_offset, const int64_t *bmin, const int64_t *bmax,
                                           const double *e_state, const double *tab_q, const double *tab_s,
                                           double wtq, int32_t nT, const double *Ts, const double *etas,
                                           int32_t method, int32_t smearing, double w_cut, int64_t nstates,
                                           const int64_t *rowptr, double *S_out, double *S_in, uint32_t *row_code,
                                           void *stream) {
    EPHIP_REQUIRE(nunits >= 0 && nunits <= 65535 && cs >= 0 && nbw >= 1 && nbw <= 31 && nm >= 1 && nT >= 1 && nq >= 0,
                  "bte_accumulate_tables: bad sizes");
    EPHIP_REQUIRE(nstates < (1LL << 27), "bte_accumulate_tables: %lld states exceed the row code range",
                  (long long)nstates);
    EPHIP_REQUIRE(method >= 1 && method <= 6 && (smearing == 1 || smearing == 2),
                  "bte_accumulate_tables: bad method/smearing");
    if (nunits == 0 || cs == 0) return EPHIP_OK;
    EPHIP_REQUIRE(count && col_index && ikq && g2 && unit_state_index && state_offset && bmin && bmax && e_state &&
                      tab_q && tab_s && Ts && etas && rowptr && S_out && S_in && row_code,
                  "bte_accumulate_tables: null device pointer");
    using K = decltype(&bte_accumulate_tab_kernel<1, 1>);
#define BTE_ROW(m) {bte_accumulate_tab_kernel<m, 1>, bte_accumulate_tab_kernel<m, 2>, bte_accumulate_tab_kernel<m, 3>}
    static const K kern[6][3] = {BTE_ROW(1), BTE_ROW(2), BTE_ROW(3), BTE_ROW(4), BTE_ROW(5), BTE_ROW(6)};
#undef BTE_ROW
    kern[method - 1][nT == 1 ? 0 : nT == 2 ? 1 : 2]<<<units_first_grid(nunits, (cs + 255) / 256), 256,
                                                      (size_t)256 * nbw * sizeof(uint16_t), as_stream(stream)>>>(
        nunits, cs, nbw, nm, nq, count, col_index, ikq, g2, unit_state_index, state_offset, bmin, bmax, e_state, tab_q,
        tab_s, wtq, nT, Ts, etas, smearing, w_cut, nstates, rowptr, S_out, S_in, row_code,
        (nm & 3) == 0 && (reinterpret_cast<uintptr_t>(g2) & 15) == 0);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_band_velocity(int32_t nw, int64_t nstates, const int64_t *state_col, const int32_t *state_band,
                                   const int64_t *state_k, const void *dH, int64_t ld_dh, const void *U, double *v,
                                   void *stream) {
    EPHIP_REQUIRE(nw >= 1 && nstates >= 0 && ld_dh >= 3LL * nw * nw, "band_velocity: bad sizes");
    if (nstates == 0) return EPHIP_OK;
    EPHIP_REQUIRE(state_col && state_band && state_k && dH && U && v, "band_velocity: null device pointer");
    band_velocity_kernel<<<nbk(nstates * 3), 256, 0, as_stream(stream)>>>(
        nw, nstates, state_col, state_band, state_k, static_cast<const double2 *>(dH), ld_dh,
        static_cast<const float2 *>(U), v);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_el_velocity_direct_batched(int32_t nw, int64_t nk, const void *M, int64_t ld_m, const void *U,
                                                const double *E, const void *rbar, int64_t ld_r, void *out,
                                                int64_t ld_out, void *stream) {
    EPHIP_REQUIRE(nw >= 1 && nw <= VEL_NW_MAX && nk >= 0 && nk <= 0x7fffffffLL / 3,
                  "el_velocity_direct_batched: nw=%d (1..%d), nk=%lld", nw, VEL_NW_MAX, (long long)nk);
    EPHIP_REQUIRE(ld_m >= 3LL * nw * nw && ld_out >= 3LL * nw * nw, "el_velocity_direct_batched: ld below 3 nw^2");
    EPHIP_REQUIRE((E == nullptr) == (rbar == nullptr), "el_velocity_direct_batched: E and rbar come together");
    EPHIP_REQUIRE(rbar == nullptr || ld_r >= 3LL * nw * nw, "el_velocity_direct_batched: ld_r below 3 nw^2");
    if (nk == 0) return EPHIP_OK;
    EPHIP_REQUIRE(M && U && out, "el_velocity_direct_batched: null device pointer");
    el_velocity_full_kernel<<<(unsigned)(3 * nk), 256, 0, as_stream(stream)>>>(
        nw, static_cast<const double2 *>(M), ld_m, static_cast<const float2 *>(U), E,
        static_cast<const double2 *>(rbar), ld_r, static_cast<double2 *>(out), ld_out);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_bte_spmv(int32_t nunits, int32_t nbw, int32_t nT, int32_t iT, const int64_t *rowptr,
                              const uint32_t *row_code, const int64_t *unit_state_index, const double *S_in,
                              const double *x, double *y, void *stream) {
    EPHIP_REQUIRE(nunits >= 0 && nbw >= 1 && nT >= 1 && iT >= 0 && iT < nT, "bte_spmv: bad sizes");
    if (nunits == 0) return EPHIP_OK;
    EPHIP_REQUIRE(rowptr && row_code && unit_state_index && S_in && x && y, "bte_spmv: null device pointer");
    bte_spmv_kernel<<<(unsigned)((nunits + 3) / 4), 256, 0, as_stream(stream)>>>(nunits, nbw, nT, iT, rowptr, row_code,
                                                                                unit_state_index, S_in, x, y);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_bte_window_accumulate(int32_t fp64, double *S_out, int64_t ld_so, double *S_in, int64_t ld_si1,
                                           int64_t ld_si2, const void *g2vals, const void *wq, const int64_t *imap_i,
                                           const int64_t *imap_f, int64_t ld_f, int64_t nk_f, const int64_t *ikqs,
                                           const double *e_i, const double *e_f, const double *wf, int32_t nT,
                                           const double *mus, const double *Ts, const double *etas, int32_t method,
                                           int32_t smearing, double w_cut, int32_t nbandkq, int32_t nbandk, int32_t nm,
                                           int64_t nq, int64_t i0, uint32_t *dropped, void *stream) {
    EPHIP_REQUIRE(nbandkq >= 0 && nbandk >= 0 && nm >= 0 && nq >= 0 && nT >= 1 && i0 >= 0 && nk_f >= 0,
                  "bte_window_accumulate: bad sizes");
    EPHIP_REQUIRE(ld_f >= (nbandkq > 0 ? nbandkq : 1) && ld_si1 >= 1 && ld_si2 >= 1 && ld_so >= 1,
                  "bte_window_accumulate: bad leading dimensions");
    EPHIP_REQUIRE(method >= 1 && method <= 6 && (smearing == 1 || smearing == 2),
                  "bte_window_accumulate: bad method/smearing");
    const int64_t ne = (int64_t)nbandkq * nbandk * nq;
    if (ne == 0) return EPHIP_OK;
    EPHIP_REQUIRE(S_out && S_in && g2vals && wq && imap_i && imap_f && ikqs && e_i && e_f && wf && mus && Ts && etas,
                  "bte_window_accumulate: null device pointer");
    EPHIP_REQUIRE(ne <= 0x7fffffffLL * 256, "bte_window_accumulate: too many entries");
    if (fp64)
        bte_window_accumulate_kernel<double><<<nbk(ne), 256, 0, as_stream(stream)>>>(
            S_out, ld_so, S_in, ld_si1, ld_si2, static_cast<const double *>(g2vals), static_cast<const double *>(wq),
            imap_i, imap_f, ld_f, nk_f, ikqs, e_i, e_f, wf, nT, mus, Ts, etas, method, smearing, w_cut, nbandkq, nbandk, nm, nq,
            i0, dropped);
    else
        bte_window_accumulate_kernel<float><<<nbk(ne), 256, 0, as_stream(stream)>>>(
            S_out, ld_so, S_in, ld_si1, ld_si2, static_cast<const float *>(g2vals), static_cast<const float *>(wq),
            imap_i, imap_f, ld_f, nk_f, ikqs, e_i, e_f, wf, nT, mus, Ts, etas, method, smearing, w_cut, nbandkq, nbandk, nm, nq,
            i0, dropped);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}

extern "C" int ephip_bte_step(int64_t n, const double *y, const double *inv_tau, const double *rhs, double mixing,
                              double *df, const double *vs, double scale, const double *old, double *work,
                              double *out, void *stream) {
    EPHIP_REQUIRE(n >= 0, "bte_step: n=%lld is negative", (long long)n);
    EPHIP_REQUIRE(work && out && old != out, "bte_step: null work or out, or old is out");
    EPHIP_REQUIRE(n == 0 || (df && vs && (!y || (inv_tau && rhs))), "bte_step: null device pointer");
    const int nblocks = (int)std::max<int64_t>(1, std::min<int64_t>(BTE_STEP_BLOCKS, (n + 255) / 256));
    bte_step_kernel<<<nblocks, 256, 0, as_stream(stream)>>>(n, y, inv_tau, rhs, mixing, df, vs, work);
    bte_step_sum_kernel<<<1, 256, 0, as_stream(stream)>>>(nblocks, work, scale, old, out);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}
