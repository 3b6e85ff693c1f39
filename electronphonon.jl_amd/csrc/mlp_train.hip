// One gradient of the band-energy network in three launches: forward and data-backward pass of a block of points
// through all three layers, weight and bias gradients as per-workgroup partial sums, and their reduction. The
// layers are those of mlp.hip (features -> W1, b1 -> SiLU -> W2, b2 -> SiLU -> W3, b3, mean squared error).
//
// Everything is FP32 on 16x16x4 MFMAs. Such an MFMA adds its four products one by one, each a rounded FMA in order of
// k (checked bit for bit on gfx950 against the chain of fmaf), so the sums over k, taken in ascending order, are those
// of gemm_f32_kernel: z, a and y come out the same. Layer by layer (23 launches of a VALU GEMM at 7 TFLOP/s, SiLU, column
// sums) a gradient of 33824 points, 64 features, 128 hidden, 16 outputs took 843 us of kernels; here 124 (80, 36 and 7.6),
// with the matrix cores' floor at 31: one workgroup a CU (its weights and activations fill the LDS), whose staging,
// products and SiLU follow one another.
#include "common.hpp"

namespace ephip {

constexpr int MT_DIM = 128;   // largest feature and hidden size
constexpr int MT_OUT = 64;    // largest output size
constexpr int MT_WAVES = 9;   // most waves of a workgroup, 16 points each
// LDS pitches, fixed so that a product's operand offsets are immediates: activations and out x in weights put 16 rows of
// 4 consecutive k on the 64 banks, in x out weights 4 k rows of 16 columns
constexpr int MT_PITCH_A = MT_DIM + 4, MT_PITCH_T = MT_DIM + 4, MT_PITCH_N = MT_DIM + 16;

struct MtArgs {
    int64_t n;
    const double *xk;
    int nf2, nf, nh, no;
    const int *mvec;
    const float *W1, *b1, *W2, *b2, *W3, *b3, *target;
    float scale;
    float *f, *z1, *a1, *z2, *a2, *y, *gy, *gz2, *gz1;
    double *partial;
};

__device__ __forceinline__ float mt_silu(float z) { return z / (1.f + __expf(-z)); }
__device__ __forceinline__ float mt_dsilu(float z) {
    const float s = 1.f / (1.f + __expf(-z));
    return s * (1.f + z * (1.f - s));
}

// W (rows x cols, row-major) into LDS with the given pitch
__device__ __forceinline__ void mt_stage(const float *__restrict__ W, int rows, int cols, float *lds, int pitch) {
    const int n = rows * cols / 4, bd = blockDim.x;
    const unsigned magic = (unsigned)(((1ull << 32) + cols - 1) / cols);  // floor(x / cols) = umulhi for x < 2^16
    for (int e0 = threadIdx.x; e0 < n; e0 += 8 * bd) {  // eight loads in flight
        float4 v[8];
#pragma unroll
        for (int x = 0; x < 8; x++) v[x] = reinterpret_cast<const float4 *>(W)[min(e0 + x * bd, n - 1)];
#pragma unroll
        for (int x = 0; x < 8; x++) {
            const int e = e0 + x * bd, r = (int)__umulhi(4u * e, magic), c = 4 * e - r * cols;
            if (e < n) *reinterpret_cast<float4 *>(lds + r * pitch + c) = v[x];
        }
    }
}

// acc[cb] += A (16 x K, the wave's rows) op(W) for NCB column blocks: TRANS W out x in (B[k][n] = W[n][k]), else in x
// out. NCB is a constant: with a test per block every MFMA waited for its own operand read.
template <bool TRANS, int NCB>
__device__ __forceinline__ void mt_product_n(const float *A, const float *W, int K, f32x4 (&acc)[MT_DIM / 16]) {
    const int lane = threadIdx.x & 63, il = lane & 15, kq = lane >> 4;
    const float *ap = A + il * MT_PITCH_A + kq, *wp = TRANS ? W + il * MT_PITCH_T + kq : W + kq * MT_PITCH_N + il;
    for (int k0 = 0; k0 < K; k0 += 16) {  // K a multiple of 16
#pragma unroll
        for (int kk = 0; kk < 16; kk += 4) {
            const int k = k0 + kk;
            const float a = ap[k];
            const float *w = TRANS ? wp + k : wp + k * MT_PITCH_N;
#pragma unroll
            for (int cb = 0; cb < NCB; cb++)
                acc[cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, w[TRANS ? 16 * cb * MT_PITCH_T : 16 * cb], acc[cb], 0, 0, 0);
        }
    }
}

template <bool TRANS>
__device__ __forceinline__ void mt_product(const float *A, const float *W, int K, int ncb, f32x4 (&acc)[MT_DIM / 16]) {
    switch (ncb) {  // uniform
        case 1: return mt_product_n<TRANS, 1>(A, W, K, acc);
        case 2: return mt_product_n<TRANS, 2>(A, W, K, acc);
        case 3: return mt_product_n<TRANS, 3>(A, W, K, acc);
        case 4: return mt_product_n<TRANS, 4>(A, W, K, acc);
        case 5: return mt_product_n<TRANS, 5>(A, W, K, acc);
        case 6: return mt_product_n<TRANS, 6>(A, W, K, acc);
        case 7: return mt_product_n<TRANS, 7>(A, W, K, acc);
        default: return mt_product_n<TRANS, 8>(A, W, K, acc);
    }
}

// One workgroup: 16 points per wave; every wave carries its points through all layers, the activations of its rows
// in its part of LDS, z2 in registers for the backward pass; the weights of a layer are staged for all waves.
__global__ __launch_bounds__(64 * MT_WAVES) void mlp_train_kernel(MtArgs a) {
    extern __shared__ float mt_lds[];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nwave = blockDim.x >> 6;
    const int il = lane & 15, q = lane >> 4;
    const int nf = a.nf, nh = a.nh, no = a.no;
    float *act = mt_lds + wave * 16 * MT_PITCH_A;
    float *W = mt_lds + nwave * 16 * MT_PITCH_A;
    const int64_t p0 = ((int64_t)blockIdx.x * nwave + wave) * 16;
    float *actw = act + 4 * q * MT_PITCH_A + il;  // this thread's products: rows 4 q + r, column il of each block
    const f32x4 zero{0.f, 0.f, 0.f, 0.f};
    f32x4 acc[MT_DIM / 16], z2[MT_DIM / 16];

    // features of the wave's points
    for (int e = lane; e < 16 * a.nf2; e += 64) {
        const int i = e / a.nf2, j = e - i * a.nf2;
        const int64_t p = p0 + i;
        float c = 0.f, s = 0.f;
        if (p < a.n) {
            const double x = a.mvec[3 * j] * a.xk[3 * p] + a.mvec[3 * j + 1] * a.xk[3 * p + 1] +
                             a.mvec[3 * j + 2] * a.xk[3 * p + 2];
            cis2pi(x, c, s);
            a.f[p * nf + j] = c;
            a.f[p * nf + a.nf2 + j] = s;
        }
        act[i * MT_PITCH_A + j] = c;
        act[i * MT_PITCH_A + a.nf2 + j] = s;
    }
    // hidden layers
    for (int layer = 0; layer < 2; layer++) {
        const int K = layer ? nh : nf;
        if (layer) __syncthreads();  // the last layer's weights no longer read
        mt_stage(layer ? a.W2 : a.W1, nh, K, W, MT_PITCH_T);
        __syncthreads();
#pragma unroll
        for (int cb = 0; cb < MT_DIM / 16; cb++) acc[cb] = zero;
        mt_product<true>(act, W, K, nh / 16, acc);
        wave_lds_sync();  // the wave's activations are replaced below
        const float *bias = layer ? a.b2 : a.b1;
        float *zr[4], *ar[4];  // the rows this thread stores, at its column
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int64_t o = min(p0 + 4 * q + r, a.n - 1) * nh + il;
            zr[r] = (layer ? a.z2 : a.z1) + o;
            ar[r] = (layer ? a.a2 : a.a1) + o;
        }
#pragma unroll
        for (int cb = 0; cb < MT_DIM / 16; cb++) {
            if (16 * cb < nh) {
                const int c = 16 * cb + il;
                const float b = bias[c];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float z = acc[cb][r] + b, v = mt_silu(z);
                    acc[cb][r] = z;
                    actw[r * MT_PITCH_A + 16 * cb] = v;
                    if (p0 + 4 * q + r < a.n) {
                        zr[r][16 * cb] = z;
                        ar[r][16 * cb] = v;
                    }
                }
            }
            if (layer) z2[cb] = acc[cb];
        }
        wave_lds_sync();
    }
    // output layer, error and its gradient
    __syncthreads();
    mt_stage(a.W3, no, nh, W, MT_PITCH_T);
    __syncthreads();
#pragma unroll
    for (int cb = 0; cb < MT_DIM / 16; cb++) acc[cb] = zero;
    mt_product<true>(act, W, nh, no / 16, acc);
    wave_lds_sync();
#pragma unroll
    for (int cb = 0; cb < MT_OUT / 16; cb++) {
        if (16 * cb < no) {
            const int c = 16 * cb + il;
            const float b = a.b3[c];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int64_t p = p0 + 4 * q + r;
                float d = 0.f;
                if (p < a.n) {
                    const float y = acc[cb][r] + b;
                    d = y - a.target[p * no + c];
                    a.y[p * no + c] = y;
                    a.gy[p * no + c] = 2.f * d * a.scale;
                }
                act[(4 * q + r) * MT_PITCH_A + c] = d;
            }
        }
    }
    wave_lds_sync();
    // sums of d^2 over 256 consecutive entries of the flat (point, output) array: the wave's 16 points hold no / 16
    for (int b = 0; b < no / 16; b++) {
        double s = 0.0;
#pragma unroll
        for (int x = 0; x < 4; x++) {
            const int e = 256 * b + 4 * lane + x;
            const float d = act[(e / no) * MT_PITCH_A + e % no];
            s += (double)d * d;
        }
        s = wave_sum(s);
        if (lane == 0 && p0 * no + 256 * b < a.n * no) a.partial[p0 * no / 256 + b] = s;
    }
    wave_lds_sync();
#pragma unroll
    for (int cb = 0; cb < MT_OUT / 16; cb++)
        if (16 * cb < no)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float &d = act[(4 * q + r) * MT_PITCH_A + 16 * cb + il];
                d = 2.f * d * a.scale;
            }
    wave_lds_sync();
    // backward through the output and the second hidden layer
    for (int layer = 2; layer >= 1; layer--) {
        const int K = layer == 2 ? no : nh;
        __syncthreads();  // the staged weights no longer read
        mt_stage(layer == 2 ? a.W3 : a.W2, K, nh, W, MT_PITCH_N);
        __syncthreads();
#pragma unroll
        for (int cb = 0; cb < MT_DIM / 16; cb++) acc[cb] = zero;
        mt_product<false>(act, W, K, nh / 16, acc);
        wave_lds_sync();
        float *gr[4];
        const float *zr[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int64_t o = min(p0 + 4 * q + r, a.n - 1) * nh + il;
            gr[r] = (layer == 2 ? a.gz2 : a.gz1) + o;
            zr[r] = a.z1 + o;
        }
#pragma unroll
        for (int cb = 0; cb < MT_DIM / 16; cb++) {
            if (16 * cb < nh) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    // z1 is read back (this thread wrote it): kept as well, the registers spill
                    const float z = layer == 2 ? z2[cb][r] : zr[r][16 * cb];
                    const float g = acc[cb][r] * mt_dsilu(z);
                    actw[r * MT_PITCH_A + 16 * cb] = g;
                    if (p0 + 4 * q + r < a.n) gr[r][16 * cb] = g;
                }
            }
        }
        wave_lds_sync();
    }
}

// Weight gradients gW = gz^T x (out x in) and bias gradients (column sums of gz) of the three layers over one
// workgroup's share of the points, as a partial of the flat parameter vector (W1, b1, W2, b2, W3, b3). The points are
// staged MG_PTS at a time, natural row order with pitches of 16 over a multiple of 64 (four points of 16 columns on
// 64 banks), the next points' loads in flight during the products. Wave w owns row block w of gW1 and gW2 and column
// block w of gW3 (one operand read serves the block's tiles), all in accumulators. With the tiles dealt one by one and
// no loads ahead it took 82 us (both operands read per tile, spills).
constexpr int MG_PTS = 32, MG_WAVES = MT_DIM / 16;
__host__ __device__ constexpr int mg_pitch(int n) { return (n + 63) / 64 * 64 + 16; }

// TH, TF, TO: the blocks of hidden, features and outputs rounded up to 2, 4, 8 (1, 2, 4); the blocks past the sizes
// read the rows' padding and are not stored.
template <int TH, int TF, int TO>
__global__ __launch_bounds__(64 * MG_WAVES) void mlp_wgrad_kernel(int64_t n, int nf, int nh, int no,
                                                                  const float *__restrict__ f,
                                                                  const float *__restrict__ a1,
                                                                  const float *__restrict__ a2,
                                                                  const float *__restrict__ gy,
                                                                  const float *__restrict__ gz2,
                                                                  const float *__restrict__ gz1, int64_t nparam,
                                                                  float *__restrict__ part) {
    extern __shared__ float mg_lds[];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, bd = blockDim.x, il = lane & 15, kq = lane >> 4;
    const int ph = mg_pitch(nh), pf = mg_pitch(nf), po = mg_pitch(no);
    float *sg1 = mg_lds, *sf = sg1 + MG_PTS * ph, *sg2 = sf + MG_PTS * pf, *sa1 = sg2 + MG_PTS * ph,
          *sa2 = sa1 + MG_PTS * ph, *sgy = sa2 + MG_PTS * ph;
    const int th = nh / 16, tf = nf / 16, to = no / 16;
    f32x4 acc1[TF], acc2[TH], acc3[TO];
#pragma unroll
    for (int x = 0; x < TF; x++) acc1[x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < TH; x++) acc2[x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < TO; x++) acc3[x] = f32x4{0.f, 0.f, 0.f, 0.f};
    float bs = 0.f;  // thread t < 2 nh + no: the sum of one column of gz1, gz2 or gy
    const int64_t pa = n * blockIdx.x / gridDim.x, pz = n * (blockIdx.x + 1) / gridDim.x;
    // the next points' rows: a thread's float4 of each array (two of the hidden-size ones and f, one of gy), zero past
    // the workgroup's points
    constexpr int LH = MG_PTS * MT_DIM / 4 / (64 * MG_WAVES), LO = MG_PTS * MT_OUT / 4 / (64 * MG_WAVES);
    float4 pre[4][LH], pre_f[LH], pre_y[LO];
    auto load_one = [&](const float *src, int cols, int64_t p0, int e) {
        const int r = 4 * e / cols, c = 4 * e - r * cols;
        const bool on = r < MG_PTS && p0 + r < pz;
        const float4 v = *reinterpret_cast<const float4 *>(src + (on ? (p0 + r) * cols + c : 0));
        return on ? v : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    auto store_one = [&](float *dst, int cols, int pitch, int e, float4 v) {
        const int r = 4 * e / cols, c = 4 * e - r * cols;
        if (r < MG_PTS) *reinterpret_cast<float4 *>(dst + r * pitch + c) = v;
    };
    auto load = [&](int64_t p0) {
#pragma unroll
        for (int x = 0; x < LH; x++) {
            const int e = t + x * bd;
            pre[0][x] = load_one(gz1, nh, p0, e);
            pre[1][x] = load_one(gz2, nh, p0, e);
            pre[2][x] = load_one(a1, nh, p0, e);
            pre[3][x] = load_one(a2, nh, p0, e);
            pre_f[x] = load_one(f, nf, p0, e);
        }
#pragma unroll
        for (int x = 0; x < LO; x++) pre_y[x] = load_one(gy, no, p0, t + x * bd);
    };
    if (pa < pz) load(pa);
    for (int64_t p0 = pa; p0 < pz; p0 += MG_PTS) {
#pragma unroll
        for (int x = 0; x < LH; x++) {
            const int e = t + x * bd;
            store_one(sg1, nh, ph, e, pre[0][x]);
            store_one(sg2, nh, ph, e, pre[1][x]);
            store_one(sa1, nh, ph, e, pre[2][x]);
            store_one(sa2, nh, ph, e, pre[3][x]);
            store_one(sf, nf, pf, e, pre_f[x]);
        }
#pragma unroll
        for (int x = 0; x < LO; x++) store_one(sgy, no, po, t + x * bd, pre_y[x]);
        __syncthreads();
        if (p0 + MG_PTS < pz) load(p0 + MG_PTS);
        if (wave < th) {  // uniform
            const float *g1 = sg1 + kq * ph + 16 * wave + il, *g2 = sg2 + kq * ph + 16 * wave + il;
            const float *x3 = sa2 + kq * ph + 16 * wave + il, *x1 = sf + kq * pf + il, *x2 = sa1 + kq * ph + il;
            const float *g3 = sgy + kq * po + il;
#pragma unroll 2
            for (int k = 0; k < MG_PTS; k += 4) {
                const float u1 = g1[k * ph], u2 = g2[k * ph], u3 = x3[k * ph];
#pragma unroll
                for (int c = 0; c < TH; c++)
                    acc2[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(u2, x2[k * ph + 16 * c], acc2[c], 0, 0, 0);
#pragma unroll
                for (int c = 0; c < TF; c++)
                    acc1[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(u1, x1[k * pf + 16 * c], acc1[c], 0, 0, 0);
#pragma unroll
                for (int r = 0; r < TO; r++)
                    acc3[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(g3[k * po + 16 * r], u3, acc3[r], 0, 0, 0);
            }
        }
        if (t < 2 * nh + no) {
            const float *g = t < nh ? sg1 + t : t < 2 * nh ? sg2 + t - nh : sgy + t - 2 * nh;
            const int pg = t < 2 * nh ? ph : po;
            for (int k = 0; k < MG_PTS; k++) bs += g[k * pg];
        }
        __syncthreads();
    }
    // flat offsets: W1 (nh x nf), b1, W2 (nh x nh), b2, W3 (no x nh), b3
    float *out = part + nparam * blockIdx.x;
    const int ob1 = nh * nf, oW2 = ob1 + nh, ob2 = oW2 + nh * nh, oW3 = ob2 + nh, ob3 = oW3 + no * nh;
    if (wave < th) {
#pragma unroll
        for (int y = 0; y < 4; y++) {
            const int r = 16 * wave + 4 * kq + y;
#pragma unroll
            for (int c = 0; c < TF; c++)
                if (c < tf) out[r * nf + 16 * c + il] = acc1[c][y];
#pragma unroll
            for (int c = 0; c < TH; c++)
                if (c < th) out[oW2 + r * nh + 16 * c + il] = acc2[c][y];
#pragma unroll
            for (int c = 0; c < TO; c++)
                if (c < to) out[oW3 + (16 * c + 4 * kq + y) * nh + 16 * wave + il] = acc3[c][y];
        }
    }
    if (t < nh) out[ob1 + t] = bs;
    else if (t < 2 * nh) out[ob2 + t - nh] = bs;
    else if (t < 2 * nh + no) out[ob3 + t - 2 * nh] = bs;
}

// g[e] = sum over the partials, a block per 64 parameters: sixteen waves take every sixteenth partial
__global__ __launch_bounds__(1024) void mlp_reduce_kernel(int nparts, int64_t nparam, const float *__restrict__ part,
                                                          float *__restrict__ g) {
    __shared__ float red[16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t e = (int64_t)blockIdx.x * 64 + lane;
    float s[4] = {0.f, 0.f, 0.f, 0.f};  // four loads in flight
    if (e < nparam)
        for (int b = 4 * wave; b < nparts; b += 64)
#pragma unroll
            for (int x = 0; x < 4; x++)
                if (b + x < nparts) s[x] += part[(b + x) * nparam + e];
    red[wave][lane] = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    if (wave == 0 && e < nparam) {
        float v = 0.f;
        for (int w = 0; w < 16; w++) v += red[w][lane];
        g[e] = v;
    }
}

}  // namespace ephip

using namespace ephip;

static size_t mt_lds_bytes(int waves, int nh, int no) {
    return sizeof(float) * ((size_t)waves * 16 * MT_PITCH_A + (size_t)max(nh, no) * MT_PITCH_N);
}

extern "C" int ephip_mlp_train_step(int64_t npts, const double *xk, int32_t nf2, const int32_t *mvec, int32_t hidden,
                                    int32_t nout, const float *params, const float *target, float *f, float *z1,
                                    float *a1, float *z2, float *a2, float *y, float *gy, float *gz2, float *gz1,
                                    double *partial, int32_t nparts, float *part, float *grad, void *stream) {
    const int nf = 2 * nf2;
    EPHIP_REQUIRE(npts >= 0 && npts < ((int64_t)1 << 36), "mlp_train_step: bad point count");
    EPHIP_REQUIRE(nf2 >= 8 && nf % 16 == 0 && nf <= MT_DIM && hidden >= 16 && hidden % 16 == 0 && hidden <= MT_DIM &&
                      nout >= 16 && nout % 16 == 0 && nout <= MT_OUT,
                  "mlp_train_step: features %d and hidden %d multiples of 16 up to %d, outputs %d up to %d", nf, hidden,
                  MT_DIM, nout, MT_OUT);
    EPHIP_REQUIRE(nparts >= 1 && nparts <= 65535, "mlp_train_step: %d partials", nparts);
    if (npts == 0) return EPHIP_OK;
    EPHIP_REQUIRE(xk && mvec && params && target && f && z1 && a1 && z2 && a2 && y && gy && gz2 && gz1 && partial &&
                      part && grad,
                  "mlp_train_step: null device pointer");
    EPHIP_REQUIRE((reinterpret_cast<uintptr_t>(params) & 15) == 0 && ((nf * hidden + hidden) & 3) == 0,
                  "mlp_train_step: parameters must be 16-byte aligned");
    MtArgs a{};
    a.n = npts, a.xk = xk, a.nf2 = nf2, a.nf = nf, a.nh = hidden, a.no = nout, a.mvec = mvec;
    a.W1 = params, a.b1 = a.W1 + hidden * nf, a.W2 = a.b1 + hidden, a.b2 = a.W2 + hidden * hidden;
    a.W3 = a.b2 + hidden, a.b3 = a.W3 + nout * hidden, a.target = target;
    a.scale = (float)(1.0 / ((double)npts * nout));
    a.f = f, a.z1 = z1, a.a1 = a1, a.z2 = z2, a.a2 = a2, a.y = y, a.gy = gy, a.gz2 = gz2, a.gz1 = gz1;
    a.partial = partial;
    hipStream_t st = as_stream(stream);
    // waves (16 points each) per workgroup: the fewest rounds over the 256 CUs times the waves that share a SIMD
    int waves = 4;
    double best = 0.0;
    for (int w = 4; w <= MT_WAVES; w++) {
        const size_t lds = mt_lds_bytes(w, hidden, nout);
        if (lds > 152 * 1024) break;
        const int64_t blocks = (npts + 16 * w - 1) / (16 * w), per_cu = max((int64_t)1, (int64_t)(160 * 1024 / lds));
        const int64_t rounds = (blocks + 256 * per_cu - 1) / (256 * per_cu);
        const double cost = rounds * (0.5 + (double)((min(per_cu, (blocks + 255) / 256) * w + 3) / 4));
        if (best == 0.0 || cost < best) best = cost, waves = w;
    }
    const size_t lds = mt_lds_bytes(waves, hidden, nout);
    if (lds > 64 * 1024)
        EPHIP_TRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(mlp_train_kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    mlp_train_kernel<<<(unsigned)((npts + 16 * waves - 1) / (16 * waves)), 64 * waves, lds, st>>>(a);
    EPHIP_LAUNCHED();
    const int64_t nparam = (int64_t)hidden * nf + hidden + (int64_t)hidden * hidden + hidden + (int64_t)nout * hidden + nout;
    const size_t ldg = sizeof(float) * MG_PTS * (4 * (size_t)mg_pitch(hidden) + mg_pitch(nf) + mg_pitch(nout));
    using KG = decltype(&mlp_wgrad_kernel<2, 2, 1>);
#define MG_ROW(h, f) {mlp_wgrad_kernel<h, f, 1>, mlp_wgrad_kernel<h, f, 2>, mlp_wgrad_kernel<h, f, 4>}
#define MG_TAB(h) {MG_ROW(h, 2), MG_ROW(h, 4), MG_ROW(h, 8)}
    static const KG kg[3][3][3] = {MG_TAB(2), MG_TAB(4), MG_TAB(8)};
#undef MG_TAB
#undef MG_ROW
    auto size = [](int n) { return n <= 32 ? 0 : n <= 64 ? 1 : 2; };
    const KG wgrad = kg[size(hidden)][size(nf)][size(2 * nout)];
    if (ldg > 64 * 1024)
        EPHIP_TRY_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(wgrad),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)ldg));
    wgrad<<<(unsigned)nparts, 64 * MG_WAVES, ldg, st>>>(npts, nf, hidden, nout, f, a1, a2, gy, gz2, gz1, nparam,
                                                                 part);
    EPHIP_LAUNCHED();
    mlp_reduce_kernel<<<(unsigned)((nparam + 63) / 64), 1024, 0, st>>>(nparts, nparam, part, grad);
    EPHIP_LAUNCHED();
    return EPHIP_OK;
}
