// Learned closure: training-data kernels and training kernels (see mlp.h).
//
// Training data come from the solver's own fine runs.  A fine lattice is box
// filtered 2x2x2 onto the coarse grid (k_filter: means of rho, u and of the
// products u_a u_b).  For each coarse node (k_features) the resolved strain
// S is taken by central differences of the filtered velocity (no-slip walls
// half a cell beyond the first and last nodes), the subgrid stress is
// tau_ab = <u_a u_b> - <u_a><u_b>, and the target is the eddy viscosity that
// best carries it, nu_t = -tau:S / (2 S:S), as nu_t/nu clipped to [-10, 10]
// (backscatter is kept: the network's non-negative output then fits the
// conditional mean instead of the mean of the positive part).
// The features are the non-equilibrium moments the coarse MRT would carry
// for that strain to first order (Chapman-Enskog: m_neq = -(2/(3 s)) times
// the strain combination of the moment; zero for e, eps, 3pi_xx, pi_ww), in
// the same scaling the fused collision uses, plus y+.
//
// Training: minibatch gradient of the mean squared error of softplus(o)
// against the target on the matrix cores in FP32, 32 samples a wave at a
// time, per-wave and per-block sums in a fixed order, then a fixed-order sum
// over blocks and an Adam step.
#include <algorithm>
#include <cmath>
#include <utility>

#include "kernels_impl.h"
#include "mlp_train.h"

namespace d3q19 {

namespace {

template <int P>
__global__ void __launch_bounds__(256) k_filter(FilterArgs a)
{
    using S = typename Prec<P>::S;
    using T = typename Prec<P>::T;
    const uint32_t nc = blockIdx.x * 256 + threadIdx.x;
    const uint32_t Nc = a.lxc * a.lyc * a.lzc;
    if (nc >= Nc)
        return;
    const uint32_t cx = nc % a.lxc, cy = (nc / a.lxc) % a.lyc, cz = nc / (a.lxc * a.lyc);
    double s[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int dz = 0; dz < 2; dz++)
        for (int dy = 0; dy < 2; dy++)
            for (int dx = 0; dx < 2; dx++) {
                const uint32_t n = (2 * cx + dx) + a.gf.lx * ((2 * cy + dy) + a.gf.ly * (2 * cz + dz));
                const Nbr b = make_nbr(n, a.gf);
                T f[19];
                pull_all<P>((const S *)a.L, a.gf.S, b, f);
                T rho9, ux9, uy9, uz9;
                macro_sums(f, rho9, ux9, uy9, uz9);
                const double ux = (double)ux9 + 0.5 * a.fx, uy = (double)uy9 + 0.5 * a.fy,
                             uz = (double)uz9 + 0.5 * a.fz;
                s[0] += (double)rho9;
                s[1] += ux;
                s[2] += uy;
                s[3] += uz;
                s[4] += ux * ux;
                s[5] += uy * uy;
                s[6] += uz * uz;
                s[7] += ux * uy;
                s[8] += uy * uz;
                s[9] += ux * uz;
            }
#pragma unroll
    for (int q = 0; q < 10; q++)
        a.out[(uint64_t)q * Nc + nc] = (float)(s[q] * 0.125);
}

__global__ void __launch_bounds__(256) k_features(FeatArgs a)
{
    const uint32_t n = blockIdx.x * 256 + threadIdx.x;
    const uint32_t N = a.lx * a.ly * a.lz;
    if (n >= N)
        return;
    const uint32_t ix = n % a.lx, iy = (n / a.lx) % a.ly, iz = n / (a.lx * a.ly);
    const float *U[3] = {a.fields + 1 * (uint64_t)N, a.fields + 2 * (uint64_t)N, a.fields + 3 * (uint64_t)N};
    // d/dx with no-slip walls half a cell outside: ghost value -u at x = -1, lx
    auto at = [&](int c, int x, uint32_t y, uint32_t z) -> float {
        if (x < 0 || x >= (int)a.lx)
            return -U[c][(x < 0 ? 0 : a.lx - 1) + a.lx * (y + a.ly * z)];
        return U[c][x + a.lx * (y + a.ly * z)];
    };
    float g[3][3]; // g[c][d] = d u_c / d x_d
    const uint32_t yp = (iy + 1) % a.ly, ym = (iy + a.ly - 1) % a.ly;
    const uint32_t zp = (iz + 1) % a.lz, zm = (iz + a.lz - 1) % a.lz;
    for (int c = 0; c < 3; c++) {
        g[c][0] = 0.5f * (at(c, (int)ix + 1, iy, iz) - at(c, (int)ix - 1, iy, iz));
        g[c][1] = 0.5f * (at(c, (int)ix, yp, iz) - at(c, (int)ix, ym, iz));
        g[c][2] = 0.5f * (at(c, (int)ix, iy, zp) - at(c, (int)ix, iy, zm));
    }
    float S[3][3];
    for (int c = 0; c < 3; c++)
        for (int d = 0; d < 3; d++)
            S[c][d] = 0.5f * (g[c][d] + g[d][c]);
    const float u[3] = {U[0][n], U[1][n], U[2][n]};
    // filtered products: uxux, uyuy, uzuz, uxuy, uyuz, uxuz
    const float *F = a.fields;
    float tau[3][3];
    tau[0][0] = F[4 * (uint64_t)N + n] - u[0] * u[0];
    tau[1][1] = F[5 * (uint64_t)N + n] - u[1] * u[1];
    tau[2][2] = F[6 * (uint64_t)N + n] - u[2] * u[2];
    tau[0][1] = tau[1][0] = F[7 * (uint64_t)N + n] - u[0] * u[1];
    tau[1][2] = tau[2][1] = F[8 * (uint64_t)N + n] - u[1] * u[2];
    tau[0][2] = tau[2][0] = F[9 * (uint64_t)N + n] - u[0] * u[2];
    float ts = 0.f, ss = 0.f;
    for (int c = 0; c < 3; c++)
        for (int d = 0; d < 3; d++) {
            ts += tau[c][d] * S[c][d];
            ss += S[c][d] * S[c][d];
        }
    float y = ss > 1e-30f ? -ts / (2.0f * ss) / a.nu : 0.0f;
    y = fminf(fmaxf(y, -10.0f), 10.0f);
    if (a.ts) {
        a.ts[n] = ts;
        a.ss[n] = ss;
    }
    // first-order non-equilibrium moments of the coarse MRT for strain S
    const float k = -2.0f / (3.0f * a.s9);
    const float neq[9] = {0.0f,
                          0.0f,
                          k * (2.0f * S[0][0] - S[1][1] - S[2][2]),
                          0.0f,
                          k * (S[1][1] - S[2][2]),
                          0.0f,
                          k * S[0][1],
                          k * S[1][2],
                          k * S[0][2]};
    float *o = a.feat + (uint64_t)(a.offset + n) * MLP_IN;
    for (int q = 0; q < 9; q++)
        o[q] = neq[q] / a.scale[q];
    const float wd = fminf((float)ix + 0.5f, (float)a.lx - (float)ix - 0.5f);
    o[9] = wd * a.inv_ystar / a.yscale;
    a.target[a.offset + n] = y;
}

// ---------------------------------------------------------------------------
// Training and prediction on the matrix cores, FP32 throughout.
//
// One wave works on 32 samples at a time with v_mfma_f32_32x32x2_f32, whose
// operands take A[i][k] from lane 32 k + i and B[k][j] from lane 32 k + j (one
// float each, k = 0, 1) and which returns D[row][j] to lane 32 h + j, register
// r holding row mfma_row(r, h).  Samples are the columns: D of one layer (a
// lane's own sample, 16 of its 32 hidden units) is operand B of the next as
// it stands when step t of the product takes k = mfma_row(t, h), so the
// forward pass and the back-propagation need no exchange between lanes; the
// weights are loaded in that order once per wave.  The weight gradients sum
// over samples, so their operands have the hidden unit in the lane: those
// pass through LDS (TS floats a sample: 16-byte stores, conflict-free reads).
//
// Bound: 53 matrix instructions of 64 cycles and 16 of 32 (the gradient of W1,
// whose ten columns and b1 fill a 16-wide product) a group of 32 samples, with
// 32 tanh and the LDS traffic between them; the samples (44 B each) stay in
// cache.  An iteration of 65 536 samples takes 14.4 us, 287 us with one lane
// per sample on the vector ALUs (48 us) and one thread per parameter adding 1
// 024 partials (231 us).
constexpr int GROUP = 32;
constexpr int MLP_WAVES = 4;             // waves per block of the prediction
constexpr int TS = 36;                   // LDS stride of a sample's 32 values
constexpr int TX = 12;                   // LDS stride of a sample's inputs
constexpr int MLP_OUT = MLP_NPARAM + 1;  // gradient and loss

typedef float mlp_float16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ constexpr int mfma_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// The forward weights of one wave: rows of W1 and W2 as operand A, biases and
// W3 in the layout of D.
struct MlpRegs {
    float a1[5], a2[16], b1[16], b2[16], w3[16], b3;
    __device__ __forceinline__ void load(const float *__restrict__ w, int j, int h)
    {
#pragma unroll
        for (int t = 0; t < 5; t++)
            a1[t] = w[MLP_W1 + j * MLP_IN + 5 * h + t];
#pragma unroll
        for (int t = 0; t < 16; t++) {
            a2[t] = w[MLP_W2 + j * MLP_H + mfma_row(t, h)];
            b1[t] = w[MLP_B1 + mfma_row(t, h)];
            b2[t] = w[MLP_B2 + mfma_row(t, h)];
            w3[t] = w[MLP_W3 + mfma_row(t, h)];
        }
        b3 = w[MLP_B3];
    }
    // Hidden units h1, h2 and output of the lane's sample; half h of the wave
    // holds its inputs 5 h .. 5 h + 4.
    __device__ __forceinline__ float forward(const float (&x)[5], mlp_float16 &h1, mlp_float16 &h2) const
    {
#pragma unroll
        for (int r = 0; r < 16; r++) {
            h1[r] = b1[r];
            h2[r] = b2[r];
        }
#pragma unroll
        for (int t = 0; t < 5; t++)
            h1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[t], x[t], h1, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; r++)
            h1[r] = fast_tanh(h1[r]);
#pragma unroll
        for (int t = 0; t < 16; t++)
            h2 = __builtin_amdgcn_mfma_f32_32x32x2f32(a2[t], h1[t], h2, 0, 0, 0);
        float o = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            h2[r] = fast_tanh(h2[r]);
            o = fmaf(w3[r], h2[r], o);
        }
        return o + __shfl_xor(o, 32) + b3;
    }
};

// Orders a wave's own LDS stores before its later LDS loads by other lanes:
// the LDS serves one wave's instructions in order, so the compiler's order is
// all there is to keep.
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Gradient of mean((softplus(o) + m - y)^2) over samples [first, first+count):
// wave v of the grid takes groups v, v + waves, ... of 32 samples; the block
// adds its waves in order and writes partial[block * MLP_OUT + i] (i =
// NPARAM: loss).  253 VGPRs and 19.5 KiB of LDS a wave: W = 4 or 8 waves, one
// block per CU (mlp_shape).
template <int W>
__global__ void __launch_bounds__(64 * W, 2)
k_mlp_grad(const float *__restrict__ w, const float *__restrict__ feat, const float *__restrict__ target,
           uint32_t first, uint32_t count, float *__restrict__ partial)
{
    __shared__ __attribute__((aligned(16))) float lds[W][GROUP * (4 * TS + TX)];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, j = lane & 31, h = lane >> 5;
    float *const th1 = lds[wv], *const tg2 = th1 + GROUP * TS, *const tg1 = tg2 + GROUP * TS,
                 *const th3 = tg1 + GROUP * TS, *const tx = th3 + GROUP * TS;
    const float inv_count = 1.0f / (float)count;
    const uint32_t groups = (count + GROUP - 1) / GROUP, waves = gridDim.x * W;
    // the lane's sample of group g: half its inputs and the target, loaded one
    // group ahead (the first with the weights)
    auto sample = [&](uint32_t g, float (&x)[5], float &y) {
        const uint32_t s = g * GROUP + j;
        const bool valid = s < count; // also false past the last group
#pragma unroll
        for (int t = 0; t < 5; t++)
            x[t] = valid ? feat[((uint64_t)first + s) * MLP_IN + 5 * h + t] : 0.0f;
        y = valid ? target[(uint64_t)first + s] : 0.0f;
    };
    float xn[5], yn;
    sample(blockIdx.x * W + wv, xn, yn);
    MlpRegs n;
    n.load(w, j, h);
    float a2t[16]; // columns of W2: the transposed product of the back-propagation
#pragma unroll
    for (int t = 0; t < 16; t++)
        a2t[t] = w[MLP_W2 + mfma_row(t, h) * MLP_H + j];

    mlp_float16 dw2;
    mlp_float4 dw1[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int r = 0; r < 16; r++)
        dw2[r] = 0.0f;
    float db2 = 0.0f, dw3 = 0.0f, db3 = 0.0f, loss = 0.0f;
    for (uint32_t g = blockIdx.x * W + wv; g < groups; g += waves) {
        const bool valid = g * GROUP + j < count;
        float x[5];
#pragma unroll
        for (int t = 0; t < 5; t++)
            x[t] = xn[t];
        const float y = yn;
        sample(g + waves, xn, yn);
        mlp_float16 h1, h2;
        const float o = n.forward(x, h1, h2);
        const float err = mlp_nut(w, o) - y;
        const float sig = 1.0f / (1.0f + __expf(-o));
        const float go = valid ? 2.0f * err * sig * inv_count : 0.0f;
        loss += valid ? err * err * inv_count : 0.0f;
        db3 += go;
        mlp_float16 g2, g1;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            g2[r] = go * n.w3[r] * (1.0f - h2[r] * h2[r]);
            h2[r] = go * h2[r];
            g1[r] = 0.0f;
        }
#pragma unroll
        for (int t = 0; t < 16; t++)
            g1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a2t[t], g2[t], g1, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; r++)
            g1[r] = g1[r] * (1.0f - h1[r] * h1[r]);
        wave_lds_order(); // the previous group's loads come first
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int e = j * TS + mfma_row(4 * q, h);
            *(mlp_float4 *)(th1 + e) = mlp_float4{h1[4 * q], h1[4 * q + 1], h1[4 * q + 2], h1[4 * q + 3]};
            *(mlp_float4 *)(tg2 + e) = mlp_float4{g2[4 * q], g2[4 * q + 1], g2[4 * q + 2], g2[4 * q + 3]};
            *(mlp_float4 *)(tg1 + e) = mlp_float4{g1[4 * q], g1[4 * q + 1], g1[4 * q + 2], g1[4 * q + 3]};
            *(mlp_float4 *)(th3 + e) = mlp_float4{h2[4 * q], h2[4 * q + 1], h2[4 * q + 2], h2[4 * q + 3]};
        }
#pragma unroll
        for (int t = 0; t < 5; t++)
            tx[j * TX + 5 * h + t] = x[t];
        if (h == 0)
            tx[j * TX + MLP_IN] = 1.0f; // column 10 of dw1: the gradient of b1
        wave_lds_order();
#pragma unroll
        for (int t = 0; t < 16; t++) {
            const int k = 2 * t + h; // samples k of the group
            const float ga = tg2[k * TS + j];
            dw2 = __builtin_amdgcn_mfma_f32_32x32x2f32(ga, th1[k * TS + j], dw2, 0, 0, 0);
            db2 += ga;
            dw3 += th3[k * TS + j];
        }
        // v_mfma_f32_16x16x4_f32: A[i][k], B[k][j] in lane 16 k + i, 16 k + j
        const int c16 = lane & 15, k16 = lane >> 4;
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int k = 4 * t + k16;
            const float xb = c16 <= MLP_IN ? tx[k * TX + (c16 <= MLP_IN ? c16 : 0)] : 0.0f;
            dw1[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(tg1[k * TS + c16], xb, dw1[0], 0, 0, 0);
            dw1[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(tg1[k * TS + 16 + c16], xb, dw1[1], 0, 0, 0);
        }
    }

    // each wave's sums into its own LDS rows, then the waves in order
    static_assert(MLP_OUT <= GROUP * (4 * TS + TX), "a wave's sums fit its LDS");
    db2 += __shfl_xor(db2, 32);
    dw3 += __shfl_xor(dw3, 32);
#pragma unroll
    for (int m = 16; m > 0; m >>= 1) { // both halves of the wave hold the same samples
        db3 += __shfl_xor(db3, m);
        loss += __shfl_xor(loss, m);
    }
    wave_lds_order();
    float *out = lds[wv];
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int i = mfma_row(r, h);
        out[MLP_W2 + i * MLP_H + j] = dw2[r];
    }
#pragma unroll
    for (int q = 0; q < 8; q++) { // D of 16x16: column lane % 16, row 4 (lane / 16) + q % 4
        const int i = 16 * (q >> 2) + 4 * (lane >> 4) + (q & 3), c = lane & 15;
        if (c < MLP_IN)
            out[MLP_W1 + i * MLP_IN + c] = dw1[q >> 2][q & 3];
        else if (c == MLP_IN)
            out[MLP_B1 + i] = dw1[q >> 2][q & 3];
    }
    if (h == 0) {
        out[MLP_B2 + j] = db2;
        out[MLP_W3 + j] = dw3;
    }
    if (lane == 0) {
        out[MLP_B3] = db3;
        out[MLP_NPARAM] = loss;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < MLP_OUT; i += 64 * W) {
        float v = lds[0][i];
#pragma unroll
        for (int k = 1; k < W; k++)
            v += lds[k][i];
        partial[(uint64_t)blockIdx.x * MLP_OUT + i] = v;
    }
}

// Sum of the blocks' partials in a fixed order (SUM_ROWS strided sums a
// parameter, then those in order) and the optional Adam step.  c1, c2: the
// bias corrections 1 / (1 - beta^step).  One thread per parameter walking
// 1024 partials took 231 us; the loads of a strided sum are independent, so
// this one is bound by their latency.
constexpr int SUM_PARAMS = 64, SUM_ROWS = 16;
__global__ void __launch_bounds__(SUM_PARAMS *SUM_ROWS)
k_mlp_sum_adam(const float *__restrict__ partial, uint32_t rows, float *__restrict__ grad, float *w, float *m,
               float *v, float c1, float c2, float lr, int adam)
{
    __shared__ float sums[SUM_ROWS][SUM_PARAMS];
    const int p = threadIdx.x % SUM_PARAMS, q = threadIdx.x / SUM_PARAMS;
    const int i = blockIdx.x * SUM_PARAMS + p;
    float g = 0.0f;
    // the step's own operands load with the partials
    const bool step = adam && q == 0 && i < MLP_NPARAM;
    const float m0 = step ? m[i] : 0.0f, v0 = step ? v[i] : 0.0f, w0 = step ? w[i] : 0.0f;
    if (i < MLP_OUT) {
        // MLP_GRAD_BLOCKS rows at most: a thread's loads are all in flight at once
        float t[MLP_GRAD_BLOCKS / SUM_ROWS];
#pragma unroll
        for (uint32_t b = 0; b < MLP_GRAD_BLOCKS / SUM_ROWS; b++)
            t[b] = q + b * SUM_ROWS < rows ? partial[(uint64_t)(q + b * SUM_ROWS) * MLP_OUT + i] : 0.0f;
#pragma unroll
        for (uint32_t b = 0; b < MLP_GRAD_BLOCKS / SUM_ROWS; b++)
            g += t[b];
    }
    sums[q][p] = g;
    __syncthreads();
    if (q != 0 || i >= MLP_OUT)
        return;
#pragma unroll
    for (int k = 1; k < SUM_ROWS; k++)
        g += sums[k][p];
    grad[i] = g;
    if (step) {
        const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
        const float mi = b1 * m0 + (1.0f - b1) * g;
        const float vi = b2 * v0 + (1.0f - b2) * g * g;
        m[i] = mi;
        v[i] = vi;
        w[i] = w0 - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
    }
}

// target[first + i] = values[i mod nx] for i < count.
__global__ void k_fill_plane_targets(float *__restrict__ target, uint64_t first, uint64_t count, uint32_t nx,
                                     const float *__restrict__ values)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count)
        target[first + i] = values[i % nx];
}

// Network outputs for samples [first, first+count) (evaluation), groups of 32
// samples to waves as in k_mlp_grad.
__global__ void __launch_bounds__(64 * MLP_WAVES)
k_mlp_predict(const float *__restrict__ w, const float *__restrict__ feat, uint32_t first, uint32_t count,
              float *__restrict__ out)
{
    const int lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
    MlpRegs n;
    n.load(w, j, h);
    const uint32_t groups = (count + GROUP - 1) / GROUP, waves = gridDim.x * MLP_WAVES;
    for (uint32_t g = blockIdx.x * MLP_WAVES + (threadIdx.x >> 6); g < groups; g += waves) {
        const uint32_t s = g * GROUP + j;
        float x[5];
#pragma unroll
        for (int t = 0; t < 5; t++)
            x[t] = s < count ? feat[((uint64_t)first + s) * MLP_IN + 5 * h + t] : 0.0f;
        mlp_float16 h1, h2;
        const float o = n.forward(x, h1, h2);
        if (h == 0 && s < count)
            out[s] = mlp_nut(w, o);
    }
}

} // namespace

template <int P>
hipError_t MlpLaunch<P>::filter(const FilterArgs &a, hipStream_t s)
{
    const uint32_t Nc = a.lxc * a.lyc * a.lzc;
    hipLaunchKernelGGL((k_filter<P>), dim3((Nc + 255) / 256), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t mlp_features(const FeatArgs &a, hipStream_t s)
{
    const uint32_t N = a.lx * a.ly * a.lz;
    hipLaunchKernelGGL(k_features, dim3((N + 255) / 256), dim3(256), 0, s, a);
    return hipGetLastError();
}

// One block per coarse x plane: FP64 sums of tau:S and S:S over the plane in
// a fixed order (strided per thread, then a fixed LDS tree), the plane's
// least-squares eddy viscosity, written to every node of the plane.
__global__ void __launch_bounds__(256) k_plane_targets(uint32_t lx, uint32_t ly, uint32_t lz,
                                                       const float *__restrict__ ts, const float *__restrict__ ss,
                                                       float nu, float *__restrict__ target, uint64_t offset)
{
    const uint32_t ix = blockIdx.x;
    const uint32_t rows = ly * lz;
    double a = 0.0, b = 0.0;
    for (uint32_t r = threadIdx.x; r < rows; r += 256) {
        const uint64_t n = ix + (uint64_t)lx * r;
        a += (double)ts[n];
        b += (double)ss[n];
    }
    __shared__ double sa[256], sb[256];
    sa[threadIdx.x] = a;
    sb[threadIdx.x] = b;
    __syncthreads();
    for (uint32_t h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) {
            sa[threadIdx.x] += sa[threadIdx.x + h];
            sb[threadIdx.x] += sb[threadIdx.x + h];
        }
        __syncthreads();
    }
    float y = sb[0] > 1e-30 ? (float)(-sa[0] / (2.0 * sb[0]) / (double)nu) : 0.0f;
    y = fminf(fmaxf(y, -10.0f), 10.0f);
    for (uint32_t r = threadIdx.x; r < rows; r += 256)
        target[offset + ix + (uint64_t)lx * r] = y;
}

hipError_t mlp_plane_targets(uint32_t lx, uint32_t ly, uint32_t lz, const float *ts, const float *ss, float nu,
                             float *target, uint64_t offset, hipStream_t s)
{
    hipLaunchKernelGGL(k_plane_targets, dim3(lx), dim3(256), 0, s, lx, ly, lz, ts, ss, nu, target, offset);
    return hipGetLastError();
}

// Blocks and waves per block of a gradient over `count` samples: a wave for
// every group of 32 up to a block of four waves per CU, beyond that blocks of
// eight, whose two waves per SIMD overlap matrix and vector instructions while
// the CU still writes one partial gradient; more than 65 536 samples take
// several groups a wave.  us an iteration with blocks of four waves, two per
// CU from 262 144 samples on / with these: 32 800 samples 14.0 / 13.5, 65 536
// 14.8 / 14.4, 131 072 22.2 / 21.3, 262 144 35.3 / 33.4, 524 288 59.2 / 57.6;
// 9.2 us of each are the two launches with their chains of loads.
struct MlpShape {
    uint32_t blocks, waves;
};
static MlpShape mlp_shape(uint32_t count)
{
    const uint32_t groups = (count + GROUP - 1) / GROUP;
    const uint32_t waves = groups <= 4 * MLP_GRAD_BLOCKS ? 4 : 8;
    return MlpShape{std::min<uint32_t>((groups + waves - 1) / waves, MLP_GRAD_BLOCKS), waves};
}

hipError_t mlp_grad(const float *w, const float *feat, const float *target, uint32_t first, uint32_t count,
                    float *partial, float *grad, float *wmut, float *m, float *v, int step, float lr, int adam,
                    hipStream_t s)
{
    const MlpShape sh = mlp_shape(count);
    // Adam's bias corrections, in double on the host
    const float c1 = (float)(1.0 / (1.0 - std::pow((double)0.9f, step)));
    const float c2 = (float)(1.0 / (1.0 - std::pow((double)0.999f, step)));
    if (sh.waves == 4)
        hipLaunchKernelGGL(k_mlp_grad<4>, dim3(sh.blocks), dim3(64 * 4), 0, s, w, feat, target, first, count, partial);
    else
        hipLaunchKernelGGL(k_mlp_grad<8>, dim3(sh.blocks), dim3(64 * 8), 0, s, w, feat, target, first, count, partial);
    hipLaunchKernelGGL(k_mlp_sum_adam, dim3((MLP_OUT + SUM_PARAMS - 1) / SUM_PARAMS), dim3(SUM_PARAMS * SUM_ROWS), 0, s,
                       partial, sh.blocks, grad, wmut, m, v, c1, c2, lr, adam);
    return hipGetLastError();
}

hipError_t mlp_fill_plane_targets(float *target, uint64_t first, uint64_t count, uint32_t nx, const float *values,
                                  hipStream_t s)
{
    hipLaunchKernelGGL(k_fill_plane_targets, dim3((uint32_t)((count + 255) / 256)), dim3(256), 0, s, target, first,
                       count, nx, values);
    return hipGetLastError();
}

hipError_t mlp_predict(const float *w, const float *feat, uint32_t first, uint32_t count, float *out, hipStream_t s)
{
    // a wave for every group up to two blocks of four per CU
    const uint32_t groups = (count + GROUP - 1) / GROUP;
    const uint32_t nb = std::min<uint32_t>((groups + MLP_WAVES - 1) / MLP_WAVES, 512);
    hipLaunchKernelGGL(k_mlp_predict, dim3(nb), dim3(64 * MLP_WAVES), 0, s, w, feat, first, count, out);
    return hipGetLastError();
}

template struct MlpLaunch<0>;
template struct MlpLaunch<1>;
template struct MlpLaunch<2>;
template struct MlpLaunch<3>;

} // namespace d3q19
