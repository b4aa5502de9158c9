// Adjoint (vector-Jacobian product) of the fast-path muon polarisation
//   P_b(t) = (1/4d) sum_jk |O_jk|^2 cos(2 pi (E_j - E_k) t),  O = U^H sigma U,
// with respect to the Hamiltonian, for fitting (the reference fits by finite
// differences, muspinsim/fitting.py:99-105).  For upstream weights r_b(t) =
// dL/dP_b(t), L = sum_bt r_b(t) P_b(t) has the eigenbasis gradient G'
// (dL = Re tr(G' U^H dH U)):
//   G'_jj = -(pi/d) sum_k |O_jk|^2 S_jk                      (eigenvalue part)
//   G'_jm = (1/2d) Y_jm / (E_j - E_m),  Y = [R o O, O]       (eigenvector part)
//   G'_jm = (1/2d) sum_k O_jk O_km (-2 pi S_jk)  for E_j ~ E_m (the limit of
//           the divided difference, so degenerate levels are well defined)
// with R_jk = sum_t r(t) cos(w_jk t), S_jk = sum_t r(t) t sin(w_jk t),
// w_jk = 2 pi (E_j - E_k).  G = U G' U^H, summed over instances, gives
// dL/dtheta = Re tr(G dH/dtheta) for any parameter of the field-independent H.
#include <hip/hip_runtime.h>

#include "msp_kernels.h"
#include "msp_mfma.h"
#include "msp_team.h"

namespace {

constexpr int kTile = 64;        // (j, k) tile edge
constexpr int kTC = 8;           // times per chunk
constexpr int kLd = kTile + 16;  // row stride of the LDS phases (two rows cover all banks)
constexpr int kPairs = 16;       // k_adjoint_freq_pairs: (j, k) tile edge
constexpr int kPairTimes = 64;   // and times per chunk

// R and S of one 64 x 64 tile (j0 <= k0) of one instance, and of its mirror
// (R symmetric, S antisymmetric): with w_jk = w_j - w_k both are sums over times
// of products of one-index phases,
//   R_jk = sum_t (r c_j) c_k + (r s_j) s_k,
//   S_jk = sum_t (r t s_j) c_k - (r t c_j) s_k,
// so they run on FP64 MFMA (four products per k-step and 16 x 16 tile).  Eight
// waves: two groups of four take alternate chunks of 8 times (each forms its
// chunk's phases in LDS, group wave v owns rows 16 v of the tile) and are added
// at the end.  Bound by the phases' sine and cosine and the matrix products
// about equally at one workgroup per instance.  n = 64, 2000 times, 256
// instances: 1.51 ms with a thread per (j, k) and the phases of a 16 x 16 tile
// formed per tile (each phase eight times over), 0.42 here.
__global__ void __launch_bounds__(512) k_adjoint_freq(int n, int ntimes, const double *E,
                                                      const double *times, const double *r,
                                                      const int32_t *slot, const double *w,
                                                      double scale, double *R, double *S)
{
    // per group: c, s of the tile's rows and of its columns, [time][index]
    __shared__ double ph[2][4][kTC * kLd];
    __shared__ double rt[2][kTC], tt[2][kTC];
    const int b = blockIdx.y;
    // tile of the upper triangle
    int jt = 0, rest = blockIdx.x;
    const int nt = (n + kTile - 1) / kTile;
    while (rest >= nt - jt) {
        rest -= nt - jt;
        ++jt;
    }
    const int j0 = jt * kTile, k0 = (jt + rest) * kTile;
    const bool diag = j0 == k0;
    const int tid = threadIdx.x & 255;
    const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, li = lane & 15, lq = lane >> 4;
    const double *Eb = E + (size_t)b * n;
    const double Ec = 0.5 * (Eb[0] + Eb[n - 1]);
    const double *rb = r + (size_t)(slot ? slot[b] : 0) * ntimes;
    const double twopi = 6.283185307179586;
    double(*P)[kTC * kLd] = ph[grp];
    const double *Ck = P[diag ? 0 : 2], *Sk = P[diag ? 1 : 3];
    msp_d4 aR[4], aS[4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) aR[ct] = aS[ct] = d4zero();
    const bool rows = j0 + 16 * wave < n;
    for (int c0 = 0; c0 < ntimes; c0 += 2 * kTC) {
        const int t0 = c0 + kTC * grp;
        __syncthreads();
        if (tid < kTC) {
            const int t = t0 + tid;
            rt[grp][tid] = t < ntimes ? rb[t] : 0.0;
            tt[grp][tid] = t < ntimes ? times[t] : 0.0;
        }
        // thread: index tid % 64 of the rows (then of the columns), four times
        for (int side = 0; side < (diag ? 1 : 2); ++side) {
            const int idx = (side ? k0 : j0) + (tid & 63);
            const double e = idx < n ? twopi * (Eb[idx] - Ec) : 0.0;
#pragma unroll
            for (int u = 0; u < kTC / 4; ++u) {
                const int c = (tid >> 6) + 4 * u, t = t0 + c;
                double sn = 0.0, cs = 0.0;
                if (idx < n && t < ntimes) sincos(e * times[t], &sn, &cs);
                P[2 * side][c * kLd + (tid & 63)] = cs;
                P[2 * side + 1][c * kLd + (tid & 63)] = sn;
            }
        }
        __syncthreads();
        if (!rows) continue;
#pragma unroll
        for (int h = 0; h < kTC / 4; ++h) {
            const int c = 4 * h + lq;
            const double rc = rt[grp][c], rtc = rc * tt[grp][c];
            const double cj = P[0][c * kLd + 16 * wave + li], sj = P[1][c * kLd + 16 * wave + li];
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) {
                if (k0 + 16 * ct >= n) break;
                const double ck = Ck[c * kLd + 16 * ct + li], sk = Sk[c * kLd + 16 * ct + li];
                aR[ct] = mfma_f64(rc * cj, ck, aR[ct]);
                aS[ct] = mfma_f64(rtc * sj, ck, aS[ct]);
                aR[ct] = mfma_f64(rc * sj, sk, aR[ct]);
                aS[ct] = mfma_f64(-rtc * cj, sk, aS[ct]);
            }
        }
    }
    // group 1's sums to group 0 through the phases' place, R and then S
    double *sum = &ph[0][0][0];
    static_assert(sizeof(ph) >= sizeof(double) * kTile * kTile, "a tile of sums fits");
    const double f = scale * (w ? w[b] : 1.0);
    double *Rb = R + (size_t)b * n * n, *Sb = S + (size_t)b * n * n;
#pragma unroll
    for (int part = 0; part < 2; ++part) {
        __syncthreads();
        if (grp == 1 && rows) {
#pragma unroll
            for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    sum[(16 * wave + 4 * q + lq) * kTile + 16 * ct + li] = part ? aS[ct][q] : aR[ct][q];
        }
        __syncthreads();
        if (grp == 1 || !rows) continue;
#pragma unroll
        for (int ct = 0; ct < 4; ++ct)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j = j0 + 16 * wave + 4 * q + lq, k = k0 + 16 * ct + li;
                if (j >= n || k >= n) continue;
                const double other = sum[(16 * wave + 4 * q + lq) * kTile + 16 * ct + li];
                if (part == 0) {
                    const double v = f * (aR[ct][q] + other);
                    Rb[(size_t)j * n + k] = v;
                    if (!diag) Rb[(size_t)k * n + j] = v;
                } else {
                    const double v = f * (aS[ct][q] + other);
                    Sb[(size_t)j * n + k] = j == k ? 0.0 : v;
                    if (!diag) Sb[(size_t)k * n + j] = -v;
                }
            }
    }
}

// The same by one thread per (j, k), a workgroup per 16 x 16 tile: for few
// instances, over which the tiles above would leave most CUs idle.
__global__ void __launch_bounds__(256) k_adjoint_freq_pairs(int n, int ntimes, const double *E,
                                                            const double *times, const double *r,
                                                            const int32_t *slot, const double *w,
                                                            double scale, double *R, double *S)
{
    __shared__ cdbl Pj[kPairs][kPairTimes + 1];
    __shared__ cdbl Pk[kPairs][kPairTimes + 1];
    __shared__ double rt[kPairTimes], tt[kPairTimes];
    const int b = blockIdx.z;
    const int j0 = blockIdx.y * kPairs, k0 = blockIdx.x * kPairs;
    const int tid = threadIdx.x, jj = tid / kPairs, kk = tid % kPairs;
    const double *Eb = E + (size_t)b * n;
    const double Ec = 0.5 * (Eb[0] + Eb[n - 1]);
    const double *rb = r + (size_t)(slot ? slot[b] : 0) * ntimes;
    const double twopi = 6.283185307179586;
    double sr = 0.0, ss = 0.0;
    for (int t0 = 0; t0 < ntimes; t0 += kPairTimes) {
        __syncthreads();
        for (int l = tid; l < kPairTimes; l += 256) {
            const int t = t0 + l;
            rt[l] = (t < ntimes) ? rb[t] : 0.0;
            tt[l] = (t < ntimes) ? times[t] : 0.0;
        }
        for (int l = tid; l < 2 * kPairs * kPairTimes; l += 256) {
            const int which = l / (kPairs * kPairTimes), rem = l % (kPairs * kPairTimes);
            const int a = rem / kPairTimes, c = rem % kPairTimes;
            const int t = t0 + c;
            const int idx = (which ? k0 : j0) + a;
            double sn = 0.0, cs = 1.0;
            if (idx < n && t < ntimes) sincos(twopi * (Eb[idx] - Ec) * times[t], &sn, &cs);
            if (which) Pk[a][c] = cmk(cs, sn);
            else Pj[a][c] = cmk(cs, sn);
        }
        __syncthreads();
        const int lim = (ntimes - t0 < kPairTimes) ? ntimes - t0 : kPairTimes;
        for (int c = 0; c < lim; ++c) {
            // exp(i w_jk t) = Pj conj(Pk)
            const cdbl pj = Pj[jj][c], pk = Pk[kk][c];
            const double re = pj.re * pk.re + pj.im * pk.im;
            const double im = pj.im * pk.re - pj.re * pk.im;
            sr = fma(rt[c], re, sr);
            ss = fma(rt[c] * tt[c], im, ss);
        }
    }
    const int j = j0 + jj, k = k0 + kk;
    if (j < n && k < n) {
        const double f = scale * (w ? w[b] : 1.0);
        R[(size_t)b * n * n + (size_t)j * n + k] = f * sr;
        S[(size_t)b * n * n + (size_t)j * n + k] = f * ss;
    }
}

// M = R o O (elementwise, R real, O complex)
__global__ void k_hadamard_real(int n, int batch, const double *R, const double *O, double *M)
{
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)batch * n * n) return;
    ((cdbl *)M)[e] = cscale(((const cdbl *)O)[e], R[e]);
}

// G'_jm from Y = M O - O M, the eigenvalues, S and O (see the file header);
// the result is made Hermitian, G' <- (G' + G'^H)/2, which leaves Re tr(G' D)
// unchanged for Hermitian D.
__global__ void k_adjoint_gprime(int n, int batch, const double *E, const double *O,
                                 const double *MO, const double *OM, const double *S, double d,
                                 double degtol, double *G)
{
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)batch * n * n) return;
    const int b = (int)(e / ((size_t)n * n));
    const int jm = (int)(e % ((size_t)n * n));
    const int j = jm / n, m = jm % n;
    const double *Eb = E + (size_t)b * n;
    const cdbl *Ob = (const cdbl *)O + (size_t)b * n * n;
    const double *Sb = S + (size_t)b * n * n;
    const double twopi = 6.283185307179586;
    const double scaleE = fmax(fabs(Eb[0]), fabs(Eb[n - 1]));
    cdbl g[2];
    // entry (j, m) and its mirror (m, j), averaged conjugated
    for (int side = 0; side < 2; ++side) {
        const int p = side ? m : j, q = side ? j : m;
        cdbl v;
        if (p == q) {
            double a = 0.0;
            for (int k = 0; k < n; ++k) a += cabs2(Ob[(size_t)p * n + k]) * Sb[(size_t)p * n + k];
            v = cmk(-0.5 * twopi / d * a, 0.0);
        } else {
            const double dE = Eb[p] - Eb[q];
            if (fabs(dE) > degtol * fmax(scaleE, 1.0)) {
                const size_t o = (size_t)b * n * n + (size_t)p * n + q;
                const cdbl y = csub(((const cdbl *)MO)[o], ((const cdbl *)OM)[o]);
                v = cscale(y, 0.5 / (d * dE));
            } else {
                cdbl acc = cmk(0.0, 0.0);
                for (int k = 0; k < n; ++k)
                    acc = cadd(acc, cscale(cmul(Ob[(size_t)p * n + k], Ob[(size_t)k * n + q]),
                                           -twopi * Sb[(size_t)p * n + k]));
                v = cscale(acc, 0.5 / d);
            }
        }
        g[side] = v;
    }
    // G'_jm <- (G'_jm + conj(G'_mj)) / 2
    ((cdbl *)G)[e] = cscale(cadd(g[0], cconj(g[1])), 0.5);
}

// out[i] = sum_b X[b][i] (deterministic order), complex
__global__ void k_batch_sum(int len, int batch, const double *X, double *out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= len) return;
    cdbl acc = cmk(0.0, 0.0);
    for (int b = 0; b < batch; ++b) acc = cadd(acc, ((const cdbl *)X)[(size_t)b * len + i]);
    ((cdbl *)out)[i] = cadd(((cdbl *)out)[i], acc);
}

// out[p] = Re sum_ab G_ab dH_p[b][a], one workgroup per parameter
__global__ void __launch_bounds__(256) k_trace_products(int n, const double *G, const double *dH,
                                                        double *out)
{
    __shared__ double red[8];
    const int p = blockIdx.x;
    const cdbl *Gm = (const cdbl *)G;
    const cdbl *D = (const cdbl *)dH + (size_t)p * n * n;
    double s = 0.0;
    for (int idx = threadIdx.x; idx < n * n; idx += 256) {
        const int a = idx / n, c = idx % n;
        const cdbl g = Gm[idx], h = D[(size_t)c * n + a];
        s += g.re * h.re - g.im * h.im;
    }
    s = team_sum(s, red);
    if (threadIdx.x == 0) out[p] = s;
}

inline unsigned cdivu(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

}  // namespace

hipError_t launch_adjoint_freq(int n, int batch, int ntimes, const double *E, const double *times,
                               const double *r, const int32_t *slot, const double *w, double scale,
                               double *R, double *S, hipStream_t s)
{
    ProfScope ps_("k_adjoint_freq", s);
    // The matrix form has one workgroup per 64 x 64 tile of an instance's upper
    // triangle, the thread-per-pair form one per 16 x 16 tile of all of it: the
    // first is ahead once the second's workgroups fill the chip about 4.5 times
    // over (2.8 times up to n = 48, where it forms fewer phases twice), and never
    // when n fits one small tile.  ms pairs / matrix form, 1000 times: n = 16, 512
    // instances 0.12 / 0.19; n = 32, 128 0.091 / 0.090, 256 0.18 / 0.12; n = 64, 48
    // 0.14 / 0.17, 96 0.28 / 0.18; n = 128, 16 0.21 / 0.24, 24 0.32 / 0.25; n = 256, 4
    // 0.22 / 0.24, 8 0.41 / 0.25; n = 64, one instance, 4000 times 0.37 / 0.70
    const unsigned np = cdivu(n, kPairs);
    const size_t pair_wgs = (size_t)np * np * batch;
    if (n <= kPairs || pair_wgs <= (n <= 48 ? 720 : 1152)) {
        hipLaunchKernelGGL(k_adjoint_freq_pairs, dim3(np, np, batch), dim3(256), 0, s, n, ntimes, E,
                           times, r, slot, w, scale, R, S);
        return hipGetLastError();
    }
    const unsigned nt = cdivu(n, kTile);
    hipLaunchKernelGGL(k_adjoint_freq, dim3(nt * (nt + 1) / 2, batch), dim3(512), 0, s, n, ntimes, E, times, r, slot, w,
                       scale, R, S);
    return hipGetLastError();
}

hipError_t launch_hadamard_real(int n, int batch, const double *R, const double *O, double *M,
                                hipStream_t s)
{
    ProfScope ps_("k_hadamard_real", s);
    hipLaunchKernelGGL(k_hadamard_real, dim3(cdivu((size_t)batch * n * n, 256)), dim3(256), 0, s,
                       n, batch, R, O, M);
    return hipGetLastError();
}

hipError_t launch_adjoint_gprime(int n, int batch, const double *E, const double *O,
                                 const double *MO, const double *OM, const double *S, double d,
                                 double degtol, double *G, hipStream_t s)
{
    ProfScope ps_("k_adjoint_gprime", s);
    hipLaunchKernelGGL(k_adjoint_gprime, dim3(cdivu((size_t)batch * n * n, 256)), dim3(256), 0, s,
                       n, batch, E, O, MO, OM, S, d, degtol, G);
    return hipGetLastError();
}

hipError_t launch_batch_sum(int len, int batch, const double *X, double *out, hipStream_t s)
{
    ProfScope ps_("k_batch_sum", s);
    hipLaunchKernelGGL(k_batch_sum, dim3(cdivu(len, 256)), dim3(256), 0, s, len, batch, X, out);
    return hipGetLastError();
}

hipError_t launch_trace_products(int n, int nparam, const double *G, const double *dH, double *out,
                                 hipStream_t s)
{
    ProfScope ps_("k_trace_products", s);
    hipLaunchKernelGGL(k_trace_products, dim3(nparam), dim3(256), 0, s, n, G, dH, out);
    return hipGetLastError();
}
