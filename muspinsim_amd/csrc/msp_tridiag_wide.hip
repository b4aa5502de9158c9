// Householder tridiagonalisation of a few large matrices, each spread over many
// workgroups (gfx950).
//
// Same reduction and output as k_tridiag_lp (A = Q T Q^H, reflector tails below
// the subdiagonal, d / e / tau out; only the lower triangle is read), two
// launches per column: k_tdw_matvec forms A22 v over 64 x 64 tiles of the lower
// triangle, k_tdw_vector (one workgroup per matrix, a thread per row) finishes
// column k's w and forms column k + 1's reflector.  The trailing update is
// deferred over panels of kNB columns and applied by the first matvec of the
// next panel as it reads the tiles, so a panel costs kNB reads and one write of
// the trailing triangle.  No workgroup waits for another inside a launch.
//
// A tile's row sums and column sums go to slots of their own (block row X,
// slot s: from tile (X, s) or, s > X, from the column side of tile (s, X)), so
// the order of every sum is fixed.
//
// Bound by the launches (6 us each, one after the other) for a few matrices and
// by HBM for many: with k_tdw_vector's share taken off, the tiles of 91 matrices
// of n = 1024 are read and written at 4.5 TB/s.  ms, one workgroup per matrix
// before -> here: n = 512, one matrix 15.6 -> 6.2, 42 matrices 16.4 -> 10.2;
// n = 768, one 51 -> 10.0, 84 58 -> 35; n = 1024, one 111 -> 14.4, 91 130 -> 80.
#include <hip/hip_runtime.h>

#include "msp_kernels.h"
#include "msp_team.h"
#include "msp_tridiag.h"

namespace {

constexpr int kNB = 8;      // panel width (two panel pairs fill the workspace's panel area)
constexpr int kT = 64;      // tile edge
static_assert(4 * kNB <= 2 * MSP_TD_NB, "two panel pairs of kNB columns in the panel area");

struct Wide {
    cdbl *part;     // nt x n: partial sums of A22 v by slot
    cdbl *nxt;      // n: column k + 1 at the start of its panel's updates
    cdbl *y;        // 2 kNB: Wp^H v, then Vp^H v
    cdbl *pan;      // two pairs (Vp, Wp), each kNB columns of n
};

// (the divide and conquer's arrays are free until it starts: at n > 256 its
// first 4 n^2 doubles hold the (n / 64 + 1) n partial sums many times over)
__device__ inline Wide wide_carve(int n, double *base)
{
    Wide w;
    w.part = (cdbl *)(base + 4 * (size_t)n);
    w.nxt = w.part + (size_t)((n + kT - 1) / kT) * n;
    w.y = w.nxt + n;
    w.pan = dc_panels(n, base);
    return w;
}

__device__ inline cdbl *panel_v(int n, cdbl *pan, int k) { return pan + (size_t)((k / kNB) & 1) * 2 * kNB * n; }

// Sums over the wave of 32 values per lane: lane l returns the total of value
// (l >> 1) (lane swaps halve the values at each level).
__device__ inline double wave_sum32(double (&x)[32], int lane)
{
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        swap32(x[i], x[i + 16]);
        x[i] += x[i + 16];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        swap16(x[i], x[i + 8]);
        x[i] += x[i + 8];
    }
    const bool b3 = lane & 8, b2 = lane & 4, b1 = lane & 2;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const double keep = b3 ? x[i + 4] : x[i], send = b3 ? x[i] : x[i + 4];
        x[i] = keep + dpp_f64<0x128, 0xF>(send);     // row_ror 8
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const double keep = b2 ? x[i + 2] : x[i], send = b2 ? x[i] : x[i + 2];
        x[i] = keep + dpp_f64<0x141, 0xF>(send);     // row_half_mirror
    }
    const double keep = b1 ? x[1] : x[0], send = b1 ? x[0] : x[1];
    const double v = keep + dpp_f64<0x4E, 0xF>(send);  // quad_perm [2,3,0,1]
    return v + dpp_f64<0xB1, 0xF>(v);                  // quad_perm [1,0,3,2]
}

// A22 v of column k.  Workgroups blockIdx.x < ny: the products of v with the
// panel's earlier columns, one per wave; the others: one 64 x 64 tile, wave w
// on rows 16 w .., lane on its column.  UPD: the previous panel's update is
// applied to the tile first and written back.
template <bool UPD>
__global__ void __launch_bounds__(256) k_tdw_matvec(int n, int k, int ny, double *H, double *work)
{
    __shared__ cdbl vr[kT], vc[kT], cpart[4][kT], rsum[kT];
    __shared__ cdbl prow[UPD ? 2 * kNB : 1][kT];
    const int b = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double *base = work + (size_t)b * dc_work_doubles(n);
    const Wide ws = wide_carve(n, base);
    const int j = k % kNB;
    const cdbl *Vp = panel_v(n, ws.pan, k);
    const cdbl *Wp = Vp + (size_t)kNB * n;
    const cdbl *v = Vp + (size_t)j * n;
    if ((int)blockIdx.x < ny) {
        const int l = 4 * blockIdx.x + wave;
        if (l >= 2 * j) return;
        const cdbl *M = (l < j) ? Wp + (size_t)l * n : Vp + (size_t)(l - j) * n;
        double sr = 0.0, si = 0.0;
#pragma unroll 4
        for (int i = k + 1 + lane; i < n; i += 64) {
            const cdbl t = cmulc(M[i], v[i]);
            sr += t.re;
            si += t.im;
        }
        sr = wave_sum_all(sr);
        si = wave_sum_all(si);
        if (lane == 0) ws.y[l] = cmk(sr, si);
        return;
    }
    // tile (I, J), J <= I, of the blocks from tb on
    const int tb = (k + 1) / kT;
    const int t = blockIdx.x - ny;
    int I = (int)((sqrtf(8.0f * t + 1.0f) - 1.0f) * 0.5f);
    while (I * (I + 1) / 2 > t) --I;
    while ((I + 1) * (I + 2) / 2 <= t) ++I;
    const int J = tb + t - I * (I + 1) / 2;
    I += tb;
    cdbl *A = (cdbl *)H + (size_t)b * n * n;
    const int i0 = kT * I + 16 * wave, c = kT * J + lane;
    cdbl a[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int i = (i0 + u < n) ? i0 + u : n - 1;
        a[u] = A[(size_t)i * n + ((c <= i) ? c : i)];
    }
    if (tid < 2 * kT) {
        const int i = kT * (tid < kT ? I : J) + lane;
        (tid < kT ? vr : vc)[lane] = (i < n) ? v[i] : cmk(0.0, 0.0);
    }
    cdbl pc[UPD ? 2 * kNB : 1];
    if constexpr (UPD) {
        const cdbl *P = panel_v(n, ws.pan, k - 1);       // Vp, then Wp
        for (int idx = tid; idx < 2 * kNB * kT; idx += 256) {
            const int i = kT * I + (idx & 63);
            prow[idx >> 6][idx & 63] = P[(size_t)(idx >> 6) * n + (i < n ? i : n - 1)];
        }
        const int cc = (c < n) ? c : n - 1;
#pragma unroll
        for (int l = 0; l < 2 * kNB; ++l) pc[l] = cconj(P[(size_t)l * n + cc]);
    }
    __syncthreads();
    const cdbl vl = vc[lane];
    cdbl col = cmk(0.0, 0.0);
    double x[32];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int i = i0 + u;
        const bool use = i < n && c > k && c <= i;       // (c <= i, c > k: so is i)
        cdbl e = a[u];
        if constexpr (UPD) {
#pragma unroll
            for (int l = 0; l < kNB; ++l) {
                e = csub(e, cmul(prow[l][16 * wave + u], pc[kNB + l]));
                e = csub(e, cmul(prow[kNB + l][16 * wave + u], pc[l]));
            }
            if (use) A[(size_t)i * n + c] = e;
        }
        if (!use) e = cmk(0.0, 0.0);
        if (use && c == k + 1) ws.nxt[i] = e;
        x[2 * u] = e.re * vl.re - e.im * vl.im;
        x[2 * u + 1] = e.re * vl.im + e.im * vl.re;
        if (c != i) cfmac(col, e, vr[16 * wave + u]);
    }
    const double r = wave_sum32(x, lane);
    if ((lane & 1) == 0) ((double *)rsum)[32 * wave + (lane >> 1)] = r;
    cpart[wave][lane] = col;
    __syncthreads();
    if (wave == 0) {
        cdbl s = cadd(cadd(cpart[0][lane], cpart[1][lane]), cadd(cpart[2][lane], cpart[3][lane]));
        if (I == J) s = cadd(s, rsum[lane]);
        if (c < n) ws.part[(size_t)I * n + c] = s;
    } else if (wave == 1 && I != J) {
        const int i = kT * I + lane;
        if (i < n) ws.part[(size_t)J * n + i] = rsum[lane];
    }
}

// Block sum of two doubles per thread over nw waves (red: 2 x 16 doubles).
__device__ inline void block_sum2(double &a, double &b, double *red, int wave, int lane, int nw)
{
    a = wave_sum_all(a);
    b = wave_sum_all(b);
    if (lane == 0) {
        red[wave] = a;
        red[16 + wave] = b;
    }
    __syncthreads();
    a = red[0];
    b = red[16];
    for (int w = 1; w < nw; ++w) {
        a += red[w];
        b += red[16 + w];
    }
}

// Column k's w = p - (tau / 2)(p^H v) v with p = tau (A22 v - Vp y1 - Wp y2)
// (k = -1: none), then column k + 1 brought up to date and its reflector.  One
// thread per row from the row block of k + 1 on; both corrections by the
// panel's earlier columns are formed in one pass over them.
__global__ void __launch_bounds__(1024) k_tdw_vector(int n, int k, double *H, double *E, double *work)
{
    __shared__ double red[2][32];
    __shared__ cdbl pub[3];          // v and w at row k + 1, the next column at row k + 2
    const int b = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
    cdbl *A = (cdbl *)H + (size_t)b * n * n;
    double *base = work + (size_t)b * dc_work_doubles(n);
    const Wide ws = wide_carve(n, base);
    double *e;
    cdbl *tau;
    dc_carve(n, base, &e, &tau);
    double *d = E + (size_t)b * n;
    const int k1 = k + 1;
    const int tb = k1 / kT, nt = (n + kT - 1) / kT;
    const int i = kT * tb + tid;
    const bool on = i >= k1 && i < n;
    const int ic = (i < n) ? i : n - 1;
    cdbl col;
    if (k < 0) {
        col = A[(size_t)ic * n];
    } else {
        const int j = k % kNB;
        cdbl *Vp = panel_v(n, ws.pan, k);
        cdbl *Wp = Vp + (size_t)kNB * n;
        const cdbl v = on ? Vp[(size_t)j * n + ic] : cmk(0.0, 0.0);
        const cdbl tk = tau[k];
        col = ws.nxt[ic];
        cdbl acc = cmk(0.0, 0.0);
#pragma unroll 4
        for (int s = tb; s < nt; ++s) acc = cadd(acc, ws.part[(size_t)s * n + ic]);
#pragma unroll 2
        for (int l = 0; l < j; ++l) {
            const cdbl vi = Vp[(size_t)l * n + ic], wi = Wp[(size_t)l * n + ic];
            acc = csub(acc, cmul(vi, ws.y[l]));
            acc = csub(acc, cmul(wi, ws.y[j + l]));
            col = csub(col, cmul(vi, cconj(Wp[(size_t)l * n + k1])));
            col = csub(col, cmul(wi, cconj(Vp[(size_t)l * n + k1])));
        }
        acc = on ? cmul(tk, acc) : cmk(0.0, 0.0);
        const cdbl pv = cmulc(acc, v);
        double sr = pv.re, si = pv.im;
        block_sum2(sr, si, red[0], wave, lane, nw);
        const cdbl a2 = cmul(cmk(-0.5 * tk.re, -0.5 * tk.im), cmk(sr, si));
        const cdbl w = cadd(acc, cmul(a2, v));
        if (on) Wp[(size_t)j * n + i] = w;
        if (i == k1) {
            pub[0] = v;
            pub[1] = w;
        }
        __syncthreads();
        col = csub(col, cmul(v, cconj(pub[1])));
        col = csub(col, cmul(w, cconj(pub[0])));
    }
    if (i == k1) d[k1] = col.re;
    if (k1 == n - 1) return;
    if (i == k1 + 1) pub[2] = col;
    double xn2 = (i >= k1 + 2 && i < n) ? cabs2(col) : 0.0, zero = 0.0;
    block_sum2(xn2, zero, red[1], wave, lane, nw);
    // reflector of A[k1 + 1.., k1], as k_tridiag_lp forms it
    const cdbl alpha = pub[2];
    double beta;
    cdbl tk, scale;
    if (xn2 == 0.0 && alpha.im == 0.0) {
        tk = cmk(0.0, 0.0);
        beta = alpha.re;
        scale = cmk(0.0, 0.0);
    } else {
        const double nrm = sqrt(alpha.re * alpha.re + alpha.im * alpha.im + xn2);
        beta = alpha.re >= 0.0 ? -nrm : nrm;
        const double ib = msp_recip(beta);
        tk = cmk((beta - alpha.re) * ib, -alpha.im * ib);
        const cdbl dd = cmk(alpha.re * ib - 1.0, alpha.im * ib);
        const double id = ib * msp_recip(dd.re * dd.re + dd.im * dd.im);
        scale = cmk(dd.re * id, -dd.im * id);
    }
    const bool act = tk.re != 0.0 || tk.im != 0.0;
    const cdbl v1 = !act || i <= k1 ? cmk(0.0, 0.0) : i == k1 + 1 ? cmk(1.0, 0.0) : cmul(col, scale);
    if (i < n) {
        (panel_v(n, ws.pan, k1) + (size_t)(k1 % kNB) * n)[i] = v1;
        if (i >= k1 + 2) A[(size_t)i * n + k1] = v1;
    }
    if (i == k1) {
        e[k1] = beta;
        tau[k1] = tk;
    }
}

}  // namespace

// 2 n - 1 launches; every workgroup ends by itself.  n <= 1024 (one thread per row).
hipError_t launch_tridiag_wide(int n, int batch, double *H, double *E, double *work, hipStream_t s)
{
    if (n > 1024) return hipErrorNotSupported;
    const int nt = (n + kT - 1) / kT;
    for (int k = -1; k < n - 1; ++k) {
        const int nb = nt - (k + 1) / kT;
        if (k >= 0) {
            const int ny = (2 * (k % kNB) + 3) / 4;
            const dim3 grid(ny + nb * (nb + 1) / 2, batch);
            if (k > 0 && k % kNB == 0)
                hipLaunchKernelGGL(k_tdw_matvec<true>, grid, dim3(256), 0, s, n, k, ny, H, work);
            else
                hipLaunchKernelGGL(k_tdw_matvec<false>, grid, dim3(256), 0, s, n, k, ny, H, work);
        }
        hipLaunchKernelGGL(k_tdw_vector, dim3(batch), dim3(kT * nb), 0, s, n, k, H, E, work);
    }
    return hipGetLastError();
}
