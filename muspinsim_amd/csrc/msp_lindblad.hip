// Lindbladian path on gfx950 (muspinsim/lindbladian.py:19-173):
//
//   k_liouvillian     L = -i (H (x) 1 - 1 (x) H^T)
//                         + sum_k g_k (A_k (x) A_k* - 1/2 (A_k^H A_k (x) 1 + 1 (x) (A_k^H A_k)^T))
//                     on row-major vec(rho), one workgroup per instance
//   k_lindblad_modes  eigendecomposition L = V diag(lambda) V^{-1} (msp_nonsym.h) and
//                     the mode amplitudes amp_km = (u_k^T V)_m (V^{-1} r)_m; the
//                     matrix lives in LDS when N <= 64, else in global memory
//                     (kSplitMinN <= N <= 64 without V, up to N = 20 for batches
//                     of at most 2048: the same steps in three
//                     launches, k_lindblad_hess, _schur and _amps)
//   k_mode_sum        P_k(t) = sum_m amp_km exp(2 pi lambda_m t)
//   k_mode_integral   I_k = sum_m amp_km / (1/tau - 2 pi lambda_m)
//   k_mode_states     rho(t) = V (c exp(2 pi lambda t)) (states without operators)
#include <hip/hip_runtime.h>

#include "msp_kernels.h"
#include "msp_nonsym.h"

namespace {

constexpr int kNT = 256;
constexpr int kLdsMaxN = 64;    // N at or below this keeps L and Z in LDS
constexpr int kSplitMinN = 16;  // from here to kLdsMaxN the three-launch form runs without V
constexpr int kSplitMaxOps = 3; // and up to this many operators
constexpr int kSplitSmallN = 20;      // up to here only for batches of at most this many:
constexpr int kSplitSmallBatch = 2048;

__global__ void __launch_bounds__(kNT) k_liouvillian(int n, const double *H, int n_jump,
                                                     const double *Aj, const double *rate,
                                                     double *Lout)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int b = blockIdx.x;
    const int N = n * n;
    cdbl *Hs = (cdbl *)smem;                 // n x n
    cdbl *M = Hs + N;                        // n x n: sum_k g_k A_k^H A_k
    const cdbl *Hb = (const cdbl *)H + (size_t)b * N;
    const cdbl *Ab = (const cdbl *)Aj + (size_t)b * n_jump * N;
    const double *gb = rate + (size_t)b * n_jump;
    MSP_PFOR(idx, N)
    {
        Hs[idx] = Hb[idx];
        const int a = idx / n, c = idx - (idx / n) * n;
        cdbl s = cmk(0.0, 0.0);
        for (int k = 0; k < n_jump; ++k) {
            const cdbl *A = Ab + (size_t)k * N;
            cdbl t = cmk(0.0, 0.0);
            for (int m = 0; m < n; ++m) cfmac(t, A[m * n + a], A[m * n + c]);
            s = cadd(s, cscale(t, gb[k]));
        }
        M[idx] = s;
    }
    __syncthreads();
    cdbl *L = (cdbl *)Lout + (size_t)b * N * N;
    // element ((a,b2),(c,d)) at row a*n+b2, column c*n+d
    for (size_t e = threadIdx.x; e < (size_t)N * N; e += kNT) {
        const int row = (int)(e / N), col = (int)(e - (e / N) * N);
        const int a = row / n, b2 = row - (row / n) * n;
        const int c = col / n, d = col - (col / n) * n;
        cdbl v = cmk(0.0, 0.0);
        // -i (H_ac delta_bd - delta_ac H_db)
        cdbl h = cmk(0.0, 0.0);
        if (b2 == d) h = Hs[a * n + c];
        if (a == c) h = csub(h, Hs[d * n + b2]);
        v = cmk(h.im, -h.re);
        // dissipators
        for (int k = 0; k < n_jump; ++k) {
            const cdbl *A = Ab + (size_t)k * N;
            v = cadd(v, cscale(cmul(A[a * n + c], cconj(A[b2 * n + d])), gb[k]));
        }
        if (b2 == d) v = csub(v, cscale(M[a * n + c], 0.5));
        if (a == c) v = csub(v, cscale(M[d * n + b2], 0.5));
        L[e] = v;
    }
}

// Per-instance scratch of the modes kernel: vectors v, w, y, t, r, u (N each),
// plus Z (N x N) when the matrix is not in LDS.
__host__ __device__ inline size_t modes_vec_elems(int N) { return 6 * (size_t)N; }

// NT threads per instance: one wave when the matrix is in LDS (N <= 64: a
// sweep step's rows and columns are one element per lane, and the phase
// boundaries are those of a single wave), four above.  LDS and VMODE are
// template parameters so that the LDS form's pointers derive from the LDS
// block alone and compile to LDS instructions (a pointer that may be LDS or
// global is accessed with slower flat instructions).  VMODE (LDS, no
// eigenvectors to return): Z^H r and u_q^T Z are carried through the
// reduction instead of Z, which halves the LDS.
template <int NT, bool LDS, bool VMODE>
__global__ void __launch_bounds__(NT) k_lindblad_modes(int N, double *Lg, const double *r,
                                                       int n_ops, const double *u, double *lam,
                                                       double *amp, double *cout, double *Vout,
                                                       int32_t *info, double *work, int max_its)
{
    static_assert(LDS || !VMODE, "the vector form is the LDS form");
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double red[NT];
    const int b = blockIdx.x;
    cdbl *A, *Z, *vec;
    int ld;
    constexpr bool vmode = VMODE;
    if constexpr (LDS) {
        ld = N + 1;
        A = (cdbl *)smem;
        Z = vmode ? nullptr : A + (size_t)N * ld;
        vec = vmode ? A + (size_t)N * ld : Z + (size_t)N * ld;
        const cdbl *Lb = (const cdbl *)Lg + (size_t)b * N * N;
        MSP_PFOR(idx, N * N)
        {
            const int i = idx / N, j = idx - (idx / N) * N;
            A[i * ld + j] = Lb[idx];
        }
    } else {
        ld = N;
        A = (cdbl *)Lg + (size_t)b * N * N;
        cdbl *wb = (cdbl *)work + (size_t)b * ((size_t)N * N + modes_vec_elems(N));
        Z = wb;
        vec = wb + (size_t)N * N;
    }
    cdbl *v = vec, *w = vec + N, *y = vec + 2 * N, *t = vec + 3 * N, *rv = vec + 4 * N,
         *lv = vec + 5 * N;
    ModeVecs mv{nullptr, nullptr, 0};
    if (vmode) {
        mv.rho = rv;
        mv.omega = vec + 6 * N;
        mv.n_omega = n_ops;
        MSP_PFOR(i, N) rv[i] = ((const cdbl *)r)[(size_t)b * N + i];
        MSP_PFOR(i, n_ops * N) mv.omega[i] = ((const cdbl *)u)[(size_t)b * n_ops * N + i];
    }
    MSP_SYNC();
    hessenberg_team(N, A, ld, Z, ld, v, w, red, mv);
    const int st = schur_team(N, A, ld, Z, ld, lv, max_its, red, mv);
    if (threadIdx.x == 0) info[b] = st;
    if (st != 0) return;                      // uniform across the workgroup
    schur_vectors_team(N, A, ld, lv);
    if (!vmode) {
        MSP_PFOR(i, N) rv[i] = ((const cdbl *)r)[(size_t)b * N + i];
        MSP_SYNC();
    }
    modes_coeff_team(N, A, ld, Z, ld, rv, y);          // y = c
    for (int k = 0; k < n_ops; ++k) {
        const cdbl *uk = vmode ? mv.omega + (size_t)k * N : rv;
        if (!vmode) {
            MSP_PFOR(i, N) rv[i] = ((const cdbl *)u)[((size_t)b * n_ops + k) * N + i];
            MSP_SYNC();
        }
        modes_proj_team(N, A, ld, Z, ld, uk, t, w);    // w = o
        MSP_PFOR(m, N) ((cdbl *)amp)[((size_t)b * n_ops + k) * N + m] = cmul(w[m], y[m]);
        MSP_SYNC();
    }
    MSP_PFOR(m, N)
    {
        ((cdbl *)lam)[(size_t)b * N + m] = lv[m];
        if (cout) ((cdbl *)cout)[(size_t)b * N + m] = y[m];
    }
    if (Vout) {
        modes_vectors_team(N, A, ld, Z, ld);
        cdbl *Vb = (cdbl *)Vout + (size_t)b * N * N;
        MSP_PFOR(idx, N * N)
        {
            const int i = idx / N, j = idx - (idx / N) * N;
            Vb[idx] = Z[i * ld + j];
        }
    }
}

// ---------------------------------------------------------------------------
// The same decomposition for kSplitMinN <= N <= 64 when no eigenvectors are
// wanted, in three launches, each with the layout its step needs.  The one
// launch above holds the N x N matrix in LDS throughout (two one-wave instances
// per CU at N = 64) and pays a chain of LDS round trips per Givens rotation.
// ms per 1024 / 4096 random matrices, one launch against three (hess + schur +
// amps): N = 64 14.5 / 56.9 against 5.1 / 17.4 (2.3 + 14.0 + 0.9), 36 2.6 / 8.5
// against 1.3 / 4.5, 16 0.62 / 1.03 against 0.37 / 0.99; N = 9 0.23 / 0.36
// against 0.17 / 0.43, which keeps the one launch.  1024 Liouvillians of a
// relaxing electron (N = 64): 8.4 against 3.2.  Up to N = 20 the one launch holds
// enough instances per CU to hide its round trips once there are many: N = 17,
// 2048 matrices 0.76 / 0.76, 4096 1.09 / 1.19; 2048 Liouvillians of N = 16 0.47 /
// 0.45, 4096 0.67 / 0.71; N = 21, 4096 matrices 2.2 / 1.7.

__device__ inline cdbl lane_c(cdbl v, int l) { return cmk(readlane_f64(v.re, l), readlane_f64(v.im, l)); }

// Sums over the 64 lanes of 16 doubles per lane, halving the values held per
// step (by swaps of lane halves and rows, then by selects at the row mirror
// and the half-row mirror), then plain sums.  Lane l returns the total of
// value 8 b5 + 4 b4 + 2 b3 + b2 with b the bits of l.
__device__ inline double wave_sum16(double (&x)[16], int lane)
{
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        swap32(x[j], x[j + 8]);
        x[j] += x[j + 8];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        swap16(x[j], x[j + 4]);
        x[j] += x[j + 4];
    }
    const bool h3 = lane & 8, h2 = lane & 4;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const double send = h3 ? x[j] : x[j + 2];
        x[j] = (h3 ? x[j + 2] : x[j]) + dpp_f64<0x140, 0xF>(send);   // row_mirror
    }
    const double send = h2 ? x[0] : x[1];
    double t = (h2 ? x[1] : x[0]) + dpp_f64<0x141, 0xF>(send);       // row_half_mirror
    t += dpp_f64<0x4E, 0xF>(t);                                      // quad_perm [2,3,0,1]
    return t + dpp_f64<0xB1, 0xF>(t);                                // quad_perm [1,0,3,2]
}

// Hessenberg reduction, four waves per instance, the matrix in registers:
// lane j holds column j, slot a of wave p row 4 a + p (N <= 4 kRows).  Step k forms y = A v
// (16 rows per wave, butterflies over the lanes) and z = v^H A (per lane, added
// over the waves in LDS) from the same A and applies both sides of
// H^H A H, H = I - tau v v^H, as one rank-2 update
//   A -= v (conj(tau) z) + (tau y - |tau|^2 (z v) v) v^H.
// The annihilated entries are not cleared: nothing reads them again (v is zero
// at finished columns).  rho = Q^H r goes to lam, omega_q = u_q^T Q to amp.
template <int kRows>
__global__ void __launch_bounds__(256, 2) k_lindblad_hess(int N, double *Lg, const double *r,
                                                          int n_ops, const double *u, double *lam,
                                                          double *amp)
{
    extern __shared__ __align__(16) unsigned char smem[];
    cdbl *vec = (cdbl *)smem;                  // rho, then omega_q: 64 each
    __shared__ cdbl col[64], vb[4][64], part[4][64], yb[64], sub[64];
    const int b = blockIdx.x, lane = threadIdx.x & 63;
    const int p = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    cdbl *L = (cdbl *)Lg + (size_t)b * N * N;
    const bool inj = lane < N;
    cdbl A[kRows];
#pragma unroll
    for (int a = 0; a < kRows; ++a) {
        const int i = 4 * a + p;
        A[a] = (i < N && inj) ? L[(size_t)i * N + lane] : cmk(0.0, 0.0);
    }
    // each vector belongs to one wave, each entry to one lane
    for (int q = p; q < 1 + n_ops; q += 4) {
        const cdbl *src = q == 0 ? (const cdbl *)r + (size_t)b * N
                                 : (const cdbl *)u + ((size_t)b * n_ops + q - 1) * N;
        vec[64 * q + lane] = inj ? src[lane] : cmk(0.0, 0.0);
    }
    for (int k = 0; k + 2 < N; ++k) {
        if (lane == k) {
#pragma unroll
            for (int a = 0; a < kRows; ++a) col[4 * a + p] = A[a];
        }
        __syncthreads();
        // the reflector, in every wave; tau = 0 (v = 0) leaves A as it is
        const cdbl x = inj ? col[lane] : cmk(0.0, 0.0), alpha = col[k + 1];
        const double xn2 = wave_sum_all(lane > k + 1 ? cabs2(x) : 0.0);
        cdbl tau = cmk(0.0, 0.0), scal = tau;
        double beta = alpha.re, one = 0.0;
        if (!(xn2 == 0.0 && alpha.im == 0.0)) {
            const double nrm = sqrt(alpha.re * alpha.re + alpha.im * alpha.im + xn2);
            beta = alpha.re >= 0.0 ? -nrm : nrm;
            tau = cmk((beta - alpha.re) / beta, -alpha.im / beta);
            scal = cdivc(cmk(1.0, 0.0), cmk(alpha.re - beta, alpha.im));
            one = 1.0;
        }
        const cdbl v = lane > k + 1 ? cmul(x, scal) : cmk(lane == k + 1 ? one : 0.0, 0.0);
        if (threadIdx.x == 0) sub[k] = cmk(beta, 0.0);
        vb[p][lane] = v;                       // this wave's copy: no barrier
        cdbl z = cmk(0.0, 0.0);
#pragma unroll
        for (int hf = 0; hf < (kRows + 7) / 8; ++hf) {
            double s[16];
#pragma unroll
            for (int a = 0; a < 8; ++a) {
                s[2 * a] = s[2 * a + 1] = 0.0;
                if (8 * hf + a >= kRows) continue;
                const cdbl m = A[8 * hf + a];
                cfmac(z, vb[p][4 * (8 * hf + a) + p], m);
                s[2 * a] = fma(m.re, v.re, -m.im * v.im);
                s[2 * a + 1] = fma(m.re, v.im, m.im * v.re);
            }
            const double t = wave_sum16(s, lane);
            const int vi = lane >> 2;          // 2 a + (re, im)
            if (!(lane & 3) && 8 * hf + (vi >> 1) < kRows)
                ((double *)yb)[2 * (4 * (8 * hf + (vi >> 1)) + p) + (vi & 1)] = t;
        }
        part[p][lane] = z;
        // vectors of this wave: rho -= conj(tau) (v^H rho) v, omega -= tau (omega v) v^H
        for (int q = p; q < 1 + n_ops; q += 4) {
            const cdbl m = vec[64 * q + lane];
            cdbl t = q == 0 ? cmulc(v, m) : cmul(m, v);
            t = cmk(wave_sum_all(t.re), wave_sum_all(t.im));
            vec[64 * q + lane] = q == 0 ? csub(m, cmul(v, cmul(cconj(tau), t)))
                                        : csub(m, cmul(cmul(t, tau), cconj(v)));
        }
        __syncthreads();
        z = cmk(0.0, 0.0);
#pragma unroll
        for (int w = 0; w < 4; ++w) z = cadd(z, part[w][lane]);
        cdbl zv = cmul(z, v);
        zv = cmk(wave_sum_all(zv.re), wave_sum_all(zv.im));
        const cdbl g = cscale(zv, cabs2(tau)), ze = cmul(cconj(tau), z);
#pragma unroll
        for (int a = 0; a < kRows; ++a) {
            const cdbl va = vb[p][4 * a + p];
            const cdbl ua = csub(cmul(tau, yb[4 * a + p]), cmul(g, va));
            cdbl m = A[a];
            m.re = fma(-va.re, ze.re, m.re);
            m.im = fma(-va.re, ze.im, m.im);
            m.re = fma(va.im, ze.im, m.re);
            m.im = fma(-va.im, ze.re, m.im);
            m.re = fma(-ua.re, v.re, m.re);
            m.im = fma(ua.re, v.im, m.im);
            m.re = fma(-ua.im, v.im, m.re);
            m.im = fma(-ua.im, v.re, m.im);
            A[a] = m;
        }
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < kRows; ++a) {
        const int i = 4 * a + p;
        cdbl m = A[a];
        if (i == lane + 1 && lane < N - 2) {
            m.re = sub[lane].re;
            m.im = 0.0;
        }
        if (i < N && inj && i <= lane + 1) L[(size_t)i * N + lane] = m;
    }
    for (int q = p; q < 1 + n_ops; q += 4)
        if (inj)
            ((cdbl *)(q == 0 ? lam : amp))[(q == 0 ? (size_t)b : (size_t)b * n_ops + q - 1) * N + lane] =
                vec[64 * q + lane];
}

// Packed upper Hessenberg storage: entry (r, j), j >= r - 1, at base(r) + j.
__device__ inline int uh_base(int N, int r)
{
    return r == 0 ? 0 : N + (r - 1) * (N + 1) - r * (r - 1) / 2 - (r - 1);
}
__host__ __device__ inline size_t uh_elems(int N)
{
    return (size_t)N + (size_t)(N - 1) * (N + 1) - (size_t)N * (N - 1) / 2;
}

// c a + s b and c b - conj(s) a
__device__ inline cdbl rot_first(double c, cdbl s, cdbl a, cdbl b)
{
    return cmk(fma(c, a.re, fma(s.re, b.re, -s.im * b.im)), fma(c, a.im, fma(s.re, b.im, s.im * b.re)));
}
__device__ inline cdbl rot_second(double c, cdbl s, cdbl a, cdbl b)
{
    return cmk(fma(c, b.re, -fma(s.re, a.re, s.im * a.im)), fma(c, b.im, -fma(s.re, a.im, -s.im * a.re)));
}

// One DPP move of a double; lanes without a source keep `old`.
template <int CTRL, int ROWMASK>
__device__ inline double dpp_keep(double old, double v)
{
    const long long x = __double_as_longlong(v), o = __double_as_longlong(old);
    int lo = (int)(x & 0xffffffffll), hi = (int)(x >> 32);
    lo = __builtin_amdgcn_update_dpp((int)(o & 0xffffffffll), lo, CTRL, ROWMASK, 0xF, false);
    hi = __builtin_amdgcn_update_dpp((int)(o >> 32), hi, CTRL, ROWMASK, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
// One step of an inclusive scan of the affine maps x -> a x + b over the lanes.
template <int CTRL, int ROWMASK>
__device__ inline void affine_step(cdbl &a, cdbl &b)
{
    const cdbl a1 = cmk(dpp_keep<CTRL, ROWMASK>(1.0, a.re), dpp_keep<CTRL, ROWMASK>(0.0, a.im));
    const cdbl b1 = cmk(dpp_keep<CTRL, ROWMASK>(0.0, b.re), dpp_keep<CTRL, ROWMASK>(0.0, b.im));
    cfma(b, a, b1);
    a = cmul(a, a1);
}
// Rotations k = l .. ihi - 1 (lane k holds c and s of rotation k) applied in
// turn to the lane-distributed vector m: (m_k, m_{k+1}) <- (c m_k + s m_{k+1},
// c m_{k+1} - conj(s) m_k).  The entry carried from one rotation to the next
// obeys an affine recurrence, summed by a scan over the lanes instead of step
// by step.  buf: 64 entries of LDS.
__device__ inline cdbl rotate_vector(cdbl m, double c, cdbl s, int l, int ihi, int lane, cdbl *buf)
{
    buf[lane] = m;
    NS_SYNC();
    const cdbl mn = buf[min(lane + 1, 63)], ml = buf[l];
    const bool in = lane >= l && lane < ihi;
    cdbl a = in ? cmk(-s.re, s.im) : cmk(1.0, 0.0);
    cdbl b = in ? cscale(mn, c) : cmk(0.0, 0.0);
    affine_step<0x111, 0xF>(a, b);             // row_shr 1, 2, 4, 8
    affine_step<0x112, 0xF>(a, b);
    affine_step<0x114, 0xF>(a, b);
    affine_step<0x118, 0xF>(a, b);
    affine_step<0x142, 0xA>(a, b);             // row_bcast15 -> rows 1, 3
    affine_step<0x143, 0xC>(a, b);             // row_bcast31 -> rows 2, 3
    cfma(b, a, ml);                            // carried entry after rotation `lane`
    NS_SYNC();
    buf[lane] = b;
    NS_SYNC();
    const cdbl ca = lane > l ? buf[max(lane - 1, 0)] : ml;
    NS_SYNC();
    if (lane == ihi) return ca;
    return in ? cadd(cscale(ca, c), cmul(s, mn)) : m;
}

// Upper Hessenberg H (in L) -> Schur form T, one wave per instance, by explicit
// single-shift QR sweeps: H - sigma = Q R by row rotations (lane = column, the
// carried row in registers, the next rows prefetched), then R Q + sigma by
// column rotations (lane = row, the carried column in registers).  A rotation
// then depends on the one before only through registers and lane reads, not
// through LDS round trips; rotation k is kept by lane k between the passes.
// Shifts, deflation test and exceptional shifts are those of schur_team.  The
// matrix is scaled by a power of two to a largest entry near 1 (so that the
// rotations need no scaling of their own) and packed (34 KB at N = 64), four
// instances per CU, one on each SIMD.  T goes to L's upper triangle, rho and
// omega_q (in lam and amp) are rotated along.
// What bounds it: about 500 cycles per rotation in the row pass and 330 in the
// column pass of one wave per SIMD (dependent FP64 operations), and the slowest
// instance of the launch (1.6 times the mean).
template <int NOPS>
__global__ void __launch_bounds__(64) k_lindblad_schur(int N, double *Lg, int n_ops, double *lam,
                                                       double *amp, int32_t *info, int max_its)
{
    extern __shared__ __align__(16) unsigned char smem[];
    cdbl *S = (cdbl *)smem, *buf = S + uh_elems(N);
    const int b = blockIdx.x, lane = threadIdx.x;
    const int jl = min(lane, N - 1);           // lanes past N shadow the last
    const bool inj = lane < N;
    cdbl *L = (cdbl *)Lg + (size_t)b * N * N;
    double big = 0.0;
    for (int i = 0; i < N; ++i)
        if (jl >= i - 1) {
            const cdbl m = L[(size_t)i * N + jl];
            big = fmax(big, fmax(fabs(m.re), fabs(m.im)));
        }
    big = ns_team_max(big, nullptr);
    int ex = 0;
    if (big > 0.0 && big < INFINITY) (void)frexp(big, &ex);
    for (int i = 0; i < N; ++i)
        if (inj && lane >= i - 1) {
            const cdbl m = L[(size_t)i * N + lane];
            S[uh_base(N, i) + lane] = cmk(ldexp(m.re, -ex), ldexp(m.im, -ex));
        }
    cdbl rho = ((const cdbl *)lam)[(size_t)b * N + jl];
    cdbl om[NOPS];
#pragma unroll
    for (int q = 0; q < NOPS; ++q)
        om[q] = q < n_ops ? ((const cdbl *)amp)[((size_t)b * n_ops + q) * N + jl] : cmk(0.0, 0.0);
    NS_SYNC();

    const double ulp = 1.1102230246251565e-16;
    const double smlnum = 2.2250738585072014e-308 * ((double)N / ulp);
    const int bl = uh_base(N, jl), bl1 = uh_base(N, max(jl - 1, 0));
    int ihi = N - 1, its = 0, total = 0, st = 0;
    while (ihi >= 0) {
        // split point: largest l <= ihi with a negligible subdiagonal entry
        bool neg = false;
        if (lane >= 1 && lane <= ihi) {
            const double sb = cabs1(S[bl + lane - 1]);
            double tst = cabs1(S[bl1 + lane - 1]) + cabs1(S[bl + lane]);
            if (tst == 0.0) {
                if (lane >= 2) tst += fabs(S[bl1 + lane - 2].re);
                if (lane + 1 <= ihi) tst += fabs(S[uh_base(N, lane + 1) + lane].re);
            }
            neg = sb <= smlnum || sb <= ulp * tst;
        }
        const unsigned long long nm = __ballot(neg);
        const int l = nm ? 63 - __builtin_clzll(nm) : 0;
        if (l > 0 && lane == l) S[bl + l - 1] = cmk(0.0, 0.0);
        if (l == ihi) {
            --ihi;
            its = 0;
            continue;
        }
        if (++total > max_its * N) {
            st = ihi + 1;
            break;
        }
        NS_SYNC();
        cdbl sft;
        {
            const int bi = uh_base(N, ihi), bi1 = uh_base(N, ihi - 1);
            if (its == 10) {
                const cdbl a = S[uh_base(N, l) + l];
                sft = cmk(a.re + 0.75 * fabs(S[uh_base(N, l + 1) + l].re), a.im);
            } else if (its == 20) {
                const cdbl a = S[bi + ihi];
                sft = cmk(a.re + 0.75 * fabs(S[bi + ihi - 1].re), a.im);
            } else {
                // eigenvalue of the trailing 2 x 2 block closest to its last diagonal
                const cdbl a = S[bi1 + ihi - 1], bb = S[bi1 + ihi];
                const cdbl c = S[bi + ihi - 1], d = S[bi + ihi];
                const cdbl hm = cscale(csub(a, d), 0.5);
                const cdbl disc = cadd(cmul(hm, hm), cmul(bb, c));
                const double m = sqrt(cabs2(disc));
                double sr = sqrt(0.5 * (m + fabs(disc.re)));
                double si = (sr > 0.0) ? 0.5 * disc.im / sr : 0.0;
                if (disc.re < 0.0) {
                    const double t = sr;
                    sr = fabs(si);
                    si = (disc.im >= 0.0) ? t : -t;
                }
                const cdbl e1 = cmk(hm.re - sr, hm.im - si), e2 = cmk(hm.re + sr, hm.im + si);
                sft = cadd(d, (cabs1(e1) <= cabs1(e2)) ? e1 : e2);
            }
        }
        ++its;

        // H - sigma in the window
        const bool win = lane >= l && lane <= ihi;
        if (win) S[bl + lane] = csub(S[bl + lane], sft);
        NS_SYNC();

        // rows: H - sigma = Q R.  Row k + 1 enters at step k; lanes left of a
        // row's first entry hold values that nothing uses.
        double cv = 1.0;
        cdbl sv = cmk(0.0, 0.0);               // rotation of step `lane`
        int bk = uh_base(N, l);
        cdbl x = S[bk + jl];
        int bn = bk + N - l;                   // base(l + 1)
        cdbl y = S[bn + jl];
        for (int k = l; k < ihi; ++k) {
            const int bn2 = bn + N - k - 1;    // base(k + 2)
            const cdbl yn = S[(k + 2 <= ihi ? bn2 : bn) + jl];
            const cdbl f = lane_c(x, k), g = lane_c(y, k);
            // c = |f| / nrm, s = f conj(g) / (|f| nrm)
            const double f2 = cabs2(f), g2 = cabs2(g);
            // (the usual case computed straight through and the test put after
            // it, so that the serial chain does not wait for a branch)
            const bool usual = f2 * g2 > 1e-280;
            const double inv = ns_rsqrt(f2 * (f2 + g2));
            double c = f2 * inv;
            cdbl s = cscale(cmul(f, cconj(g)), inv);
            cdbl t = rot_first(c, s, x, y), xn = rot_second(c, s, x, y);
            asm volatile("" : "+v"(t.re), "+v"(t.im), "+v"(xn.re), "+v"(xn.im));
            if (!usual) {
                cdbl rr;
                givens(f, g, c, s, rr);
                t = rot_first(c, s, x, y);
                xn = rot_second(c, s, x, y);
            }
            x = xn;
            // (lanes with nothing to store write to buf: without a branch the
            // prefetch above is not waited for together with this store)
            *(inj && lane >= k ? S + bk + lane : buf + lane) = t;
            if (lane == k) {
                cv = c;
                sv = s;
            }
            bk = bn;
            bn = bn2;
            y = yn;
        }
        if (inj && lane >= ihi) S[bk + lane] = x;
        if (lane > l && lane <= ihi) S[bl + lane - 1] = cmk(0.0, 0.0);
        rho = rotate_vector(rho, cv, sv, l, ihi, lane, buf);
#pragma unroll
        for (int q = 0; q < NOPS; ++q) om[q] = rotate_vector(om[q], cv, cconj(sv), l, ihi, lane, buf);
        NS_SYNC();

        // columns: R Q, rows 0 .. ihi
        cdbl pc = lane <= l ? S[bl + l] : cmk(0.0, 0.0);
        cdbl qc = S[bl + l + 1];
        for (int k = l; k < ihi; ++k) {
            const cdbl qn = S[bl + (k + 2 <= ihi ? k + 2 : k + 1)];
            if (lane > k + 1) qc = cmk(0.0, 0.0);
            const double c = readlane_f64(cv, k);
            const cdbl s = lane_c(sv, k);
            // [p q] <- [c p + conj(s) q, -s p + c q]
            const cdbl t = rot_first(c, cconj(s), pc, qc);
            pc = rot_second(c, cconj(s), pc, qc);
            *(lane <= k + 1 ? S + bl + k : buf + lane) = t;
            qc = qn;
        }
        if (lane <= ihi) S[bl + ihi] = pc;
        NS_SYNC();
        // back from H - sigma
        if (win) S[bl + lane] = cadd(S[bl + lane], sft);
        NS_SYNC();
    }
    if (lane == 0) info[b] = st;
    if (st != 0) return;
    for (int i = 0; i < N; ++i)
        if (inj && lane >= i) {
            const cdbl m = S[uh_base(N, i) + lane];
            L[(size_t)i * N + lane] = cmk(ldexp(m.re, ex), ldexp(m.im, ex));
        }
    if (!inj) return;
    ((cdbl *)lam)[(size_t)b * N + lane] = rho;
#pragma unroll
    for (int q = 0; q < NOPS; ++q)
        if (q < n_ops) ((cdbl *)amp)[((size_t)b * n_ops + q) * N + lane] = om[q];
}

// Eigenvectors of T, lambda, c = X^-1 rho and the amplitudes, one wave per
// instance (T from L, rho from lam, omega_q from amp).
__global__ void __launch_bounds__(64) k_lindblad_amps(int N, const double *Lg, int n_ops,
                                                      double *lam, double *amp, double *cout,
                                                      const int32_t *info)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int b = blockIdx.x, ld = N + 1;
    if (info[b] != 0) return;                  // uniform across the workgroup
    cdbl *A = (cdbl *)smem, *lv = A + (size_t)N * ld, *y = lv + N, *t = y + N, *w = t + N, *om = w + N;
    const cdbl *L = (const cdbl *)Lg + (size_t)b * N * N;
    for (int i = 0; i < N; ++i)
        for (int j = i + (int)threadIdx.x; j < N; j += 64) A[i * ld + j] = L[(size_t)i * N + j];
    MSP_PFOR(i, N) om[i] = ((const cdbl *)lam)[(size_t)b * N + i];
    MSP_SYNC();
    MSP_PFOR(i, N) lv[i] = A[i * ld + i];
    MSP_SYNC();
    schur_vectors_team(N, A, ld, lv);
    modes_coeff_team(N, A, ld, nullptr, 0, om, y);          // y = c
    for (int k = 0; k < n_ops; ++k) {
        cdbl *ak = (cdbl *)amp + ((size_t)b * n_ops + k) * N;
        MSP_PFOR(i, N) om[i] = ak[i];
        MSP_SYNC();
        modes_proj_team(N, A, ld, nullptr, 0, om, t, w);    // w = o
        MSP_PFOR(m, N) ak[m] = cmul(w[m], y[m]);
        MSP_SYNC();
    }
    MSP_PFOR(m, N)
    {
        ((cdbl *)lam)[(size_t)b * N + m] = lv[m];
        if (cout) ((cdbl *)cout)[(size_t)b * N + m] = y[m];
    }
}

// exp(2 pi lambda t)
__device__ inline cdbl mode_phase(cdbl l, double t)
{
    const double mag = exp(6.283185307179586 * l.re * t);
    // the phase in turns, reduced exactly, needs no range reduction by pi
    const double turn = l.im * t;
    double sn, cs;
    sincospi(2.0 * (turn - rint(turn)), &sn, &cs);
    return cmk(mag * cs, mag * sn);
}

// one thread per (instance, operator, time)
__global__ void k_mode_sum(int N, int batch, int n_ops, int ntimes, const double *lam,
                           const double *amp, const double *times, const double *w,
                           int out_complex, double *out)
{
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t total = (size_t)batch * n_ops * ntimes;
    if (e >= total) return;
    const int ti = (int)(e % ntimes);
    const size_t bk = e / ntimes;
    const int b = (int)(bk / n_ops);
    const cdbl *l = (const cdbl *)lam + (size_t)b * N;
    const cdbl *a = (const cdbl *)amp + bk * N;
    const double tt = times[ti];
    cdbl s = cmk(0.0, 0.0);
    for (int m = 0; m < N; ++m) s = cadd(s, cmul(a[m], mode_phase(l[m], tt)));
    if (out_complex) ((cdbl *)out)[e] = s;
    else out[e] = (w ? w[b] : 1.0) * s.re;
}

__global__ void k_mode_integral(int N, int batch, int n_ops, const double *lam, const double *amp,
                                double tau, double out_scale, const double *w, int out_complex,
                                double *out)
{
    const int bk = blockIdx.x * blockDim.x + threadIdx.x;
    if (bk >= batch * n_ops) return;
    const int b = bk / n_ops;
    const cdbl *l = (const cdbl *)lam + (size_t)b * N;
    const cdbl *a = (const cdbl *)amp + (size_t)bk * N;
    const double twopi = 6.283185307179586;
    cdbl s = cmk(0.0, 0.0);
    for (int m = 0; m < N; ++m)
        s = cadd(s, cdivc(a[m], cmk(1.0 / tau - twopi * l[m].re, -twopi * l[m].im)));
    s = cscale(s, out_scale);
    if (out_complex) ((cdbl *)out)[bk] = s;
    else out[bk] = (w ? w[b] : 1.0) * s.re;
}

// out[t][i] = sum_m V_im c_m exp(2 pi lambda_m t), one instance
__global__ void k_mode_states(int N, int ntimes, const double *lam, const double *c,
                              const double *V, const double *times, double *out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int ti = blockIdx.y;
    if (i >= N || ti >= ntimes) return;
    const cdbl *l = (const cdbl *)lam, *cc = (const cdbl *)c, *Vm = (const cdbl *)V;
    cdbl s = cmk(0.0, 0.0);
    for (int m = 0; m < N; ++m)
        s = cadd(s, cmul(Vm[(size_t)i * N + m], cmul(cc[m], mode_phase(l[m], times[ti]))));
    ((cdbl *)out)[(size_t)ti * N + i] = s;
}

inline unsigned cdivu(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

}  // namespace

size_t lindblad_modes_workspace(int N, int batch)
{
    if (N <= kLdsMaxN) return 0;
    return sizeof(cdbl) * ((size_t)N * N + modes_vec_elems(N)) * (size_t)batch;
}

hipError_t launch_liouvillian(int n, int batch, const double *H, int n_jump, const double *A,
                              const double *rate, double *L, hipStream_t s)
{
    const size_t lds = sizeof(cdbl) * 2 * (size_t)n * n;
    ProfScope ps_("k_liouvillian", s);
    hipLaunchKernelGGL(k_liouvillian, dim3(batch), dim3(kNT), lds, s, n, H, n_jump, A, rate, L);
    return hipGetLastError();
}

hipError_t launch_lindblad_modes(int N, int batch, double *L, const double *r, int n_ops,
                                 const double *u, double *lam, double *amp, double *c, double *V,
                                 int32_t *info, double *work, int max_its, hipStream_t s)
{
    if (N >= kSplitMinN && N <= kLdsMaxN && !V && n_ops <= kSplitMaxOps &&
        (N > kSplitSmallN || batch <= kSplitSmallBatch)) {
        ProfScope ps_("k_lindblad_modes", s);
        const size_t lh = sizeof(cdbl) * 64 * (1 + (size_t)n_ops), ls = sizeof(cdbl) * (uh_elems(N) + 64);
        const size_t la = sizeof(cdbl) * ((size_t)N * (N + 1) + 5 * (size_t)N);
        hipError_t err = msp_set_lds((const void *)k_lindblad_amps, la);
        if (err != hipSuccess) return err;
        if (N <= 16)
            hipLaunchKernelGGL((k_lindblad_hess<4>), dim3(batch), dim3(256), lh, s, N, L, r, n_ops, u, lam, amp);
        else if (N <= 40)
            hipLaunchKernelGGL((k_lindblad_hess<10>), dim3(batch), dim3(256), lh, s, N, L, r, n_ops, u, lam, amp);
        else
            hipLaunchKernelGGL((k_lindblad_hess<16>), dim3(batch), dim3(256), lh, s, N, L, r, n_ops, u, lam, amp);
        if (n_ops <= 1)
            hipLaunchKernelGGL((k_lindblad_schur<1>), dim3(batch), dim3(64), ls, s, N, L, n_ops, lam,
                               amp, info, max_its);
        else
            hipLaunchKernelGGL((k_lindblad_schur<kSplitMaxOps>), dim3(batch), dim3(64), ls, s, N, L,
                               n_ops, lam, amp, info, max_its);
        hipLaunchKernelGGL(k_lindblad_amps, dim3(batch), dim3(64), la, s, N, L, n_ops, lam, amp, c, info);
        return hipGetLastError();
    }
    const int in_lds = N <= kLdsMaxN;
    // (without V the LDS form holds the matrix, the vectors and the n_ops rows
    // u_q^T Z, not Z)
    const size_t lds = !in_lds ? 0
                       : V ? sizeof(cdbl) * (2 * (size_t)N * (N + 1) + modes_vec_elems(N))
                           : sizeof(cdbl) * ((size_t)N * (N + 1) + modes_vec_elems(N) + (size_t)n_ops * N);
    const void *fn = !in_lds ? (const void *)k_lindblad_modes<kNT, false, false>
                     : V     ? (const void *)k_lindblad_modes<64, true, false>
                             : (const void *)k_lindblad_modes<64, true, true>;
    hipError_t err = msp_set_lds(fn, lds);
    if (err != hipSuccess) return err;
    ProfScope ps_("k_lindblad_modes", s);
    if (!in_lds)
        hipLaunchKernelGGL((k_lindblad_modes<kNT, false, false>), dim3(batch), dim3(kNT), lds, s, N, L,
                           r, n_ops, u, lam, amp, c, V, info, work, max_its);
    else if (V)
        hipLaunchKernelGGL((k_lindblad_modes<64, true, false>), dim3(batch), dim3(64), lds, s, N, L, r,
                           n_ops, u, lam, amp, c, V, info, work, max_its);
    else
        hipLaunchKernelGGL((k_lindblad_modes<64, true, true>), dim3(batch), dim3(64), lds, s, N, L, r,
                           n_ops, u, lam, amp, c, V, info, work, max_its);
    return hipGetLastError();
}

hipError_t launch_mode_sum(int N, int batch, int n_ops, int ntimes, const double *lam,
                           const double *amp, const double *times, const double *w,
                           int out_complex, double *out, hipStream_t s)
{
    const size_t total = (size_t)batch * n_ops * ntimes;
    ProfScope ps_("k_mode_sum", s);
    hipLaunchKernelGGL(k_mode_sum, dim3(cdivu(total, 256)), dim3(256), 0, s, N, batch, n_ops,
                       ntimes, lam, amp, times, w, out_complex, out);
    return hipGetLastError();
}

hipError_t launch_mode_integral(int N, int batch, int n_ops, const double *lam, const double *amp,
                                double tau, double out_scale, const double *w, int out_complex,
                                double *out, hipStream_t s)
{
    ProfScope ps_("k_mode_integral", s);
    hipLaunchKernelGGL(k_mode_integral, dim3(cdivu((size_t)batch * n_ops, 256)), dim3(256), 0, s,
                       N, batch, n_ops, lam, amp, tau, out_scale, w, out_complex, out);
    return hipGetLastError();
}

hipError_t launch_mode_states(int N, int ntimes, const double *lam, const double *c,
                              const double *V, const double *times, double *out, hipStream_t s)
{
    ProfScope ps_("k_mode_states", s);
    hipLaunchKernelGGL(k_mode_states, dim3(cdivu(N, 256), ntimes), dim3(256), 0, s, N, ntimes,
                       lam, c, V, times, out);
    return hipGetLastError();
}
