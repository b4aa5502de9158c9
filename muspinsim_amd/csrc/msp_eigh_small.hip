// Hermitian eigensolver for n <= 16: cyclic Jacobi, one wave for one matrix
// (n > 8), four (n > 4) or sixteen.  Reads the lower triangle only; no workspace.
//
// A round rotates the N / 2 disjoint pairs of a round-robin tournament on N = n
// (or n + 1) indices at once: lane (i, j) forms the rotations of pairs i and j
// itself, from the diagonal and pair elements in LDS, applies both to its 2 x 2
// block of A (rows of pair i, columns of pair j), and pair j's to rows 2 i and
// 2 i + 1 of V.  No lane waits for another's rotation and the wave needs no
// barrier; N - 1 rounds are a sweep.
//
// What bounds it: the latency of a round, about 1000 cycles for some 190
// instructions of one wave (an LDS round trip, the two square roots of a
// rotation, 72 FMAs a lane), times about eight sweeps.
// ms for 256 / 16384 random matrices, the LDS Jacobi kernel (a workgroup per
// matrix, three barriers a round), the tridiagonal pipeline, and this one:
//   n = 16 0.165 / 1.48, 0.140 / 3.48, 0.075 / 0.88
//   n = 12 0.121 / 0.90, 0.119 / 2.77, 0.055 / 0.56
//   n = 8  0.070 / 0.43, 0.081 / 1.85, 0.032 / 0.12
//   n = 4  0.024 / 0.14, 0.056 / 0.89, 0.013 / 0.02
// and for n = 24 and 32 the pipeline is ahead (two or four blocks a lane).
// Measured and not taken: the register-resident reduction, implicit QL and
// back-transformation in one wave (n = 16 0.095 / 0.90, n = 12 0.059 / 0.54: 400
// cycles a QL rotation, one after the other); incremental row pointers
// (n = 12 0.62 against 0.56 ms).
#include <hip/hip_runtime.h>

#include "msp_kernels.h"
#include "msp_team.h"

namespace {

// 1/sqrt(t): hardware estimate and two Newton steps, each adding a small
// correction to y.  The product y (1.5 - t y^2 / 2) of the same length rounds its
// factor near one instead and is biased: at n = 16 the squared norms of the
// vectors were off by -2.2e-15 on average (+6e-16 so, LDS Jacobi +1.6e-15), the
// eigenvalues by 3.7e-16 ||H|| rms (2.1e-16 so, LDS Jacobi 2.0e-16).
__device__ inline double small_rsqrt(double t)
{
    double y = __builtin_amdgcn_rsq(t);
    const double h = 0.5 * t;
    y = fma(y, fma(-h * y, y, 0.5), y);
    return fma(y, fma(-h * y, y, 0.5), y);
}

// a wave executes LDS operations in order: the compiler must keep them so
__device__ inline void wave_sync() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// Rotation J = [c s; -conj(s) c] with J^H [alpha beta; conj(beta) gamma] J
// diagonal, of the smaller angle; the identity (and false) for |beta|^2 <= skip.
// The new diagonal is alpha - shift, gamma + shift: with the small shift added,
// instead of the products of the rotation rounded at full size, a diagonal stops
// moving once its rotations are small (error of zero-field series at n = 16,
// phases to 1e5, geometric mean over six inputs: 3.6e-12, by divide and conquer
// 5.0e-12; on the one input tried with the products 1e-11).
__device__ inline bool rotation(double alpha, double gamma, cdbl beta, double skip, double &c, cdbl &s,
                                double &shift)
{
    const double dl = 0.5 * (gamma - alpha), b2 = cabs2(beta);
    const bool on = b2 > skip;
    const double ir = small_rsqrt(on ? fma(dl, dl, b2) : 1.0);
    const double c2 = on ? fma(0.5 * fabs(dl), ir, 0.5) : 1.0;
    const double ic = small_rsqrt(c2);
    c = c2 * ic;
    const double f = on ? (dl >= 0.0 ? 0.5 : -0.5) * ir * ic : 0.0;
    s = cscale(beta, f);
    shift = f * b2 * ic;
    return on;
}

// [p q] <- [c p - conj(s) q, s p + c q]
__device__ inline void mix(double c, cdbl s, cdbl &p, cdbl &q)
{
    const cdbl p1 = cmk(fma(c, p.re, -fma(s.re, q.re, s.im * q.im)),
                        fma(c, p.im, -fma(s.re, q.im, -s.im * q.re)));
    q = cmk(fma(c, q.re, fma(s.re, p.re, -s.im * p.im)), fma(c, q.im, fma(s.re, p.im, s.im * p.re)));
    p = p1;
}

// M x M lanes per matrix, n <= 2 M.
template <int M>
__global__ void __launch_bounds__(64) k_eigh_small(int n, int batch, const double *H, double *E,
                                                   double *U, int32_t *info, int max_sweeps)
{
    constexpr int PER = 64 / (M * M), LD = 2 * M + 1, SZ = 2 * M * LD;
    __shared__ cdbl lds[PER][2 * SZ];
    __shared__ int order[PER][2 * M];
    const int lane = threadIdx.x, sub = lane / (M * M), l = lane - sub * M * M;
    const int b = blockIdx.x * PER + sub;
    const bool real_one = b < batch;           // the last wave's spare lanes repeat a matrix
    const cdbl *Hb = (const cdbl *)H + (size_t)min(b, batch - 1) * n * n;
    cdbl *A = lds[sub], *V = A + SZ;
    const int N = n + (n & 1), m = N / 2;      // an odd n gets an isolated zero index
    double big = 0.0;
    for (int x = l; x < 4 * M * M; x += M * M) {
        const int r = x / (2 * M), k = x - r * 2 * M;
        cdbl a = cmk(0.0, 0.0);
        if (r < n && k < n) {
            a = r >= k ? Hb[(size_t)r * n + k] : Hb[(size_t)k * n + r];
            if (r < k) a.im = -a.im;
            if (r == k) a.im = 0.0;
        }
        A[r * LD + k] = a;
        V[r * LD + k] = cmk(r == k ? 1.0 : 0.0, 0.0);
        big = fmax(big, fmax(fabs(a.re), fabs(a.im)));
    }
#pragma unroll
    for (int o = M * M / 2; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
    // scaled by a power of two to a largest component near 1
    int ex = 0;
    if (big > 0.0 && big < INFINITY) (void)frexp(big, &ex);
    wave_sync();
    double fro = 0.0;
    for (int x = l; x < 4 * M * M; x += M * M) {
        cdbl &a = A[(x / (2 * M)) * LD + x % (2 * M)];
        a = cmk(ldexp(a.re, -ex), ldexp(a.im, -ex));
        fro += cabs2(a);
    }
#pragma unroll
    for (int o = M * M / 2; o > 0; o >>= 1) fro += __shfl_xor(fro, o, 64);
    // pair elements at or below 2^-53 ||A||_F are left alone
    const double skip = fro * 0x1p-106;
    // a NaN or infinite entry: no rotation is made (every comparison with skip is
    // false); info = 1 and NaN results below
    const bool bad = !(fro < INFINITY);
    const int i = l / M, j = l - i * M;
    const bool on = i < m && j < m;
    wave_sync();

    int st = 1;
    for (int sweep = 0; sweep < max_sweeps; ++sweep) {
        bool moved = false;
        // pair 0 is the fixed index N - 1 with t, pair x is t + x with t - x mod N - 1
        const int last = N - 2;
        int ti = i, tj = j, si = N - 1 - i, sj = N - 1 - j;
        for (int t = 0; t <= last; ++t) {
            const int pi = i == 0 ? N - 1 : ti, qi = i == 0 ? t : si;
            const int pj = j == 0 ? N - 1 : tj, qj = j == 0 ? t : sj;
            if (on) {
                double ci, cj, di, dj;
                cdbl ri, rj;
                const cdbl bi = A[pi * LD + qi], bj = A[pj * LD + qj];
                const double alpha = A[pi * LD + pi].re, gamma = A[qi * LD + qi].re;
                const bool turned = rotation(alpha, gamma, bi, skip, ci, ri, di);
                rotation(A[pj * LD + pj].re, A[qj * LD + qj].re, bj, skip, cj, rj, dj);
                cdbl x00 = A[pi * LD + pj], x01 = A[pi * LD + qj];
                cdbl x10 = A[qi * LD + pj], x11 = A[qi * LD + qj];
                cdbl v0 = V[2 * i * LD + pj], w0 = V[2 * i * LD + qj];
                cdbl v1 = V[(2 * i + 1) * LD + pj], w1 = V[(2 * i + 1) * LD + qj];
                moved |= turned;
                mix(cj, rj, x00, x01);
                mix(cj, rj, x10, x11);
                const cdbl rc = cconj(ri);
                mix(ci, rc, x00, x10);
                mix(ci, rc, x01, x11);
                mix(cj, rj, v0, w0);
                mix(cj, rj, v1, w1);
                if (i == j) {
                    x00 = cmk(alpha - di, 0.0);
                    x11 = cmk(gamma + di, 0.0);
                    if (turned) x01 = x10 = cmk(0.0, 0.0);
                }
                wave_sync();
                A[pi * LD + pj] = x00;
                A[pi * LD + qj] = x01;
                A[qi * LD + pj] = x10;
                A[qi * LD + qj] = x11;
                V[2 * i * LD + pj] = v0;
                V[2 * i * LD + qj] = w0;
                V[(2 * i + 1) * LD + pj] = v1;
                V[(2 * i + 1) * LD + qj] = w1;
            }
            wave_sync();
            ti = ti == last ? 0 : ti + 1;
            tj = tj == last ? 0 : tj + 1;
            si = si == last ? 0 : si + 1;
            sj = sj == last ? 0 : sj + 1;
        }
        if (__ballot(moved) == 0) {
            st = 0;
            break;
        }
    }
    if (st != 0) {
        // which of the wave's matrices still turned is not kept apart: a later
        // sweep leaves a finished matrix alone, so test each against skip
        double off = 0.0;
        for (int x = l; x < N * N; x += M * M) {
            const int r = x / N, k = x - r * N;
            if (r != k) off = fmax(off, cabs2(A[r * LD + k]));
        }
#pragma unroll
        for (int o = M * M / 2; o > 0; o >>= 1) off = fmax(off, __shfl_xor(off, o, 64));
        st = off <= skip ? 0 : 1;
    }
    if (l == 0 && real_one) info[b] = bad ? 1 : st;

    // ascending order (a NaN diagonal has none)
    for (int r = l; r < n; r += M * M) {
        const double d = A[r * LD + r].re;
        int rank = 0;
        for (int k = 0; k < n; ++k) {
            const double dk = A[k * LD + k].re;
            rank += (dk < d || (dk == d && k < r)) ? 1 : 0;
        }
        if (bad) rank = r;
        order[sub][rank] = r;
        if (real_one) E[(size_t)b * n + rank] = bad ? NAN : ldexp(d, ex);
    }
    wave_sync();
    if (!real_one) return;
    cdbl *Ub = (cdbl *)U + (size_t)b * n * n;
    for (int x = l; x < n * n; x += M * M) {
        const int r = x / n, k = x - r * n;
        Ub[x] = bad ? cmk(NAN, NAN) : V[r * LD + order[sub][k]];
    }
}

template <int M>
void small_launch(int n, int batch, const double *H, double *E, double *U, int32_t *info,
                  int max_sweeps, hipStream_t s)
{
    constexpr int PER = 64 / (M * M);
    hipLaunchKernelGGL((k_eigh_small<M>), dim3((batch + PER - 1) / PER), dim3(64), 0, s, n, batch, H, E, U,
                       info, max_sweeps);
}

}  // namespace

hipError_t launch_eigh_small(int n, int batch, const double *H, double *E, double *U, int32_t *info,
                             hipStream_t s)
{
    constexpr int kSweeps = 40;
    ProfScope ps_("k_eigh_small", s);
    if (n <= 4) small_launch<2>(n, batch, H, E, U, info, kSweeps, s);
    else if (n <= 8) small_launch<4>(n, batch, H, E, U, info, kSweeps, s);
    else if (n <= kSmallMax) small_launch<8>(n, batch, H, E, U, info, kSweeps, s);
    else return hipErrorNotSupported;
    return hipGetLastError();
}
