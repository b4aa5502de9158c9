// Householder tridiagonalisation with the matrix resident in the registers of
// one CU (gfx950, n <= 256).  Same reduction and outputs as the panel kernel
// (msp_tridiag_lp.hip): reflectors v with v_{k+1} = 1, tails below the
// subdiagonal of the row-major matrix, d to E, e and tau to the workspace.
//
// Layout: rows go in strips of 4 W (W waves); lane l of wave w holds row
// 4 w + l / 16 of every strip and column l % 16 of every 16-column block up to
// the strip's diagonal region, which is held whole.  Every wave has the same
// static code and the same share of the live matrix at every step; row sums
// stay in one wave, column sums cross the W waves once per step through LDS.
// Above n = 192 the registers hold the trailing 192 columns; the one or two
// pairs of 16-column blocks before them stay in global memory, updated there
// (each element by one lane) until their 32 or 64 columns are done.
//
// Column step k:
//   1. wave 0 brings column k up to date and forms its reflector, the others
//      meanwhile apply the previous step's rank-2 update to the live blocks;
//   2. A22 x' over the live blocks, row sums and (by Hermitian symmetry)
//      column sums; x' is the column with its first entry replaced by
//      alpha - beta, so v = x' / (alpha - beta); column k + 1 goes to LDS;
//   3. per row: the sums are added and v and
//      w = tau A22 v - (|tau|^2 / 2)(v^H A22 v) v, whose scalar is real, formed.
// Three workgroup barriers per column; global memory is read once.
//
// What bounds it: at n = 192 about 480 vector instructions per wave and column
// (300 of them FP64 FMAs, 190 of those the live lower triangle's) keep the
// SIMDs half busy; the rest is the reflector's serial chain, the barriers and
// LDS (43 % busy, a fifth of it bank conflicts).  At one 8-wave workgroup per CU nothing covers the barriers;
// below n = 128 two to sixteen workgroups share a CU.
// The panel kernel re-reads the trailing triangle once per column (at n = 192
// 5.2 TB/s past L2); here the matrix is read once.  ms per 4096 matrices, panel
// kernel (below n = 65: registers in 64-column slots) against this one:
//   n = 192 18.6 / 10.3, 144 10.7 / 6.6, 128 8.3 / 3.2, 108 6.2 / 2.5,
//   96 5.1 / 1.7, 72 3.3 / 1.1, 64 2.25 / 0.74, 48 1.82 / 0.37, 32 0.91 / 0.19;
//   one matrix: n = 192 1.88 / 0.62, 64 0.18 / 0.11; n = 256
//   3.3 / 1.65, and for 256 matrices 3.7 / 2.3.
// Measured and not taken: 16 x 16 tiles in MFMA accumulators dealt to the waves
// with the rank-2 update on MFMA (n = 192 14.6 ms: FP64 MFMA and FP64 VALU
// share one pipe, so the products delay the other waves' serial chains, and a
// branch per tile costs register copies); row sums by DPP halving instead of
// through LDS (10.5 ms).
#include <hip/hip_runtime.h>

#include <utility>

#include "msp_kernels.h"
#include "msp_tridiag.h"

namespace {

__device__ inline void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Square root and its reciprocal of t > 0: hardware estimate, two coupled
// Newton steps, and a last correction of the root.
__device__ inline void sqrt_recip(double t, double &root, double &rec)
{
    const double y = __builtin_amdgcn_rsq(t);
    double gg = t * y, h = 0.5 * y;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const double r = fma(-gg, h, 0.5);
        gg = fma(gg, r, gg);
        h = fma(h, r, h);
    }
    root = fma(fma(-gg, gg, t), h, gg);
    rec = 2.0 * h;
}

// Value of lane L of this lane's row of 16 lanes.
template <int L>
__device__ inline double row_bcast(double v)
{
    return __longlong_as_double(
        __builtin_amdgcn_update_dpp(0ll, __double_as_longlong(v), 0x150 + L, 0xF, 0xF, true));
}
// m -= v w^H + w v^H at one element, as FMA chains
__device__ __forceinline__ void rank2(cdbl &m, cdbl vi, cdbl wi, cdbl vj, cdbl wj)
{
    m.re = fma(-vi.re, wj.re, m.re);
    m.im = fma(-vi.im, wj.re, m.im);
    m.re = fma(-vi.im, wj.im, m.re);
    m.im = fma(vi.re, wj.im, m.im);
    m.re = fma(-wi.re, vj.re, m.re);
    m.im = fma(-wi.im, vj.re, m.im);
    m.re = fma(-wi.im, vj.im, m.re);
    m.im = fma(wi.re, vj.im, m.im);
}
// o[a] = x of lane FIRST + STEP a of each row of 16 lanes
template <int FIRST, int STEP, int NS, int... I>
__device__ inline void spread(cdbl x, cdbl (&o)[NS], std::integer_sequence<int, I...>)
{
    ((o[I] = cmk(row_bcast<FIRST + STEP * I>(x.re), row_bcast<FIRST + STEP * I>(x.im))), ...);
}

// W: waves, NS: strips of 4 W rows (n <= 4 W NS), OCC: waves per SIMD asked for.
// JC: pairs of leading 16-column blocks that are kept in place in global memory
// (the matrix's own, read and written by the lanes that would hold them) while
// their columns last.
template <int W, int NS, int JC>
struct RtShape {
    static constexpr int SR = 4 * W;                       // rows per strip
    static constexpr int NR = SR * NS;
    // first and last column block of strip a's diagonal region
    static constexpr int j0(int a) { return a * W / 4; }
    static constexpr int dl(int a) { return W >= 4 ? j0(a) + W / 4 - 1 : j0(a); }
    static constexpr int slot(int a, int J)
    {
        int s = 0;
        for (int b = 0; b < a; ++b) s += dl(b) + 1 > 2 * JC ? dl(b) + 1 - 2 * JC : 0;
        return s + J - 2 * JC;
    }
    static constexpr int NJ = dl(NS - 1) + 1;
    static constexpr int NSLOT = slot(NS, 2 * JC);
    static constexpr int NC = (NR + 63) / 64;              // entries per lane of a vector
    static constexpr int NP = 64 * NC;
    // LDS: x', column k + 1, v and w, column sums per wave, row sums per lane,
    // scale, tau scale, -|tau scale|^2 / 2, and a share of v^H A22 v per wave
    static constexpr int CDBL = 4 * NP + W * NP + 64 * W * NS + 3;
    static constexpr size_t LDS = sizeof(cdbl) * CDBL + sizeof(double) * W;
};

template <int W, int NS, int OCC, int JC>
__global__ void __launch_bounds__(64 * W, OCC) k_tridiag_rt(int n, double *H, double *E, double *work)
{
    using T = RtShape<W, NS, JC>;
    constexpr int SR = T::SR, NJ = T::NJ, NC = T::NC, NP = T::NP;
    static_assert(NS <= 8 && W % 2 == 0, "two lanes per row of a wave, each on half the waves' sums");
    static_assert(JC == 0 || W == 8, "a strip's diagonal region is one pair of blocks");
    extern __shared__ __align__(16) unsigned char smem[];
    cdbl *col = (cdbl *)smem;                  // x': zero up to row k
    cdbl *cn = col + NP;                       // column k + 1 before step k's update
    cdbl *V = cn + NP, *Wv = V + NP;           // v and w of the pending update
    cdbl *P = Wv + NP;                         // column sums per wave
    cdbl *R = P + W * NP;                      // row sums per lane: [wave][strip][g][c]
    cdbl *scal = R + 64 * W * NS;              // scale, tau scale, (-|tau scale|^2 / 2, -)
    double *dot = (double *)(scal + 3);

    const int tid = threadIdx.x;
    const int lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    cdbl *A = (cdbl *)H + (size_t)blockIdx.x * n * n;
    double *base = work + (size_t)blockIdx.x * dc_work_doubles(n);
    double *e;
    cdbl *tau;
    dc_carve(n, base, &e, &tau);
    double *d = E + (size_t)blockIdx.x * n;

    cdbl M[T::NSLOT];
    double big = 0.0;
    const auto element = [&](int row, int cc) {
        cdbl x = cmk(0.0, 0.0);
        if (row < n && cc < n) {
            x = (row >= cc) ? A[(size_t)row * n + cc] : A[(size_t)cc * n + row];
            if (row < cc) x.im = -x.im;
            if (row == cc) x.im = 0.0;
        }
        big = fmax(big, fmax(fabs(x.re), fabs(x.im)));
        return x;
    };
#pragma unroll
    for (int a = 0; a < NS; ++a)
#pragma unroll
        for (int J = 2 * JC; J <= T::dl(a); ++J)
            M[T::slot(a, J)] = element(SR * a + 4 * wave + g, 16 * J + c);
    for (int a = 0; a < NS; ++a)
        for (int J = 0; J < 2 * JC && J <= T::dl(a); ++J) (void)element(SR * a + 4 * wave + g, 16 * J + c);
    // scaled by a power of two to a largest component near 1: x'^H A22 x' is
    // cubic in the entries
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
    if (lane == 0) dot[wave] = big;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < W; ++w) big = fmax(big, dot[w]);
    int ex = 0;
    if (big > 0.0 && big < INFINITY) (void)frexp(big, &ex);
    ex = __builtin_amdgcn_readfirstlane(ex);
#pragma unroll
    for (int s = 0; s < T::NSLOT; ++s) M[s] = cmk(ldexp(M[s].re, -ex), ldexp(M[s].im, -ex));
    for (int i = tid; i < NP; i += 64 * W) {
        V[i] = Wv[i] = cmk(0.0, 0.0);
        const cdbl x = (i < n) ? A[(size_t)i * n] : cmk(0.0, 0.0);
        cn[i] = cmk(ldexp(x.re, -ex), ldexp(x.im, -ex));
    }
    if constexpr (JC > 0) {
        // scaled in place; the diagonal regions made whole (the mirror of an
        // element below the diagonal is another lane's, so all are read before
        // any is written)
        cdbl cold[2 * JC * JC];
#pragma unroll
        for (int a = 0; a < JC; ++a)
#pragma unroll
            for (int J = 0; J < 2 * JC && J <= T::dl(a); ++J)
                cold[2 * JC * a + J] = element(SR * a + 4 * wave + g, 16 * J + c);
        __syncthreads();
        const auto put = [&](int row, int J, cdbl x) {
            if (row < n) A[(size_t)row * n + 16 * J + c] = cmk(ldexp(x.re, -ex), ldexp(x.im, -ex));
        };
#pragma unroll
        for (int a = 0; a < JC; ++a)
#pragma unroll
            for (int J = 0; J < 2 * JC && J <= T::dl(a); ++J)
                put(SR * a + 4 * wave + g, J, cold[2 * JC * a + J]);
        for (int a = JC; a < NS; ++a)
            for (int J = 0; J < 2 * JC; ++J) {
                const int row = SR * a + 4 * wave + g;
                put(row, J, row < n ? A[(size_t)row * n + 16 * J + c] : cmk(0.0, 0.0));
            }
    }
    for (int i = tid; i < W * NP + 64 * W * NS; i += 64 * W) P[i] = cmk(0.0, 0.0);
    // LDS places of this lane: its rows and columns, its share of the sums
    const cdbl *vrp = V + NP * (c & 1) + SR * min(c >> 1, NS - 1) + 4 * wave + g;
    const cdbl *xrp = col + SR * min(c, NS - 1) + 4 * wave + g;
    double *Pw = (double *)(P + wave * NP + 16 * (g >> 1) + c) + (g & 1);
    cdbl *Rw = R + 64 * wave * NS + lane;
    // stage 3: lane halves share a row, half h adds the column sums of its
    // waves and the row sums of its eight columns, from a different column in
    // each lane so that the lanes read different banks
    const int h = lane >> 5, rr = lane & 31;
    const int i3 = SR * (rr >> 2) + 4 * wave + (rr & 3);
    const cdbl *Rs = R + 64 * wave * NS + 16 * min(rr, 4 * NS - 1);
    const int u3 = rr + 8 * h;
    __syncthreads();

    for (int k = 0;; ++k) {
        const int jp1 = (k + 1) >> 5;          // pairs of column blocks before it are done
        // (1) wave 0: column k with the pending update and its reflector
        if (wave == 0) {
            __builtin_amdgcn_s_setprio(2);
            cdbl x[NC];
            const double vkr = V[k].re, vki = V[k].im, wkr = Wv[k].re, wki = Wv[k].im;
#pragma unroll
            for (int t = 0; t < NC; ++t) {
                const int i = 64 * t + lane;
                const double vr = V[i].re, vi = V[i].im, wr = Wv[i].re, wi = Wv[i].im;
                x[t] = cn[i];
                x[t].re = fma(-vr, wkr, x[t].re);
                x[t].im = fma(-vi, wkr, x[t].im);
                x[t].re = fma(-vi, wki, x[t].re);
                x[t].im = fma(vr, wki, x[t].im);
                x[t].re = fma(-wr, vkr, x[t].re);
                x[t].im = fma(-wi, vkr, x[t].im);
                x[t].re = fma(-wi, vki, x[t].re);
                x[t].im = fma(wr, vki, x[t].im);
            }
            double part = 0.0, dk = 0.0;
            cdbl alpha = cmk(0.0, 0.0);
#pragma unroll
            for (int t = 0; t < NC; ++t) {
                const int i = 64 * t + lane;
                part += (i > k + 1) ? cabs2(x[t]) : 0.0;
                dk = (i == k) ? x[t].re : dk;
                const cdbl a = cmk(readlane_f64(x[t].re, (k + 1) & 63), readlane_f64(x[t].im, (k + 1) & 63));
                if (((k + 1) >> 6) == t) alpha = a;
            }
            if (lane == (k & 63)) d[k] = ldexp(dk, ex);
            if (k == n - 1) break;
            const double xn2 = wave_sum_all(part);
            cdbl tk = cmk(0.0, 0.0), scale = tk, xh = tk;
            double beta = alpha.re;
            if (!(xn2 == 0.0 && alpha.im == 0.0)) {
                double nrm, rb;
                sqrt_recip(fma(alpha.re, alpha.re, fma(alpha.im, alpha.im, xn2)), nrm, rb);
                beta = alpha.re >= 0.0 ? -nrm : nrm;
                rb = alpha.re >= 0.0 ? -rb : rb;
                // tau = (beta - alpha)/beta, 1/(alpha - beta) = (1/beta)/d with
                // d = alpha/beta - 1, 1 <= |d| <= 2
                tk = cmk((beta - alpha.re) * rb, -alpha.im * rb);
                const double dr = fma(alpha.re, rb, -1.0), di = alpha.im * rb;
                const double rd = rb * msp_recip(fma(dr, dr, di * di));
                scale = cmk(dr * rd, -di * rd);
                xh = cmk(alpha.re - beta, alpha.im);
            }
#pragma unroll
            for (int t = 0; t < NC; ++t) {
                const int i = 64 * t + lane;
                col[i] = (i > k + 1) ? x[t] : (i == k + 1 ? xh : cmk(0.0, 0.0));
            }
            if (lane == 0) {
                const cdbl u = cmul(tk, scale);
                scal[0] = scale;
                scal[1] = u;
                scal[2] = cmk(-0.5 * cabs2(u), 0.0);
                e[k] = ldexp(beta, ex);
                tau[k] = tk;
            }
            __builtin_amdgcn_s_setprio(0);
            lds_barrier();
        } else if (k == n - 1) {
            break;
        }

        // pending update A22 -= v w^H + w v^H of the live blocks
        if (k > 0) {
            // lane c of a row of 16 reads v (c even) or w (c odd) of strip c / 2
            const cdbl ro = *vrp;
            if constexpr (JC > 0) {
                // blocks in global memory, a pair per strip, the next strip's
                // loads issued before this strip's stores; finished columns hold
                // reflector tails, which the lanes leave alone
#pragma unroll 1
                for (int jp = jp1; jp < JC; ++jp) {
                    const cdbl v0 = V[32 * jp + c], w0 = Wv[32 * jp + c];
                    const cdbl v1 = V[32 * jp + 16 + c], w1 = Wv[32 * jp + 16 + c];
                    const bool l0 = 32 * jp + c > k, l1 = 32 * jp + 16 + c > k;
                    int row = SR * jp + 4 * wave + g;
                    cdbl *p0 = A + row * n + 32 * jp + c;
                    cdbl y0 = cmk(0.0, 0.0), y1 = y0;
                    if (row < n) {
                        y0 = p0[0];
                        y1 = p0[16];
                    }
#pragma unroll 1
                    for (int a = jp; a < NS; ++a) {
                        cdbl x0 = y0, x1 = y1, *pn = p0 + SR * n;
                        if (row + SR < n) {
                            y0 = pn[0];
                            y1 = pn[16];
                        }
                        const cdbl va = V[row], wa = Wv[row];
                        rank2(x0, va, wa, v0, w0);
                        rank2(x1, va, wa, v1, w1);
                        if (row < n && l0) p0[0] = x0;
                        if (row < n && l1) p0[16] = x1;
                        row += SR;
                        p0 = pn;
                    }
                }
            }
            cdbl vr[NS], wr[NS];
            spread<0, 2>(ro, vr, std::make_integer_sequence<int, NS>());
            spread<1, 2>(ro, wr, std::make_integer_sequence<int, NS>());
#pragma unroll
            for (int jp = JC; jp < (NJ + 1) / 2; ++jp) {
                if (jp < jp1) continue;
#pragma unroll
                for (int J = 2 * jp; J < 2 * jp + 2 && J < NJ; ++J) {
                    const cdbl vj = V[16 * J + c], wj = Wv[16 * J + c];
#pragma unroll
                    for (int a = 0; a < NS; ++a)
                        if (J <= T::dl(a)) rank2(M[T::slot(a, J)], vr[a], wr[a], vj, wj);
                }
            }
        }
        if (wave != 0) lds_barrier();

        // (2) A22 x' over the live blocks
        {
            cdbl xr[NS], rs[NS];
            double dacc = 0.0;
#pragma unroll
            for (int a = 0; a < NS; ++a) rs[a] = cmk(0.0, 0.0);
            const cdbl xo = *xrp;
            const auto column_sums = [&](int jp, cdbl (&cs)[2]) {
                swap32(cs[0].re, cs[1].re);
                swap32(cs[0].im, cs[1].im);
                double s = cs[0].re + cs[1].re, t = cs[0].im + cs[1].im;
                swap16(s, t);
                Pw[64 * jp] = s + t;
            };
            if constexpr (JC > 0) {
#pragma unroll 1
                for (int jp = jp1; jp < JC; ++jp) {
                    const cdbl xc0 = col[32 * jp + c], xc1 = col[32 * jp + 16 + c];
                    const bool next0 = k + 1 == 32 * jp + c, next1 = k + 1 == 32 * jp + 16 + c;
                    int row = SR * jp + 4 * wave + g;
                    const cdbl *p0 = A + row * n + 32 * jp + c;
                    cdbl y0 = cmk(0.0, 0.0), y1 = y0, cs[2];
                    cs[0] = cs[1] = y0;
                    if (row < n) {
                        y0 = p0[0];
                        y1 = p0[16];
                    }
#pragma unroll 1
                    for (int a = jp; a < NS; ++a) {
                        const cdbl x0 = row < n ? y0 : cmk(0.0, 0.0), x1 = row < n ? y1 : cmk(0.0, 0.0);
                        p0 += SR * n;
                        if (row + SR < n) {
                            y0 = p0[0];
                            y1 = p0[16];
                        }
                        const cdbl xa = col[row];
                        if (next0) cn[row] = x0;
                        if (next1) cn[row] = x1;
                        cdbl r = cmk(0.0, 0.0);
                        cfma(r, x0, xc0);
                        cfma(r, x1, xc1);
                        const double t = fma(xa.re, r.re, xa.im * r.im);
                        dacc += t;
                        if (a > jp) {          // (strip jp: its diagonal region)
                            dacc += t;
                            cfmac(cs[0], x0, xa);
                            cfmac(cs[1], x1, xa);
                        }
                        // a strip's row sums collect in its place in R
                        Rw[64 * a] = jp > jp1 ? cadd(Rw[64 * a], r) : r;
                        row += SR;
                    }
                    column_sums(jp, cs);
                }
            }
            spread<0, 1>(xo, xr, std::make_integer_sequence<int, NS>());
#pragma unroll
            for (int jp = JC; jp < (NJ + 1) / 2; ++jp) {
                if (jp < jp1) continue;
                cdbl cs[2];
                cs[0] = cs[1] = cmk(0.0, 0.0);
#pragma unroll
                for (int J = 2 * jp; J < 2 * jp + 2 && J < NJ; ++J) {
                    const cdbl xc = col[16 * J + c];
#pragma unroll
                    for (int a = 0; a < NS; ++a) {
                        if (J > T::dl(a)) continue;
                        const cdbl m = M[T::slot(a, J)];
                        if (J < T::j0(a)) cfmac(cs[J & 1], m, xr[a]);
                        // v^H A22 v counts the blocks left of the diagonal region twice
                        if (J == T::j0(a)) dacc = fma(xr[a].re, rs[a].re, fma(xr[a].im, rs[a].im, dacc));
                        cfma(rs[a], m, xc);
                    }
                }
                // column k + 1 for the next step
#pragma unroll
                for (int J = 2 * jp; J < 2 * jp + 2 && J < NJ; ++J) {
                    if (J != ((k + 1) >> 4)) continue;
                    if (c == ((k + 1) & 15)) {
#pragma unroll
                        for (int a = 0; a < NS; ++a)
                            if (J <= T::dl(a)) cn[SR * a + 4 * wave + g] = M[T::slot(a, J)];
                    }
                }
                if (2 * jp < T::j0(NS - 1)) column_sums(jp, cs);
            }
#pragma unroll
            for (int a = 0; a < NS; ++a) dacc = fma(xr[a].re, rs[a].re, fma(xr[a].im, rs[a].im, dacc));
            // row sums of the live strips, left to stage 3 (this wave's rows)
            if (JC > 0 && jp1 < JC) {
#pragma unroll
                for (int a = 0; a < NS; ++a)
                    if (T::dl(a) >= 2 * JC) Rw[64 * a] = cadd(Rw[64 * a], rs[a]);
            } else {
                if (k + 1 < SR * (NS / 2)) {
#pragma unroll
                    for (int a = 0; a < NS / 2; ++a) Rw[64 * a] = rs[a];
                }
#pragma unroll
                for (int a = NS / 2; a < NS; ++a) Rw[64 * a] = rs[a];
            }
            dacc = wave_sum_all(dacc);
            if (lane == 0) dot[wave] = dacc;
        }
        lds_barrier();

        // (3) v and w of this wave's rows
        if (SR * (NS - 1) + 4 * wave + 3 >= k) {
            const bool in = rr < 4 * NS;
            const int i = in ? i3 : 0;
            cdbl y = Rs[u3 & 15];
#pragma unroll
            for (int u = 1; u < 8; ++u) y = cadd(y, Rs[(u + u3) & 15]);
            const cdbl xi = col[i], scale = scal[0], u = scal[1];
            const double mh = scal[2].re;
            double rho = 0.0;
#pragma unroll
            for (int w = 0; w < W; ++w) rho += dot[w];
#pragma unroll
            for (int w = 0; w < W / 2; ++w) y = cadd(y, P[(w + h * (W / 2)) * NP + i]);
            double t = y.re;
            swap32(y.re, t);
            y.re += t;
            t = y.im;
            swap32(y.im, t);
            y.im += t;
            const bool act = u.re != 0.0 || u.im != 0.0;
            const cdbl v = (i == k + 1) ? cmk(act ? 1.0 : 0.0, 0.0) : cmul(xi, scale);
            const cdbl p = cmul(u, y);
            const double c0 = mh * rho;
            cdbl o = h ? cmk(fma(c0, v.re, p.re), fma(c0, v.im, p.im)) : v;
            if (!(i > k && i < n)) o = cmk(0.0, 0.0);
            if (in) V[NP * h + i] = o;
            if (in && h == 0 && i >= k + 2 && i < n) A[(size_t)i * n + k] = v;
        }
        lds_barrier();
    }
}

template <int W, int NS, int OCC, int JC = 0>
hipError_t rt_launch(int n, int batch, double *H, double *E, double *work, hipStream_t s)
{
    const size_t lds = RtShape<W, NS, JC>::LDS;
    hipError_t err = msp_set_lds((const void *)k_tridiag_rt<W, NS, OCC, JC>, lds);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL((k_tridiag_rt<W, NS, OCC, JC>), dim3(batch), dim3(64 * W), lds, s, n, H, E, work);
    return hipGetLastError();
}

}  // namespace

// Waves and strips by n (n <= 16 has an eigensolver of its own): few waves for
// small matrices, so that many matrices share a CU, four waves where two or more workgroups still fit its
// registers (n <= 128), eight above.  Strips of 4 W rows cover n closely: a
// strip too many costs 10 to 20 %.
// Up to 512 matrices run at most two to a CU and take the form with the
// shortest column step; more take the form that holds more matrices per CU.
// ms for 256 / 4096 matrices: n = 48 four waves 0.078 / 0.44, two 0.095 /
// 0.37; n = 96 at two workgroups per CU 0.205 / 1.93, at three (four registers
// spilled) 0.230 / 1.71; n = 32 two waves 0.051 / 0.19, one 0.058 / 0.19;
// n = 128 four waves 0.32 / 3.1, eight 0.31 / 4.9.
// Above n = 256 the columns left in global memory would be most of the work.
hipError_t launch_tridiag_rt(int n, int batch, double *H, double *E, double *work, hipStream_t s)
{
    const bool many = batch > 512;
    if (n <= 24) return rt_launch<2, 3, 4>(n, batch, H, E, work, s);
    if (n <= 32) return rt_launch<2, 4, 4>(n, batch, H, E, work, s);
    if (n <= 48 && many) return rt_launch<2, 6, 4>(n, batch, H, E, work, s);
    if (n <= 48) return rt_launch<4, 3, 4>(n, batch, H, E, work, s);
    if (n <= 64) return rt_launch<4, 4, 4>(n, batch, H, E, work, s);
    if (n <= 80) return rt_launch<4, 5, 3>(n, batch, H, E, work, s);
    if (n <= 96 && many) return rt_launch<4, 6, 3>(n, batch, H, E, work, s);
    if (n <= 96) return rt_launch<4, 6, 2>(n, batch, H, E, work, s);
    if (n <= 112) return rt_launch<4, 7, 2>(n, batch, H, E, work, s);
    if (n <= 128) return rt_launch<4, 8, 2>(n, batch, H, E, work, s);
    if (n <= 160) return rt_launch<8, 5, 2>(n, batch, H, E, work, s);
    if (n <= 192) return rt_launch<8, 6, 2>(n, batch, H, E, work, s);
    if (n <= 224) return rt_launch<8, 7, 2, 1>(n, batch, H, E, work, s);
    if (n <= 256) return rt_launch<8, 8, 2, 2>(n, batch, H, E, work, s);
    return hipErrorNotSupported;
}
