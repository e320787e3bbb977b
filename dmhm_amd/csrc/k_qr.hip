// gfx950 batched Householder QR of tall-skinny panels, Q formed in place
// (geqrf + orgqr semantics, one workgroup per panel, FP64 arithmetic).
#include <type_traits>
#include "kcommon.hpp"

namespace dmhm {

// A column whose squared norm (diagonal entry included) is below this is left
// unreflected (tau = 0): its entries are below ~1e-140, and squares of such
// entries reach the subnormal range, where a reflector computed from them is
// no longer orthogonal and would corrupt the later columns. The entries it
// leaves below the diagonal are that small in absolute terms.
constexpr double kTinyColumn = 1e-280;

// ---------------------------------------------------------------------------
// Batched Householder QR (one workgroup per panel, FP64 arithmetic).
// ---------------------------------------------------------------------------

// dots[c] = sum_{i > j} A(i, j) * A(i, c) for c in [c0, k)
template <typename T>
__device__ void column_dots(const T* A, int m, int j, int c0, int k, double* dots,
                            double (*red)[16])
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int cb = c0; cb < k; cb += 16) {
        double p[16];
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) p[cc] = 0.0;
        for (int i = j + 1 + tid; i < m; i += 256) {
            const double x = (double)A[i + (int64_t)j * m];
#pragma unroll
            for (int cc = 0; cc < 16; ++cc)
                if (cb + cc < k) p[cc] += x * (double)A[i + (int64_t)(cb + cc) * m];
        }
#pragma unroll
        for (int cc = 0; cc < 16; ++cc) {
            const double v = wave_sum(p[cc]);
            if (lane == 0) red[wave][cc] = v;
        }
        __syncthreads();
        if (tid < 16 && cb + tid < k) dots[cb + tid] = red[0][tid] + red[1][tid] + red[2][tid] + red[3][tid];
        __syncthreads();
    }
}

template <typename T>
__global__ void __launch_bounds__(256) qr_kernel(Bases b, const QrTask* __restrict__ tasks)
{
    __shared__ double red[4][16];
    __shared__ double dots[64];
    __shared__ double wv[64];
    __shared__ double tau_s[64];
    __shared__ double scale_s;
    const QrTask tk = tasks[blockIdx.x];
    T* A = reinterpret_cast<T*>(b.val[tk.slot]) + tk.off;
    const int m = tk.m, kstat = tk.k;
    const int k = tk.krank >= 0 ? min(kstat, b.rank[tk.kslot][tk.krank]) : kstat, kk = min(m, k);
    const int tid = threadIdx.x;
    if (m <= 0 || k <= 0) return;
    // Factor.
    for (int j = 0; j < kk; ++j) {
        column_dots(A, m, j, j, k, dots, red);
        if (tid == 0) {
            const double alpha = (double)A[j + (int64_t)j * m];
            const double xn2 = dots[j];
            double tau = 0.0, scale = 0.0, beta = alpha;
            if (xn2 > 0.0 && alpha * alpha + xn2 > kTinyColumn) {
                beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
                tau = (beta - alpha) / beta;
                scale = 1.0 / (alpha - beta);
            }
            tau_s[j] = tau; scale_s = scale;
            A[j + (int64_t)j * m] = (T)beta;
        }
        __syncthreads();
        const double scale = scale_s, tau = tau_s[j];
        if (tid > j && tid < k) {
            const int c = tid;
            const double w = tau * ((double)A[j + (int64_t)c * m] + scale * dots[c]);
            wv[c] = w;
            A[j + (int64_t)c * m] = (T)((double)A[j + (int64_t)c * m] - w);
        }
        __syncthreads();
        for (int i = j + 1 + tid; i < m; i += 256) {
            const double v = (double)A[i + (int64_t)j * m] * scale;
            for (int c = j + 1; c < k; ++c)
                A[i + (int64_t)c * m] = (T)((double)A[i + (int64_t)c * m] - wv[c] * v);
            A[i + (int64_t)j * m] = (T)v;
        }
        __syncthreads();
    }
    // R (kstat x k, ld rld: upper triangle, rows >= kk zero).
    if (tk.roff >= 0) {
        T* R = reinterpret_cast<T*>(b.val[SLOT_WS]) + tk.roff;
        for (int e = tid; e < kstat * k; e += 256) {
            const int r = e % kstat, c = e / kstat;
            R[r + (int64_t)c * tk.rld] = (r <= c && r < kk) ? A[r + (int64_t)c * m] : T(0);
        }
    }
    __syncthreads();
    // Form Q in place (orgqr); columns >= kk are zero.
    for (int c = kk + (tid >> 6); c < k; c += 4)
        for (int i = tid & 63; i < m; i += 64) A[i + (int64_t)c * m] = T(0);
    __syncthreads();
    for (int j = kk - 1; j >= 0; --j) {
        const double tau = tau_s[j];
        if (j + 1 < k) column_dots(A, m, j, j + 1, k, dots, red);
        if (tid > j && tid < k) {
            const int c = tid;
            const double w = tau * ((double)A[j + (int64_t)c * m] + dots[c]);
            wv[c] = w;
            A[j + (int64_t)c * m] = (T)((double)A[j + (int64_t)c * m] - w);
        }
        __syncthreads();
        for (int i = j + 1 + tid; i < m; i += 256) {
            const double v = (double)A[i + (int64_t)j * m];
            for (int c = j + 1; c < k; ++c)
                A[i + (int64_t)c * m] = (T)((double)A[i + (int64_t)c * m] - wv[c] * v);
            A[i + (int64_t)j * m] = (T)(-tau * v);
        }
        for (int i = tid; i < j; i += 256) A[i + (int64_t)j * m] = T(0);
        if (tid == 0) A[j + (int64_t)j * m] = (T)(1.0 - tau);
        __syncthreads();
    }
}

// Wave sum with a uniform result: DPP sums inside each row of 16 lanes, then
// the four row sums through scalar registers (no LDS round trip).
__device__ inline double wave_sum_uniform(double v)
{
    v = group_sum<16>(v);
    return (bcast(v, 0) + bcast(v, 16)) + (bcast(v, 32) + bcast(v, 48));
}

// Householder QR of one m x k panel (m <= 64 RR, k <= KMAX), lane = row (rows
// lane + 64 r), the KMAX columns split over NWV waves (wave w holds columns
// [w CW, (w + 1) CW) of every row in registers). Step j: the wave that owns
// column j forms the reflector (its column's sum of squares below the
// diagonal is one wave reduction), publishes v and tau through LDS, and
// every wave then applies it to its own columns right of j (one wave
// reduction v^T a_c per column). One barrier per step; buffers alternate by
// step parity, so a step's writes never meet the reads of the step before.
// The explicit Q is E - V T V1^T (V1: the first k rows of V), T^-1 = 1 / tau on
// the diagonal and v_l . v_j above it (the products of step j with the columns
// left of j; the inverse of the compact WY form's T: Puglisi, SIAM J. Sci. Stat.
// Comput. 13, 1992), by one triangular solve per column instead of a second pass of k
// barriers over the reflectors: panels of 1,024 rows 303 -> 250 us per 870,
// 117 -> 95 us per launch of few. Same
// reflector convention and outputs as qr_kernel (Q over the panel, R to the
// workspace); the panel and R may be strided (leading dimensions ld, rld), as
// the row blocks of a TSQR are. FP64 arithmetic.
template <typename T, int KMAX, int NWV, int RR>
__global__ void __launch_bounds__(64 * NWV) qr_split_kernel(Bases b, const QrTask* __restrict__ tasks)
{
    constexpr int CW = KMAX / NWV;
    static_assert(KMAX % NWV == 0, "whole columns per wave");
    // Rows of V that pass through LDS together when Q is formed, 64 RC of them
    // (odd leading dimension: rows and columns are both read without conflicts).
    constexpr int RC = RR < (KMAX <= 24 ? 4 : 2) ? RR : (KMAX <= 24 ? 4 : 2), VLD = 64 * RC + 1;
    constexpr int BUF = 128 * RR > KMAX * VLD ? 128 * RR : KMAX * VLD;
    static_assert(RR % RC == 0 && KMAX % 8 == 0, "whole row groups and column groups");
    __shared__ double buf[BUF];
    double (*vbuf)[64 * RR] = reinterpret_cast<double (*)[64 * RR]>(buf);
    double* Vs = buf;
    __shared__ double G[KMAX][KMAX];
    __shared__ double tbuf[2];
    __shared__ double taus[KMAX];
    const QrTask tk = tasks[blockIdx.x];
    T* A = reinterpret_cast<T*>(b.val[tk.slot]) + tk.off;
    const int m = tk.m, kstat = tk.k, ld = tk.ld;
    const int k = tk.krank >= 0 ? min(kstat, b.rank[tk.kslot][tk.krank]) : kstat, kk = min(m, k);
    if (k <= 0) return;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double a[CW][RR];
#pragma unroll
    for (int jj = 0; jj < CW; ++jj)
#pragma unroll
        for (int r = 0; r < RR; ++r) {
            const int c = w * CW + jj, i = lane + 64 * r;
            a[jj][r] = (i < m && c < k) ? (double)A[i + (int64_t)c * ld] : 0.0;
        }
    // Applies the published reflector (v, tau) of step j to this wave's columns c, j < c < k.
    auto apply = [&](int j, int par) {
        if (w * CW >= k) return;
        const double t = tbuf[par];
        double v[RR];
#pragma unroll
        for (int r = 0; r < RR; ++r) v[r] = vbuf[par][lane + 64 * r];
        double dot[CW];
#pragma unroll
        for (int jj = 0; jj < CW; ++jj) {
            double s = 0.0;
#pragma unroll
            for (int r = 0; r < RR; ++r) s += v[r] * a[jj][r];
            dot[jj] = wave_sum_uniform(s);
        }
#pragma unroll
        for (int jj = 0; jj < CW; ++jj) {
            const int c = w * CW + jj;
            if (c < j && lane == 0) G[j][c] = dot[jj];
            if (c > j && c < k) {
                const double f = t * dot[jj];
#pragma unroll
                for (int r = 0; r < RR; ++r) a[jj][r] -= f * v[r];
            }
        }
    };
#pragma unroll 1
    for (int j = 0; j < kk; ++j) {
        const int par = j & 1;
        if (w == j / CW) {
            const int js = j - w * CW;
            double x[RR];
#pragma unroll
            for (int r = 0; r < RR; ++r) {
                x[r] = 0.0;
#pragma unroll
                for (int jj = 0; jj < CW; ++jj) x[r] = jj == js ? a[jj][r] : x[r];
            }
            double s = 0.0, xj = 0.0;
#pragma unroll
            for (int r = 0; r < RR; ++r) {
                const int i = lane + 64 * r;
                const double xb = (i > j && i < m) ? x[r] : 0.0;
                s += xb * xb;
                xj = r == (j >> 6) ? x[r] : xj;
            }
            const double xn2 = wave_sum_uniform(s);
            const double alpha = bcast(xj, j & 63);
            double t = 0.0, scale = 0.0, beta = alpha;
            const double n2 = fma(alpha, alpha, xn2);
            if (xn2 > 0.0 && n2 > kTinyColumn) householder<HwEst>(alpha, n2, t, scale, beta);
#pragma unroll
            for (int r = 0; r < RR; ++r) {
                const int i = lane + 64 * r;
                const bool below = i > j && i < m;
                vbuf[par][i] = below ? x[r] * scale : (i == j ? 1.0 : 0.0);
                const double nx = i == j ? beta : (i > j ? x[r] * scale : x[r]);
#pragma unroll
                for (int jj = 0; jj < CW; ++jj) a[jj][r] = jj == js ? nx : a[jj][r];
            }
            if (lane == 0) { tbuf[par] = t; taus[j] = t; }
        }
        __syncthreads();
        apply(j, par);
    }
    if (tk.roff >= 0) {
        T* R = reinterpret_cast<T*>(b.val[SLOT_WS]) + tk.roff;
#pragma unroll
        for (int jj = 0; jj < CW; ++jj)
#pragma unroll
            for (int r = 0; r < RR; ++r) {
                const int c = w * CW + jj, i = lane + 64 * r;
                if (c < k && i < kstat) R[i + (int64_t)c * tk.rld] = (i <= c && i < kk) ? (T)a[jj][r] : T(0);
            }
    }
    // Explicit Q: columns c >= kk are zero, the others e_c - V x with S x = row c
    // of V, S the upper triangle of G with 1 / tau on its diagonal. V passes
    // through LDS RC row groups at a time; each wave solves for its own columns
    // (lane = entry of x) before the first group's products.
    double x[CW];
#pragma unroll 1
    for (int r0 = 0; r0 < RR; r0 += RC) {
        __syncthreads();                        // the last readers of buf
#pragma unroll
        for (int jj = 0; jj < CW; ++jj)
#pragma unroll
            for (int q = 0; q < RR; ++q) {
                if (q < r0 || q >= r0 + RC) continue;
                const int c = w * CW + jj, i = lane + 64 * q;
                Vs[c * VLD + i - 64 * r0] = i == c ? 1.0 : (i > c && c < kk ? a[jj][q] : 0.0);
            }
        __syncthreads();
        if (r0 == 0) {
            const double tau = lane < kk ? taus[lane] : 0.0;
#pragma unroll
            for (int jj = 0; jj < CW; ++jj) {
                const int c = w * CW + jj;
                x[jj] = lane <= c && c < kk ? Vs[min(lane, KMAX - 1) * VLD + c] : 0.0;
            }
#pragma unroll 1
            for (int l0 = KMAX - 8; l0 >= 0; l0 -= 8) {
                if (l0 > w * CW + CW - 1) continue;
                double g[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) g[u] = lane < l0 + u && l0 + u < kk ? G[l0 + u][min(lane, KMAX - 1)] : 0.0;
#pragma unroll
                for (int u = 7; u >= 0; --u)
#pragma unroll
                    for (int jj = 0; jj < CW; ++jj) {
                        x[jj] = lane == l0 + u ? tau * x[jj] : x[jj];
                        x[jj] = fma(-g[u], bcast(x[jj], l0 + u), x[jj]);
                    }
            }
        }
        const int top = min(kk, w * CW + CW);
        double q[CW][RC];
#pragma unroll
        for (int jj = 0; jj < CW; ++jj)
#pragma unroll
            for (int r = 0; r < RC; ++r) {
                const int c = w * CW + jj;
                q[jj][r] = lane + 64 * (r0 + r) == c && c < kk ? 1.0 : 0.0;
            }
#pragma unroll 4
        for (int l = 0; l < top; ++l) {
            double v[RC];
#pragma unroll
            for (int r = 0; r < RC; ++r) v[r] = Vs[l * VLD + lane + 64 * r];
#pragma unroll
            for (int jj = 0; jj < CW; ++jj) {
                const double xl = bcast(x[jj], l);
#pragma unroll
                for (int r = 0; r < RC; ++r) q[jj][r] = fma(-v[r], xl, q[jj][r]);
            }
        }
#pragma unroll
        for (int jj = 0; jj < CW; ++jj)
#pragma unroll
            for (int r = 0; r < RC; ++r) {
                const int c = w * CW + jj, i = lane + 64 * (r0 + r);
                if (c < k && i < m) A[i + (int64_t)c * ld] = (T)q[jj][r];
            }
    }
}

// Householder QR of one m x k panel, m <= 64, k <= KMAX: one column per group
// of LPC = 8 lanes, 8 rows per lane (rows 2 sub + 16 r and the next), a panel
// per workgroup of 8 KMAX threads.
// What bounds these panels is the instructions of a step, about 9 cycles each
// with one wave per SIMD, not memory: a sum over the 64 lanes of a wave costs
// 23 instructions per column, over a group of 8 lanes 9 for all the columns of
// a wave. Measured against lane = row with the columns split over the waves
// (FP64, k = 20): 80 panels of 64 rows 19.4 -> 15.3 us, 12,831 of them 466 ->
// 234 us.
// Step j: column j is in LDS as it stands; every lane forms its norm, its
// products with the lane's own column and, from these, tau and the scale of
// the reflector v, all in one pass of three sums, updates its column and the
// group of column j + 1 publishes. One barrier per step.
// Q is not accumulated by a second pass over the reflectors: Q = E - V T V1^T
// with V1 the first k rows of V, and T^-1 is 1 / tau on the diagonal and the
// products v_l . v_j above it, which step j yields for the columns left of j.
// Each group solves for its own column of T V1^T (KMAX entries, held by every
// lane) and multiplies by V from LDS.
template <typename T, int KMAX>
__global__ void __launch_bounds__(KMAX * 8) qr_group_kernel(Bases b, const QrTask* __restrict__ tasks)
{
    constexpr int LPC = 8, NP = 4;              // lanes per column, row pairs per lane
    constexpr int ROWS = 2 * LPC * NP, VLD = ROWS + 2;
    static_assert(KMAX <= ROWS && KMAX % 4 == 0 && (KMAX * LPC) % 64 == 0, "panel shape");
    typedef double d2 __attribute__((ext_vector_type(2)));
    __shared__ __align__(16) double xb[2][ROWS];
    __shared__ __align__(16) double Vs[KMAX][VLD];
    __shared__ __align__(16) double G[KMAX][KMAX];      // G[j][l] = -v_l . v_j, l < j
    __shared__ __align__(16) double taus[KMAX], scales[KMAX], betas[KMAX];
    const QrTask tk = tasks[blockIdx.x];
    T* A = reinterpret_cast<T*>(b.val[tk.slot]) + tk.off;
    const int m = tk.m, kstat = tk.k, ld = tk.ld;
    const int k = tk.krank >= 0 ? min(kstat, b.rank[tk.kslot][tk.krank]) : kstat, kk = min(m, k);
    if (k <= 0) return;
    const int c = threadIdx.x / LPC, sub = threadIdx.x % LPC;
    auto row = [&](int r, int e) { return 2 * sub + 2 * LPC * r + e; };
    double a[NP][2];
#pragma unroll
    for (int r = 0; r < NP; ++r)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int i = row(r, e);
            a[r][e] = (i < m && c < k) ? (double)A[i + (int64_t)c * ld] : 0.0;
        }
    auto publish = [&](double* x) {
#pragma unroll
        for (int r = 0; r < NP; ++r) *reinterpret_cast<d2*>(x + row(r, 0)) = d2{a[r][0], a[r][1]};
    };
    if (c == 0) publish(xb[0]);
    // The last group of columns solved for may reach beyond the reflectors.
    if (threadIdx.x < KMAX) taus[threadIdx.x] = scales[threadIdx.x] = 0.0;
    for (int e = threadIdx.x; e < KMAX * KMAX; e += KMAX * LPC) G[e / KMAX][e % KMAX] = 0.0;
    __syncthreads();
    // Rows 2 LPC rb .. of the diagonal are register pair rb: the pairs above
    // it are done with, those below it need no masks.
    auto steps = [&](auto rbc) {
        constexpr int rb = decltype(rbc)::value;
#pragma unroll 1
        for (int j = 2 * LPC * rb; j < min(kk, 2 * LPC * (rb + 1)); ++j) {
            const double* xp = xb[j & 1];
            const double alpha = xp[j];
            d2 x[NP];
#pragma unroll
            for (int r = rb; r < NP; ++r) x[r] = *reinterpret_cast<const d2*>(xp + row(r, 0));
            const bool at0 = row(rb, 0) == j, at1 = row(rb, 1) == j;
            double aj = at0 ? a[rb][0] : 0.0;
            aj = group_sum<LPC>(at1 ? a[rb][1] : aj);
            x[rb][0] = row(rb, 0) > j ? x[rb][0] : 0.0;
            x[rb][1] = row(rb, 1) > j ? x[rb][1] : 0.0;
            d2 xx = {0.0, 0.0}, xa = {0.0, 0.0};
#pragma unroll
            for (int r = rb; r < NP; ++r)
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    xx[e] = fma(x[r][e], x[r][e], xx[e]);
                    xa[e] = fma(x[r][e], a[r][e], xa[e]);
                }
            const double xn2 = group_sum<LPC>(xx[0] + xx[1]);
            const double dot = group_sum<LPC>(xa[0] + xa[1]);
            double t = 0.0, scale = 0.0, beta = alpha;
            const double n2 = fma(alpha, alpha, xn2);
            if (xn2 > 0.0 && n2 > kTinyColumn) householder<HwEst>(alpha, n2, t, scale, beta);
            const double d = fma(scale, dot, aj);       // v . (this column)
            if (c > j) {
                const double f = t * d, fs = f * scale;
#pragma unroll
                for (int r = rb; r < NP; ++r)
#pragma unroll
                    for (int e = 0; e < 2; ++e) a[r][e] = fma(-fs, x[r][e], a[r][e]);
                a[rb][0] -= at0 ? f : 0.0;
                a[rb][1] -= at1 ? f : 0.0;
                if (c == j + 1) publish(xb[(j + 1) & 1]);
            } else if (sub == 0) {
                // Column j stays as it is (times scale: v); its beta and scale are kept.
                if (c < j) G[j][c] = d;
                else { taus[j] = t; scales[j] = scale; betas[j] = beta; }
            }
            __syncthreads();
        }
    };
    steps(std::integral_constant<int, 0>{});
    if constexpr (2 * LPC < KMAX) steps(std::integral_constant<int, 1>{});
    if constexpr (4 * LPC < KMAX) steps(std::integral_constant<int, 2>{});
    static_assert(6 * LPC >= KMAX, "diagonal blocks");
    const double own = scales[c];
    if (tk.roff >= 0) {
        T* R = reinterpret_cast<T*>(b.val[SLOT_WS]) + tk.roff;
        const double beta = betas[c];
#pragma unroll
        for (int r = 0; r < NP; ++r)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int i = row(r, e);
                if (2 * LPC * r < KMAX && c < k && i < kstat)
                    R[i + (int64_t)c * tk.rld] = (T)(i < kk && i <= c ? (i == c ? beta : a[r][e]) : 0.0);
            }
    }
#pragma unroll
    for (int r = 0; r < NP; ++r) {
        d2 v;
#pragma unroll
        for (int e = 0; e < 2; ++e) v[e] = row(r, e) == c ? 1.0 : (row(r, e) > c ? a[r][e] * own : 0.0);
        *reinterpret_cast<d2*>(&Vs[c][row(r, 0)]) = v;
    }
    // The products of step j met column l before its scale.
    for (int e = threadIdx.x; e < KMAX * KMAX; e += KMAX * LPC) G[e / KMAX][e % KMAX] *= -scales[e % KMAX];
    __syncthreads();
    // x := T V1^T e_c by back substitution (columns from kk on: zero).
    double x[KMAX];
#pragma unroll
    for (int l = 0; l < KMAX; ++l) x[l] = c < kk ? Vs[l][c] : 0.0;
#pragma unroll
    for (int g = KMAX / 4 - 1; g >= 0; --g) {
        if (4 * g < kk) {
#pragma unroll
            for (int u = 3; u >= 0; --u) {
                const int l = 4 * g + u;
                x[l] *= taus[l];
#pragma unroll
                for (int i = 0; i < l; ++i) x[i] = fma(G[l][i], x[l], x[i]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < NP; ++r)
#pragma unroll
        for (int e = 0; e < 2; ++e) a[r][e] = row(r, e) == c && c < kk ? 1.0 : 0.0;
#pragma unroll
    for (int g = 0; g < KMAX / 4; ++g) {
        if (4 * g < kk) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int r = 0; r < NP; ++r) {
                    const int l = 4 * g + u;
                    const d2 v = *reinterpret_cast<const d2*>(&Vs[l][row(r, 0)]);
                    a[r][0] = fma(-x[l], v[0], a[r][0]);
                    a[r][1] = fma(-x[l], v[1], a[r][1]);
                }
        }
    }
#pragma unroll
    for (int r = 0; r < NP; ++r)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int i = row(r, e);
            if (c < k && i < m) A[i + (int64_t)c * ld] = (T)a[r][e];
        }
}

// Panel classes of a QR phase (tasks are sorted by class at upload):
// 0: m <= 64, 1: m <= 256, 2: m <= 512 (k <= 40), 3: m <= 1024 with k <= 24,
// 4: the rest (qr_kernel). Class 0 takes the kernel with a column per 8 lanes,
// 1-3 the column-split kernel with 256, 512 and 1024 rows in registers: the
// share of the sums over lanes, which the first one shortens, falls with the
// rows (panels of 200 rows with 16 lanes per column: 2,967 of them 271 us
// against 217, 80 of them 21.5 against 23.5).
template <typename T, int KMAX>
static void launch_qr_classes(const QrTask* tasks, const int* classEnd, const Bases& b, hipStream_t s)
{
    constexpr int NWV = KMAX == 24 ? 12 : 10;      // 2 or 4 columns per wave
    int begin = 0;
    for (int c = 0; c < 4; ++c) {
        const int n = classEnd[c] - begin;
        if (n > 0) {
            const QrTask* t = tasks + begin;
            if (c == 0) {
                qr_group_kernel<T, KMAX><<<n, 8 * KMAX, 0, s>>>(b, t);
            } else if (c == 1) {
                qr_split_kernel<T, KMAX, NWV, 4><<<n, 64 * NWV, 0, s>>>(b, t);
            } else if (c == 2) {
                qr_split_kernel<T, KMAX, NWV, 8><<<n, 64 * NWV, 0, s>>>(b, t);
            } else {
                qr_split_kernel<T, 24, 12, 16><<<n, 768, 0, s>>>(b, t);    // class 3 has k <= 24
            }
        }
        begin = classEnd[c];
    }
}

template <typename T>
void launch_qr_phase(const Phase& ph, const Bases& b, hipStream_t s)
{
    const int n = (int)ph.qr.size();
    if (n == 0) return;
    const QrTask* tasks = static_cast<const QrTask*>(ph.dTasks);
    if (ph.qrClassEnd[3] > 0) {
        if (ph.qrRegK <= 24) launch_qr_classes<T, 24>(tasks, ph.qrClassEnd, b, s);
        else launch_qr_classes<T, 40>(tasks, ph.qrClassEnd, b, s);
    }
    const int big = ph.qrClassEnd[3];
    if (n > big) qr_kernel<T><<<n - big, 256, 0, s>>>(b, tasks + big);
    HIP_LAUNCH_CHECK();
}
template void launch_qr_phase<double>(const Phase&, const Bases&, hipStream_t);
template void launch_qr_phase<float>(const Phase&, const Bases&, hipStream_t);

} // namespace dmhm
