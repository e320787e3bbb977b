// gfx950 kernels of the recursive direct inversion (HMat2d/HMat3d::
// DirectInvert, src/HMat2d/Invert-incl.hpp:17-125) and of merged plans: the
// dense leaf inverse (hmat_tools::Invert on a Dense, src/hmat_tools/
// Invert.cpp:14-42, there LAPACK getrf + getri), and copies and fills of index
// ranges inside one allocation (sub-matrix copies: a subtree of the block
// tree is one contiguous range of each storage pool).
#include "kcommon.hpp"

namespace dmhm {

// vals[d + e] = vals[s + e] (copy) or vals[d + e] = 0 (fill) for every range
// (s, d, len) of one step, the value ranges (blockIdx.y < nVal) and the rank
// ranges in one launch.
template <typename T, bool FILL>
__global__ void ranges2_kernel(T* __restrict__ vals, int* __restrict__ ranks, const CopyRange* __restrict__ rs, int nVal)
{
    const int y = blockIdx.y;
    const CopyRange r = rs[y];
    if (y < nVal) {
        for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < r.len; e += (int64_t)gridDim.x * blockDim.x)
            vals[r.dst + e] = FILL ? T(0) : vals[r.src + e];
    } else {
        for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < r.len; e += (int64_t)gridDim.x * blockDim.x)
            ranks[r.dst + e] = FILL ? 0 : ranks[r.src + e];
    }
}

template <typename T>
void launch_arena_ranges(T* vals, int* ranks, const CopyRange* ranges, int nVal, int nRank, int64_t maxLen, bool fill,
                         hipStream_t s)
{
    const int count = nVal + nRank;
    if (count <= 0 || maxLen <= 0) return;
    if (count > 65535) throw std::invalid_argument("too many ranges in one launch");
    const dim3 grid((unsigned)std::min<int64_t>((maxLen + 255) / 256, 2048), (unsigned)count);
    if (fill) ranges2_kernel<T, true><<<grid, 256, 0, s>>>(vals, ranks, ranges, nVal);
    else ranges2_kernel<T, false><<<grid, 256, 0, s>>>(vals, ranks, ranges, nVal);
    HIP_LAUNCH_CHECK();
}

// In-place Gauss-Jordan inversion with partial pivoting of one m x m
// column-major matrix (leading dimension m) by one workgroup of NT threads:
// at step k the pivot row p (largest |a(i,k)|, i >= k) is swapped into row k,
// then every entry is updated from the saved column k and the scaled row k;
// the row swaps are undone as column swaps in reverse order at the end. The
// matrix is worked on in dst (copied from src first). A zero pivot sets *singular.
template <typename T, int NT>
__global__ __launch_bounds__(NT) void dense_inverse_kernel(const T* __restrict__ src, T* __restrict__ dst, int m,
                                                           int* __restrict__ singular)
{
    extern __shared__ __align__(16) unsigned char smem[];
    T* col = reinterpret_cast<T*>(smem);              // saved column k (m)
    T* row = col + m;                                 // scaled row k (m)
    int* piv = reinterpret_cast<int*>(row + m);       // pivot rows (m)
    __shared__ int pivot;
    T* a = dst;
    const int tid = threadIdx.x;
    const int mm = m * m;
    for (int e = tid; e < mm; e += NT) a[e] = src[e];
    __syncthreads();
    for (int k = 0; k < m; ++k) {
        if (tid < 64) {
            // Pivot search by the first wave: largest magnitude, lowest row on ties.
            double best = -1.0;
            int bi = k;
            for (int i = k + tid; i < m; i += 64) {
                const double v = fabs((double)a[i + (int64_t)k * m]);
                if (v > best) { best = v; bi = i; }
            }
            for (int o = 32; o > 0; o >>= 1) {
                const double ov = __shfl_xor(best, o, 64);
                const int oi = __shfl_xor(bi, o, 64);
                if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
            }
            if (tid == 0) { pivot = bi; piv[k] = bi; }
        }
        __syncthreads();
        const int p = pivot;
        if (p != k)
            for (int j = tid; j < m; j += NT) {
                const T t = a[k + (int64_t)j * m];
                a[k + (int64_t)j * m] = a[p + (int64_t)j * m];
                a[p + (int64_t)j * m] = t;
            }
        __syncthreads();
        const T d = a[k + (int64_t)k * m];
        if (d == T(0) && tid == 0) atomicExch(singular, 1);
        const T inv = d == T(0) ? T(0) : T(1) / d;
        for (int i = tid; i < m; i += NT) {
            col[i] = a[i + (int64_t)k * m];
            row[i] = a[k + (int64_t)i * m] * inv;
        }
        __syncthreads();
        for (int e = tid; e < mm; e += NT) {
            const int i = e % m, j = e / m;
            T v;
            if (i == k) v = j == k ? inv : row[j];
            else v = j == k ? -col[i] * inv : a[e] - col[i] * row[j];
            a[e] = v;
        }
        __syncthreads();
    }
    for (int k = m - 1; k >= 0; --k) {
        const int p = piv[k];
        if (p != k)
            for (int i = tid; i < m; i += NT) {
                const T t = a[i + (int64_t)k * m];
                a[i + (int64_t)k * m] = a[i + (int64_t)p * m];
                a[i + (int64_t)p * m] = t;
            }
        __syncthreads();
    }
}

// Largest unsigned value over the wave (DPP within rows of 16, then the four
// row maxima through scalar registers); the result is uniform.
__device__ inline uint32_t wave_max_u32(uint32_t x)
{
    x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, kDppXor1, 0xF, 0xF, false));
    x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, kDppXor2, 0xF, 0xF, false));
    x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, kDppMirror8, 0xF, 0xF, false));
    x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, kDppMirror16, 0xF, 0xF, false));
    const uint32_t a = __builtin_amdgcn_readlane(x, 0), b = __builtin_amdgcn_readlane(x, 16);
    const uint32_t c = __builtin_amdgcn_readlane(x, 32), e = __builtin_amdgcn_readlane(x, 48);
    return max(max(a, b), max(c, e));
}

// Inverse of one m x m leaf (m <= 64): Gauss-Jordan with partial pivoting,
// lane = row, the 64 columns split over NWV waves (wave w holds columns
// [w CW, (w + 1) CW) of every row in registers). Three departures from the
// textbook form keep a panel of CW steps to one barrier and one LDS exchange:
// - rows are not exchanged: step k takes the largest |u(i,k)| over the rows
//   not yet used as pivots (compared on the high word of the double: sign
//   cleared, exponent and 20 mantissa bits, ties to the lowest row) and
//   records the pivot row p_k. The elimination then leaves
//   inv(A)(k, p_j) = T(p_k, j) for the final array T, applied at the store;
// - the pivot row is not scaled by 1/u(p,k) at its step: the factor of every
//   other row is u(i,k) / u(p,k) either way, so the scale is kept per row and
//   applied at the store (the row's entries stay, its column-k entry is 1);
// - the wave that owns columns k .. k + CW - 1 takes all their steps on its own
//   columns alone (they need no other wave's) and publishes the CW pivot rows'
//   indices and every row's factors through LDS; the other waves then apply the
//   CW steps to their own columns, reading their share of each pivot row from
//   their own lane p (v_readlane), the next panel's wave ahead of the others.
//   Buffers alternate by panel parity, so a panel's writes never meet the
//   previous one's reads: one barrier per panel.
// Padding rows and columns beyond m hold the identity; their steps (up to
// CW - 1 in the last panel) change nothing.
template <typename T, int NWV>
__global__ void __launch_bounds__(64 * NWV) dense_inverse_split_kernel(const T* __restrict__ src,
                                                                      T* __restrict__ dst, int m,
                                                                      int* __restrict__ singular)
{
    constexpr int CW = 64 / NWV;
    __shared__ double gbuf[2][CW][64], scales[64];      // scales: of the steps' pivot rows
    __shared__ int pivs[64], steps[64];                 // pivot row of a step, step of a row
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double u[CW];
#pragma unroll
    for (int j = 0; j < CW; ++j) {
        const int c = w * CW + j;
        u[j] = (c < m && lane < m) ? (double)src[lane + (int64_t)c * m] : (c == lane ? 1.0 : 0.0);
    }
    bool sing = false;
    uint64_t used = 0;              // rows that have been pivots
    const int panels = (m + CW - 1) / CW;
#pragma unroll 1
    for (int kb = 0; kb < panels; ++kb) {
        const int par = kb & 1;
        if (w == kb) {
#pragma unroll
            for (int kk = 0; kk < CW; ++kk) {
                const double v = u[kk];
                const uint32_t hi = used >> lane & 1 ? 0u : ((uint32_t)__double2hiint(v) & 0x7fffffffu);
                const uint32_t mx = wave_max_u32(hi);
                const uint64_t cand = __ballot(hi == mx) & ~used;
                const int p = __builtin_ctzll(cand);
                const double dd = bcast(v, p);
                const double inv = dd == 0.0 ? 0.0 : rcp_nr(dd);
                const double g = lane == p ? 0.0 : v * inv;
                gbuf[par][kk][lane] = g;
                if (lane == p) {
                    pivs[kb * CW + kk] = p;
                    scales[kb * CW + kk] = inv;
                    steps[p] = kb * CW + kk;
                }
                sing = sing || dd == 0.0;
                used |= uint64_t(1) << p;
#pragma unroll
                for (int j = 0; j < CW; ++j)
                    u[j] = j == kk ? (lane == p ? 1.0 : -g) : fma(-g, bcast(u[j], p), u[j]);
            }
        }
        __syncthreads();
        if (w == kb) {
            __builtin_amdgcn_s_setprio(0);
            continue;
        }
        if (w == kb + 1) __builtin_amdgcn_s_setprio(3);
        const int pl = pivs[kb * CW + lane % CW];
#pragma unroll
        for (int kk = 0; kk < CW; ++kk) {
            const int p = __builtin_amdgcn_readlane(pl, kk);
            const double g = gbuf[par][kk][lane];
            used |= uint64_t(1) << p;
#pragma unroll
            for (int j = 0; j < CW; ++j) u[j] = fma(-g, bcast(u[j], p), u[j]);
        }
    }
    if (sing && lane == 0) atomicExch(singular, 1);
    // A row beyond m is its own pivot in a step beyond m, or in none.
    const int step = used >> lane & 1 ? steps[lane] : 64;
    const double scale = step < m ? scales[step] : 0.0;
    const bool row = lane < m && step < m;
#pragma unroll
    for (int j = 0; j < CW; ++j) {
        const int c = w * CW + j;
        if (row && c < m && pivs[c] < m) dst[step + (int64_t)pivs[c] * m] = (T)(u[j] * scale);
    }
}

// The same elimination for a leaf of up to 64 RR rows, worked on in memory
// (`work`, overwritten) in panels of NB columns: the first wave takes a panel's
// steps in registers (rows lane + 64 r) and publishes its pivots and factors,
// then every wave applies the NB steps to whole columns in one read and one
// write of each. One step per pass over the matrix, as dense_inverse_kernel
// takes, is bound by that traffic through one CU. Direct inversion of 88^2 in
// leaves of 121 points (FP64, rank 8): 89.7 -> 22.2 ms, of 120^2 in leaves of
// 225 points 415 -> 117 ms (290 ms with panels of 8 at four rows a lane, 128 ms
// with 8 columns and 8 waves; in panels of 4 too the compiler keeps 144 bytes
// per lane of the four rows' arrays in scratch).
template <typename T, int RR>
__global__ void __launch_bounds__(1024) dense_inverse_panel_kernel(T* work, T* __restrict__ dst, int m,
                                                                   int* __restrict__ singular)
{
    constexpr int NB = RR <= 2 ? 8 : 4, NW = 16;
    __shared__ double G[NB][64 * RR], scales[64 * RR];
    __shared__ int pivs[64 * RR], steps[64 * RR];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Entry of row p of a column held as rows lane + 64 r (p uniform).
    auto at = [&](const double (&x)[RR], int p) {
        double v = x[0];
#pragma unroll
        for (int r = 1; r < RR; ++r) v = p >> 6 == r ? x[r] : v;
        return bcast(v, p & 63);
    };
    uint64_t used[RR] = {};         // rows that have been pivots (kept by the first wave)
    bool sing = false;
#pragma unroll 1
    for (int k0 = 0; k0 < m; k0 += NB) {
        const int nb = min(NB, m - k0);
        if (w == 0) {
            double u[NB][RR];
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int r = 0; r < RR; ++r) {
                    const int i = lane + 64 * r;
                    u[j][r] = j < nb && i < m ? (double)work[i + (int64_t)(k0 + j) * m] : 0.0;
                }
#pragma unroll
            for (int kk = 0; kk < NB; ++kk) {
                if (kk >= nb) continue;
                uint32_t hi[RR], mine = 0;
#pragma unroll
                for (int r = 0; r < RR; ++r) {
                    const bool open = lane + 64 * r < m && !(used[r] >> lane & 1);
                    hi[r] = open ? (uint32_t)__double2hiint(u[kk][r]) & 0x7fffffffu : 0u;
                    mine = max(mine, hi[r]);
                }
                const uint32_t mx = wave_max_u32(mine);
                uint64_t cand[RR];
                int tied = 0;
#pragma unroll
                for (int r = 0; r < RR; ++r) {
                    cand[r] = __ballot(lane + 64 * r < m && hi[r] == mx) & ~used[r];
                    tied += __popcll(cand[r]);
                }
                if (tied > 1) {                 // equal to 20 bits: the low words decide
                    uint32_t lo[RR];
                    mine = 0;
#pragma unroll
                    for (int r = 0; r < RR; ++r) {
                        lo[r] = (uint32_t)__double2loint(u[kk][r]);
                        mine = cand[r] >> lane & 1 ? max(mine, lo[r]) : mine;
                    }
                    const uint32_t ml = wave_max_u32(mine);
#pragma unroll
                    for (int r = 0; r < RR; ++r) cand[r] &= __ballot(lo[r] == ml);
                }
                int p = -1;
#pragma unroll
                for (int r = 0; r < RR; ++r)
                    if (p < 0 && cand[r]) {
                        p = 64 * r + __builtin_ctzll(cand[r]);
                        used[r] |= cand[r] & (~cand[r] + 1);
                    }
                p = __builtin_amdgcn_readfirstlane(p);
                const double dd = at(u[kk], p);
                const double inv = dd == 0.0 ? 0.0 : rcp_nr(dd);
                sing = sing || dd == 0.0;
                double g[RR];
#pragma unroll
                for (int r = 0; r < RR; ++r) {
                    g[r] = lane + 64 * r == p ? 0.0 : u[kk][r] * inv;
                    G[kk][lane + 64 * r] = g[r];
                }
                if (lane == 0) { pivs[k0 + kk] = p; scales[k0 + kk] = inv; steps[p] = k0 + kk; }
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    const double x = at(u[j], p);
#pragma unroll
                    for (int r = 0; r < RR; ++r)
                        u[j][r] = j == kk ? (lane + 64 * r == p ? 1.0 : -g[r]) : fma(-g[r], x, u[j][r]);
                }
            }
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int r = 0; r < RR; ++r) {
                    const int i = lane + 64 * r;
                    if (j < nb && i < m) work[i + (int64_t)(k0 + j) * m] = (T)u[j][r];
                }
        }
        __syncthreads();
        double g[NB][RR];
#pragma unroll
        for (int kk = 0; kk < NB; ++kk)
#pragma unroll
            for (int r = 0; r < RR; ++r) g[kk][r] = kk < nb ? G[kk][lane + 64 * r] : 0.0;
        const int pl = pivs[k0 + min(lane, nb - 1)];
#pragma unroll 1
        for (int c = w; c < m; c += NW) {
            if (c >= k0 && c < k0 + nb) continue;
            T* col = work + (int64_t)c * m;
            double x[RR];
#pragma unroll
            for (int r = 0; r < RR; ++r) x[r] = lane + 64 * r < m ? (double)col[lane + 64 * r] : 0.0;
#pragma unroll
            for (int kk = 0; kk < NB; ++kk) {
                if (kk >= nb) continue;
                const double v = at(x, __builtin_amdgcn_readlane(pl, kk));
#pragma unroll
                for (int r = 0; r < RR; ++r) x[r] = fma(-g[kk][r], v, x[r]);
            }
#pragma unroll
            for (int r = 0; r < RR; ++r)
                if (lane + 64 * r < m) col[lane + 64 * r] = (T)x[r];
        }
        __syncthreads();
    }
    if (sing && threadIdx.x == 0) atomicExch(singular, 1);
    for (int c = w; c < m; c += NW) {
        const int pc = pivs[c];
#pragma unroll
        for (int r = 0; r < RR; ++r) {
            const int i = lane + 64 * r;
            if (i < m) dst[steps[i] + (int64_t)pc * m] = (T)((double)work[i + (int64_t)c * m] * scales[steps[i]]);
        }
    }
}

// Waves of the leaf inversion. What bounds it is the instructions of the wave
// that owns the panel: its own steps (the pivot search and reciprocal, then a
// lane read and an FMA per column) and the steps of the panel before it. A 64 x
// 64 FP64 leaf: 29.0 us with a barrier and an exchange per column, 25.5 us per
// panel of 8 columns (8 waves), 20.9 us per panel of 4 (16 waves), a launch of
// about 4 us included; 108 us for lane = column with rows split over 8 waves.
constexpr int kInvWaves = 16;

// `src` is overwritten (m in 65 .. 256).
template <typename T>
void launch_dense_inverse(T* src, T* dst, int m, int* singular, hipStream_t s)
{
    if (m <= 0) return;
    if (m <= 64) {
        dense_inverse_split_kernel<T, kInvWaves><<<1, 64 * kInvWaves, 0, s>>>(src, dst, m, singular);
        HIP_LAUNCH_CHECK();
        return;
    }
    if (m <= 256) {
        if (m <= 128) dense_inverse_panel_kernel<T, 2><<<1, 1024, 0, s>>>(src, dst, m, singular);
        else dense_inverse_panel_kernel<T, 4><<<1, 1024, 0, s>>>(src, dst, m, singular);
        HIP_LAUNCH_CHECK();
        return;
    }
    const size_t vecs = 2 * (size_t)m * sizeof(T) + (((size_t)m + 3) & ~size_t(3)) * sizeof(int);
    if (vecs > 64 * 1024) throw std::invalid_argument("dense leaf too large to invert");
    dense_inverse_kernel<T, 512><<<1, 512, vecs, s>>>(src, dst, m, singular);
    HIP_LAUNCH_CHECK();
}

#define INST(T)                                                                                          \
    template void launch_arena_ranges<T>(T*, int*, const CopyRange*, int, int, int64_t, bool, hipStream_t); \
    template void launch_dense_inverse<T>(T*, T*, int, int*, hipStream_t);
INST(double)
INST(float)

} // namespace dmhm
