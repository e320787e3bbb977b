// gfx950 streaming H*X and H^T*X kernels for few right-hand sides (HBM-bound).
#include "kcommon.hpp"

namespace dmhm {

// ---------------------------------------------------------------------------
// Streaming H*X and H^T*X (K right-hand sides). Every factor entry is read
// once; what bounds both launches is HBM once the matrix is larger than the
// 256 MB cache, and otherwise the chain of dependent loads of one wave.
//
// mv_proj: P(j, kk) = sum_r V(r, j) X(r, kk) per admissible block (U and the
//   target rows for H^T). A block of at most kMvBigRows rows is one wave's, a
//   taller one a workgroup's, whose four waves take every fourth 64 rows and
//   add their sums through LDS: P is written once, with no atomics and nothing
//   to clear. The factor is read with 16-byte loads: a lane owns VW = 16 /
//   sizeof(T) consecutive rows, LPC = 64 / VW lanes cover 64 rows of one
//   column and the VW lane groups of a wave walk different columns (1 KiB per
//   load instruction); DPP row sums finish each column.
// mv_acc: one workgroup of NW waves per output row atom (<= 64 rows, lane =
//   row). The atom's contributions (dense leaves D X, low-rank U P) come as
//   records of at most 16 columns, dealt to the waves in turn and read 64 at
//   a time, one record per lane; a wave issues the 16 column loads of its next
//   record (and the one or two loads that bring its R values, one per lane)
//   before the FMAs of the current one, whose R values are broadcast by lane
//   reads. One LDS reduction across the waves at the end.
//   For H^T the low-rank part is the same (V P over source rows); the dense
//   leaves contribute D^T X: a wave takes every NW-th leaf, reads its columns
//   as mv_proj does and keeps one sum per column until all its leaves are
//   done, so the cross-lane sums cost one pass per atom.
//
// The number of waves follows the number of atoms (mv_waves). Measured against
// one wave per 512 rows with atomic sums, four waves per atom walking whole
// contributions without prefetch, and tile products for H^T (one vector):
// H^T x 256^2 FP64 1073 -> 270 us (1.53 GB, 5.7 TB/s), H x 256^2 FP32 150 ->
// 138 us, 512^2 FP32 1277 -> 1235 us (7.26 GB, 5.9 TB/s), 64^2 FP64 42 -> 19 us,
// and six vectors on the 3D 27 x 33 x 30 inverse (FP32, 867 MB) 655 -> 188 us.
// ---------------------------------------------------------------------------
template <typename T> struct MvVec;
template <> struct MvVec<float> { typedef float type __attribute__((ext_vector_type(4), aligned(4))); };
template <> struct MvVec<double> { typedef double type __attribute__((ext_vector_type(2), aligned(8))); };

// acc[u][kk] += A(rows, c0 + cg + VW u) . X(rows, kk) over this lane's rows (VW
// consecutive ones at r0 + rg VW, + step, ..., below `rows`) of a column-major
// panel. CLAMP: column indices are clamped below ncol.
template <typename T, int K, int NA, bool CLAMP>
__device__ __forceinline__ void mv_columns_(const T* __restrict__ A, int64_t ld, const T* __restrict__ X, int64_t ldx,
                                            int c0, int ncol, int r0, int step, int rows, int rg, int cg,
                                            T (&acc)[NA][K])
{
    constexpr int VW = 16 / (int)sizeof(T);
    typedef typename MvVec<T>::type vec;
    const T* __restrict__ base = A + (CLAMP ? 0 : (c0 + cg) * ld);
    auto col = [&](int u) { return CLAMP ? min(c0 + cg + VW * u, ncol - 1) * ld : VW * u * ld; };
    for (int r = r0 + rg * VW; r < rows; r += step) {
        T xv[K][VW];
        vec lv[NA];
        if (r + VW <= rows) {
#pragma unroll
            for (int u = 0; u < NA; ++u) lv[u] = *reinterpret_cast<const vec*>(base + r + col(u));
#pragma unroll
            for (int kk = 0; kk < K; ++kk) {
                const vec v = *reinterpret_cast<const vec*>(X + r + kk * ldx);
#pragma unroll
                for (int e = 0; e < VW; ++e) xv[kk][e] = v[e];
            }
        } else {
            // The rows' last lane: entries beyond the end count as zero.
#pragma unroll
            for (int u = 0; u < NA; ++u)
#pragma unroll
                for (int e = 0; e < VW; ++e) lv[u][e] = r + e < rows ? base[r + e + col(u)] : T(0);
#pragma unroll
            for (int kk = 0; kk < K; ++kk)
#pragma unroll
                for (int e = 0; e < VW; ++e) xv[kk][e] = r + e < rows ? X[r + e + kk * ldx] : T(0);
        }
#pragma unroll
        for (int u = 0; u < NA; ++u)
#pragma unroll
            for (int kk = 0; kk < K; ++kk)
#pragma unroll
                for (int e = 0; e < VW; ++e) acc[u][kk] += lv[u][e] * xv[kk][e];
    }
}
template <typename T, int K, int NA>
__device__ __forceinline__ void mv_columns(const T* __restrict__ A, int64_t ld, const T* __restrict__ X, int64_t ldx,
                                           int c0, int ncol, int r0, int step, int rows, int rg, int cg,
                                           T (&acc)[NA][K])
{
    if (c0 + NA * (16 / (int)sizeof(T)) <= ncol) mv_columns_<T, K, NA, false>(A, ld, X, ldx, c0, ncol, r0, step, rows, rg, cg, acc);
    else mv_columns_<T, K, NA, true>(A, ld, X, ldx, c0, ncol, r0, step, rows, rg, cg, acc);
}

// Sum over the LPC lanes that share a column.
template <typename T>
__device__ __forceinline__ T mv_column_sum(T v)
{
    v = group_sum<16>(v);
    if constexpr (sizeof(T) == 8) v += __shfl_xor(v, 16, 64);
    return v;
}

template <typename T, int K>
__global__ void __launch_bounds__(256) mv_proj_kernel(Bases b, const MvProjItem* __restrict__ items, int n, int nBig,
                                                      int ldx)
{
    constexpr int VW = 16 / (int)sizeof(T);
    constexpr int LPC = 64 / VW;                // lanes per column
    constexpr int NC = K <= 2 ? 16 : 8;         // columns per pass
    constexpr int UN = NC / VW;                 // of one lane
    __shared__ T part[4][NC][K];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = (int)blockIdx.x;
    const bool big = g < nBig;                  // uniform across the workgroup
    const int id = big ? g : nBig + (g - nBig) * 4 + w;
    if (id >= n) return;
    const MvProjItem it = items[id];
    const int rank = min(it.cap, b.rank[SLOT_A][it.rankIdx]);
    if (rank <= 0) return;
    const int rg = lane % LPC, cg = lane / LPC;
    const T* __restrict__ V = reinterpret_cast<const T*>(b.val[SLOT_A]) + it.voff;
    const T* __restrict__ X = reinterpret_cast<const T*>(b.val[SLOT_X]) + it.xrow;
    T* P = reinterpret_cast<T*>(b.val[SLOT_WS]) + it.poff;
    for (int j0 = 0; j0 < rank; j0 += NC) {
        T acc[UN][K];
#pragma unroll
        for (int u = 0; u < UN; ++u)
#pragma unroll
            for (int kk = 0; kk < K; ++kk) acc[u][kk] = T(0);
        mv_columns<T, K, UN>(V, it.ldv, X, ldx, j0, rank, big ? 64 * w : 0, big ? 256 : 64, it.rows, rg, cg, acc);
#pragma unroll
        for (int u = 0; u < UN; ++u)
#pragma unroll
            for (int kk = 0; kk < K; ++kk) acc[u][kk] = mv_column_sum(acc[u][kk]);
        if (!big) {
            if (rg == 0)
#pragma unroll
                for (int u = 0; u < UN; ++u) {
                    const int j = j0 + cg + VW * u;
                    if (j >= rank) continue;
#pragma unroll
                    for (int kk = 0; kk < K; ++kk) P[j + (int64_t)kk * it.cap] = acc[u][kk];
                }
            continue;
        }
        if (rg == 0)
#pragma unroll
            for (int u = 0; u < UN; ++u)
#pragma unroll
                for (int kk = 0; kk < K; ++kk) part[w][cg + VW * u][kk] = acc[u][kk];
        __syncthreads();
        for (int e = threadIdx.x; e < NC * K; e += 256) {
            const int c = e % NC, kk = e / NC;
            if (j0 + c < rank)
                P[j0 + c + (int64_t)kk * it.cap] = (part[0][c][kk] + part[1][c][kk]) + (part[2][c][kk] + part[3][c][kk]);
        }
        __syncthreads();
    }
}

// One wave's records of an output atom: columns of L (lane = row) times R.
template <typename T, int K>
struct MvAcc {
    static constexpr int NR = (K + 3) / 4;      // loads that bring 16 x K values, one per lane
    struct Frag { T l[16]; T r[NR]; int q; };
    const T* __restrict__ H;
    const T* __restrict__ X;
    const T* __restrict__ WS;
    int lane, row, ldx;         // row: the lane's row, clamped to the atom
    // lane records
    int64_t dl, dr;
    int dld, dldr, dq, dkind;
    T acc[K];

    static __device__ __forceinline__ int64_t lane_i64(int64_t v, int i)
    {
        const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)v, i);
        const uint32_t hi = __builtin_amdgcn_readlane((int)(v >> 32), i);
        return (int64_t)((uint64_t)hi << 32 | lo);
    }
    // Loads of record i; columns beyond its q are read at the last one.
    template <bool TAIL>
    __device__ __forceinline__ void fetch(int i, Frag& f)
    {
        const int64_t ld = __builtin_amdgcn_readlane(dld, i);
        const int q = __builtin_amdgcn_readlane(dq, i);
        const int kind = __builtin_amdgcn_readlane(dkind, i);
        const int64_t ldr = kind == 0 ? ldx : __builtin_amdgcn_readlane(dldr, i);
        const T* __restrict__ L = H + lane_i64(dl, i) + row;
        const T* __restrict__ R = (kind == 0 ? X : WS) + lane_i64(dr, i);
        f.q = q;
#pragma unroll
        for (int j = 0; j < NR; ++j)
            f.r[j] = R[min(lane & 15, q - 1) + min(4 * j + (lane >> 4), K - 1) * ldr];
#pragma unroll
        for (int u = 0; u < 16; ++u) f.l[u] = L[(TAIL ? min(u, q - 1) : u) * ld];
    }
    // A record's products are summed by themselves: a wave's sum over all its
    // records is hundreds of terms long, and as one chain it was off by 4.0e-7
    // (256^2, FP32, one vector, relative to the result).
    template <bool TAIL>
    __device__ __forceinline__ void use(const Frag& f)
    {
        T sum[K];
#pragma unroll
        for (int kk = 0; kk < K; ++kk) sum[kk] = f.l[0] * bcast(f.r[kk >> 2], 16 * (kk & 3));
#pragma unroll
        for (int u = 1; u < 16; ++u) {
            if (TAIL && u >= f.q) continue;     // uniform
#pragma unroll
            for (int kk = 0; kk < K; ++kk) sum[kk] += f.l[u] * bcast(f.r[kk >> 2], 16 * (kk & 3) + u);
        }
#pragma unroll
        for (int kk = 0; kk < K; ++kk) acc[kk] += sum[kk];
    }
    template <bool TAIL>
    __device__ __forceinline__ void run(uint64_t left)
    {
        if (left == 0) return;
        // After the last record the fetch repeats it, so that the wait before
        // use(f) is "all but the newest record" on every path.
        int i = 0;
        auto next = [&]() -> bool {
            if (left == 0) return false;
            i = __builtin_ctzll(left);
            left &= left - 1;
            return true;
        };
        Frag f0, f1;
        next();
        fetch<TAIL>(i, f0);
        while (true) {
            const bool more1 = next();
            fetch<TAIL>(i, f1);
            use<TAIL>(f0);
            if (!more1) break;
            const bool more0 = next();
            fetch<TAIL>(i, f0);
            use<TAIL>(f1);
            if (!more0) break;
        }
    }
    // Records c0, c0 + step, ... below ce.
    __device__ __forceinline__ void records(const MvContrib* __restrict__ cs, const int* __restrict__ ranks, int c0,
                                            int ce, int step)
    {
        for (int at = c0; at < ce; at += 64 * step) {
            const int c = at + lane * step;
            const bool in = c < ce;
            const MvContrib& C = cs[in ? c : at];
            dl = C.loff; dr = C.roff; dld = C.ld; dldr = C.ldr; dkind = C.kind; dq = C.q;
            if (C.kind == 1) dq = min(dq, ranks[C.rankIdx] - C.p0);
            run<false>(__ballot(in && dq == 16));
            run<true>(__ballot(in && dq > 0 && dq < 16));
        }
    }
};

template <typename T, int K, int NW, bool TR>
__global__ void __launch_bounds__(64 * NW) mv_acc_kernel(Bases b, const MvAtom* __restrict__ atoms,
                                                         const MvContrib* __restrict__ cs, int ldx, int ldy, T alpha,
                                                         T beta)
{
    __shared__ T red[NW][K][64];
    const MvAtom at = atoms[blockIdx.x];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = threadIdx.x & 63;
    MvAcc<T, K> a;
    a.H = reinterpret_cast<const T*>(b.val[SLOT_A]);
    a.X = reinterpret_cast<const T*>(b.val[SLOT_X]);
    a.WS = reinterpret_cast<const T*>(b.val[SLOT_WS]);
    a.lane = i; a.row = min(i, at.m - 1); a.ldx = ldx;
#pragma unroll
    for (int kk = 0; kk < K; ++kk) a.acc[kk] = T(0);
    a.records(cs, b.rank[SLOT_A], at.cb + w, at.ce, NW);
#pragma unroll
    for (int kk = 0; kk < K; ++kk) red[w][kk][i] = a.acc[kk];
    if constexpr (TR) {
        // Dense leaves: y(c) += D(:, c)^T x, NA x VW columns per pass.
        constexpr int VW = 16 / (int)sizeof(T), LPC = 64 / VW;
        constexpr int NA = K <= 2 ? (NW == 16 ? 4 : 8) / K : 2;     // 16 waves have 128 registers each
        const int rg = i % LPC, cg = i / LPC;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");     // red[w] was written by the wave's other lanes
        for (int c0 = 0; c0 < at.m; c0 += NA * VW) {
            T acc[NA][K];
#pragma unroll
            for (int u = 0; u < NA; ++u)
#pragma unroll
                for (int kk = 0; kk < K; ++kk) acc[u][kk] = T(0);
            for (int c = at.db + w; c < at.de; c += NW) {
                const MvContrib& C = cs[c];
                mv_columns<T, K, NA>(a.H + C.loff, C.ld, a.X + C.roff, ldx, c0, at.m, 0, 64, C.ld, rg, cg, acc);
            }
#pragma unroll
            for (int u = 0; u < NA; ++u)
#pragma unroll
                for (int kk = 0; kk < K; ++kk) {
                    const T v = mv_column_sum(acc[u][kk]);
                    const int c = c0 + cg + VW * u;
                    if (rg == 0 && c < at.m) red[w][kk][c] += v;
                }
        }
    }
    __syncthreads();
    // Rows of the result, summed over the waves in order.
    for (int e = threadIdx.x; e < 64 * K; e += 64 * NW) {
        const int r = e & 63, kk = e >> 6;
        if (r >= at.m) continue;
        T sum = red[0][kk][r];
#pragma unroll
        for (int x = 1; x < NW; ++x) sum += red[x][kk][r];
        T* y = reinterpret_cast<T*>(b.val[SLOT_Y]) + at.yrow + r + (int64_t)kk * ldy;
        *y = (beta != T(0) ? beta * *y : T(0)) + alpha * sum;
    }
}

// Waves per atom, by the number of atoms. Whole calls with 4, 8 and 16 waves,
// mean over both directions, both precisions, one and six vectors, in us:
//   2D, rank 16:   256 atoms (128^2) 68.4 63.1 62.6; 512 (150^2) 103.3 103.5
//   104.4; 768 (200^2) 174.5 180.3 178.5; 1,024 (256^2) 237.9 238.0 248.2;
//   2,048 (300^2, rank 8) 292 307 330;
//   3D, rank 16:   440 (27 x 33 x 30) 346 306 277; 512 (32^3) 409 368 361; 664
//   (34 x 36 x 33) 643 577 552; 768 (36^3) 806 758 730; 944 1141 1099 1088;
//   1,024 (40^3) 1294 1246 1242.
// From 768 on the 2D matrices gain from four; the 3D ones, whose atoms carry
// several times the records, would still gain 4 to 10% from sixteen there.
// (H^T with 7 and 8 vectors and sixteen waves keeps 6 to 29 of its registers in
// scratch.)
static int mv_waves(int atoms) { return atoms >= 768 ? 4 : 16; }

template <typename T, int K, bool TR>
static void launch_mv_acc(int n, const Phase& ph, const Bases& b, T alpha, T beta, hipStream_t s)
{
    const MvAtom* at = static_cast<const MvAtom*>(ph.dTasks);
    const MvContrib* cs = static_cast<const MvContrib*>(ph.dAux);
    switch (mv_waves(n)) {
    case 4: mv_acc_kernel<T, K, 4, TR><<<n, 256, 0, s>>>(b, at, cs, ph.ldx, ph.ldy, alpha, beta); break;
    default: mv_acc_kernel<T, K, 16, TR><<<n, 1024, 0, s>>>(b, at, cs, ph.ldx, ph.ldy, alpha, beta); break;
    }
}

template <typename T, int K>
static void launch_mv_k(const Phase& ph, const Bases& b, T alpha, T beta, hipStream_t s)
{
    if (ph.kind == PH_MV_PROJ) {
        const int n = (int)ph.mvProj.size(), big = ph.mvBig;
        if (n)
            mv_proj_kernel<T, K><<<big + (n - big + 3) / 4, 256, 0, s>>>(b, static_cast<const MvProjItem*>(ph.dTasks),
                                                                        n, big, ph.ldx);
    } else {
        const int n = (int)ph.mvAtoms.size();
        if (n == 0) return;
        if (ph.mvTrans) launch_mv_acc<T, K, true>(n, ph, b, alpha, beta, s);
        else launch_mv_acc<T, K, false>(n, ph, b, alpha, beta, s);
    }
}

template <typename T>
void launch_mv_phase(const Phase& ph, const Bases& b, T alpha, T beta, hipStream_t s)
{
    switch (ph.mvK) {
    case 1: launch_mv_k<T, 1>(ph, b, alpha, beta, s); break;
    case 2: launch_mv_k<T, 2>(ph, b, alpha, beta, s); break;
    case 3: launch_mv_k<T, 3>(ph, b, alpha, beta, s); break;
    case 4: launch_mv_k<T, 4>(ph, b, alpha, beta, s); break;
    case 5: launch_mv_k<T, 5>(ph, b, alpha, beta, s); break;
    case 6: launch_mv_k<T, 6>(ph, b, alpha, beta, s); break;
    case 7: launch_mv_k<T, 7>(ph, b, alpha, beta, s); break;
    case 8: launch_mv_k<T, 8>(ph, b, alpha, beta, s); break;
    default: throw std::runtime_error("streaming H*X supports 1..8 columns");
    }
    HIP_LAUNCH_CHECK();
}

template void launch_mv_phase<double>(const Phase&, const Bases&, double, double, hipStream_t);
template void launch_mv_phase<float>(const Phase&, const Bases&, float, float, hipStream_t);

} // namespace dmhm
