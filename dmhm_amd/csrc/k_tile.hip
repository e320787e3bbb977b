// gfx950 tile GEMM engine: grouped output-owned small GEMMs (H*X, sub-H
// products, projections, dense-leaf accumulation, factor formation).
#include <climits>
#include <cstddef>
#include "chunks.hpp"
#include "kcommon.hpp"

namespace dmhm {

// ---------------------------------------------------------------------------
// Tile GEMM engine.
// Workgroup = 256 threads; a tile is at most MR x NC (MR = 64 or 16 rows,
// NC = 16, 32 or 64 columns). Thread (ti, tj) = (tid % RT, tid / RT) owns
// the TM x TN micro-tile at rows TM*ti.., columns TN*tj.., accumulated in
// registers (TM + TN LDS reads per TM*TN FMAs). L and R are staged through
// LDS in chunks of QC along the inner dimension, double-buffered: the global
// loads of the next chunk (possibly of the next contribution) are issued
// before the current chunk is multiplied, so one barrier per chunk suffices
// and load latency overlaps the arithmetic. Out-of-range entries are staged
// as zeros, so every chunk multiplies a full QC slice. R is pre-scaled by
// the contribution's alpha when it is stored to LDS.
// ---------------------------------------------------------------------------
// Inner-dimension chunk. (Chunks twice as deep for 16-row tiles measured the
// same on the 256^2 rank-16 product: 117 ms FP64 either way.)
template <typename T, int MR> struct TileCfg { static constexpr int QC = 32; };
template <int MR> struct TileCfg<double, MR> { static constexpr int QC = 16; };

// Operand bases as the tile bodies read them, by run-time slot numbers that
// are uniform across the workgroup: a plain launch's own (kernel arguments),
// or a segmented launch's shifted by the member segment's offsets (kernel
// arguments plus the segment's table entry). Both resolve through uniform
// loads, with no private array indexed at run time and no LDS copy.
struct ArgBases {
    const Bases& b;
    template <typename T> __device__ __forceinline__ T* val(int s) const { return reinterpret_cast<T*>(b.val[s]); }
    __device__ __forceinline__ const int* rank(int s) const { return b.rank[s]; }
};
struct SegBases {
    const Bases& b;
    const TileSeg* __restrict__ sg;
    template <typename T> __device__ __forceinline__ T* val(int s) const
    {
        return reinterpret_cast<T*>(b.val[s]) + sg->val[s];
    }
    __device__ __forceinline__ const int* rank(int s) const { return b.rank[s] + sg->rank[s]; }
};

template <typename BV>
__device__ __forceinline__ int contrib_q(const BV& b, const Contrib& C)
{
    int q = C.q;
    if (C.qrank >= 0) q = min(q, b.rank(C.qslot)[C.qrank]);
    return q;
}

template <typename T, int MR, int NC, int QC, int LN, int RN, typename BV>
__device__ __forceinline__ void tile_load(const BV& b, const Tile& tl, const Contrib& C,
                                          const int64_t* __restrict__ gtab, int p0, int q, int m, int k, T alpha, T beta, T (&lr)[LN], T (&rr)[RN], T& a)
{
    const int tid = threadIdx.x;
    const int qc = min(QC, q - p0);
    const T* __restrict__ L = b.template val<const T>(C.lslot) + C.loff;
    const T* __restrict__ R = b.template val<const T>(C.rslot) + C.roff;
    a = (C.flags & CF_RUNTIME_ALPHA) ? alpha * T(C.alpha)
      : (C.flags & CF_RUNTIME_BETA) ? beta * T(C.alpha) : T(C.alpha);
    const bool tL = C.flags & CF_TRANS_L, tR = C.flags & CF_TRANS_R, gR = C.flags & CF_GATHER_R;
#pragma unroll
    for (int u = 0; u < LN; ++u) {
        const int e = tid + 256 * u;
        int ii, pp;
        if (!tL) { ii = e % MR; pp = e / MR; } else { pp = e % QC; ii = e / QC; }
        const bool ok = e < MR * QC && ii < m && pp < qc;
        lr[u] = ok ? (!tL ? L[ii + (int64_t)(p0 + pp) * C.ldl] : L[(p0 + pp) + (int64_t)ii * C.ldl]) : T(0);
    }
#pragma unroll
    for (int u = 0; u < RN; ++u) {
        const int e = tid + 256 * u;
        int jj, pp;
        if (!tR) { pp = e % QC; jj = e / QC; } else { jj = e % NC; pp = e / NC; }
        const bool ok = e < QC * NC && jj < k && pp < qc;
        rr[u] = ok ? (!tR ? R[(p0 + pp) + (gR ? gather_column(tl, gtab, jj) : (int64_t)jj * C.ldr)] : R[jj + (int64_t)(p0 + pp) * C.ldr])
                   : T(0);
    }
}

template <typename T, int MR, int NC, int QC, int LN, int RN, int LP, int RP>
__device__ __forceinline__ void tile_store(T* __restrict__ Lb, T* __restrict__ Rb, const T (&lr)[LN],
                                           const T (&rr)[RN], T a, uint8_t flags)
{
    const int tid = threadIdx.x;
    const bool tL = flags & CF_TRANS_L, tR = flags & CF_TRANS_R;
#pragma unroll
    for (int u = 0; u < LN; ++u) {
        const int e = tid + 256 * u;
        if (e < MR * QC) {
            int ii, pp;
            if (!tL) { ii = e % MR; pp = e / MR; } else { pp = e % QC; ii = e / QC; }
            Lb[pp * LP + ii] = lr[u];
        }
    }
#pragma unroll
    for (int u = 0; u < RN; ++u) {
        const int e = tid + 256 * u;
        if (e < QC * NC) {
            int jj, pp;
            if (!tR) { pp = e % QC; jj = e / QC; } else { jj = e % NC; pp = e / NC; }
            Rb[pp * RP + jj] = a * rr[u];
        }
    }
}

template <typename T, int MR, int NC, int TM, int TN, typename BV>
__device__ __forceinline__ void tile_body(const BV& b, const Tile& tl, const Contrib* __restrict__ cs,
                                          const int64_t* __restrict__ gtab, T alpha, T beta)
{
    constexpr int QC = TileCfg<T, MR>::QC;
    constexpr int RT = MR / TM;
    static_assert(RT * (NC / TN) == 256, "the thread grid must cover 256 threads");
    constexpr int LN = (MR * QC + 255) / 256;
    constexpr int RN = (QC * NC + 255) / 256;
    constexpr int LP = MR + 4, RP = NC + 4;     // padded LDS rows (16-byte multiples)
    __shared__ T Ls[2][QC * LP];
    __shared__ T Rs[2][QC * RP];
    int m = tl.m, k = tl.k;
    if (tl.mrank >= 0) m = min(m, max(0, b.rank(tl.mslot)[tl.mrank] - tl.moff));
    if (tl.krank >= 0) k = min(k, max(0, b.rank(tl.kslot)[tl.krank] - tl.koff));
    if (m <= 0 || k <= 0) return;
    const int tid = threadIdx.x, ti = tid % RT, tj = tid / RT;
    T acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = T(0);

    // Chunk iterator over (contribution c, offset p0 < q); uniform across the workgroup.
    int c = tl.cb, q = 0, p0 = 0;
    for (; c < tl.ce; ++c) {
        q = contrib_q(b, cs[c]);
        if (q > 0) break;
    }
    T lr[LN], rr[RN], a = T(0);
    uint8_t flags = 0;
    if (c < tl.ce) {
        const Contrib C = cs[c];
        tile_load<T, MR, NC, QC, LN, RN>(b, tl, C, gtab, p0, q, m, k, alpha, beta, lr, rr, a);
        flags = C.flags;
    }
    int buf = 0;
    while (c < tl.ce) {
        tile_store<T, MR, NC, QC, LN, RN, LP, RP>(Ls[buf], Rs[buf], lr, rr, a, flags);
        __syncthreads();
        // Advance and prefetch the next chunk while this one is multiplied.
        p0 += QC;
        if (p0 >= q) {
            p0 = 0;
            for (++c; c < tl.ce; ++c) {
                q = contrib_q(b, cs[c]);
                if (q > 0) break;
            }
        }
        if (c < tl.ce) {
            const Contrib C = cs[c];
            tile_load<T, MR, NC, QC, LN, RN>(b, tl, C, gtab, p0, q, m, k, alpha, beta, lr, rr, a);
            flags = C.flags;
        }
        const T* __restrict__ Lb = Ls[buf];
        const T* __restrict__ Rb = Rs[buf];
#pragma unroll 4
        for (int p = 0; p < QC; ++p) {
            T lv[TM], rv[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) lv[i] = Lb[p * LP + ti * TM + i];
#pragma unroll
            for (int j = 0; j < TN; ++j) rv[j] = Rb[p * RP + tj * TN + j];
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] += lv[i] * rv[j];
        }
        buf ^= 1;
    }
    T* out = b.template val<T>(tl.slot) + tl.off;
    const bool useBeta = (tl.flags & TF_RUNTIME_BETA) && beta != T(0);
    const bool accum = (tl.flags & TF_ACCUMULATE);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int r = ti * TM + i;
        if (r >= m) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int col = tj * TN + j;
            if (col < k) {
                T* o = out + r + (int64_t)col * tl.ld;
                if (useBeta) *o = beta * *o + acc[i][j];
                else if (accum) *o += acc[i][j];
                else *o = acc[i][j];
            }
        }
    }
}

// Segmented launches (merged plans of independent members): the member
// segment holding workgroup g, the last one whose first workgroup (first(sg))
// is at or before g.
template <typename F>
__device__ __forceinline__ const TileSeg* seg_of(const TileSeg* __restrict__ segs, int nseg, int g, F first)
{
    if (nseg <= 64) {
        // One load per lane and a ballot.
        const int l = threadIdx.x & 63;
        const int f = l < nseg ? first(segs[l]) : INT_MAX;
        return segs + (int)__popcll(__ballot(f <= g)) - 1;
    }
    int lo = 0, hi = nseg - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first(segs[mid]) <= g) lo = mid;
        else hi = mid - 1;
    }
    return segs + lo;
}

template <typename T, int MR, int NC, int TM, int TN, int ROLE>
__global__ void __launch_bounds__(256) tile_kernel(Bases b, const Tile* __restrict__ tiles,
                                                   const Contrib* __restrict__ cs,
                                                   const int64_t* __restrict__ gtab, T alpha, T beta)
{
    tile_body<T, MR, NC, TM, TN>(ArgBases{b}, tiles[blockIdx.x], cs, gtab, alpha, beta);
}

template <typename T, int MR, int NC, int TM, int TN>
__global__ void __launch_bounds__(256) tile_seg_kernel(Bases b, const TileSeg* __restrict__ segs, int nseg, T alpha,
                                                       T beta)
{
    const TileSeg* sg = seg_of(segs, nseg, (int)blockIdx.x, [](const TileSeg& s) { return s.first; });
    const int local = (int)blockIdx.x - sg->first;
    if (local >= sg->count) return;
    tile_body<T, MR, NC, TM, TN>(SegBases{b, sg}, sg->tiles[local], sg->cs, sg->gtab, alpha, beta);
}

// ---------------------------------------------------------------------------
// MFMA engine. A wave computes one unit of an output tile, RB x CB blocks of
// 16 x 16 entries, straight from global memory: no LDS, no barriers. It
// computes the unit transposed, D^T = R^T L^T: the first MFMA operand is a
// 16-column block of R^T, the second a 16-row block of L^T, and lane
// l = (li, lk) = (l % 16, l / 16) holds D(row li, column c) in accumulator
// register r, c = 4*lk + r for FP32 and BF16, lk + 4*r for FP64 (measured on
// gfx950), so each group of 16 lanes stores 16 rows of a column.
//
// Inner chunks of 16: lane lk supplies the four inner indices mf_k(s, lk),
// s < 4, to both operands, one per K = 4 instruction (v_mfma_f64_16x16x4f64,
// v_mfma_f32_16x16x4f32) or all four to one v_mfma_f32_16x16x16_bf16 (MODE 1:
// FP32 operands rounded to BF16, FP32 accumulation). The map makes 16 bytes
// along the inner dimension belong to one lane, so an operand stored with the
// inner dimension contiguous is read with 16-byte loads; an operand stored
// with rows (columns) contiguous is read two neighbouring rows at a time:
// row block b of a pair takes the rows of parity b. Rows and columns outside
// the tile are clamped to its last one (their results are never stored);
// inner indices outside the contribution are read at its last one and zeroed.
// Loads of the next chunk (possibly of the next contribution) are written
// before the MFMAs of the current one, into the other of two register sets
// (MfUnit::run says what the compiler keeps of that).
//
// Contribution records and run-time ranks are read 64 at a time, one per
// lane, and handed out by lane reads: two memory latencies per 64
// contributions, not two per contribution.
//
// S = 4: the four waves of a workgroup share one unit and split its
// contributions (every fourth one, or every fourth chunk where a tile has
// fewer than four contributions) and add their sums through LDS in wave order.
//
// What bounds it: operand bytes through L2 and the 256 MB cache, the FP64 MFMA
// (64 cycles each) where tiles are 64 x 64, and for tiles of few contributions
// the chain of dependent loads before the first operand. Units of 32 x 32 read
// every operand twice per 64 x 64 tile through L1 and leave room for three
// waves per SIMD with two chunks of operands in flight each. Measured against
// the LDS engine (FP64, 256^2, rank 16, one product): projections of 16 x 20
// tiles (20 GB of operands) 5.9 -> 2.7 ms, dense accumulation of 64 x 64 tiles
// 5.7 -> 3.4 ms (46 TFLOP/s of 73 that a large product reaches), all tile
// phases 82 -> 43 ms; FP32 3D update 19.5 -> 8.8 ms. Operand loads under
// branches on the form are slower (62 ms in all against 50), since every join
// then waits for all of them.
// ---------------------------------------------------------------------------
typedef double mf_d4 __attribute__((ext_vector_type(4)));
typedef float mf_f4 __attribute__((ext_vector_type(4)));
typedef __bf16 mf_b4 __attribute__((ext_vector_type(4)));

template <typename T> struct MfAcc;
template <> struct MfAcc<double> { typedef mf_d4 type; };
template <> struct MfAcc<float> { typedef mf_f4 type; };

__device__ __forceinline__ mf_d4 mf_step(double a, double b, mf_d4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ mf_f4 mf_step(float a, float b, mf_f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ mf_f4 mf_step_bf16(const float (&a)[4], const float (&b)[4], mf_f4 c)
{
    mf_b4 x, y;
#pragma unroll
    for (int e = 0; e < 4; ++e) { x[e] = (__bf16)a[e]; y[e] = (__bf16)b[e]; }
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x, y, c, 0, 0, 0);
}

// Global-memory pointers (plain global loads, not flat ones) and vectors that
// need only the element's alignment.
template <typename T> using GPtr = const __attribute__((address_space(1))) T*;
template <typename T> struct MfVec;
template <> struct MfVec<double> {
    static constexpr int VP = 2;                // elements in 16 bytes
    typedef double v2 __attribute__((ext_vector_type(2), aligned(8)));
    typedef v2 vp;
};
template <> struct MfVec<float> {
    static constexpr int VP = 4;
    typedef float v2 __attribute__((ext_vector_type(2), aligned(4)));
    typedef float vp __attribute__((ext_vector_type(4), aligned(4)));
};

// Inner index (within a chunk) that lane group lk supplies to step s.
template <typename T>
__device__ __forceinline__ int mf_k(int s, int lk)
{
    constexpr int VP = MfVec<T>::VP;
    return (s / VP) * (4 * VP) + lk * VP + s % VP;
}

// Row (column) that entry j of block b covers, relative to the unit's first.
template <int NB>
__device__ __forceinline__ int mf_row(int b, int j)
{
    return NB == 1 ? j : 32 * (b >> 1) + 2 * j + (b & 1);
}

// One operand of a contribution as a wave reads it: rows (columns) n0 +
// mf_row(b, li) clamped below nmax. PC: the inner dimension is contiguous,
// X(n, p) = X[p + n ld] (gathered columns: X[p + col[b]], the lane's own
// offsets), else X[n + p ld]. In the second form two neighbouring rows are read
// together (nmax >= 2): pointer 2g serves blocks 2g and 2g + 1, and a pair that
// would cross the last row starts one row earlier (mf_moved).
template <typename T, bool PC, int NB>
__device__ __forceinline__ void mf_lanes(GPtr<T> X, int64_t ld, bool gathered, const int64_t (&col)[NB], int n0,
                                         int nmax, int li, int lk, GPtr<T> (&x)[NB])
{
    constexpr int VP = MfVec<T>::VP;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (!PC && NB > 1 && (b & 1)) continue;
        const int n = min(n0 + mf_row<NB>(b, li), nmax - (!PC && NB > 1 ? 2 : 1));
        x[b] = X + (PC ? lk * VP + (gathered ? col[b] : n * ld) : lk * VP * ld + n);
    }
}

// Issues the loads of the chunk at p, x + inner index (TAIL: qc < 16 indices,
// read at the last one beyond). Nothing here waits for a load: the fragments
// are finished in mf_finish when they are used.
template <typename T, bool PC, bool TAIL, int NB>
__device__ __forceinline__ void mf_issue(const GPtr<T> (&x)[NB], int64_t ld, int p, int qc, int lk, T (&f)[NB][4])
{
    constexpr int VP = MfVec<T>::VP;
    typedef typename MfVec<T>::v2 v2;
    typedef typename MfVec<T>::vp vp;
    auto rel = [&](int s) { return TAIL ? min(mf_k<T>(s, lk), qc - 1) - lk * VP : mf_k<T>(s, 0); };
    if (PC && !TAIL) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int h = 0; h < 4 / VP; ++h) {
                const vp v = *(const __attribute__((address_space(1))) vp*)(x[b] + p + h * 4 * VP);
#pragma unroll
                for (int e = 0; e < VP; ++e) f[b][h * VP + e] = v[e];
            }
    } else if (PC) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int s = 0; s < 4; ++s) f[b][s] = x[b][p + rel(s)];
    } else if (NB > 1) {
#pragma unroll
        for (int g = 0; g < NB / 2; ++g)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const v2 v = *(const __attribute__((address_space(1))) v2*)(x[2 * g] + (p + rel(s)) * ld);
                f[2 * g][s] = v[0];
                f[2 * g + 1][s] = v[1];
            }
    } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) f[0][s] = x[0][(p + rel(s)) * ld];
    }
}

template <typename T, bool PC, bool TAIL, int NB>
__device__ __forceinline__ void mf_finish(T (&f)[NB][4], int n0, int nmax, int qc, int li, int lk)
{
    if (!PC && NB > 1) {
        // The even row of a pair moved down is the pair's second entry.
#pragma unroll
        for (int g = 0; g < NB / 2; ++g) {
            const bool moved = n0 + 32 * g + 2 * li > nmax - 2;
#pragma unroll
            for (int s = 0; s < 4; ++s) f[2 * g][s] = moved ? f[2 * g + 1][s] : f[2 * g][s];
        }
    }
    if (TAIL) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int s = 0; s < 4; ++s) f[b][s] = mf_k<T>(s, lk) < qc ? f[b][s] : T(0);
    }
}

template <typename T, int RB, int CB>
struct MfFrag {
    T l[RB][4], r[CB][4];
    T a;
    int qc;
};

// Records as whole vectors: loads by field (single bytes among them) are
// issued one after another as their fields are used.
typedef uint32_t mf_u2 __attribute__((ext_vector_type(2), aligned(8)));
typedef uint32_t mf_u4 __attribute__((ext_vector_type(4), aligned(8)));
static_assert(sizeof(Tile) == 56 && offsetof(Tile, k) == 16 && offsetof(Tile, koff) == 32 &&
              offsetof(Tile, gather) == 48 && offsetof(Tile, gcols) == 52 && offsetof(Tile, slot) == 44, "tile record layout");
static_assert(sizeof(Contrib) == 40 && offsetof(Contrib, ldl) == 16 && offsetof(Contrib, lslot) == 32 &&
              offsetof(Contrib, flags) == 35, "contribution record layout");
__device__ __forceinline__ int64_t mf_i64(uint32_t lo, uint32_t hi) { return (int64_t)((uint64_t)hi << 32 | lo); }
__device__ __forceinline__ Tile mf_tile(const Tile* __restrict__ p)
{
    const mf_u4* v = reinterpret_cast<const mf_u4*>(p);
    const mf_u4 a = v[0], b = v[1], c = v[2];
    Tile t;
    const mf_u2 d = reinterpret_cast<const mf_u2*>(p)[6];
    t.off = mf_i64(a[0], a[1]); t.ld = (int)a[2]; t.m = (int)a[3];
    t.k = (int)b[0]; t.mrank = (int)b[1]; t.krank = (int)b[2]; t.moff = (int)b[3];
    t.koff = (int)c[0]; t.cb = (int)c[1]; t.ce = (int)c[2];
    t.gather = (int)d[0]; t.gcols = (int)d[1];
    t.slot = (uint8_t)c[3]; t.mslot = (uint8_t)(c[3] >> 8); t.kslot = (uint8_t)(c[3] >> 16);
    t.flags = (uint8_t)(c[3] >> 24);
    return t;
}

// One unit of a tile: walks the tile's contributions 64 at a time, one record
// per lane, and within them by form (which operands have the inner dimension
// contiguous; whole chunks, then the remainders of inner dimensions that 16
// does not divide), so that each inner loop is free of branches on the form
// and its loads stay in flight across the other register set's MFMAs.
template <typename T, int MODE, int RB, int CB, int S, typename BV>
struct MfUnit {
    typedef typename MfAcc<T>::type Acc;
    typedef MfFrag<T, RB, CB> Frag;
    const BV& b;
    T alpha, beta;
    int w, li, lk;
    int row0, col0, m, n;       // the unit's first row and column, the tile's extent
    ChunkWalk<S> walk;          // byChunk: S waves split chunks, not contributions
    int64_t gcol[CB];           // offsets of the unit's columns in gathered right operands
    // lane records
    int64_t dl, dr;
    int dldl, dldr, dq, dqrank;
    uint32_t dmeta;             // left, right and rank slot, flags (bytes)
    float dalpha;
    Acc acc[RB][CB];

    static __device__ __forceinline__ int64_t lane_i64(int64_t v, int i)
    {
        const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)v, i);
        const uint32_t hi = __builtin_amdgcn_readlane((int)(v >> 32), i);
        return (int64_t)((uint64_t)hi << 32 | lo);
    }

    __device__ __forceinline__ void mma(Frag& f)
    {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int s = 0; s < 4; ++s) f.l[rb][s] *= f.a;
        if constexpr (MODE == 1) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = mf_step_bf16(f.r[cb], f.l[rb], acc[rb][cb]);
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                    for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = mf_step(f.r[cb][s], f.l[rb][s], acc[rb][cb]);
        }
    }

    // The whole chunks (TAIL: the remainders) of the contributions in `left`.
    template <bool PL, bool PR, bool TAIL>
    __device__ __forceinline__ void run(uint64_t left)
    {
        GPtr<T> L[RB], R[CB];
        int64_t ldl = 0, ldr = 0;
        T a = T(0);
        walk.start();
        // Moves to the wave's next chunk; at the end it stays on the last one.
        auto next = [&]() -> bool {
            return walk.template next<TAIL>(left, [&](int i) { return __builtin_amdgcn_readlane(dq, i); }, [&](int i) {
                const uint32_t meta = __builtin_amdgcn_readlane(dmeta, i);
                const int fl = meta >> 24;
                const float ca = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dalpha), i));
                a = (fl & CF_RUNTIME_ALPHA) ? alpha * T(ca) : (fl & CF_RUNTIME_BETA) ? beta * T(ca) : T(ca);
                ldl = __builtin_amdgcn_readlane(dldl, i);
                ldr = __builtin_amdgcn_readlane(dldr, i);
                const int64_t none[RB] = {};
                mf_lanes<T, PL, RB>((GPtr<T>)(b.template val<const T>(meta & 255) + lane_i64(dl, i)), ldl, false, none,
                                    row0, m, li, lk, L);
                mf_lanes<T, PR, CB>((GPtr<T>)(b.template val<const T>((meta >> 8) & 255) + lane_i64(dr, i)), ldr,
                                    fl & CF_GATHER_R, gcol, col0, n, li, lk, R);
            });
        };
        auto fetch = [&](Frag& f) {
            f.a = a;
            f.qc = walk.q - walk.p;
            mf_issue<T, PL, TAIL, RB>(L, ldl, walk.p, f.qc, lk, f.l);
            mf_issue<T, PR, TAIL, CB>(R, ldr, walk.p, f.qc, lk, f.r);
        };
        auto use = [&](Frag& f) {
            mf_finish<T, PL, TAIL, RB>(f.l, row0, m, f.qc, li, lk);
            mf_finish<T, PR, TAIL, CB>(f.r, col0, n, f.qc, li, lk);
            mma(f);
        };
        Frag f0, f1;
        if (!next()) return;
        fetch(f0);
        // After the last chunk the fetch repeats it, so that no fetch is under a
        // branch (a fetch under one, 62 against 50 ms per 256^2 FP64 product),
        // and one use per register set keeps one set of accumulators. The
        // compiler overlaps one half of the loop only: the wait before use(f1)
        // leaves f0's loads in flight, but f1's, which nothing needs once the
        // loop ends, it moves behind use(f0) and the first exit.
        while (true) {
            const bool more1 = next();
            fetch(f1);
            use(f0);
            if (!more1) break;
            const bool more0 = next();
            fetch(f0);
            use(f1);
            if (!more0) break;
        }
    }

    // Any contributions, one chunk and one load at a time: the forms the tile
    // plans do not use (L with, R without contiguous inner dimension) and
    // row-contiguous operands of tiles of one row or column.
    __device__ __forceinline__ void runAny(uint64_t left)
    {
        while (left) {
            const int i = __builtin_ctzll(left);
            left &= left - 1;
            const int q = __builtin_amdgcn_readlane(dq, i);
            const uint32_t meta = __builtin_amdgcn_readlane(dmeta, i);
            const int fl = meta >> 24;
            const float ca = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dalpha), i));
            const int64_t ldl = __builtin_amdgcn_readlane(dldl, i), ldr = __builtin_amdgcn_readlane(dldr, i);
            const bool tL = fl & CF_TRANS_L, tR = fl & CF_TRANS_R;
            const GPtr<T> L = (GPtr<T>)(b.template val<const T>(meta & 255) + lane_i64(dl, i));
            const GPtr<T> R = (GPtr<T>)(b.template val<const T>((meta >> 8) & 255) + lane_i64(dr, i));
            Frag f;
            f.a = (fl & CF_RUNTIME_ALPHA) ? alpha * T(ca) : (fl & CF_RUNTIME_BETA) ? beta * T(ca) : T(ca);
#pragma unroll 1
            for (int p = 0; p < q; p += 16) {
                if (S > 1 && walk.byChunk && (walk.turn++ & (S - 1)) != w) continue;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const int k = p + mf_k<T>(s, lk), kc = min(k, q - 1);
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) {
                        const int r = min(row0 + mf_row<RB>(rb, li), m - 1);
                        const T v = L[tL ? kc + r * ldl : r + kc * ldl];
                        f.l[rb][s] = k < q ? v : T(0);
                    }
#pragma unroll
                    for (int cb = 0; cb < CB; ++cb) {
                        const int c = min(col0 + mf_row<CB>(cb, li), n - 1);
                        const T v = R[tR ? c + kc * ldr : kc + ((fl & CF_GATHER_R) ? gcol[cb] : c * ldr)];
                        f.r[cb][s] = k < q ? v : T(0);
                    }
                }
                mma(f);
            }
        }
    }

    // Issues the loads of the lane's record among the 64 from c0 on.
    __device__ __forceinline__ void record(const Tile& tl, const Contrib* __restrict__ cs, int c0)
    {
        if (tl.cb == tl.ce) return;
        const Contrib* C = cs + min(c0 + 16 * lk + li, tl.ce - 1);
        const mf_u4 x = reinterpret_cast<const mf_u4*>(C)[0], y = reinterpret_cast<const mf_u4*>(C)[1];
        const mf_u2 z = reinterpret_cast<const mf_u2*>(C)[4];
        dl = mf_i64(x[0], x[1]); dr = mf_i64(x[2], x[3]);
        dldl = (int)y[0]; dldr = (int)y[1]; dq = (int)y[2]; dqrank = (int)y[3];
        dmeta = z[0];
        dalpha = __int_as_float((int)z[1]);
    }

    // record() has been called for the first 64.
    __device__ __forceinline__ void contributions(const Tile& tl, const Contrib* __restrict__ cs)
    {
        const int lane = 16 * lk + li;
        for (int c0 = tl.cb; c0 < tl.ce; c0 += 64) {
            if (c0 != tl.cb) record(tl, cs, c0);
            const bool in = c0 + lane < tl.ce;
            if (dqrank >= 0) {
                // The slots that have ranks, picked per lane without a load.
                const uint32_t sl = (dmeta >> 16) & 255;
                const int* r = b.rank(SLOT_A);
                r = sl == SLOT_B ? b.rank(SLOT_B) : r;
                r = sl == SLOT_C ? b.rank(SLOT_C) : r;
                r = sl == SLOT_X ? b.rank(SLOT_X) : r;
                r = sl == SLOT_WIDTH ? b.rank(SLOT_WIDTH) : r;
                dq = min(dq, r[dqrank]);
            }
            const bool mine = in && dq > 0 && (S == 1 || walk.byChunk || (lane & (S - 1)) == w);
            const bool pl = dmeta >> 24 & CF_TRANS_L, pr = !(dmeta >> 24 & CF_TRANS_R);
            const bool any = (pl && !pr) || (RB > 1 && !pl && m < 2) || (CB > 1 && !pr && n < 2);
            const bool whole = mine && !any && dq >= 16, rest = mine && !any && (dq & 15);
            run<false, true, false>(__ballot(whole && !pl && pr));
            run<false, true, true>(__ballot(rest && !pl && pr));
            run<true, true, false>(__ballot(whole && pl && pr));
            run<true, true, true>(__ballot(rest && pl && pr));
            run<false, false, false>(__ballot(whole && !pl && !pr));
            run<false, false, true>(__ballot(rest && !pl && !pr));
            runAny(__ballot(mine && any));
        }
    }
};

// One unit (row group ur, column group uc) of tile tl; w: the wave's share of
// the contributions (S > 1).
template <typename T, int MODE, int RB, int CB, int S, typename BV>
__device__ __forceinline__ void mfma_body(const BV& b, const Tile& tl, const Contrib* __restrict__ cs,
                                          const int64_t* __restrict__ gtab, int ur, int uc, int w, T alpha, T beta)
{
    static_assert(MODE == 0 || sizeof(T) == 4, "the BF16 mode reads FP32 operands");
    static_assert(S == 1 || S == 4, "one wave or the four waves of a workgroup per unit");
    const int row0 = ur * 16 * RB, col0 = uc * 16 * CB;
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    MfUnit<T, MODE, RB, CB, S, BV> u{b, alpha, beta, w, li, lk, row0, col0, 0, 0,
                                      {w, S > 1 && tl.ce - tl.cb < S}};
    // The first records' loads are in flight while the ranks are read.
    u.record(tl, cs, tl.cb);
    int m = tl.m, n = tl.k;
    if (tl.mrank >= 0) m = min(m, max(0, b.rank(tl.mslot)[tl.mrank] - tl.moff));
    if (tl.krank >= 0) n = min(n, max(0, b.rank(tl.kslot)[tl.krank] - tl.koff));
    if (m <= row0 || n <= col0) return;         // uniform over the waves that share the unit
    u.m = m;
    u.n = n;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
        u.gcol[cb] = tl.gather >= 0 ? gather_column(tl, gtab, min(col0 + mf_row<CB>(cb, li), n - 1)) : 0;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int r = 0; r < 4; ++r) u.acc[rb][cb][r] = T(0);
    u.contributions(tl, cs);

    T* out = b.template val<T>(tl.slot) + tl.off;
    const bool useBeta = (tl.flags & TF_RUNTIME_BETA) && beta != T(0);
    const bool accum = (tl.flags & TF_ACCUMULATE);
    const int64_t ld = tl.ld;
    auto put = [&](int row, int col, T v) {
        if (row >= m || col >= n) return;
        T* o = out + row + col * ld;
        if (useBeta) *o = beta * *o + v;
        else if (accum) *o += v;
        else *o = v;
    };
    auto cidx = [&](int r) { return sizeof(T) == 8 ? lk + 4 * r : 4 * lk + r; };
    if constexpr (S == 1) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
                    put(row0 + mf_row<RB>(rb, li), col0 + mf_row<CB>(cb, cidx(r)), u.acc[rb][cb][r]);
    } else {
        // Wave w adds up register w of every wave's blocks, in wave order.
        __shared__ T part[S][RB * CB][4][64];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int r = 0; r < 4; ++r) part[w][rb * CB + cb][r][lane] = u.acc[rb][cb][r];
        __syncthreads();
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                T v = part[0][rb * CB + cb][w][lane];
#pragma unroll
                for (int x = 1; x < S; ++x) v += part[x][rb * CB + cb][w][lane];
                put(row0 + mf_row<RB>(rb, li), col0 + mf_row<CB>(cb, cidx(w)), v);
            }
    }
}

// Units of a phase's tiles: ur x uc per tile (the phase's largest tile over
// the unit's size), numbered tile-major.
struct MfGrid { int ur, uc; };

// Workgroups are dealt to the eight XCDs in turn; kXcdRun consecutive ones of
// the tile order go to one XCD, so that neighbouring tiles, which share
// operands, meet in one L2 (FP32 3D update 13.7 ms with the plain order, 13.1
// with runs of 16, 13.0 with 64; the 256^2 FP64 product 62.9, 62.1 and 62.8).
constexpr int kXcdRun = 16;
template <int RUN>
__device__ __forceinline__ int xcd_order(int g, int n)
{
    const int full = n / (8 * RUN) * (8 * RUN);
    if (g >= full) return g;
    const int j = g >> 3;
    return (j / RUN) * (8 * RUN) + (g & 7) * RUN + j % RUN;
}

// Unit of workgroup g and wave w of a tile list: every unit a workgroup's (ALL),
// or the units of the first nLong tiles a workgroup's and the others a wave's.
template <typename T, int MODE, int RB, int CB, bool ALL, typename BV>
__device__ __forceinline__ void mfma_unit(const BV& b, const Tile* __restrict__ tiles,
                                          const Contrib* __restrict__ cs, const int64_t* __restrict__ gtab, int ntiles,
                                          int nLong, MfGrid gr, int g, int w, T alpha, T beta)
{
    const int per = gr.ur * gr.uc;
    if (ALL || g < nLong * per) {
        const int id = g / per, sub = g - id * per;
        if (id >= ntiles) return;
        mfma_body<T, MODE, RB, CB, 4>(b, mf_tile(tiles + id), cs, gtab, sub / gr.uc, sub % gr.uc, w, alpha, beta);
    } else {
        const int u = (g - nLong * per) * 4 + w, at = u / per, id = nLong + at, sub = u - at * per;
        if (id >= ntiles) return;
        mfma_body<T, MODE, RB, CB, 1>(b, mf_tile(tiles + id), cs, gtab, sub / gr.uc, sub % gr.uc, w, alpha, beta);
    }
}

template <typename T, int MODE, int RB, int CB, bool ALL>
__global__ void __launch_bounds__(256) tile_mfma_kernel(Bases b, const Tile* __restrict__ tiles,
                                                        const Contrib* __restrict__ cs,
                                                        const int64_t* __restrict__ gtab, int ntiles, int nLong,
                                                        MfGrid gr, T alpha, T beta)
{
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lng = ALL ? 0 : nLong * gr.ur * gr.uc, g0 = (int)blockIdx.x;
    const int g = g0 < lng ? xcd_order<4>(g0, lng) : lng + xcd_order<kXcdRun>(g0 - lng, (int)gridDim.x - lng);
    mfma_unit<T, MODE, RB, CB, ALL>(ArgBases{b}, tiles, cs, gtab, ntiles, nLong, gr, g, w, alpha, beta);
}

template <typename T, int MODE, int RB, int CB, bool ALL>
__global__ void __launch_bounds__(256) tile_mfma_seg_kernel(Bases b, const TileSeg* __restrict__ segs, int nseg,
                                                            MfGrid gr, int unitLog, T alpha, T beta)
{
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int per = gr.ur * gr.uc;
    auto first = [=](const TileSeg& s) { return ALL ? s.first * per : s.firstUnit[unitLog]; };
    const TileSeg* sg = seg_of(segs, nseg, (int)blockIdx.x, first);
    mfma_unit<T, MODE, RB, CB, ALL>(SegBases{b, sg}, sg->tiles, sg->cs, sg->gtab, sg->count, sg->nLong, gr,
                                    (int)blockIdx.x - first(*sg), w, alpha, beta);
}

template <typename T, int MODE, int RB, int CB, bool ALL>
static void launch_mfma_u(const Phase& ph, const Bases& b, T alpha, T beta, hipStream_t s)
{
    const MfGrid gr{(ph.maxMTile + 16 * RB - 1) / (16 * RB), (ph.maxKTile + 16 * CB - 1) / (16 * CB)};
    const int per = gr.ur * gr.uc;
    if (!ph.segSrc.empty()) {
        const int lg = per == 1 ? 0 : per == 2 ? 1 : 2;
        if (!ALL && per != 1 << lg) throw std::runtime_error("segmented tile units");
        const int64_t grid = ALL ? (int64_t)ph.segTiles * per : ph.segBlocks[lg];
        if (grid == 0) return;
        tile_mfma_seg_kernel<T, MODE, RB, CB, ALL><<<(unsigned)grid, 256, 0, s>>>(
            b, static_cast<const TileSeg*>(ph.dSegs), (int)ph.segSrc.size(), gr, lg, alpha, beta);
        return;
    }
    const int64_t n = (int64_t)ph.tiles.size(), lng = ALL ? n : ph.nLong;
    const int64_t grid = lng * per + ((n - lng) * per + 3) / 4;
    tile_mfma_kernel<T, MODE, RB, CB, ALL><<<(unsigned)grid, 256, 0, s>>>(
        b, static_cast<const Tile*>(ph.dTiles), static_cast<const Contrib*>(ph.dContribs),
        static_cast<const int64_t*>(ph.dGather), (int)n, ph.nLong, gr, alpha, beta);
}

// Units of the launch: 32 x 32 entries (a row or column block less where the
// tiles are narrower), one per wave but for the long tiles, where the phase
// has tiles enough to give each of the 1,024 SIMDs one such wave, else 16 x 16
// split over the four waves of a workgroup: such a phase is one tile's
// latency, and the split cuts it (direct inversion of 64^2 at rank 8, 940
// launches of at most a few hundred tiles: 15.4 -> 10.6 ms; of 256^2 at rank
// 16 with its refinement: 648 -> 500 ms. With the line at 512, 1,024, 2,048
// and 4,096 units: 8.20, 8.20, 8.30 and 8.46 ms, and 370, 370, 373 and 379 ms).
// From 8,192 units of tiles that are mostly wide (Phase::wide), units of 64
// columns: a quarter (16 rows: a sixth) fewer operand loads per MFMA and half as
// many waves that begin with a chain of dependent loads, for two waves per SIMD
// instead of three (H X with 64 columns on the 256^2 inverse 891 -> 846 us,
// 256^2 FP64 product 47.0 -> 45.6 ms, FP32 3D update 9.91 -> 8.61 ms, 9.00 with
// the line at 4,096).
constexpr int64_t kMfmaWaves = 1024, kMfmaWide = 8192;

template <typename T, int MODE>
static void launch_mfma(const Phase& ph, const Bases& b, T alpha, T beta, hipStream_t s)
{
    const int64_t n = ph.segSrc.empty() ? (int64_t)ph.tiles.size() : ph.segTiles;
    const int rb = ph.maxMTile <= 16 ? 1 : 2;
    int cb = ph.maxKTile <= 16 ? 1 : 2;
    const int64_t units = n * ((ph.maxMTile + 16 * rb - 1) / (16 * rb)) * ((ph.maxKTile + 16 * cb - 1) / (16 * cb));
    if (units >= kMfmaWide && ph.wide) cb = 4;
    if (units < kMfmaWaves) launch_mfma_u<T, MODE, 1, 1, true>(ph, b, alpha, beta, s);
    else if (rb == 1 && cb == 1) launch_mfma_u<T, MODE, 1, 1, false>(ph, b, alpha, beta, s);
    else if (rb == 2 && cb == 4) launch_mfma_u<T, MODE, 2, 4, false>(ph, b, alpha, beta, s);
    else if (cb == 4) launch_mfma_u<T, MODE, 1, 4, false>(ph, b, alpha, beta, s);
    else if (rb == 1) launch_mfma_u<T, MODE, 1, 2, false>(ph, b, alpha, beta, s);
    else if (cb == 1) launch_mfma_u<T, MODE, 2, 1, false>(ph, b, alpha, beta, s);
    else launch_mfma_u<T, MODE, 2, 2, false>(ph, b, alpha, beta, s);
}

// Segmented launches of a merged phase (its members' segment table).
template <typename T, int MR>
static void launch_tile_seg_mr(const Phase& ph, const Bases& b, T alpha, T beta, hipStream_t s)
{
    constexpr int TM = MR == 64 ? 4 : 1;
    const int grid = ph.segTiles;
    const int nseg = (int)ph.segSrc.size();
    const TileSeg* sg = static_cast<const TileSeg*>(ph.dSegs);
    const int kmax = ph.maxKTile;
    if (grid == 0) return;
    if (kmax <= 16) tile_seg_kernel<T, MR, 16, TM, 1><<<grid, 256, 0, s>>>(b, sg, nseg, alpha, beta);
    else if (kmax <= 32) tile_seg_kernel<T, MR, 32, TM, 2><<<grid, 256, 0, s>>>(b, sg, nseg, alpha, beta);
    else tile_seg_kernel<T, MR, 64, TM, 4><<<grid, 256, 0, s>>>(b, sg, nseg, alpha, beta);
}

template <typename T, int ROLE, int MR>
static void launch_tile_mr(int n, int kmax, const Bases& b, const Tile* t, const Contrib* c, const int64_t* g, T alpha,
                           T beta, hipStream_t s)
{
    constexpr int TM = MR == 64 ? 4 : 1;
    if (kmax <= 16) tile_kernel<T, MR, 16, TM, 1, ROLE><<<n, 256, 0, s>>>(b, t, c, g, alpha, beta);
    else if (kmax <= 32) tile_kernel<T, MR, 32, TM, 2, ROLE><<<n, 256, 0, s>>>(b, t, c, g, alpha, beta);
    else tile_kernel<T, MR, 64, TM, 4, ROLE><<<n, 256, 0, s>>>(b, t, c, g, alpha, beta);
}

template <typename T>
static void launch_mfma_engine(const Phase& ph, const Bases& b, T alpha, T beta, hipStream_t s, int engine)
{
    if constexpr (sizeof(T) == 4) {
        if (engine == TILE_MFMA_BF16 || engine == TILE_MFMA_BF16_PF) {
            launch_mfma<float, 1>(ph, b, alpha, beta, s);
            return;
        }
    }
    launch_mfma<T, 0>(ph, b, alpha, beta, s);
}

// Member segments of at least this many tiles launch one by one.
constexpr size_t kSegSplitTiles = 8192;

template <typename T>
void launch_tile_phase(const Phase& ph, const Bases& b, T alpha, T beta, hipStream_t s, int engine)
{
    if (!ph.segSrc.empty()) {
        if (ph.maxKTile > 64 || ph.maxMTile > 64) throw std::runtime_error("tile larger than 64 x 64");
        if (!ph.dSegs) throw std::runtime_error("segmented tile phase not uploaded");
        // Members whose own tile lists fill the chip several times over run
        // as one plain launch each, on their own bases: one launch over all
        // of them saves nothing and interleaves the members' operands in the
        // caches (measured on 12 3D members of 16^3-20^3: 30% slower).
        size_t smallest = SIZE_MAX;
        for (const auto& sg : ph.segSrc) smallest = std::min(smallest, sg.src->tiles.size());
        if (smallest >= kSegSplitTiles) {
            for (const auto& sg : ph.segSrc) {
                Bases mb;
                for (int k = 0; k < NUM_SLOTS; ++k) {
                    mb.val[k] = b.val[k] ? static_cast<void*>(static_cast<T*>(b.val[k]) + sg.val[k]) : nullptr;
                    mb.rank[k] = b.rank[k] ? b.rank[k] + sg.rank[k] : nullptr;
                }
                launch_tile_phase<T>(*sg.src, mb, alpha, beta, s, engine);
            }
            return;
        }
        if (engine != TILE_LDS) {
            launch_mfma_engine<T>(ph, b, alpha, beta, s, engine);
        } else if (ph.maxMTile <= 16) {
            launch_tile_seg_mr<T, 16>(ph, b, alpha, beta, s);
        } else {
            launch_tile_seg_mr<T, 64>(ph, b, alpha, beta, s);
        }
        HIP_LAUNCH_CHECK();
        return;
    }
    const int n = (int)ph.tiles.size();
    if (n == 0) return;
    const Tile* t = static_cast<const Tile*>(ph.dTiles);
    const Contrib* c = static_cast<const Contrib*>(ph.dContribs);
    const int64_t* g = static_cast<const int64_t*>(ph.dGather);
    const int kmax = ph.maxKTile;
    if (kmax > 64 || ph.maxMTile > 64) throw std::runtime_error("tile larger than 64 x 64");
    if (engine != TILE_LDS) {
        launch_mfma_engine<T>(ph, b, alpha, beta, s, engine);
        HIP_LAUNCH_CHECK();
        return;
    }
    // ROLE only distinguishes projection and accumulation launches in profiles;
    // MR = 16 serves phases whose tiles all have at most 16 rows.
    if (ph.maxMTile <= 16) {
        if (ph.role == 1) launch_tile_mr<T, 1, 16>(n, kmax, b, t, c, g, alpha, beta, s);
        else launch_tile_mr<T, 0, 16>(n, kmax, b, t, c, g, alpha, beta, s);
    } else {
        if (ph.role == 1) launch_tile_mr<T, 1, 64>(n, kmax, b, t, c, g, alpha, beta, s);
        else launch_tile_mr<T, 0, 64>(n, kmax, b, t, c, g, alpha, beta, s);
    }
    HIP_LAUNCH_CHECK();
}

template void launch_tile_phase<double>(const Phase&, const Bases&, double, double, hipStream_t, int);
template void launch_tile_phase<float>(const Phase&, const Bases&, float, float, hipStream_t, int);

} // namespace dmhm
