// Replays the MFMA tile kernel's walk over inner chunks (ChunkWalk) on the
// host, fetch by fetch, for every pair and triple of inner dimensions: each
// fetch lies inside the contribution whose operands are set, and each chunk is
// multiplied once over the waves. Exits with 1 and a line at the first fault.
#include <cstdio>
#include <cstring>
#include "chunks.hpp"

static int used[3][17];

template <int S, bool TAIL>
static bool walk(const int* q, int n, int wave, bool byChunk)
{
    uint64_t left = 0;
    for (int i = 0; i < n; ++i)
        if ((TAIL ? q[i] & 15 : q[i] >= 16) && (S == 1 || byChunk || i % S == wave)) left |= uint64_t(1) << i;
    dmhm::ChunkWalk<S> w{wave, byChunk};
    int at = -1;                                // the contribution whose operands are set
    bool ok = true;
    auto next = [&] { return w.template next<TAIL>(left, [&](int i) { return q[i]; }, [&](int i) { at = i; }); };
    struct Fetch { int i, p; };
    auto fetch = [&]() -> Fetch {
        ok = ok && at >= 0 && w.q == q[at] && w.p >= 0 && w.p % 16 == 0 && (TAIL ? w.p < w.q : w.p + 16 <= w.q);
        return {at, w.p};
    };
    auto use = [&](Fetch f) { if (f.i >= 0) ++used[f.i][f.p / 16]; };
    // The loop of the kernel: two register sets, the last fetch repeated.
    if (!next()) return true;
    Fetch f0 = fetch(), f1;
    while (ok) {
        const bool more1 = next();
        f1 = fetch();
        use(f0);
        if (!more1) break;
        const bool more0 = next();
        f0 = fetch();
        use(f1);
        if (!more0) break;
    }
    return ok;
}

template <int S>
static bool check(const int* q, int n, bool byChunk)
{
    std::memset(used, 0, sizeof used);
    bool ok = true;
    for (int w = 0; w < S; ++w) ok = walk<S, false>(q, n, w, byChunk) && ok;
    for (int w = 0; w < S; ++w) ok = walk<S, true>(q, n, w, byChunk) && ok;
    for (int i = 0; i < n; ++i)
        for (int c = 0; c < 17; ++c) ok = ok && used[i][c] == (16 * c < q[i]);
    if (!ok) std::printf("S %d byChunk %d q %d %d %d of %d\n", S, byChunk, q[0], n > 1 ? q[1] : 0, n > 2 ? q[2] : 0, n);
    return ok;
}

int main()
{
    for (int a = 1; a <= 256; ++a)
        for (int b = 1; b <= 256; ++b) {
            const int two[2] = {a, b};
            if (!check<4>(two, 2, true) || !check<4>(two, 2, false) || !check<1>(two, 2, false)) return 1;
            for (int c = 1; c <= 256; ++c) {
                const int three[3] = {a, b, c};
                if (!check<4>(three, 3, true)) return 1;
            }
        }
    std::puts("ok");
    return 0;
}
