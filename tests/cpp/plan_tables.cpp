// The table through which a product's plan reads its stacked factors: one entry
// per factor and one per stack of two or more, whatever the rank, hence at most
// 1.5 per low-rank term of the product, and every column of every tile it
// serves starts where a stored factor has a column. Exits with 1 and a line.
#include <cstdio>
#include <unordered_set>
#include "plan.hpp"

using namespace dmhm;
namespace dmhm {
void Plan::upload() {}
void Plan::release() {}
} // namespace dmhm

static bool check(int dim, int n, int levels, int rank)
{
    const int sizes[3] = {n, n, n};
    Geometry g(dim, sizes, levels, true);
    const Layout lay = Layout::make(g, std::vector<int>(g.lrBlocks.size(), rank), 0);
    Planner planner(g);
    planner.setWorkspaceBudget(int64_t(1) << 33);
    planner.setStacking(true, true);
    std::unique_ptr<Plan> plan(planner.hhProduct(lay, lay, lay, rank, 4));
    std::unordered_set<int64_t> starts;
    for (size_t i = 0; i < g.lrBlocks.size(); ++i)
        for (int c = 0; c < rank; ++c) {
            starts.insert(lay.uOff[i] + (int64_t)c * g.tbox(g.lrBlocks[i]).size);
            starts.insert(lay.vOff[i] + (int64_t)c * g.sbox(g.lrBlocks[i]).size);
        }
    size_t columns = 0;
    const size_t entries = plan->gtab.size(), terms = enumerateProductTerms(g).w.size();
    for (const Phase& ph : plan->phases) {
        for (const Tile& t : ph.tiles)
            for (int j = 0; t.gather >= 0 && j < t.k; ++j, ++columns)
                if (!starts.count(gather_column(t, plan->gtab.data(), j))) {
                    std::printf("dim %d n %d: column %d of a tile is no column of a factor\n", dim, n, j);
                    return false;
                }
    }
    std::printf("dim %d n %d: %zu entries, %zu terms, %zu columns\n", dim, n, entries, terms, columns);
    return columns > 0 && 2 * entries <= 3 * terms;
}

int main() { return check(2, 64, 4, 8) && check(2, 128, 5, 16) && check(3, 16, 3, 20) && check(3, 12, 3, 7) ? 0 : 1; }
