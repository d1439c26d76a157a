// Properties of the prefill work lists (relux_amd/csrc/rlx_prefill_plan.h) over
// generated calls.  Exit status 0: they hold.
#include "rlx_prefill_plan.h"

#include <cstdio>
#include <map>
#include <numeric>
#include <random>
#include <tuple>

struct I2 {
    int x, y;
};
struct I4 {
    int x, y, z, w;
};

#define CHECK(c)                                                                             \
    do {                                                                                     \
        if (!(c)) {                                                                          \
            std::printf("line %d: %s (seqs %d heads %d target %d)\n", __LINE__, #c, t.seqs(), heads, target); \
            return 1;                                                                        \
        }                                                                                    \
    } while (0)

static int check(const rlx::PfTiles &t, int heads, int target, int cus) {
    const auto plan = rlx::prefill_plan<I2, I4>(t, heads, target);
    CHECK(plan.work.size() % rlx::kXcds == 0);
    // every item once; where it runs
    std::map<std::tuple<int, int, int>, std::vector<int>> items;  // (seq, head, tile) -> slots
    std::map<std::pair<int, int>, int> xcd;                       // (seq, head) of whole calls
    std::vector<int> per_xcd(rlx::kXcds);
    for (size_t i = 0; i < plan.work.size(); i++) {
        const I4 w = plan.work[i];
        if (w.x < 0) continue;
        CHECK(w.x < t.seqs() && w.y >= 0 && w.y < heads && w.z >= 0 && w.z < t.first[w.x + 1] - t.first[w.x]);
        CHECK(w.w >= -1 && w.w < (int)plan.ranges.size());
        items[{w.x, w.y, w.z}].push_back(w.w);
        per_xcd[i % rlx::kXcds]++;
        if (target == 0) {
            const auto at = xcd.emplace(std::make_pair(w.x, w.y), (int)(i % rlx::kXcds));
            CHECK(at.first->second == (int)(i % rlx::kXcds));  // one XCD's L2 serves the tiles of a head
        }
    }
    // merge: (seq, head, tile | parts << 20, first slot)
    std::map<std::tuple<int, int, int>, std::pair<int, int>> merged;
    for (const I4 &m : plan.merge) {
        CHECK(merged.emplace(std::make_tuple(m.x, m.y, m.z & 0xFFFFF), std::make_pair(m.z >> 20, m.w)).second);
    }
    std::vector<int> used(plan.ranges.size());
    size_t n = 0;
    for (int i = 0; i < t.seqs(); i++)
        for (int h = 0; h < heads; h++)
            for (int q = 0; q < t.first[i + 1] - t.first[i]; q++) {
                auto it = items.find({i, h, q});
                CHECK(it != items.end());
                const int b = rlx::pf_blocks(t.keys[t.first[i] + q]);
                std::vector<int> &s = it->second;
                n += s.size();
                std::sort(s.begin(), s.end());
                if (s[0] == -1) {  // whole
                    CHECK(s.size() == 1 && !merged.count({i, h, q}) && (target == 0 || b <= target));
                    continue;
                }
                const auto m = merged.find({i, h, q});
                CHECK(m != merged.end() && m->second.first == (int)s.size() && m->second.second == s[0]);
                int at = 0;  // the parts' ranges, in order, are the tile's blocks
                for (size_t k = 0; k < s.size(); k++) {
                    CHECK(s[k] == s[0] + (int)k && ++used[s[k]] == 1);
                    const I2 r = plan.ranges[s[k]];
                    CHECK(r.x == at && r.y > r.x && r.y - r.x <= target);
                    at = r.y;
                }
                CHECK(at == b);
            }
    CHECK(n == (size_t)std::accumulate(per_xcd.begin(), per_xcd.end(), 0));
    for (int u : used) CHECK(u == 1);
    CHECK(plan.merge.size() == merged.size());
    // a cut call's work-groups fit one round of every XCD's CUs if they fit the chip's
    if (!plan.ranges.empty() && (int)n <= cus)
        for (int x : per_xcd) CHECK(x <= cus / rlx::kXcds);
    return 0;
}

int main() {
    std::mt19937 rng(7);
    auto upto = [&](int n) { return (int)(rng() % n) + 1; };
    int cut = 0;
    for (int round = 0; round < 3000; round++) {
        rlx::PfTiles t;
        const int S = upto(6), heads = 1 << (rng() % 6), toks = 256 >> (rng() % 5);
        for (int i = 0; i < S; i++) {
            const int old = rng() % 3 ? (int)(rng() % 9000) : 0, nq = upto(1500);
            for (int q = 0; q * toks < nq; q++) t.add(old + std::min(nq, (q + 1) * toks));
            t.end_seq();
        }
        const int target = rlx::prefill_target(t, heads, 256, 1.0);
        cut += target > 0;
        if (check(t, heads, 0, 256) || (target > 0 && check(t, heads, target, 256)) ||
            check(t, heads, upto(40), 256))
            return 1;
        // the heads of a smaller launch, and a sequence whose queries see no key
        if (target > 0 && check(t, upto(heads), target, 256)) return 1;
        t.add(0);
        t.end_seq();
        if (check(t, heads, target, 256)) return 1;
    }
    if (cut < 300) {
        std::printf("only %d calls were cut\n", cut);
        return 1;
    }
    return 0;
}
