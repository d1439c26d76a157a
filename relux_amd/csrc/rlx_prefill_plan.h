// Work lists of a chunked prefill call: which query tiles are cut along the
// keys, and the order of the work items over the XCDs.  Host code; the element
// types of the lists (four and two ints) are the caller's.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace rlx {

constexpr int kXcds = 8;

// The query tiles of a call's sequences (the same for every head), by the keys
// each attends.
struct PfTiles {
    std::vector<int> first{0};  // index of each sequence's first tile, and the end
    std::vector<int> keys;
    int seqs() const { return (int)first.size() - 1; }
    void add(int n) { keys.push_back(n); }
    void end_seq() { first.push_back((int)keys.size()); }
};
inline int pf_blocks(int keys) { return (keys + 63) / 64; }  // key blocks of the kernel

// Cuts of a prefill call's tiles along the keys.  A work-group (one per CU)
// walks its tile's keys in blocks of 64, so a call with fewer tiles than CUs,
// or a few long ones, leaves most of the chip waiting: B 1, 8 kv heads, 16 new
// tokens on 8192 ran 8 work-groups of 128 blocks.  Tiles of more than `target`
// blocks are cut into equal parts, merged by their (max, sum) afterwards;
// the target is the one of a few whose estimate is least: the longest
// work-group or the CUs' share of the work, kPfStart blocks of start-up per
// work-group, the merge's launch and its traffic counted in (a block takes
// about 2 us), if it saves a tenth.  Calls that fill the chip stay whole.
// Measured (32 heads over 8, D 128, T 8192, us whole / cut): 16 new tokens 231 /
// 39, 128 235 / 56, 512 251 / 112; T 0: 1024 60 / 55.
// fill: the share of a tile's 256 rows that hold queries (what the merge moves).
// Returns the target, 0: every tile stays whole.
constexpr double kPfStart = 2.5, kPfMerge = 2.2, kPfMergePart = 0.035;
constexpr int kPfMaxParts = 480;  // 64 MB of partial sums
inline int prefill_target(const PfTiles &t, int heads, int cus, double fill) {
    int64_t total = 0;
    int most = 0;
    for (int keys : t.keys) {
        total += pf_blocks(keys);
        most = std::max(most, pf_blocks(keys));
    }
    total *= heads;
    const int64_t tiles = (int64_t)t.keys.size() * heads;
    if (tiles == 0 || tiles >= 2 * (int64_t)cus) return 0;
    auto estimate = [&](int64_t n, double longest) {
        const double share = ((double)total + (double)n * kPfStart) / cus;
        const double last = n > cus ? 0.5 * ((double)total / n + kPfStart) : 0.0;
        return std::max(longest + kPfStart, share + last);
    };
    int target = 0;
    double best = 0.9 * estimate(tiles, most);
    const int base = (int)std::max<int64_t>(4, (total + cus - 1) / cus);
    for (int k = 4; k <= 10; k++) {
        const int at = base * k / 4;
        if (at >= most) break;
        int64_t n = 0, cut = 0;
        int longest = 0;
        for (int keys : t.keys) {
            const int b = pf_blocks(keys), m = std::max(1, (b + at - 1) / at);
            n += m;
            if (m > 1) cut += m;
            longest = std::max(longest, (b + m - 1) / m);
        }
        n *= heads;
        cut *= heads;
        if (cut > kPfMaxParts) continue;
        const double e = estimate(n, longest) + kPfMerge + kPfMergePart * fill * (double)cut;
        if (e < best) {
            best = e;
            target = at;
        }
    }
    return target;
}

template <class I2, class I4>
struct PrefillPlan {
    std::vector<I4> work;    // (sequence, head, tile, part slot or -1: the whole tile); sequence -1: nothing
    std::vector<I2> ranges;  // part slot -> key blocks
    std::vector<I4> merge;   // cut tiles: (sequence, head, tile | parts << 20, first slot)
};

// The lists of `heads` heads.  Work-group b runs on XCD b % 8 and each XCD has
// its own L2, so all query tiles of one (sequence, head) -- which stream the
// same K/V blocks in the same order -- are placed on one XCD at consecutive
// positions: the XCD then fetches each block from HBM once.  Cut tiles are
// grouped by part, so that parts of the same keys stay together.  Groups go to
// the least-loaded XCD, largest first; shorter XCD lists are padded with empty
// items.  A cut call has about a work-group per CU, so there no XCD may get
// more than its eighth of them (a second round on a few CUs costs as much as
// the first): the ends of the longer lists move to the shorter ones.
// plain: the tiles in order, nothing placed (tuning).
template <class I2, class I4>
PrefillPlan<I2, I4> prefill_plan(const PfTiles &t, int heads, int target, bool plain = false) {
    PrefillPlan<I2, I4> plan;
    const int S = t.seqs(), T = (int)t.keys.size();
    // Parts of every tile, and the slot of its first part within its head.
    std::vector<int> parts(T), slot(T), head_slots(S);
    struct Group {
        double cost;
        int seq, part;
    };
    std::vector<Group> groups;
    for (int i = 0; i < S; i++) {
        int n = 0, most = 1;
        for (int q = t.first[i + 1] - 1; q >= t.first[i]; q--) {
            const int b = pf_blocks(t.keys[q]);
            parts[q] = target > 0 ? std::max(1, (b + target - 1) / target) : 1;
            most = std::max(most, parts[q]);
            slot[q] = n;
            if (parts[q] > 1) n += parts[q];
        }
        head_slots[i] = n;
        for (int k = 0; k < most; k++) {
            double cost = 0.0;
            for (int q = t.first[i]; q < t.first[i + 1]; q++)
                if (parts[q] > k) cost += (double)t.keys[q] / parts[q];
            groups.push_back(Group{cost, i, k});
        }
    }
    int base = 0;
    std::vector<int> seq_slot(S);
    for (int i = 0; i < S; i++) {
        seq_slot[i] = base;
        base += head_slots[i] * heads;
    }
    plan.ranges.resize(base);
    for (int i = 0; i < S; i++)
        for (int h = 0; h < heads; h++)
            for (int q = t.first[i + 1] - 1; q >= t.first[i]; q--) {
                const int m = parts[q], b = pf_blocks(t.keys[q]), s0 = seq_slot[i] + h * head_slots[i] + slot[q];
                if (m == 1) continue;
                for (int k = 0; k < m; k++)
                    plan.ranges[s0 + k] = I2{(int)((int64_t)b * k / m), (int)((int64_t)b * (k + 1) / m)};
                plan.merge.push_back(I4{i, h, (q - t.first[i]) | m << 20, s0});
            }
    auto put = [&](std::vector<I4> &list, const Group &g, int h) {
        for (int q = t.first[g.seq + 1] - 1; q >= t.first[g.seq]; q--)
            if (parts[q] > g.part)
                list.push_back(I4{g.seq, h, q - t.first[g.seq],
                                  parts[q] == 1 ? -1 : seq_slot[g.seq] + h * head_slots[g.seq] + slot[q] + g.part});
    };
    if (plain) {
        for (const Group &g : groups)
            for (int h = 0; h < heads; h++) put(plan.work, g, h);
        return plan;
    }
    std::stable_sort(groups.begin(), groups.end(), [](const Group &a, const Group &b) { return a.cost > b.cost; });
    std::vector<I4> lists[kXcds];
    double load[kXcds] = {};
    for (const Group &g : groups)
        for (int h = 0; h < heads; h++) {
            const int x = (int)(std::min_element(load, load + kXcds) - load);
            load[x] += g.cost;
            put(lists[x], g, h);
        }
    size_t total = 0;
    for (auto &l : lists) total += l.size();
    if (base > 0) {
        const size_t most = (total + kXcds - 1) / kXcds;
        int to = 0;
        for (auto &l : lists)
            while (l.size() > most) {
                while (lists[to].size() >= most) to++;
                lists[to].push_back(l.back());
                l.pop_back();
            }
    }
    size_t n = 0;
    for (auto &l : lists) n = std::max(n, l.size());
    plan.work.assign(n * kXcds, I4{-1, 0, 0, 0});
    for (int x = 0; x < kXcds; x++)
        for (size_t i = 0; i < lists[x].size(); i++) plan.work[i * kXcds + x] = lists[x][i];
    return plan;
}

}  // namespace rlx
