#include "als_sched.hpp"

#include <algorithm>
#include <numeric>

#include "als_launch.hpp"

namespace als {

constexpr int64_t GPU_SIMDS = 1024;  // 256 CUs of four

int64_t row_solve_cost(int prec) { return prec == PREC_FP32 ? 96 : 1024; }

Schedule build_schedule(int64_t rows, const int *ptr, int64_t split_len, int64_t batch_work, int grid, int prec,
                        const std::vector<int> *subset, bool shrinks, bool slow_ratings) {
    Schedule s;
    const int64_t solve = row_solve_cost(prec);
    const int64_t nrows = subset ? (int64_t)subset->size() : rows;
    auto row_at = [&](int64_t i) -> int64_t { return subset ? (int64_t)(*subset)[i] : i; };
    int64_t total = 0;
    for (int64_t i = 0; i < nrows; i++) {
        const int64_t r = row_at(i);
        total += (int64_t)(ptr[r + 1] - ptr[r]) + solve;
    }
    const int64_t waves = std::max<int64_t>(1, grid);
    // Parts small enough that the heaviest row spreads over many waves, large
    // enough that the traffic of the partial tiles stays small next to the
    // gathers: an eighth of what each SIMD gets, however many waves of the
    // kernel at hand fit on it (their gathers share its time). Counted by waves
    // instead, kernels of fewer blocks, which fit more often, cut rows shorter:
    // 16-bit Gram and CG, items of a quarter of the netflix shape, f = 80 at
    // three waves a SIMD, parts of 2,048 653 us, of 4,322 500; f = 112 at two,
    // 742 and 555.
    s.split_len = split_len > 0 ? split_len : std::max<int64_t>(2048, total / (std::min(waves, GPU_SIMDS) * 8));
    s.batch_work = batch_work > 0 ? batch_work : std::max<int64_t>(solve, total / (waves * 16));

    struct Item { Unit u; int64_t cost; };
    std::vector<Item> items;
    items.reserve(nrows + total / s.split_len + 1);
    for (int64_t i = 0; i < nrows; i++) {
        const int64_t r = row_at(i);
        const int64_t n = ptr[r + 1] - ptr[r];
        if (n <= s.split_len) {
            items.push_back({{(int)r, ptr[r], ptr[r + 1], -1}, n + solve});
            continue;
        }
        const int64_t P = (n + s.split_len - 1) / s.split_len;
        const int64_t len = (n + P - 1) / P;
        Split sp{(int)s.nslots, (int)P, (int)len, 0};
        const int sid = (int)s.splits.size();
        s.splits.push_back(sp);
        s.nslots += P;
        for (int64_t p = 0; p < P; p++) {
            const int64_t kb = ptr[r] + p * len, ke = std::min<int64_t>(ptr[r + 1], kb + len);
            items.push_back({{(int)r, (int)kb, (int)ke, sid}, (ke - kb) + (p == P - 1 ? solve : 0)});
        }
    }
    std::stable_sort(items.begin(), items.end(), [](const Item &a, const Item &b) { return a.cost > b.cost; });
    s.units.reserve(items.size());
    // Batches of batch_work, heaviest rows first. Each batch but a wave's first
    // costs an atomic on a counter that all waves share, some 12 ns, one after
    // the other. Where they may shrink (shrinks) and an average batch is
    // little more work than the GPU gets through in that time, the waves would
    // wait for the counter: there the batches start large and shrink to
    // batch_work, each taking half of what an even share of the work still left
    // would be, and small ones are left for the end, to even out what the cost
    // model got wrong. One half-sweep of the
    // users, even batches -> shrinking: ml10M shape, f = 64 FP32 838 -> 580
    // us (62,600 -> 32,300 batches), f = 16 805 -> 490, f = 80 16-bit Gram and
    // CG 437 -> 289; a quarter of the netflix-shaped users, f = 100 FP32 2.22 ->
    // 2.02 ms. At the whole netflix shape with the 16-bit Gram (items, batches
    // of 6,100 on average) there is nothing to gain, and large first batches
    // lose: 6.54 -> 6.64 ms a sweep.
    // No batch is larger than `most`, a size at which the counter is no
    // bottleneck any more: of a larger one the model's error is all that is
    // felt. Without it 16-bit users with two refinement steps lost what the
    // short rows gain (f = 32 708 -> 773 us, f = 140 4.62 -> 5.20 ms; a quarter
    // of the netflix shape, f = 48 1.72 -> 2.07). Where a rating takes about
    // twice the model's time, at 8 and 9 blocks and with classic refinement,
    // which reads a row's ratings again for each step, half the size is the
    // better one: BF16 users at f = 128 656 us without a bound, 657 at the whole
    // of it, 631 at half (even 952); CG items at f = 140 738, 737, 692 (even
    // 690); refined 16-bit users at f = 32 773, 799, 682. At fewer blocks it is
    // not: BF16 users at f = 80 724, 740, 776 (even 984), a quarter of the
    // netflix shape.
    const int64_t small = prec == PREC_FP32 ? 768 : 4608;
    const int64_t most = slow_ratings ? small : 2 * small;
    for (const Item &it : items) s.units.push_back(it.u);
    int64_t all = 0;
    for (const Item &it : items) all += it.cost;
    auto cut = [&](bool shrink) {
        s.batch_begin.assign(1, 0);
        int64_t left = all, acc = 0;
        auto size_at = [&] { return std::max(s.batch_work, shrink ? std::min(most, left / (2 * waves)) : 0); };
        int64_t want = size_at();
        for (size_t i = 0; i < items.size(); i++) {
            acc += items[i].cost;
            if (acc >= want) {
                s.batch_begin.push_back((int)(i + 1));
                left -= acc;
                acc = 0;
                want = size_at();
            }
        }
    };
    cut(false);
    s.shrunk = shrinks && all < small * (int64_t)s.batch_begin.size();
    if (s.shrunk) cut(true);
    if (s.batch_begin.back() != (int)items.size()) s.batch_begin.push_back((int)items.size());
    return s;
}

}  // namespace als
