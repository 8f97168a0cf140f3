// Prints the batches of one schedule (als_sched.hpp): its batch_work, then
// batch_begin. Arguments: split_len batch_work grid prec shrinks
// slow_ratings; rating counts of the rows on standard input.
#include <cstdio>
#include <cstdlib>

#include "als_sched.hpp"

int main(int argc, char **argv) {
    if (argc != 7) return 2;
    std::vector<int> ptr{0};
    for (int n; std::scanf("%d", &n) == 1;) ptr.push_back(ptr.back() + n);
    const als::Schedule s = als::build_schedule((int64_t)ptr.size() - 1, ptr.data(), std::atoll(argv[1]), std::atoll(argv[2]),
                                                std::atoi(argv[3]), std::atoi(argv[4]), nullptr, std::atoi(argv[5]) != 0,
                                                std::atoi(argv[6]) != 0);
    std::printf("%lld", (long long)s.batch_work);
    for (int b : s.batch_begin) std::printf(" %d", b);
    return 0;
}
