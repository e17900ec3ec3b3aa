// Host build of the dispatch rules (philip_amd/csrc/dg_rules.hpp): reads lines of a rule's name and
// its arguments from stdin, prints what it answers.
#include <iostream>
#include <string>
#include "../../philip_amd/csrc/dg_rules.hpp"
using namespace dgx;

int main()
{
    std::string rule;
    while (std::cin >> rule) {
        int dim, n;
        std::cin >> dim >> n;
        if (rule == "store") {
            int fp64, line, curved;
            double mb;
            std::cin >> fp64 >> line >> curved >> mb;
            std::cout << store_stays_cached(dim, n, fp64, line, curved, mb) << "\n";
        } else if (rule == "small") {  // of a mesh of `cells` on 256 compute units
            int fp64, form, cells;
            std::cin >> fp64 >> form >> cells;
            const int b = block_elements(dim, n), s = small_elements(dim, n);
            std::cout << takes_small_block(dim, n, fp64, form, (cells + b - 1) / b, (cells + s - 1) / s, 256) << "\n";
        } else if (rule == "conservative") {
            int boundary, stage, cells;
            std::cin >> boundary >> stage >> cells;
            const int b = block_elements(dim, n);
            std::cout << takes_conservative_line(dim, n, boundary, stage, (cells + b - 1) / b, 256) << "\n";
        } else if (rule == "batch") {
            int fp64;
            long blocks;
            std::cin >> fp64 >> blocks;
            std::cout << batch_takes_small_tile(dim, n, fp64, blocks, 256) << "\n";
        } else if (rule == "prefetch") {
            int fp64;
            std::cin >> fp64;
            std::cout << butcher_prefetch(dim, n, fp64) << "\n";
        } else {
            return 1;
        }
    }
    return 0;
}
