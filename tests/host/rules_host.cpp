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
            int line, curved;
            double mb;
            std::cin >> line >> curved >> mb;
            std::cout << store_stays_cached(dim, n, line, curved, mb) << "\n";
        } else {
            return 1;
        }
    }
    return 0;
}
