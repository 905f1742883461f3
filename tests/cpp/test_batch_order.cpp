// The order in which workgroups take a batch's tile runs (batch_run_of): every
// run once, and in each 64 workgroups, eight per XCD, the next 64 of the list.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "batch.hpp"

int main() {
    for (int n : {1, 7, 8, 63, 64, 65, 127, 128, 1000, 4096, 9999}) {
        std::vector<int> seen(size_t(n), 0);
        for (int g = 0; g < n; ++g) {
            const int r = ndc::batch_run_of(g, n);
            if (r < 0 || r >= n || seen[size_t(r)]++ || r / 64 != g / 64) {
                std::printf("n %d: workgroup %d takes run %d\n", n, g, r);
                return 1;
            }
        }
    }
    return 0;
}
