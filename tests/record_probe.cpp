// Test helper: prints record_fits for "steps step rest free total" lines and
// tape_rest for "rest field plane q calc near target" lines of the input.
#include <cstdio>
#include <cstring>

#include "record.hpp"

using namespace lbm_amd;

int main() {
    char kind[8];
    unsigned long long a[6];
    while (std::scanf("%7s", kind) == 1) {
        if (!std::strcmp(kind, "rest")) {
            for (auto& v : a)
                if (std::scanf("%llu", &v) != 1) return 1;
            std::printf("%zu\n", tape_rest(a[0], a[1], static_cast<int>(a[2]), a[3], a[4], a[5]));
        } else {
            for (int i = 0; i < 5; ++i)
                if (std::scanf("%llu", &a[i]) != 1) return 1;
            std::printf("%d\n", record_fits(a[0], a[1], a[2], a[3], a[4]) ? 1 : 0);
        }
    }
    return 0;
}
