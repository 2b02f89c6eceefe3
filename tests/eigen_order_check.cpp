// Places of eigenpairs for every diagonal of up to six entries drawn from
// infinities, NaN, zeros of both signs and ordinary values: a permutation
// always, and the stable descending sort where there is no NaN.
#include "eigen_order.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <numeric>

using namespace vnlbhip;

template <class T> int check(const char* type) {
    const T inf = static_cast<T>(INFINITY);
    const T draws[] = {static_cast<T>(NAN), inf, -inf, static_cast<T>(-1), static_cast<T>(-0.0), static_cast<T>(0),
                       static_cast<T>(2)};
    constexpr int kDraws = 7;
    for (int n = 1; n <= 6; ++n) {
        int cases = 1;
        for (int i = 0; i < n; ++i) {
            cases *= kDraws;
        }
        for (int index = 0; index < cases; ++index) {
            T values[6];
            int rest = index;
            bool nan = false;
            for (int i = 0; i < n; ++i, rest /= kDraws) {
                values[i] = draws[rest % kDraws];
                nan = nan || values[i] != values[i];
            }
            int entry[6] = {-1, -1, -1, -1, -1, -1};
            for (int r = 0; r < n; ++r) {
                entry[descending_place(values, n, r)] = r;
            }
            int sorted[6];
            std::iota(sorted, sorted + n, 0);
            std::stable_sort(sorted, sorted + n,
                             [&](int a, int b) { return order_key(values[a]) > order_key(values[b]); });
            if (!std::equal(sorted, sorted + n, entry)) {
                std::printf("%s case %d of %d values: wrong order%s\n", type, index, n, nan ? " (NaN)" : "");
                return 1;
            }
        }
    }
    return 0;
}

int main() { return check<float>("float") + check<double>("double"); }
