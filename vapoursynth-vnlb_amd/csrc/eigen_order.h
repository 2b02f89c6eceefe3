// Order of eigenpairs: descending by value, equal ones in index order
// (topk_symmetric_eigen_jacobi's stable sort, linalg.cpp:447-519), NaN last.
// A model with an infinite sample has infinite and NaN diagonals; places that
// were no permutation then would leave an eigenpair unwritten.
#pragma once

#include <hip/hip_runtime.h>

namespace vnlbhip {

// What a value is ordered by.
template <class T> __host__ __device__ inline T order_key(T value) {
    return value == value ? value : -static_cast<T>(__builtin_huge_val());
}

// Whether the entry with key a comes before the one with key b; `first`: its
// index is the lower one.
template <class T> __host__ __device__ inline bool ordered_before(T a, T b, bool first) {
    return a > b || (first && !(b > a));
}

// Place of entry r among n values.
template <class T> __host__ __device__ inline int descending_place(const T* values, int n, int r) {
    const T own = order_key(values[r]);
    int place = 0;
    for (int j = 0; j < n; ++j) {
        place += j != r && ordered_before(order_key(values[j]), own, j < r) ? 1 : 0;
    }
    return place;
}

}  // namespace vnlbhip
