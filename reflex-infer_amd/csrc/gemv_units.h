// gemv_units.h -- which rows a wave of the Q4_K GEMV kernels takes and loads.
// Plain integer code for the kernels, their launcher and the host test that
// walks it (oracle/gemv_units_probe.cpp): every row that a wave loads lies in
// the range that it serves.
#pragma once

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define RXQ4_UNITS_FN __host__ __device__ __forceinline__
#else
#define RXQ4_UNITS_FN inline
#endif

namespace rxq4 {

// Cuts n_ranges ranges of `rows` rows into units of `per_unit` items of
// `rows_per_item` rows; a unit serves one range, range i from unit_start[i] on.
// Returns the units.
inline int cut_units(const int *rows, int n_ranges, int rows_per_item, int per_unit, int *unit_start) {
    int units = 0;
    for (int i = 0; i < 3; ++i) {
        unit_start[i] = units;
        if (i >= n_ranges) continue;
        const int items = (rows[i] + rows_per_item - 1) / rows_per_item;
        units += (items + per_unit - 1) / per_unit;
    }
    return units;
}

// The range that unit `unit` serves (u1, u2: the first units of ranges 1 and 2).
RXQ4_UNITS_FN int range_index(int unit, int n_ranges, int u1, int u2) {
    return n_ranges > 1 && unit >= u1 ? (n_ranges > 2 && unit >= u2 ? 2 : 1) : 0;
}

// The items [begin, end) of a unit of a range of n_items; none, at 0, for a wave
// past the units.
struct UnitSpan {
    int begin, end;
};
RXQ4_UNITS_FN UnitSpan unit_span(bool active, int unit, int first_unit, int per_unit, int n_items) {
    UnitSpan s{0, 0};
    if (active) {
        s.begin = (unit - first_unit) * per_unit;
        s.end = s.begin + per_unit < n_items ? s.begin + per_unit : n_items;
    }
    return s;
}

// The item whose rows are loaded for item `item` of a span that ends at `end`:
// itself, the span's last past it, item 0 for an empty span.
RXQ4_UNITS_FN int load_item(int item, int end) {
    const int i = item < end - 1 ? item : end - 1;
    return i > 0 ? i : 0;
}

// The row that lane group `sub` loads of such an item of `rows_per_item` rows
// (the range's last row `last` past it).
RXQ4_UNITS_FN int load_row(int item, int end, int rows_per_item, int sub, int last) {
    const int row = load_item(item, end) * rows_per_item + sub;
    return row < last ? row : last;
}

}  // namespace rxq4
