// Walks the units of the Q4_K GEMV kernels that keep whole rows or row groups
// (csrc/gemv_units.h) on the CPU, for every wave of every workgroup, those past
// the units among them: the rows that a wave loads (its items and two batches of
// two past them) lie in the range that it serves, and the active waves' items
// cover every row once.  Prints the launches walked, or the first that fails.
#include <cstdio>
#include <random>
#include <vector>

#include "gemv_units.h"

using namespace rxq4;

static bool walk(const int *rows, int n, int rpi, int per_unit) {
    int start[3];
    const int total = cut_units(rows, n, rpi, per_unit, start);
    std::vector<std::vector<int>> seen(n);
    for (int i = 0; i < n; ++i) seen[i].assign(rows[i], 0);
    for (int wave = 0; wave < (total + 3) / 4 * 4; ++wave) {
        const bool active = wave < total;
        const int unit = active ? wave : 0;
        const int r = range_index(unit, n, start[1], start[2]);
        const int last = rows[r] - 1;
        const UnitSpan s = unit_span(active, wave, r == 0 ? 0 : start[r], per_unit, (rows[r] + rpi - 1) / rpi);
        if (active ? s.end <= s.begin : s.end != s.begin) return false;
        for (int item = s.begin; item < s.end + 4; ++item)
            for (int sub = 0; sub < rpi; ++sub) {
                // (the whole-row kernel loads the item itself)
                const int row = rpi == 1 ? load_item(item, s.end) : load_row(item, s.end, rpi, sub, last);
                if (row < 0 || row >= rows[r]) {
                    std::printf("wave %d loads row %d of range %d\n", wave, row, r);
                    return false;
                }
                const int own = item * rpi + sub;
                if (item < s.end && own <= last) {
                    if (row != own) return false;
                    ++seen[r][own];
                }
            }
    }
    for (int i = 0; i < n; ++i)
        for (const int c : seen[i])
            if (c != 1) return false;
    return true;
}

int main() {
    std::mt19937 g(7);
    long walked = 0;
    const auto check = [&](std::vector<int> rows, int rpi, int per_unit) {
        ++walked;
        if (walk(rows.data(), (int)rows.size(), rpi, per_unit)) return true;
        std::printf("fails: %zu ranges, first of %d rows, %d rows an item, %d items a unit\n", rows.size(), rows[0],
                    rpi, per_unit);
        return false;
    };
    for (const int rpi : {1, 2, 4, 8}) {
        // the sizes whose last workgroup had waves that read past range 0
        for (const auto &rows : std::vector<std::vector<int>>{{2503, 2604}, {5101}, {1, 5099, 3}, {7, 9, 3}, {1}})
            for (int per = 1; per <= 8; ++per)
                if (!check(rows, rpi, per)) return 1;
        for (int i = 0; i < 600; ++i) {
            std::vector<int> rows(1 + g() % 3);
            for (int &m : rows) m = 1 + (int)(g() % (i % 3 ? 300 : 6000));
            if (!check(rows, rpi, 1 + (int)(g() % 12))) return 1;
        }
    }
    std::printf("walked %ld\n", walked);
    return 0;
}
