// bh_pick.hpp -- the order in which the heavy set is chosen, free of HIP.
#pragma once

#include <cstdint>
#include <limits>

namespace bh {

constexpr uint32_t kNoRow = 0xffffffffu;

// A body as the selection sees it: its weight and its row (kNoRow: none).
struct Pick {
    double m;
    uint32_t i;
};

// The weight is the mass; a NaN weighs least, so that every two picks compare
// and a set's ranks by counting are all different (with NaN weights, which
// compare with nothing, two picks could share a rank and a slot stay unset).
constexpr Pick pick(double mass, uint32_t row)
{
    return Pick{mass == mass ? mass : -std::numeric_limits<double>::infinity(), row};
}

// Descending weight, then ascending row; no row comes last.
constexpr bool heavier(const Pick& a, const Pick& b)
{
    if (a.i == kNoRow || b.i == kNoRow) return b.i == kNoRow && a.i != kNoRow;
    return a.m > b.m || (a.m == b.m && a.i < b.i);
}

}  // namespace bh
