// How many workgroups of a persistent kernel a CU holds at once, found once a
// launch shape.
#pragma once

#include <cstdint>

namespace chm {

// A gemv_ranges instantiation's launch shapes: one or four waves a workgroup,
// a power of two of steps a wave, at most 32. Its dynamic LDS follows from the
// two, but not the other way round (four steps of four waves take as much as
// sixteen of one), so the shape is the key; and every shape has its place, so
// products that take turns on one instantiation (an attention layer's QKV and
// output projection) ask the runtime once each and not once a launch.
struct ResidentTable {
    uint32_t found[2][6] = {};  // [four waves][log2 of the steps]; 0: not asked yet

    template <typename Ask>
    uint32_t of(uint32_t waves, uint32_t steps, Ask&& ask) {
        uint32_t& held = found[waves > 1][__builtin_ctz(steps)];
        if (held == 0) held = ask();
        return held;
    }
};

}  // namespace chm
