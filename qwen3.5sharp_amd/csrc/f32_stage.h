// Which thread of a 256-thread workgroup stages what of linear_f32's chunk
// (linear_q.hip).  Plain C++, so the map is checked on the CPU.
#pragma once

namespace q35 {

// A thread's i-th 16-byte unit of a tile of `rows` rows (weight rows, then
// tokens) x c4 units (c4 a multiple of 16): the columns col, col + 16, + 32,
// + 48 of the chunk, which are one reference lane's next four elements.
struct F32Unit {
    int slot;        // unit of the tile, row by row
    int row, col;
    bool store;      // false past the last unit, which then reads it again
};

constexpr F32Unit f32_unit(int tid, int i, int rows, int c4) {
    const int e = tid + 256 * i, n = rows * c4, slot = e < n ? e : n - 1;
    return {slot, slot / c4, 64 * (slot % c4 / 16) + slot % 16, n % 256 == 0 || e < n};
}

}  // namespace q35
