// Runs f32_unit (qwen3.5sharp_amd/csrc/f32_stage.h) for a workgroup and a tile
// of argv[1] rows x argv[2] units; prints a line for each fault.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "f32_stage.h"

int main(int, char** argv) {
    const int rows = atoi(argv[1]), c4 = atoi(argv[2]), n = rows * c4;
    std::vector<int> stores(n);
    for (int i = 0; i < (n + 255) / 256; ++i)
        for (int tid = 0; tid < 256; ++tid) {
            const q35::F32Unit u = q35::f32_unit(tid, i, rows, c4);
            if (u.slot < 0 || u.slot >= n) { printf("thread %d unit %d: slot %d\n", tid, i, u.slot); continue; }
            // Slot (row, 16 q + lane) holds columns 64 q + lane + 16 s.
            const int row = u.slot / c4, q = u.slot % c4 / 16, lane = u.slot % 16;
            if (u.row != row || u.col != 64 * q + lane) printf("thread %d unit %d: (%d, %d) for slot %d\n", tid, i, u.row, u.col, u.slot);
            stores[u.slot] += u.store;
        }
    for (int s = 0; s < n; ++s)
        if (stores[s] != 1) printf("slot %d stored %d times\n", s, stores[s]);
    return 0;
}
