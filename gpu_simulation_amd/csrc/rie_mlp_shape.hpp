// Launch shapes of the network's products (rie_mlp.hip), for the sizes that
// rie_mlp_create and the row calls accept.  Host arithmetic only.
#pragma once

#include <cstddef>

namespace rie {

constexpr int kMlpMaxRows = 1 << 22;
constexpr int kMlpMaxWidth = 4096;

// Grid of an M x N product.  32 x 32 tiles (sub 2) read each operand half as
// often; below 512 of them the chip has idle CUs and 16 x 16 tiles (sub 1) win.
// The column tiles are on x, so that the workgroups that read the same rows
// start together (with the rows on x a loss and gradient of 100,000 rows through
// 256 hidden units takes 5.5 ms, so 5.2).  The row tiles are on y, and beyond its
// 65535 blocks on y and z: tile blockIdx.z * gridDim.y + blockIdx.y, the last
// z's may have none.
constexpr int kMlpWideTiles = 512;

struct MlpGrid {
    int sub;
    unsigned rows;  // row tiles
    unsigned x;
    unsigned y;
    unsigned z;
};

constexpr MlpGrid mlp_grid(int M, int N) {
    const long wide = (long)((M + 31) / 32) * ((N + 31) / 32);
    const int sub = wide >= kMlpWideTiles ? 2 : 1;
    const int tile = 16 * sub;
    const unsigned rows = (unsigned)((M + tile - 1) / tile);
    const unsigned y = rows <= 65535 ? rows : 32768;
    return {sub, rows, (unsigned)((N + tile - 1) / tile), y, (rows + y - 1) / y};
}

// Workgroups of the loss product with up to `rows` rows: the 16 x 16 grid of
// fewer rows may be the larger one, of fewer than 4 kMlpWideTiles tiles.
constexpr size_t mlp_mse_partials(int rows, int cols) {
    const size_t wide = (size_t)((rows + 31) / 32) * ((cols + 31) / 32);
    return wide > 4 * (size_t)kMlpWideTiles ? wide : 4 * (size_t)kMlpWideTiles;
}

// Values that the loss is the mean of: up to 2^34.
constexpr long long mlp_elements(int rows, int cols) { return (long long)rows * cols; }

}  // namespace rie
