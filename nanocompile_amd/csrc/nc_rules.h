// Which kernel takes a problem, and what its loads may name: whole-number rules that host and device
// code share and a plain C++ compiler takes too, so that tests run them without a GPU.
#pragma once

#include <stdint.h>

namespace nc {

// The piece a prefetch of piece `at` of a table block of `pieces` reads: past the block's end its last
// one again (never used). A buffer load does not check its scalar offset against the buffer's size, so
// the index itself has to stay in the block, which may be the last of its allocation.
constexpr int head_piece(int at, int pieces) { return at < pieces ? at : pieces - 1; }

// Whether a launch runs whole: a grid has fewer than 2^32 threads along one dimension. Past that the count
// is cut to 32 bits (measured: the launch reports no error and most outputs are never written).
constexpr bool grid_fits(int64_t workgroups, int64_t threads) { return workgroups < ((int64_t)1 << 32) / threads; }

// Workgroups of the multi-row head (four waves, each one block of 64 table rows by `tile` rows of x),
// along one dimension of its grid.
constexpr int64_t head_workgroups(int64_t M, int64_t V, int tile) {
    return (M + tile - 1) / tile * (((V + 63) / 64 + 3) / 4);
}

// Rows of x a wave of the LM head takes, for M rows by a table of V: 16 once that leaves two waves a SIMD,
// 4 down to one wave a SIMD of the one-row kernels' (which read the table anew for every row, but whose
// many short waves hide what a few long ones cannot), else 0: the one-row kernels, whose grid has the rows
// along its second dimension, so they also take what the others' grid does not hold.
// Measured on MI355X, us, one row / 4 / 16 a wave:
// 128 x 151936 x 896: 10160 / 924 / 579; 16: 1272 / 167 / 124; 4: 322 / 104 / 122; 500 x 4864 x 896:
// 718 / 113 / 100; 128 x 4864 x 896: 141 / 39 / 50; 500 x 896 x 4864: 734 / 130 / 248;
// 16 x 4864 x 896: 21.1 / 20.3 / 49; 8 x 8192 x 8192: 228 / 195 / 410; 33 x 896 x 896: 10.6 / 20.6 / 49; 4 x 4864 x 896: 10.8 / 20.9 / 52.
constexpr int head_tile(int64_t M, int64_t V) {
    const int64_t blocks = (V + 63) / 64;
    const int tile = M > 4 && (M + 15) / 16 * blocks >= 2048 ? 16 : M > 1 && M * blocks >= 1000 ? 4 : 0;
    return tile && grid_fits(head_workgroups(M, V, tile), 256) ? tile : 0;
}

// Workgroups of matmul_i8_vnni's register tiles (8 rows of x by 8 `columns` weight rows each), along one
// dimension of its grid.
constexpr int64_t dp4_workgroups(int64_t M, int64_t N, int columns) {
    return (M + 7) / 8 * ((N + 8 * columns - 1) / (8 * columns));
}

// Weight rows a lane of matmul_i8_vnni's register tiles takes, or 0: the kernels that give a chain a lane
// and every row of x its own workgroups along the grid's second dimension. Those keep the calls of few
// outputs (us, they / the tiles: 4 x 896 x 4864 6.4 / 11.8, 16 x 896 x 4864 11.3 / 11.9,
// 1 x 8192 x 8192 21.3 / 23.8; 4 x 4864 x 896 6.4 / 6.1, 32 x 896 x 4864 19.0 / 12.1,
// 128 x 896 x 4864 66.5 / 24.7, 128 x 4864 x 896 85.8 / 25.3, 100 x 8192 x 8192 900 / 187), and those
// whose tiles do not fit the grid. 4 from 400 workgroups of them on, else 2 for twice the waves
// (32 x 896 x 4864 12.1 against 17.6 us; 128 x 4864 x 896 26.7 against 25.3; tiles of 4 rows by 4
// measured between the two).
constexpr int dp4_columns(int64_t M, int64_t N) {
    if (M * N < 16000) return 0;
    const int columns = dp4_workgroups(M, N, 4) >= 400 ? 4 : 2;
    return grid_fits(dp4_workgroups(M, N, columns), 256) ? columns : 0;
}

// Workgroups of matmul_i8 on the matrix cores (16 rows of x by 16 `tiles` weight rows each), along one
// dimension of its grid.
constexpr int64_t chain_workgroups(int64_t M, int64_t N, int tiles) {
    return (M + 15) / 16 * ((N + 16 * tiles - 1) / (16 * tiles));
}

// Tiles of weight rows a workgroup of matmul_i8 on the matrix cores takes, or 0: the kernels that give
// every row of x its own workgroups along the grid's second dimension. At the model's widths those run a
// chain a lane and are as quick while the outputs are few: they read a weight row anew for every row of x
// but have 16 times the waves (us, they / the matrix cores: 16 x 896 x 4864 13.0 / 14.6, 24 x 896 x 4864
// 18.5 / 14.6, 4 x 4864 x 896 5.8 / 6.1, 6 x 4864 x 896 6.5 / 6.0, 128 x 4864 x 896 88.5 / 16.4). Other
// widths' general kernel is slower throughout (1 x 8192 x 8192 65 / 27, 100 x 8192 x 8192 6167 / 142,
// 1 x 1000 x 1000 5.8 / 5.7). Two tiles once that leaves four workgroups a CU (128 x 4864 x 896: 16.4 us
// against 18.0 with one; 128 x 896 x 4864, 224 such workgroups: 20.6 against 17.9). Tiles of 32 rows of x
// measured no faster (32 x 32: 20.4, 512 x 4864 x 896 59.9 against 52.4).
constexpr int chain_tiles(int64_t M, int64_t N, int64_t K) {
    if (K < 32 || K % 8 != 0) return 0;
    if (M * N < 20000 && (K == 896 || K == 4864)) return 0;
    const int tiles = chain_workgroups(M, N, 2) >= 1000 ? 2 : 1;
    return grid_fits(chain_workgroups(M, N, tiles), 256) ? tiles : 0;
}

}  // namespace nc
