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

// The part of a packed table of V rows by H that one XCD reads when every row of x reads it anew, in bytes.
// Workgroup i of a launch runs on XCD i mod 8, so 64-row block b of the table goes to XCD (b + m blocks) mod 8
// for row m of x: always to the same one where the blocks are a multiple of 8, to all 8 where they are odd.
constexpr int64_t head_slice(int64_t V, int64_t H) {
    const int64_t blocks = (V + 63) / 64;
    const int64_t parts = blocks % 8 == 0 ? 8 : blocks % 4 == 0 ? 4 : blocks % 2 == 0 ? 2 : 1;
    return blocks * 64 * H * 4 / parts;
}

// Rows of x a wave of the LM head takes, for M rows of H by a table of V rows: 16, 4, or 0 (the one-row
// kernels, whose grid has the rows along its second dimension, so they also take what the others' grid
// does not hold).
//
// 16 once that leaves two waves a SIMD. Measured on MI355X, us, one row / 4 / 16 a wave: 128 x 151936 x 896:
// 10160 / 924 / 579; 16: 1272 / 167 / 124; 4: 322 / 104 / 122; 500 x 4864 x 896: 718 / 113 / 100;
// 128 x 4864 x 896: 141 / 39 / 50; 500 x 896 x 4864: 734 / 130 / 248; 8 x 8192 x 8192: 228 / 195 / 410.
//
// 4 against the one-row kernels: with up to about 4,000 (row, block) pairs its waves are one to a SIMD and it
// takes the time of one wave's k loop whatever their number (H = 64 / 128 / 256 / 512 / 896 / 2048 / 4096:
// 5.2 / 6.2 / 8.7 / 13.7 / 21.3 / 44 / 95 us), where the one-row kernels' time grows with the pairs, each of
// which reads 256 H bytes, and with the memory those come from: an XCD's L2 (4 MB) while its slice of the
// table stays there, slower memory past that. Pairs at which the two are equal: a slice under 1.8 MB
// 2,100-2,700 (2800 x 64 x 896 of 2,304 rows 25.6 / 21.4), 2 MB 1,400-1,800, more than 2.3 MB under 1,000,
// except at the model's width, whose ring kernel is better there (6400 rows: 1,000 pairs 18.8 / 21.3, 1,200
// 23.9 / 21.3) until the slice passes every L2; rows of 128 and less about 2,700; rows of 4,096 about 1,150
// (512 x 4096: 1,000 pairs 78 / 94, 1,400 108 / 94), of 8,192 under 1,000. A table of one block leaves three of
// a workgroup's four waves without work: four times the pairs (4000 x 64 x 896 33.7 / 45.0, 8000 77.4 / 83.8).
constexpr int64_t head_pairs(int64_t V, int64_t H) {
    const int64_t slice = head_slice(V, H);
    int64_t pairs = 2300;
    if (H >= 8192) pairs = 1000;
    else if (slice >= 2300000) pairs = H == 896 && slice < 20000000 ? 1100 : 1000;
    else if (H >= 4096) pairs = 1150;
    else if (H <= 128) pairs = 2700;
    else if (slice >= 1800000 && H != 896) pairs = 1600;
    return V <= 64 && H < 4096 ? 4 * pairs : pairs;
}

constexpr int head_tile(int64_t M, int64_t V, int64_t H) {
    const int64_t blocks = (V + 63) / 64;
    const int tile = M > 4 && (M + 15) / 16 * blocks >= 2048 ? 16
                     : M > 1 && M * blocks >= head_pairs(V, H) ? 4
                                                               : 0;
    return tile && grid_fits(head_workgroups(M, V, tile), 256) ? tile : 0;
}

// Workgroups of matmul_i8_vnni's register tiles (8 rows of x by 8 `columns` weight rows each), along one
// dimension of its grid.
constexpr int64_t dp4_workgroups(int64_t M, int64_t N, int columns) {
    return (M + 7) / 8 * ((N + 8 * columns - 1) / (8 * columns));
}

// Weight rows a lane of matmul_i8_vnni's register tiles takes, or 0: the kernels that give a chain a lane
// and every row of x its own workgroups along the grid's second dimension. Those keep (us, they / the tiles):
// * the calls of few outputs: 4 x 896 x 4864 6.4 / 11.8, 16 x 896 x 4864 11.3 / 11.9; 4 x 4864 x 896 6.4 / 6.1,
//   32 x 896 x 4864 19.0 / 12.1, 128 x 896 x 4864 66.5 / 24.7, 128 x 4864 x 896 85.8 / 25.3,
//   100 x 8192 x 8192 900 / 187;
// * one row (a tile's other seven are copies of it; with the quantizer's launch 1 x 16000 x 896 10.7 / 12.1,
//   1 x 65536 x 2048 30.7 / 42.3, 1 x 151936 x 896 32.4 / 48.9), but for long rows by few weight rows at widths
//   other than the model's, where the general kernel has too few waves (1 x 16000 x 4096 28.7 / 26.9,
//   1 x 16000 x 8192 52.4 / 46.0, 1 x 32768 x 16384 203 / 162; 1 x 24000 x 4096 32.3 / 34.4,
//   1 x 32768 x 8192 72.5 / 78.0);
// * two rows of less than 512 (2 x 65536 x 256 13.9 / 17.3; 2 x 16000 x 512 10.8 / 10.1; three rows
//   3 x 65536 x 256 17.3 / 17.3);
// * what does not fit the tiles' grid.
// 4 from 400 workgroups of them on, else 2 for twice the waves (32 x 896 x 4864 12.1 against 17.6 us;
// 128 x 4864 x 896 26.7 against 25.3; tiles of 4 rows by 4 measured between the two).
constexpr int dp4_columns(int64_t M, int64_t N, int64_t K) {
    if (M * N < 16000) return 0;
    if (M == 1 && (K == 896 || K == 4864 || N > 4 * K || (N >= 32768 && N > 2 * K))) return 0;
    if (M == 2 && K < 512) return 0;
    const int columns = dp4_workgroups(M, N, 4) >= 400 ? 4 : 2;
    return grid_fits(dp4_workgroups(M, N, columns), 256) ? columns : 0;
}

// Workgroups of matmul_i8 on the matrix cores (16 rows of x by 16 `tiles` weight rows each), along one
// dimension of its grid.
constexpr int64_t chain_workgroups(int64_t M, int64_t N, int tiles) {
    return (M + 15) / 16 * ((N + 16 * tiles - 1) / (16 * tiles));
}

// Whether matmul_i8 of M rows by N weight rows is quicker on the matrix cores, whose tiles of 16 rows of x
// read a weight row once, than on the kernels that give every row of x its own workgroups: a chain a lane at
// the model's widths, four chains a lane at any other (us, they / the matrix cores).
// Model's widths: few outputs stay with a chain a lane, which has 16 times the waves (16 x 896 x 4864
// 13.0 / 14.6, 24 x 896 x 4864 18.5 / 14.6, 6 x 4864 x 896 6.5 / 6.0, 128 x 4864 x 896 88.5 / 16.4), and so do
// few rows, of which a tile is mostly copies: one row always (20000 x 896 6.0 / 11.2, 65536 x 4864 79 / 107), two
// (40000 x 896 16.7 / 17.7, 25000 x 4864 44.8 / 46.4, 65536 x 896 26.3 / 25.4), three or four of 896
// (3 x 6667 5.9 / 6.9, 4 x 5000 5.9 / 6.9, 4 x 7500 8.0 / 6.9).
// Other widths, from four rows on: 512 and wider always (4 x 4096 x 512 5.4 / 5.1, 256 x 256 x 512 7.4 / 5.3),
// below that from some outputs on (8 x 2048 x 256 4.6 / 4.8, 8 x 4096 x 256 5.1 / 4.8).
// One to three rows: 3072 and wider always (1 x 8192 x 3072 22.1 / 13.2); 1536 to 3071 but for one row by many
// (1 x 8192 x 1536 9.0 / 8.7, 1 x 24000 x 1536 15.4 / 18.2, 1 x 24000 x 2048 20.3 / 22.5); 512 to 1535 by few
// weight rows (1 x 4096 x 1024 6.8 / 6.2, 2 x 8192 x 1000 7.3 / 7.9, 1 x 16384 x 1024 7.2 / 9.9), or by enough
// of them for the second and third row to pay (3 x 10923 x 768 9.3 / 7.6, 2 x 65536 x 1024 31.3 / 28.3); narrower
// never (1 x 65536 x 64 5.2 / 8.6).
constexpr bool chains_pay(int64_t M, int64_t N, int64_t K) {
    if (K == 896 || K == 4864)
        return M > 1 && M * N >= (M == 2 ? 100000 : M <= 4 && K == 896 ? 28000 : 20000);
    if (M >= 4) return K >= 512 || M * N >= (K >= 384 ? 16000 : 24000);
    if (K >= 3072) return true;
    if (K >= 1536) return M > 1 || N <= (K >= 2048 ? 20000 : 8192);
    if (K < 512) return false;
    return N <= 4096 || (M == 3 && K >= 768) || (M == 2 && K >= 1000 && N >= 40000);
}

// Tiles of weight rows a workgroup of matmul_i8 on the matrix cores takes, or 0: the kernels of a grid row a row
// of x. Two once that leaves four workgroups a CU (128 x 4864 x 896: 16.4 us against 18.0 with one;
// 128 x 896 x 4864, 224 such workgroups: 20.6 against 17.9). Tiles of 32 rows of x measured no faster
// (32 x 32: 20.4, 512 x 4864 x 896 59.9 against 52.4).
constexpr int chain_tiles(int64_t M, int64_t N, int64_t K) {
    if (K < 32 || K % 8 != 0 || !chains_pay(M, N, K)) return 0;
    const int tiles = chain_workgroups(M, N, 2) >= 1000 ? 2 : 1;
    return grid_fits(chain_workgroups(M, N, tiles), 256) ? tiles : 0;
}

// The SwiGLU pair's MFMA tile (nc_gemm.hip): 2 is 32 x 32, 5 is 64 x 64 with two register stages (its tiles
// stage two weight blocks, so deeper rings cost occupancy), 8 is 128 x 64.
// Short k loops: 64 x 64 from 400 such tiles, else 32 x 32 (measured at N = 4864, K = 896: M = 384 / 512 / 1024 /
// 2048: 15.7 / 19.3 / 30.5 / 54.1 us against 16.8 / 20.6 / 35.2 / 68.1 with 32 x 32 and 17.3 / 20.6 / 34.9 / 63.3
// with 32 x 64; M = 128 / 256: 8.41 / 12.13 us with 32 x 32 against 11.0 / 14.6 with 64 x 64).
// Long k loops (K >= 2048; us, 32 x 32 / 64 x 64 / 128 x 64): 128 x 64 past 256 tiles of 64 x 64 while its own
// fit one a CU (190 x 8000 x 4096 34.4 / 28.4 / 25.7, 512 x 3000 x 2048 19.9 / 18.0 / 15.7), or fill whole rounds
// of that without more padding (500 x 8192 x 2048 47.5 / 33.0 / 31.0); a round begun costs it what a full one does
// (257 x 6400 x 2048, 300 of them, 24.3 / 19.2 / 25.4; 1000 x 4864 x 2048, 608, 55.0 / 39.0 / 42.9), and up to 64
// rows half of each is padding (32 x 16500 x 2048 16.5 / 18.4 / 25.5). Else 64 x 64 from 400 tiles, or from 200
// to 256 where it pads little more than 32 x 32 (64 x 13000 x 2048 16.5 / 14.9 / 16.7; 200 x 3300 x 2048
// 11.7 / 12.8 / 14.8).
constexpr int pair_tile(int64_t M, int64_t N, int64_t K) {
    const int64_t n64 = (N + 63) / 64, t64 = (M + 63) / 64 * n64, t128 = (M + 127) / 128 * n64;
    const int64_t t32 = (M + 31) / 32 * ((N + 31) / 32);
    if (K < 2048) return t64 >= 400 ? 5 : 2;
    const int64_t rounds = (t128 + 255) / 256;
    const bool whole = 100 * t128 >= 98 * 256 * rounds && 20 * t128 <= 11 * t64;
    if (t64 > 256 && (t128 <= 256 || whole)) return 8;
    return t64 >= 400 || (t64 >= 200 && t64 <= 256 && 40 * t64 <= 11 * t32) ? 5 : 2;
}

// Query rows a workgroup of a prompt's chunk kernel takes by the library's choice, for M rows and at most `keys`
// keys: 0 is attention_rows_mfma, 4 is attention_rows_chunks<D, 4>. The matrix cores take 64 (row, head) pairs
// of a KV head's group at a time, so they need the group to fit that, and a small group needs many rows to fill
// it: with up to four heads a group and little work the vector ALU's smaller workgroups are quicker, in
// proportion to (blocks of 4 rows) x chunks x heads (us, vector ALU / matrix cores, with the combine: 8 heads of 8,
// 64 rows at past 0 8.8 / 11.1, past 400 (1,024) 10.8 / 11.6, past 1200 (2,560) 21.3 / 13.2; 4 of 4 by 32,
// 128 rows at past 400 (1,152) 10.4 / 10.9, 64 at 1200 (1,280) 11.5 / 11.3; 16 of 8, 64 rows at past 100 (768)
// 10.9 / 12.0, 128 rows (2,048) 12.6 / 12.5; 12 of 4, 128 rows at past 0 (768) 10.6 / 11.6, 256 (3,072)
// 13.5 / 12.4; 8 of 2 by 32, 64 rows at past 400 (1,024) 10.3 / 11.1, 128 (2,304) 12.3 / 11.6). Groups of 6 and
// more are quicker on the matrix cores at every size (14 of 2, 2 rows at past 0 10.3 / 9.2), of 5 as quick
// (10 of 2, 64 rows at past 0 10.9 / 11.1, at past 400 12.3 / 12.0).
constexpr int prefill_rows(int64_t M, int64_t heads, int64_t kv_heads, int64_t keys) {
    const int64_t group = heads / kv_heads;
    if (group > 64) return 4;
    return group <= 4 && (M + 3) / 4 * ((keys + 63) / 64) * heads <= 1200 ? 4 : 0;
}

}  // namespace nc
