// The reference's matmul_i8 over several rows, on the float32 matrix cores.
//
// Its order (lower.py:294-356) is 32 chains a dot product, chain 8c + l a
// running fused multiply-add over elements 32 k0 + 8c + l, k0 in order, then a
// tree. CDNA's float32 matrix instructions are exactly that chain: measured on
// gfx950 over normal, wide-ranged, subnormal and special operands, every
// element of v_mfma_f32_16x16x4_f32 is fmaf(a[k], b[k], acc) for k = 0 .. 3 in
// order, each rounded once, subnormals kept. So an instruction whose k is four
// consecutive blocks of 32 runs four steps of one chain for 16 weight rows and
// 16 rows of x, and gives the bits of the kernels that run a chain a lane.
//
// A workgroup is four waves over MT x NT tiles of 16 rows of x by 16 weight
// rows; wave w runs the chains of l = 2w and 2w + 1, every c, so a tile's 32
// accumulators are spread over four waves' registers, each wave converts only
// its own quarter of the weight bytes, and h[l] = (acc[l] + acc[8 + l]) +
// (acc[16 + l] + acc[24 + l]) is taken in registers. Then the waves trade h
// through LDS, each taking a quarter of the outputs through the rest of the
// tree: u[j] = h[j] + h[j + 4], (u0 + u1) + (u2 + u3).
//
// Both operands go through LDS, a stage of 128 k at a time, NS stages ahead in
// registers: x with each wave's eight values of a block side by side (two
// 16-byte reads a tile), the weights in the packed layout, whose dword
// [l][k0] holds the four chains of l (a stage is one of its 128-byte pieces).
//
// Measured on MI355X, 512 x 4864 x 896: 52 us, 42 T multiply-adds/s of the 77 that a
// loop of these instructions alone reaches (a chain a lane: 410 us). What it waits on
// is its short life: 7 stages at this width, then the trade. Before this layout the
// waves split the chains by c and read row-major weights from memory: 66 us, the L1
// busy 76% of the time with 8-byte reads and four times the values traded through LDS.
#include "nc_common.h"
#include "nc_epilogue.h"
#include "nc_rules.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct ChainArgs {
    float *y;
    const float *x;
    const int8_t *packed, *q;
    const float *scales, *bias, *residual, *gate;
    int M, N, K;
};

__device__ __forceinline__ float byte_float(uint32_t w, int i) { return (float)(int8_t)((w >> (8 * i)) & 0xff); }

template <int MT, int NT, int NS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void matmul_i8_chains(ChainArgs a) {
    constexpr int KS = 128;                           // k a stage: 4 blocks of 32
    constexpr int XS = KS + 4, WS = 36;               // row strides in LDS (floats, dwords): 16 rows on distinct banks
    constexpr int ROWS = 16 * MT, COLS = 16 * NT;
    constexpr int PER = ROWS * KS / 4 / 256;          // 16-byte pieces of x a thread a stage
    constexpr int U = MT * NT;                        // outputs a lane ends with (4 a tile, over 4 waves)
    constexpr int STAGE = ROWS * XS + COLS * WS;
    static_assert(2 * STAGE >= 8 * 4 * 64 * U, "the traded values must fit the staging buffers");
    __shared__ __align__(16) float lds[2 * STAGE];
    const int M = a.M, N = a.N, K = a.K;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    // workgroup i runs on XCD i mod 8: each XCD takes a contiguous range of tiles, m fastest, so
    // the workgroups of one band of weight rows share an L2
    const int mtiles = (M + ROWS - 1) / ROWS, total = gridDim.x, full = total & ~7, id = blockIdx.x;
    const int t = id < full ? (id & 7) * (total >> 3) + (id >> 3) : id;
    const int m0 = (t % mtiles) * ROWS, n0 = (t / mtiles) * COLS;
    const int blocks = K / 32, stages = (blocks + 3) / 4, whole = blocks / 4;
    const int wrow = stages * 128;                    // bytes of a packed row

    // Loads as buffer loads: the stage is a scalar offset, so it costs no vector address arithmetic.
    // Rows past M or N read the last row (not stored).
    const auto xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.x) + (size_t)m0 * K, 0,
                                                        min(ROWS, M - m0) * K * 4, 0x00020000);
    const auto wbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t *>(a.packed) + (size_t)n0 * wrow, 0,
                                                        min(COLS, N - n0) * wrow, 0x00020000);
    int xsrc[PER], xdst[PER], xpiece[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int u = threadIdx.x + 256 * i, row = u / (KS / 4), piece = u % (KS / 4);
        xsrc[i] = (min(row, M - 1 - m0) * K + 4 * piece) * 4;
        // element e = 4 piece of the row: block e / 32, c = e % 32 / 8, l = 0 or 4: pairs (l, l + 1)
        // and (l + 2, l + 3) belong to waves l / 2 and l / 2 + 1, at 8 wave + 2c of the block
        xdst[i] = row * XS + 32 * (piece / 8) + 16 * (piece & 1) + 2 * (piece / 2 & 3);
        xpiece[i] = piece;
    }
    static_assert(NT <= 2, "a packed piece a thread");
    const bool loads_w = NT > 1 || threadIdx.x < COLS * 8;
    const int wcol = (threadIdx.x / 8) & (COLS - 1), wpiece = threadIdx.x & 7;
    const int wsrc = min(wcol, N - 1 - n0) * wrow + 16 * wpiece, wdst = ROWS * XS + wcol * WS + 4 * wpiece;

    f32x4 rx[NS][PER];
    u32x4 rw[NS];
    auto load = [&](int s, f32x4 (&xs)[PER], u32x4 &ws) {
#pragma unroll
        for (int i = 0; i < PER; ++i)
            xs[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xbuf, xsrc[i], s * KS * 4, 0));
        ws = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wbuf, wsrc, s * KS, 0));
    };
    auto keep = [&](int buf, const f32x4 (&xs)[PER], const u32x4 &ws) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            float *d = &lds[buf * STAGE + xdst[i]];
            *reinterpret_cast<f32x2 *>(d) = f32x2{xs[i][0], xs[i][1]};
            *reinterpret_cast<f32x2 *>(d + 8) = f32x2{xs[i][2], xs[i][3]};
        }
        if (loads_w) *reinterpret_cast<u32x4 *>(&lds[buf * STAGE + wdst]) = ws;
    };
    f32x4 acc[2][4][MT][NT];                          // [l & 1][c]
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[l][c][i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // step c of the wave's two l: xa[i][c / 2][2 (c & 1) + l], byte c of wd[j][l]
    auto multiply = [&](const f32x4 (&xa)[MT][2], const uint32_t (&wd)[NT][2], int c) {
#pragma unroll
        for (int l = 0; l < 2; ++l) {
            float w[NT];
#pragma unroll
            for (int j = 0; j < NT; ++j) w[j] = byte_float(wd[j][l], c);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    acc[l][c][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], xa[i][c >> 1][2 * (c & 1) + l],
                                                                           acc[l][c][i][j], 0, 0, 0);
        }
    };
    const int xread = r16 * XS + 32 * kq + 8 * wave, wread = ROWS * XS + r16 * WS + 8 * wave + kq;
    auto step = [&](int buf) {
        f32x4 xa[MT][2];
        uint32_t wd[NT][2];
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int l = 0; l < 2; ++l) wd[j][l] = __float_as_uint(lds[buf * STAGE + wread + 16 * j * WS + 4 * l]);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                xa[i][h] = *reinterpret_cast<const f32x4 *>(&lds[buf * STAGE + xread + 16 * i * XS + 4 * h]);
#pragma unroll
        for (int c = 0; c < 4; ++c) multiply(xa, wd, c);
    };

    if (whole > 0) {
#pragma unroll
        for (int j = 0; j < NS; ++j) load(min(j, whole - 1), rx[j], rw[j]);
        keep(0, rx[0], rw[0]);
        __syncthreads();
        int s = 0;
        for (; s + NS <= whole; s += NS) {
#pragma unroll
            for (int j = 0; j < NS; ++j) {
                load(min(s + j + NS, whole - 1), rx[j], rw[j]);
                step(j & 1);
                keep((j + 1) & 1, rx[(j + 1) % NS], rw[(j + 1) % NS]);
                __syncthreads();
            }
        }
#pragma unroll
        for (int j = 0; j < NS - 1; ++j) {
            if (s + j < whole) {
                step(j & 1);
                keep((j + 1) & 1, rx[(j + 1) % NS], rw[(j + 1) % NS]);
                __syncthreads();
            }
        }
    }
    // The blocks past the last whole stage: a stage more, its missing blocks of x as zeros (a step of
    // w * 0 = +-0 leaves a chain, which is never -0, as it is); loads past the row's blocks read its last.
    if (blocks % 4) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int k4 = whole * (KS / 4) + xpiece[i], row = (threadIdx.x + 256 * i) / (KS / 4);
            const f32x4 v = *reinterpret_cast<const f32x4 *>(a.x + (size_t)min(m0 + row, M - 1) * K +
                                                             4 * min(k4, 8 * blocks - 1));
            rx[0][i] = k4 < 8 * blocks ? v : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        rw[0] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wbuf, wsrc, whole * KS, 0));
        keep(0, rx[0], rw[0]);
        __syncthreads();
        step(0);
        __syncthreads();
    }
    // The groups of 8 past the last whole block: element 8 k1 + l of them is a step of chain l (c = 0).
    const int groups = K % 32 / 8;
    if (groups) {
        const int at = 32 * blocks + 8 * min(kq, groups - 1) + 2 * wave;
        f32x4 xa[MT][2];
        uint32_t wd[NT][2];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const float *v = a.x + (size_t)min(m0 + 16 * i + r16, M - 1) * K + at;
            xa[i][0] = f32x4{kq < groups ? v[0] : 0.0f, kq < groups ? v[1] : 0.0f, 0.0f, 0.0f};
            xa[i][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int8_t *v = a.q + (size_t)min(n0 + 16 * j + r16, N - 1) * K + at;
            wd[j][0] = (uint8_t)v[0];
            wd[j][1] = (uint8_t)v[1];
        }
        multiply(xa, wd, 0);
    }

    // The trade: value v = 4 tile + register of each lane; wave w takes values w U .. w U + U - 1.
#pragma unroll
    for (int l = 0; l < 2; ++l)
#pragma unroll
        for (int v = 0; v < 4 * U; ++v) {
            const int i = v / 4 / NT, j = v / 4 % NT, r = v & 3;
            lds[(((2 * wave + l) * 4 + v / U) * 64 + lane) * U + v % U] =
                __fadd_rn(__fadd_rn(acc[l][0][i][j][r], acc[l][1][i][j][r]),
                          __fadd_rn(acc[l][2][i][j][r], acc[l][3][i][j][r]));
        }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
        float h[8];
#pragma unroll
        for (int l = 0; l < 8; ++l) h[l] = lds[((l * 4 + wave) * 64 + lane) * U + u];
        const float u0 = __fadd_rn(h[0], h[4]), u1 = __fadd_rn(h[1], h[5]);
        const float u2 = __fadd_rn(h[2], h[6]), u3 = __fadd_rn(h[3], h[7]);
        const float sum = __fadd_rn(__fadd_rn(u0, u1), __fadd_rn(u2, u3));
        const int v = wave * U + u, tile = v >> 2;
        const int m = m0 + 16 * (tile / NT) + r16, n = n0 + 16 * (tile % NT) + 4 * kq + (v & 3);
        if (m < M && n < N) {
            const size_t o = (size_t)m * N + n;
            float out = __fmul_rn(sum, a.scales[n]);
            if (a.bias) out = __fadd_rn(out, a.bias[n]);
            if (a.residual) out = __fadd_rn(a.residual[o], out);
            a.y[o] = a.gate ? nc::silu_mul(a.gate[o], out) : out;
        }
    }
}

template <int MT, int NT, int NS>
int32_t launch_chains(const ChainArgs &a) {
    static_assert(MT == 1, "chain_workgroups counts tiles of 16 rows");
    const unsigned workgroups = (unsigned)nc::chain_workgroups(a.M, a.N, NT);    // (chain_tiles: they fit)
    hipLaunchKernelGGL((matmul_i8_chains<MT, NT, NS>), dim3(workgroups), dim3(256), 0, nc::stream(), a);
    return nc::launched("matmul_i8_chains");
}

}  // namespace

namespace nc {

bool matmul_i8_rows_ok(const float *x, const int8_t *packed, int64_t M, int64_t N, int64_t K) {
    return chain_tiles(M, N, K) && (((uintptr_t)x | (uintptr_t)packed) & 15) == 0;
}

int32_t matmul_i8_rows(float *y, const float *x, const int8_t *packed, const int8_t *q, const float *scales,
                       const float *bias, const float *residual, const float *gate, int64_t M, int64_t N, int64_t K) {
    const ChainArgs a{y, x, packed, q, scales, bias, residual, gate, (int)M, (int)N, (int)K};
    return chain_tiles(M, N, K) == 2 ? launch_chains<1, 2, 2>(a) : launch_chains<1, 1, 4>(a);
}

}  // namespace nc
