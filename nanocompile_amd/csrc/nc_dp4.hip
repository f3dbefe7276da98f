// The reference's matmul_i8_vnni over several rows, in register tiles.
//
// Its order (lower.py:359-397) is 32 chains a dot product: chain 8c + l a running
// fused multiply-add of the Dp4 of bytes 128 k0 + 32 c + 4 l .. + 3 ((w + 128) times x,
// exact in int32) and its block's scale, k0 in order, then a tree. Each step is three
// vector instructions (a dot, a conversion, a fused multiply-add) for four products,
// which bounds it: nothing of a step can be shared between outputs but the operands.
//
// Half a wave runs the 32 chains of TM rows of x by TN weight rows, chain lane & 31: a
// tile of accumulators a lane, so an operand read once serves several outputs. x is
// staged in LDS for a workgroup's four waves as (bytes, 128 times their sum, scale), 16
// bytes a chain: one read brings a row's operands of a step, and the sum goes into the dot
// as its addend. The weights' dwords come from the packed layout, a stage ahead. The tree
// is a reduce-scatter over the 32 lanes: at each level a lane keeps half of its outputs and
// gives its partner the others, 31 additions for 32 outputs.
//
// Measured on MI355X, 128 x 896 x 4864: 24.7 us (a chain a lane, every row reading the weights anew:
// 66 us). The dots alone are 139 M / 64 instructions of about 5.5 cycles (a float add or fused
// multiply-add takes 3 with several waves on a SIMD), the steps' bound about 10 us; the rest is the
// staging and two waves a SIMD.
#include "nc_common.h"
#include "nc_epilogue.h"
#include "nc_rules.h"

namespace {

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));

struct Dp4Args {
    float *y;
    const int8_t *xq;
    const float *xs, *offset;
    const int8_t *packed, *q;
    const float *scales, *bias, *residual, *gate;
    int M, N, K, shift;                               // a block is 1 << shift values
};

// dot4 whose addend stays where it is: the saturating form (never reached: |sum| < 2^18) has a
// destination of its own, where hipcc's other choice adds into the addend's copy, a move a step.
__device__ __forceinline__ int32_t dot4_of(int32_t w, int32_t x, int32_t sum) {
    return __builtin_amdgcn_sdot4(w, x, sum, true);
}

// A conversion costs two float subtractions, so the dots carry 1.5 * 2^23's bits
// in their addend: the sum's bits are then those of the float 1.5 * 2^23 + dot, from which
// subtracting it leaves (float)dot exactly (|dot| < 2^18).
constexpr int32_t kMagicBits = 0x4B400000;
constexpr float kMagicFloat = 12582912.0f;

// 128 times the sum of four int8 values, the offset of their Dp4, on top of those bits.
__device__ __forceinline__ int32_t dp4_addend(int32_t x) { return kMagicBits + nc::dot4(x, 0x01010101, 0) * 128; }

// One level of the reduce-scatter: partners differ in lane bit OFF; v[0 .. 2 HALF - 1] becomes
// v[0 .. HALF - 1], the lower half of the outputs where the bit is clear, the upper where set.
// With one output left (HALF 0) both partners take its sum.
template <int OFF, int HALF, int OUT>
__device__ __forceinline__ void scatter_level(float (&v)[OUT], int lane) {
    if constexpr (HALF == 0) {
        v[0] = __fadd_rn(v[0], nc::xor_partner<OFF>(v[0]));
        return;
    }
#pragma unroll
    for (int i = 0; i < HALF; ++i) {
        if constexpr (OFF == 16) {
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[i]), __float_as_uint(v[HALF + i]), false,
                                                            false);
            v[i] = __fadd_rn(__uint_as_float(r[0]), __uint_as_float(r[1]));
        } else {
            const bool upper = lane & OFF;
            const float mine = upper ? v[HALF + i] : v[i], theirs = upper ? v[i] : v[HALF + i];
            v[i] = __fadd_rn(mine, nc::xor_partner<OFF>(theirs));
        }
    }
}

template <int TM, int TN>
__global__ __launch_bounds__(256) void matmul_i8_dp4(Dp4Args a) {
    constexpr int OUT = TM * TN, COLS = 8 * TN;       // outputs of a lane; weight rows of the workgroup
    constexpr int KC = 4;                             // steps a stage
    constexpr int ENTRIES = TM * KC * 32, PER = ENTRIES / 256;
    __shared__ __align__(16) i32x4 sx[2][ENTRIES];
    const int M = a.M, N = a.N, K = a.K, nb = K >> a.shift;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, chain = lane & 31, c = chain >> 3, l = chain & 7;
    // workgroup i runs on XCD i mod 8: each XCD takes a contiguous range of tiles, m fastest, so
    // the workgroups of one band of weight rows share an L2
    const int mtiles = (M + TM - 1) / TM, total = gridDim.x, full = total & ~7, id = blockIdx.x;
    const int t = id < full ? (id & 7) * (total >> 3) + (id >> 3) : id;
    const int m0 = (t % mtiles) * TM, n0 = (t / mtiles) * COLS + (wave * 2 + (lane >> 5)) * TN;
    const int strides = K / 128;

    const int8_t *wrow[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) wrow[j] = a.packed + (size_t)min(n0 + j, N - 1) * strides * 128 + 16 * l + 4 * c;
    // this thread's entries of a stage: row, step and chain fixed
    const int8_t *xrow[PER];
    const float *srow[PER];
    int at0[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int u = threadIdx.x + 256 * i, row = min(m0 + u / (KC * 32), M - 1);
        at0[i] = 4 * (u % (KC * 32));                 // byte of the stage
        xrow[i] = a.xq + (size_t)row * K;
        srow[i] = a.xs + (size_t)row * nb;
    }
    int32_t xv[PER], wv[2][KC][TN];
    float sv[PER];
    const int last = strides * 128 - 4;
    auto fetch = [&](int s) {                         // clamped: what lies past the last whole step is not used
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int at = min(s * KC * 128 + at0[i], last);
            xv[i] = *reinterpret_cast<const int32_t *>(xrow[i] + at);
            sv[i] = srow[i][at >> a.shift];
        }
    };
    auto fetch_w = [&](int s, int32_t (&w)[KC][TN]) {
#pragma unroll
        for (int k = 0; k < KC; ++k)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                w[k][j] = *reinterpret_cast<const int32_t *>(wrow[j] + (size_t)min(s * KC + k, strides - 1) * 128);
    };
    auto keep = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            sx[buf][threadIdx.x + 256 * i] = i32x4{xv[i], dp4_addend(xv[i]), __float_as_int(sv[i]), 0};
        }
    };
    float acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = 0.0f;
    // Eight dots, then their subtractions, then their steps: left to itself hipcc follows each dot with
    // its use, which has to wait three instructions' time for it.
    auto step = [&](const i32x4 (&x)[TM], const int32_t (&w)[TN]) {
        constexpr int PART = 8;
#pragma unroll
        for (int h = 0; h < OUT; h += PART) {
            float f[PART];
#pragma unroll
            for (int u = 0; u < PART; ++u)
                f[u] = __int_as_float(dot4_of(w[(h + u) % TN], x[(h + u) / TN][0], x[(h + u) / TN][1]));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < PART; ++u) f[u] = __fsub_rn(f[u], kMagicFloat);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < PART; ++u) {
                float &o = acc[(h + u) / TN][(h + u) % TN];
                o = __builtin_fmaf(f[u], __int_as_float(x[(h + u) / TN][2]), o);
            }
        }
    };
    auto stage = [&](int buf, const int32_t (&w)[KC][TN], int k) {
        i32x4 x[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) x[i] = sx[buf][(i * KC + k) * 32 + chain];
        step(x, w[k]);
    };
    if (strides > 0) {
        const int stages = (strides + KC - 1) / KC;
        fetch(0);
        fetch_w(0, wv[0]);
        keep(0);
        __syncthreads();
        for (int s = 0; s < stages; s += 2) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                if (s + b < stages) {                 // (uniform)
                    fetch(s + b + 1);
                    fetch_w(s + b + 1, wv[b ^ 1]);
#pragma unroll
                    for (int k = 0; k < KC; ++k)
                        if ((s + b) * KC + k < strides) stage(b, wv[b], k);
                    keep(b ^ 1);
                    __syncthreads();
                }
            }
        }
    }
    // The groups of 32 past the last whole 128: steps of the chains of c = 0, from the row-major weights.
    const int groups = K % 128 / 32;
    if (c == 0) {
        for (int k1 = 0; k1 < groups; ++k1) {
            const int at = strides * 128 + 32 * k1 + 4 * l;
            i32x4 x[TM];
            int32_t w[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const size_t row = min(m0 + i, M - 1);
                const int32_t v = *reinterpret_cast<const int32_t *>(a.xq + row * K + at);
                x[i] = i32x4{v, dp4_addend(v), __float_as_int(a.xs[row * nb + (at >> a.shift)]), 0};
            }
#pragma unroll
            for (int j = 0; j < TN; ++j)
                w[j] = *reinterpret_cast<const int32_t *>(a.q + (size_t)min(n0 + j, N - 1) * K + at);
            step(x, w);
        }
    }

    float v[OUT];
#pragma unroll
    for (int i = 0; i < OUT; ++i) v[i] = acc[i / TN][i % TN];
    scatter_level<8, OUT / 2>(v, lane);               // (acc[l] + acc[8 + l]), (acc[16 + l] + acc[24 + l])
    scatter_level<16, OUT / 4>(v, lane);              // their sum h[l]
    scatter_level<4, OUT / 8>(v, lane);               // u[j] = h[j] + h[j + 4]
    scatter_level<1, OUT / 16>(v, lane);              // u0 + u1, u2 + u3
    scatter_level<2, OUT / 32>(v, lane);
    const int o = (lane & 8 ? OUT / 2 : 0) + (lane & 16 ? OUT / 4 : 0) + (lane & 4 ? OUT / 8 : 0) +
                  (lane & 1 ? OUT / 16 : 0) + (lane & 2 ? OUT / 32 : 0);
    const int m = m0 + o / TN, n = n0 + o % TN;
    if (m >= M || n >= N || (OUT < 32 && (lane & 2))) return;
    const size_t at = (size_t)m * N + n;
    float out = __fmul_rn(__fsub_rn(v[0], a.offset[m]), a.scales[n]);
    if (a.bias) out = __fadd_rn(out, a.bias[n]);
    if (a.residual) out = __fadd_rn(a.residual[at], out);
    a.y[at] = a.gate ? nc::silu_mul(a.gate[at], out) : out;
}

template <int TM, int TN>
int32_t launch_dp4(const Dp4Args &a) {
    static_assert(TM == 8, "dp4_workgroups counts tiles of 8 rows");
    const unsigned workgroups = (unsigned)nc::dp4_workgroups(a.M, a.N, TN);      // (dp4_columns: they fit)
    hipLaunchKernelGGL((matmul_i8_dp4<TM, TN>), dim3(workgroups), dim3(256), 0, nc::stream(), a);
    return nc::launched("matmul_i8_dp4");
}

}  // namespace

namespace nc {

bool matmul_i8_vnni_rows_ok(const int8_t *xq, const int8_t *packed, const int8_t *q, int64_t M, int64_t N, int64_t K) {
    return dp4_columns(M, N, K) && (((uintptr_t)xq | (uintptr_t)packed | (uintptr_t)q) & 3) == 0;
}

int32_t matmul_i8_vnni_rows(float *y, const int8_t *xq, const float *xs, const float *offset, const int8_t *packed,
                            const int8_t *q, const float *scales, const float *bias, const float *residual,
                            const float *gate, int64_t M, int64_t N, int64_t K, int64_t block) {
    const Dp4Args a{y,    xq,       xs,   offset, packed, q, scales,
                    bias, residual, gate, (int)M, (int)N, (int)K, __builtin_ctzll((unsigned long long)block)};
    return dp4_columns(M, N, K) == 4 ? launch_dp4<8, 4>(a) : launch_dp4<8, 2>(a);
}

}  // namespace nc
