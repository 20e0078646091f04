// FrTensor kernels for gfx950: elementwise, conversions, layout, sums, multilinear folds and
// the inner-product sumcheck rounds.  Tensors hold standard-form residues, 32 B per element
// (8 little-endian u32 limbs), exactly the reference's Fr_t layout (fr-tensor.cu:181-184).
//
// Differences from the reference's kernels that do not change any output byte:
//  * broadcast operands and challenges are converted to Montgomery form once on the host, so a
//    product with them costs one Montgomery multiplication instead of two;
//  * sums of products are accumulated with the R^-1 factor still attached and corrected once;
//  * folds run several levels per pass (registers) and finish in one workgroup (LDS).
#include <algorithm>
#include <cstring>
#include <mutex>
#include "field.hpp"
#include "fr29.hpp"
#include "rt.hpp"
#include "../../include/zkllm_hip.h"

using namespace zk;

static constexpr int TPB = 256;

// ------------------------------------------------------------------------------------------------
// elementwise (fr-tensor.cu:71-153)
// ------------------------------------------------------------------------------------------------
enum { EW_ADD = 0, EW_SUB = 1, EW_MUL = 2, EW_MONTMUL = 3 };

template <int OP> __global__ void __launch_bounds__(TPB) k_ew(Fr* __restrict__ out, const Fr* __restrict__ a, const Fr* __restrict__ b, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    const Fr x = a[i], y = b[i];
    Fr r;
    if (OP == EW_ADD) r = add(x, y);
    else if (OP == EW_SUB) r = sub(x, y);
    else if (OP == EW_MUL) r = fr_mul_barrett(x, y);
    else r = mont_mul(x, y);
    out[i] = r;
}
// s: for EW_MUL the scalar is already in Montgomery form (s*R), so one mont_mul yields a*s.
template <int OP> __global__ void __launch_bounds__(TPB) k_ew_s(Fr* __restrict__ out, const Fr* __restrict__ a, const Fr s, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    const Fr x = a[i];
    Fr r;
    if (OP == EW_ADD) r = add(x, s);
    else if (OP == EW_SUB) r = sub(x, s);
    else r = mont_mul(x, s);
    out[i] = r;
}
// a + s b (s in Montgomery form) in one pass: 2^20 elements 72 us as a product and a sum that read it back
__global__ void __launch_bounds__(TPB) k_add_mul_s(Fr* __restrict__ out, const Fr* __restrict__ a, const Fr* __restrict__ b, const Fr s, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) out[i] = add(a[i], mont_mul(b[i], s));
}
__global__ void __launch_bounds__(TPB) k_neg(Fr* __restrict__ out, const Fr* __restrict__ a, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) out[i] = neg(a[i]);
}
__global__ void __launch_bounds__(TPB) k_fill(Fr* __restrict__ out, const Fr s, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) out[i] = s;
}
// Z[i] += bias[i % cols] (zkfc.cu:36-41)
__global__ void __launch_bounds__(TPB) k_bias(Fr* __restrict__ z, const Fr* __restrict__ bias, size_t n, uint32_t cols) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) z[i] = add(z[i], bias[i % cols]);
}

// ------------------------------------------------------------------------------------------------
// conversions (fr-tensor.cu:186-208, 691-775, 922-945)
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(TPB) k_from_i32(Fr* __restrict__ out, const int32_t* __restrict__ in, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) out[i] = fr_from_i64((int64_t)in[i]);
}
__global__ void __launch_bounds__(TPB) k_from_i64(Fr* __restrict__ out, const int64_t* __restrict__ in, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) out[i] = fr_from_i64(in[i]);
}
__global__ void __launch_bounds__(TPB) k_from_u32(Fr* __restrict__ out, const uint32_t* __restrict__ in, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) out[i] = fr_from_u64((uint64_t)in[i]);
}
// round half away from zero after scaling (float_to_scalar / double_to_scalar)
__global__ void __launch_bounds__(TPB) k_from_f32(Fr* __restrict__ out, const float* __restrict__ in, uint64_t sf, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    float x = in[i] * (float)sf;
    const int64_t v = (x >= 0) ? (int64_t)((double)x + 0.5) : (int64_t)((double)x - 0.5);
    out[i] = fr_from_i64(v);
}
__global__ void __launch_bounds__(TPB) k_from_f64(Fr* __restrict__ out, const double* __restrict__ in, uint64_t sf, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    double x = in[i] * (double)sf;
    const int64_t v = (x >= 0) ? (int64_t)(x + 0.5) : (int64_t)(x - 0.5);
    out[i] = fr_from_i64(v);
}
__global__ void __launch_bounds__(TPB) k_to_i32(int32_t* __restrict__ out, const Fr* __restrict__ in, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) out[i] = fr_to_i32(in[i]);
}
__global__ void __launch_bounds__(TPB) k_to_i64(int64_t* __restrict__ out, const Fr* __restrict__ in, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) out[i] = fr_to_i64(in[i]);
}

// ------------------------------------------------------------------------------------------------
// layout (fr-tensor.cu:800-828 pad, :885-900 transpose; tlookup.cu:446-453 gather)
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(TPB) k_pad(Fr* __restrict__ out, const Fr* __restrict__ in, size_t n_out, uint32_t last_in, uint32_t last_out, const Fr pad) {
    const size_t g = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (g >= n_out) return;
    const size_t g0 = g / last_out;
    const uint32_t g1 = (uint32_t)(g % last_out);
    out[g] = (g1 >= last_in) ? pad : in[g0 * last_in + g1];
}
// 32x32 tile through LDS so both the read and the write are contiguous along the fast axis
// blockIdx.z selects one of a stack of M x N matrices
__global__ void __launch_bounds__(TPB) k_transpose(Fr* __restrict__ out, const Fr* __restrict__ in, uint32_t M, uint32_t N) {
    __shared__ uint32_t tile[8][32][33];
    in += (size_t)blockIdx.z * M * N;
    out += (size_t)blockIdx.z * M * N;
    const uint32_t bx = blockIdx.x * 32, by = blockIdx.y * 32;
    const uint32_t tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
    for (uint32_t r = ty; r < 32; r += 8) {
        const uint32_t row = by + r, col = bx + tx;
        if (row < M && col < N) {
            const Fr v = in[(size_t)row * N + col];
#pragma unroll
            for (int l = 0; l < 8; ++l) tile[l][r][tx] = v.v[l];
        }
    }
    __syncthreads();
    for (uint32_t r = ty; r < 32; r += 8) {
        const uint32_t col = bx + r, row = by + tx;     // output row = input col
        if (row < M && col < N) {
            Fr v;
#pragma unroll
            for (int l = 0; l < 8; ++l) v.v[l] = tile[l][tx][r];
            out[(size_t)col * M + row] = v;
        }
    }
}
__global__ void __launch_bounds__(TPB) k_gather(Fr* __restrict__ out, const Fr* __restrict__ table, const uint32_t* __restrict__ idx, size_t n) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) out[i] = table[idx[i]];
}

// ------------------------------------------------------------------------------------------------
// block reduction of K running sums per thread; partials[k * gridDim.x + blockIdx.x]
// ------------------------------------------------------------------------------------------------
template <int K> __device__ __forceinline__ void block_reduce_store(Fr (&acc)[K], Fr* __restrict__ partials) {
    __shared__ uint32_t red[8][TPB];
    const uint32_t t = threadIdx.x;
#pragma unroll
    for (int k = 0; k < K; ++k) {
#pragma unroll
        for (int l = 0; l < 8; ++l) red[l][t] = acc[k].v[l];
        __syncthreads();
        for (uint32_t s = TPB / 2; s > 0; s >>= 1) {
            if (t < s) {
                Fr x, y;
#pragma unroll
                for (int l = 0; l < 8; ++l) { x.v[l] = red[l][t]; y.v[l] = red[l][t + s]; }
                x = add(x, y);
#pragma unroll
                for (int l = 0; l < 8; ++l) red[l][t] = x.v[l];
            }
            __syncthreads();
        }
        if (t == 0) {
            Fr x;
#pragma unroll
            for (int l = 0; l < 8; ++l) x.v[l] = red[l][0];
            partials[(size_t)k * gridDim.x + blockIdx.x] = x;
        }
        __syncthreads();
    }
}
// one block per k: out[k] = sum of partials[k*nb .. k*nb+nb)
__global__ void __launch_bounds__(TPB) k_finish_sums(Fr* __restrict__ out, const Fr* __restrict__ partials, uint32_t nb) {
    Fr acc[1] = {big_zero<8>()};
    const Fr* p = partials + (size_t)blockIdx.x * nb;
    for (uint32_t i = threadIdx.x; i < nb; i += TPB) acc[0] = add(acc[0], p[i]);
    block_reduce_store<1>(acc, out);   // gridDim.x == K, so out[0*K + blockIdx.x] = out[k]
}

__global__ void __launch_bounds__(TPB) k_sum(Fr* __restrict__ partials, const Fr* __restrict__ a, size_t n) {
    Fr acc[1] = {big_zero<8>()};
    for (size_t i = (size_t)blockIdx.x * TPB + threadIdx.x; i < n; i += (size_t)gridDim.x * TPB) acc[0] = add(acc[0], a[i]);
    block_reduce_store<1>(acc, partials);
}
// sum_i a_i*b_i*R^-1 (the caller applies the R^2 correction once)
__global__ void __launch_bounds__(TPB) k_dot(Fr* __restrict__ partials, const Fr* __restrict__ a, const Fr* __restrict__ b, size_t n) {
    Fr acc[1] = {big_zero<8>()};
    for (size_t i = (size_t)blockIdx.x * TPB + threadIdx.x; i < n; i += (size_t)gridDim.x * TPB) acc[0] = add(acc[0], mont_mul(a[i], b[i]));
    block_reduce_store<1>(acc, partials);
}

static inline unsigned reduce_grid(size_t n) {
    size_t b = (n + TPB - 1) / TPB;
    if (b > 2048) b = 2048;
    if (b < 1) b = 1;
    return (unsigned)b;
}
// finish K sums living in `partials` (K x nb) and bring them to the host (standard layout)
template <int K> static int finish_to_host(Fr* partials, unsigned nb, Fr* host_out, hipStream_t st) {
    void* stage = nullptr;
    int rc = staging(&stage, sizeof(Fr) * K);
    if (rc) return rc;
    hipLaunchKernelGGL(k_finish_sums, dim3(K), dim3(TPB), 0, st, (Fr*)stage, partials, nb);
    ZK_LAUNCH_CHECK();
    ZK_HIP(hipStreamSynchronize(st));
    memcpy(host_out, stage, sizeof(Fr) * K);
    return 0;
}

// ------------------------------------------------------------------------------------------------
// multilinear folds
// ------------------------------------------------------------------------------------------------
template <int L> struct FrPack { Fr x[L]; };

// Folds L levels of the middle axis of in[other][cur][window] (adjacent pairs along `cur`, index
// bit 0 first; positions past `cur` read as zero, which is the reference's odd-tail rule
// a - x*a).  xs are in Montgomery form.  (fr-tensor.cu:518-560, 588-626)
template <int L> __global__ void __launch_bounds__(TPB)
k_fold_axis(Fr* __restrict__ out, const Fr* __restrict__ in, const FrPack<L> xs, size_t n_out, uint32_t cur, uint32_t cur_out, size_t window) {
    const size_t g = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (g >= n_out) return;
    const size_t i2 = g % window;
    const size_t t = g / window;
    const uint32_t i1 = (uint32_t)(t % cur_out);
    const size_t i0 = t / cur_out;
    const Fr* base = in + (i0 * cur) * window + i2;
    const uint32_t first = i1 << L;
    Fr v[1 << L];
#pragma unroll
    for (int j = 0; j < (1 << L); ++j) v[j] = (first + j < cur) ? base[(size_t)(first + j) * window] : big_zero<8>();
#pragma unroll
    for (int l = 0; l < L; ++l) {
#pragma unroll
        for (int j = 0; j < (1 << (L - 1 - l)); ++j) v[j] = add(v[2 * j], mont_mul(xs.x[l], sub(v[2 * j + 1], v[2 * j])));
    }
    out[g] = v[0];
}
// The same L levels as one weighted sum: out = sum_j w_j in_j with w_j = prod_l (x_l if bit l of j else 1 - x_l), the
// products of every four terms sharing one Montgomery reduction (8 x 64 + 2 x 72 multiply-adds for three levels instead of
// 7 x 136).  The field value, hence the canonical result, is that of the level-by-level fold.  ws in Montgomery form.
template <int L> __global__ void __launch_bounds__(TPB)
k_fold_axis_dot(Fr* __restrict__ out, const Fr* __restrict__ in, const FrPack<(1 << L)> ws, size_t n_out, uint32_t cur, uint32_t cur_out, size_t window) {
    static_assert(L >= 2, "groups of four terms");
    const size_t g = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (g >= n_out) return;
    const size_t i2 = g % window;
    const size_t t = g / window;
    const uint32_t i1 = (uint32_t)(t % cur_out);
    const size_t i0 = t / cur_out;
    const Fr* base = in + (i0 * cur) * window + i2;
    const uint32_t first = i1 << L;
    Fr acc;
#pragma unroll
    for (int q = 0; q < (1 << L); q += 4) {
        Fr v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (first + q + j < cur) ? base[(size_t)(first + q + j) * window] : big_zero<8>();
        const Fr part = mont_dot<8, 4>(v, ws.x + q);
        acc = q ? add(acc, part) : part;
    }
    out[g] = acc;
}

// ---- a whole axis in one pass ----------------------------------------------------------------------------------------------------
// Every level of a long axis at once: out = sum_j eq(u, j) in[j].  The weights are a table (k_eq29), a product with one is only
// summed (Wide29: 81 multiply-adds in 29-bit limbs, one reduction a lane), so the tensor is read once, nothing is written but the
// result, and a wave's loads run along memory whichever axis it is.  Three levels a pass (k_fold_axis_dot) read 1 1/7 times the tensor
// and, along the innermost axis, eight elements a lane at 256-byte strides.
static constexpr int EQ29_MAX = 14;          // levels: three factors of at most five bits
struct Eq29Tabs { Fr29 t[96]; };             // 32 entries for each factor, with the factor 2^261
// entry i < n of the eq table with factor 2^261, canonical; SOA: limb l at out[l n + i], else at out[9 i + l]
template <bool SOA> __global__ void __launch_bounds__(TPB) k_eq29(int32_t* __restrict__ out, const Eq29Tabs tabs, uint32_t n, int b0, int b1) {
    const uint32_t i = blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    const Fr29 e = fr29_canon<2>(fr29_mul(fr29_mul(tabs.t[i & ((1u << b0) - 1u)], tabs.t[32 + ((i >> b0) & ((1u << b1) - 1u))]), tabs.t[64 + (i >> (b0 + b1))]));
#pragma unroll
    for (int l = 0; l < 9; ++l) out[SOA ? (size_t)l * n + i : (size_t)i * 9 + l] = e.l[l];
}
// innermost axis: out[row] = sum_p E[p] in[row][p].  WPR waves take two rows (an entry of the table serves both), 64 terms a lane at most
struct EqSoa {
    const int32_t* E;
    uint32_t n;
    __device__ __forceinline__ Fr29 operator()(uint32_t i) const {
        Fr29 e;
#pragma unroll
        for (int l = 0; l < 9; ++l) e.l[l] = E[(size_t)l * n + i];
        return e;
    }
};
struct EqAos {
    const int32_t* E;
    __device__ __forceinline__ Fr29 operator()(uint32_t i) const {
        Fr29 e;
#pragma unroll
        for (int l = 0; l < 9; ++l) e.l[l] = E[(size_t)i * 9 + l];
        return e;
    }
};
using FoldRowsLds = uint32_t[2][4][9];
template <class EQ> __device__ __forceinline__ void
fold_rows_block(FoldRowsLds& red, Fr* __restrict__ out, const Fr* __restrict__ in, const EQ& eq, size_t rows, uint32_t cur, const uint32_t wpr, uint32_t block) {
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const size_t r0 = ((size_t)block * (4 / wpr) + wave / wpr) * 2;
    const size_t ra = r0 < rows ? r0 : rows - 1, rb = r0 + 1 < rows ? r0 + 1 : rows - 1;
    const Fr *pa = in + ra * cur, *pb = in + rb * cur;
    Wide29 wa = wide29_zero(), wb = wide29_zero();
    uint32_t p = (wave % wpr) * 64u + lane, term = 0;
    Fr xa = big_zero<8>(), xb = xa;
    Fr29 e = fr29_zero();
    auto fetch = [&](uint32_t q) {
        xa = pa[q]; xb = pb[q];
        e = eq(q);
    };
    if (p < cur) fetch(p);
    while (p < cur) {
        const Fr29 a = fr29_repack(xa), b = fr29_repack(xb), ce = e;
        p += 64u * wpr;
        if (p < cur) fetch(p);
        wide29_mac(wa, ce, a);
        wide29_mac(wb, ce, b);
        if ((++term & 3u) == 0) { wide29_carry(wa); wide29_carry(wb); }
    }
    uint32_t l9[2][9];
    const Fr29 sa = fr29_canon<2>(wide29_redc(wa)), sb = fr29_canon<2>(wide29_redc(wb));
#pragma unroll
    for (int l = 0; l < 9; ++l) { l9[0][l] = (uint32_t)sa.l[l]; l9[1][l] = (uint32_t)sb.l[l]; }
    fr29_wave_sum(l9[0]);
    fr29_wave_sum(l9[1]);
    if (lane == 63u) {
#pragma unroll
        for (int l = 0; l < 9; ++l) { red[0][wave][l] = l9[0][l]; red[1][wave][l] = l9[1][l]; }
    }
    __syncthreads();
    if (threadIdx.x < 8 / wpr) {
        const uint32_t k = threadIdx.x & 1u, g = threadIdx.x >> 1;
        const size_t row = ((size_t)block * (4 / wpr) + g) * 2 + k;
        uint32_t s[9];
#pragma unroll
        for (int l = 0; l < 9; ++l) {
            s[l] = red[k][g * wpr][l];
#pragma unroll
            for (uint32_t w = 1; w < wpr; ++w) s[l] += red[k][g * wpr + w][l];
        }
        fr29_carry_u(s);
        Fr29 x;
#pragma unroll
        for (int l = 0; l < 9; ++l) x.l[l] = (int32_t)s[l];
        if (row < rows) out[row] = fr29_canon_pack<5>(fr29_mul(x, fr29_2_261()));
    }
}
template <int WPR> __global__ void __launch_bounds__(TPB)
k_fold_rows(Fr* __restrict__ out, const Fr* __restrict__ in, const int32_t* __restrict__ E, size_t rows, uint32_t cur) {
    __shared__ FoldRowsLds red;
    fold_rows_block(red, out, in, EqSoa{E, cur}, rows, cur, WPR, blockIdx.x);
}
// a middle axis: out[z][w] = sum_j E[j] in[z][j][w].  A lane takes one w and J consecutive j (the table's entry is the same for the
// whole wave), the four waves of a workgroup 4 J of them; grid (w in groups of 64, 4 J at a time, z)
using FoldColsLds = uint32_t[3][9][64];
template <class EQ> __device__ __forceinline__ void
fold_cols_block(FoldColsLds& red, Fr* __restrict__ part, const Fr* __restrict__ in, const EQ& eq, uint32_t e0, uint32_t cur, size_t window, uint32_t J,
                uint32_t bx, uint32_t by, uint32_t bz, uint32_t nz) {      // eq's first entry is e0's
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63u;
    const size_t w = (size_t)bx * 64 + lane, wc = w < window ? w : window - 1;
    const uint32_t j0 = (by * 4 + wave) * J, j1 = j0 + J < cur ? j0 + J : cur;
    const Fr* base = in + (size_t)bz * cur * window + wc;
    Wide29 acc = wide29_zero();
    for (uint32_t j = j0; j < j1; j += 4) {
        Fr x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = base[(size_t)(j + q < j1 ? j + q : j) * window];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (j + q < j1) {
                const Fr29 e = eq(j + q - e0);
                wide29_mac(acc, e, fr29_repack(x[q]));
            }
        wide29_carry(acc);
    }
    Fr29 s = wide29_redc(acc);
    if (wave) {
#pragma unroll
        for (int l = 0; l < 9; ++l) red[wave - 1][l][lane] = (uint32_t)s.l[l];
    }
    __syncthreads();
    if (wave) return;
    uint32_t l9[9];
#pragma unroll
    for (int l = 0; l < 9; ++l) l9[l] = (uint32_t)s.l[l] + red[0][l][lane] + red[1][l][lane] + red[2][l][lane];
    fr29_carry_u(l9);
#pragma unroll
    for (int l = 0; l < 9; ++l) s.l[l] = (int32_t)l9[l];
    if (w < window) part[((size_t)by * nz + bz) * window + w] = fr29_canon_pack<2>(fr29_mul(s, fr29_2_261()));
}
__global__ void __launch_bounds__(TPB)
k_fold_cols(Fr* __restrict__ part, const Fr* __restrict__ in, const int32_t* __restrict__ E, uint32_t cur, size_t window, uint32_t J) {
    __shared__ FoldColsLds red;
    fold_cols_block(red, part, in, EqAos{E}, 0u, cur, window, J, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.z);
}
// ---- the folds of a matrix product's proof, Y = X W ---------------------------------------------------------------------------------
// X over its rows at u_batch (Xf, xchunks parts of it for the reader to add up), W and Y over their columns at u_output (Wf, Yf): they need nothing of
// one another, and for all but the largest tensors each is a launch that does not fill the chip.  One launch takes the three, one before it
// both tables of weights; the parts of Xf and the value of Yf at u_batch are left to the sumcheck's launch.  Loads in flight bind
// it.  300 x 1000 x 2750: 73 us in eight launches, now 36 in two; 2048 x 4096 x 4096: 288 us in nine, now 232.
// SMALL (u of at most nine bits): the tables' two factors come in the arguments, a workgroup makes the entries that it needs in LDS, and one more
// leaves the table of u_batch for the reader of Yf.
struct EqArgs {
    Fr29 lo[32], hi[16];
    __device__ __forceinline__ Fr29 operator()(uint32_t i) const { return fr29_canon<2>(fr29_mul(lo[i & 31u], hi[i >> 5])); }
};
static constexpr int FC_SMALL_BITS = 9;
struct FcFolds {
    const Fr *X, *W, *Y;
    Fr *Xf, *Wf, *Yf;
    int32_t *Eb, *Eo;              // u_batch: nine limbs an entry; u_output: an entry's limbs O apart
    uint32_t B, D, O;
    uint32_t J, xgroups, xchunks;  // as k_fold_cols
    uint32_t wwaves, ywaves;       // waves that take two rows of W and Y (1 or 4)
    uint32_t wblocks, yblocks;     // workgroups: W's, Y's, then X's
};
template <bool SMALL> struct FcEq { };
template <> struct FcEq<true> { EqArgs batch, output; };
template <bool SMALL> __global__ void __launch_bounds__(TPB) k_fc_folds(const FcFolds a, const FcEq<SMALL> eq) {
    __shared__ union { FoldRowsLds rows; FoldColsLds cols; } lds;
    __shared__ int32_t tab[SMALL ? 9 << FC_SMALL_BITS : 1];
    uint32_t b = blockIdx.x;
    if (b < a.wblocks + a.yblocks) {
        const bool w = b < a.wblocks;
        if (!w) b -= a.wblocks;
        if constexpr (SMALL) {
            for (uint32_t i = threadIdx.x; i < a.O; i += TPB) {
                const Fr29 e = eq.output(i);
#pragma unroll
                for (int l = 0; l < 9; ++l) tab[l * a.O + i] = e.l[l];
            }
            __syncthreads();
        }
        fold_rows_block(lds.rows, w ? a.Wf : a.Yf, w ? a.W : a.Y, EqSoa{SMALL ? (const int32_t*)tab : (const int32_t*)a.Eo, a.O}, w ? a.D : a.B, a.O, w ? a.wwaves : a.ywaves, b);
        return;
    }
    b -= a.wblocks + a.yblocks;
    const uint32_t by = b / a.xgroups, bx = b - by * a.xgroups;
    if constexpr (SMALL) {
        const bool all = by == a.xchunks;                   // the workgroup behind X's
        const uint32_t j0 = all ? 0u : by * 4 * a.J, n = all ? a.B : (a.B - j0 < 4 * a.J ? a.B - j0 : 4 * a.J);
        for (uint32_t i = threadIdx.x; i < n; i += TPB) {
            const Fr29 e = eq.batch(j0 + i);
#pragma unroll
            for (int l = 0; l < 9; ++l) (all ? a.Eb : tab)[i * 9 + l] = e.l[l];
        }
        if (all) return;
        __syncthreads();
        fold_cols_block(lds.cols, a.Xf, a.X, EqAos{tab}, j0, a.B, a.D, a.J, bx, by, 0u, 1u);
    } else fold_cols_block(lds.cols, a.Xf, a.X, EqAos{a.Eb}, 0u, a.B, a.D, a.J, bx, by, 0u, 1u);
}
// both tables in one launch: four factors of at most four bits each
struct EqTwoTabs { Fr29 t[2][48]; uint32_t n[2]; int bits[2][4]; };
__global__ void __launch_bounds__(TPB) k_eq29_two(int32_t* __restrict__ Eb, int32_t* __restrict__ Eo, const EqTwoTabs a, uint32_t first) {
    const uint32_t which = blockIdx.x < first ? 0u : 1u, n = a.n[which];
    uint32_t i = (blockIdx.x - (which ? first : 0u)) * TPB + threadIdx.x;
    if (i >= n) return;
    const uint32_t at = i;
    uint32_t base = 0;
    Fr29 e = a.t[which][0];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        const uint32_t bits = (uint32_t)a.bits[which][f];
        const Fr29 x = a.t[which][base + (i & ((1u << bits) - 1u))];
        e = f ? fr29_mul(e, x) : x;
        i >>= bits;
        base += 1u << bits;
    }
    e = fr29_canon<2>(e);
#pragma unroll
    for (int l = 0; l < 9; ++l) {
        if (which) Eo[(size_t)l * n + at] = e.l[l];
        else Eb[(size_t)at * 9 + l] = e.l[l];
    }
}
// out[i] = sum of the count parts of i, sixteen lanes an output: one lane's loads behind one another took 24 us for 128 outputs of 64 parts
__global__ void __launch_bounds__(TPB) k_sum_partials(Fr* __restrict__ out, const Fr* __restrict__ part, size_t n, uint32_t count) {
    __shared__ Fr red[TPB / 16 - 1][16];
    const uint32_t q = threadIdx.x >> 4, o = threadIdx.x & 15u;
    const size_t i = (size_t)blockIdx.x * 16 + o;
    Fr s = big_zero<8>();
    if (i < n)
        for (uint32_t c = q; c < count; c += TPB / 16) s = add(s, part[(size_t)c * n + i]);
    if (q) red[q - 1][o] = s;
    __syncthreads();
    if (q || i >= n) return;
    for (uint32_t k = 0; k < TPB / 16 - 1; ++k) s = add(s, red[k][o]);
    out[i] = s;
}

// Short axes of small tensors in one launch, where a launch's cost counts and not what it does: LANES lanes take an output, at most four
// terms each, the weights out of two tables in the launch's arguments (lo: five bits, hi: the rest).
struct EqSmall { Fr29 lo[32], hi[32]; };
static constexpr uint32_t FOLD_SMALL_CUR = 1024;
static constexpr size_t FOLD_SMALL_MAX = (size_t)1 << 15;
template <int LANES> __global__ void __launch_bounds__(TPB) k_fold_small(Fr* __restrict__ out, const Fr* __restrict__ in, const EqSmall eq, uint32_t n_out, uint32_t n_in, uint32_t cur, uint32_t window) {
    __shared__ uint32_t red[4][9];
    const uint32_t t = threadIdx.x, ln = t % LANES, o = (blockIdx.x * TPB + t) / LANES;
    const bool live = o < n_out;
    const uint32_t z = live ? o / window : 0u, base = z * cur * window + (live ? o - z * window : 0u);
    Wide29 acc = wide29_zero();
    for (uint32_t j = ln; j < cur; j += LANES) {
        const uint32_t at = base + j * window;
        if (!live || at >= n_in) continue;
        Fr29 e = eq.lo[j & 31u];
        if (cur > 32u) e = fr29_mul(e, eq.hi[j >> 5]);
        wide29_mac(acc, e, fr29_repack(in[at]));
    }
    const Fr29 s = fr29_canon<2>(wide29_redc(acc));
    uint32_t l9[9];
#pragma unroll
    for (int l = 0; l < 9; ++l) l9[l] = (uint32_t)s.l[l];
    if (LANES == 16) fr29_row_sum(l9);
    else fr29_wave_sum(l9);
    if (LANES == 256) {
        if ((t & 63u) == 63u) {
#pragma unroll
            for (int l = 0; l < 9; ++l) red[t >> 6][l] = l9[l];
        }
        __syncthreads();
        if (t != TPB - 1) return;
#pragma unroll
        for (int l = 0; l < 9; ++l) l9[l] = red[0][l] + red[1][l] + red[2][l] + red[3][l];
        fr29_carry_u(l9);
    }
    if (!live || ln != LANES - 1) return;
    Fr29 x;
#pragma unroll
    for (int l = 0; l < 9; ++l) x.l[l] = (int32_t)l9[l];
    out[o] = fr29_canon_pack<5>(fr29_mul(x, fr29_2_261()));
}
// the eq tables of up to ten challenges, with the factor 2^261
static void eq_small_tables(EqSmall& e, const Fr* u_mont, int levels);
static int fold_small_queue(Fr* out, const Fr* in, const EqSmall& eq, uint32_t n_out, uint32_t n_in, uint32_t cur, uint32_t window, hipStream_t st) {
    if (cur <= 64) hipLaunchKernelGGL(k_fold_small<16>, dim3(cdiv((size_t)n_out * 16, TPB)), dim3(TPB), 0, st, out, in, eq, n_out, n_in, cur, window);
    else if (cur <= 256) hipLaunchKernelGGL(k_fold_small<64>, dim3(cdiv((size_t)n_out * 64, TPB)), dim3(TPB), 0, st, out, in, eq, n_out, n_in, cur, window);
    else hipLaunchKernelGGL(k_fold_small<256>, dim3(n_out), dim3(TPB), 0, st, out, in, eq, n_out, n_in, cur, window);
    ZK_LAUNCH_CHECK();
    return 0;
}
static void eq_small_tables(EqSmall& e, const Fr* u_mont, int levels) {
    int at = 0;
    for (int f = 0; f < 2; ++f) {
        Fr t[32];
        t[0] = fr29_pack(fr29_2_261());
        const int bits = f == 0 ? std::min(5, levels) : std::max(0, levels - 5);
        for (int b = 0; b < bits; ++b, ++at)
            for (int i = 0; i < (1 << b); ++i) {
                t[i + (1 << b)] = mont_mul(t[i], u_mont[at]);
                t[i] = sub(t[i], t[i + (1 << b)]);
            }
        for (int i = 0; i < (1 << bits); ++i) (f ? e.hi : e.lo)[i] = fr29_repack(t[i]);
    }
}

// MSB fold of the zero-extended vector: out[i] = a[i] + v*(a[i+n_out] - a[i])  (zkfc.cu:113-127,
// tlookup.cu:94-103, proof.cu:180-188)
__global__ void __launch_bounds__(TPB) k_fold_halves(Fr* __restrict__ out, const Fr* __restrict__ a, const Fr v_mont, size_t n_in, size_t n_out) {
    const size_t g = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (g >= n_out) return;
    const Fr a0 = (g < n_in) ? a[g] : big_zero<8>();
    const Fr a1 = (g + n_out < n_in) ? a[g + n_out] : big_zero<8>();
    out[g] = add(a0, mont_mul(v_mont, sub(a1, a0)));
}
// Stacked variant over [N][D] (zkfc.cu:169-185): same formula on whole rows
// (covered by k_fold_halves with n_in = N*D, n_out = N_out*D).

// ------------------------------------------------------------------------------------------------
// inner-product sumcheck (zkfc.cu:94-151)
// ------------------------------------------------------------------------------------------------
// Three sums of one round, each still carrying R^-1:
//   s0 = sum a0*b0, s1 = sum a0*(b1-b0) + b0*(a1-a0), s2 = sum (a1-a0)*(b1-b0)
__global__ void __launch_bounds__(TPB) k_ip_round(Fr* __restrict__ partials, const Fr* __restrict__ a, const Fr* __restrict__ b, size_t n_in, size_t n_out) {
    Fr acc[3] = {big_zero<8>(), big_zero<8>(), big_zero<8>()};
    for (size_t g = (size_t)blockIdx.x * TPB + threadIdx.x; g < n_out; g += (size_t)gridDim.x * TPB) {
        const Fr a0 = (g < n_in) ? a[g] : big_zero<8>();
        const Fr b0 = (g < n_in) ? b[g] : big_zero<8>();
        const Fr a1 = (g + n_out < n_in) ? a[g + n_out] : big_zero<8>();
        const Fr b1 = (g + n_out < n_in) ? b[g + n_out] : big_zero<8>();
        const Fr da = sub(a1, a0), db = sub(b1, b0);
        acc[0] = add(acc[0], mont_mul(a0, b0));
        acc[1] = add(acc[1], add(mont_mul(a0, db), mont_mul(b0, da)));
        acc[2] = add(acc[2], mont_mul(da, db));
    }
    block_reduce_store<3>(acc, partials);
}

// Stacked form (zkip_stacked_poly_kernel zkfc.cu:153-167 followed by the multilinear evaluation over the
// stacking axis, zkfc.cu:187-209): tensors are [N][D], halves are taken over N, and row n of the three
// term tensors is weighted by E[n] (eq table, Montgomery form) before everything is summed.
__global__ void __launch_bounds__(TPB) k_ip_round_w(Fr* __restrict__ partials, const Fr* __restrict__ a, const Fr* __restrict__ b, const Fr* __restrict__ E,
                                                    size_t D, size_t n_in, size_t n_out) {
    Fr acc[3] = {big_zero<8>(), big_zero<8>(), big_zero<8>()};
    for (size_t g = (size_t)blockIdx.x * TPB + threadIdx.x; g < n_out; g += (size_t)gridDim.x * TPB) {
        const Fr a0 = (g < n_in) ? a[g] : big_zero<8>();
        const Fr b0 = (g < n_in) ? b[g] : big_zero<8>();
        const Fr a1 = (g + n_out < n_in) ? a[g + n_out] : big_zero<8>();
        const Fr b1 = (g + n_out < n_in) ? b[g + n_out] : big_zero<8>();
        const Fr da = sub(a1, a0), db = sub(b1, b0);
        const Fr e = E[g / D];
        acc[0] = add(acc[0], mont_mul(e, mont_mul(a0, b0)));
        acc[1] = add(acc[1], mont_mul(e, add(mont_mul(a0, db), mont_mul(b0, da))));
        acc[2] = add(acc[2], mont_mul(e, mont_mul(da, db)));
    }
    block_reduce_store<3>(acc, partials);
}

// The whole sumcheck of short vectors (n <= 8192) in one or two launches.  The challenges are known before the first round, and a round
// pairs t with t + n/2 (the top index bit): the elements that agree in their low bits need nobody else for as many rounds as there are
// high bits.  A workgroup takes the 2^R elements of one low index (R <= 8) of both vectors, in LDS and in 29-bit limbs, and runs R
// rounds, a barrier each; a second launch of one workgroup runs what is left and adds up the first one's sums.  Every product of a pair
// has a lane of its own -- sixteen lanes (a row of the data-parallel adds) do one thing for sixteen pairs:
//   even waves: a0 b0 | a1 b1 | da db | -         odd waves: fold of a | fold of b | - | -
// so a round is the latency of one product, a row sum and a barrier: about 2 us.  One workgroup that gave a pair to a lane and
// summed through LDS took 15 us a round, 93 us for 64 elements and 225 us for 4096.  A further workgroup of the first launch may take an
// evaluation that nothing here waits for (ip_evaluate).  The middle coefficient is a1 b1 - a0 b0 - da db.
static constexpr int IP_ROUNDS = 8, IP_P = 1 << IP_ROUNDS, IP_W = 12, IP_GROUPS = 8;      // IP_GROUPS: pairs of waves, sixteen pairs each
struct IpArgs {
    const Fr *a, *b;
    Fr *na, *nb;                  // the folded vectors, nlow elements each
    Fr29 v[IP_ROUNDS];            // in round order, times 2^261
    uint32_t n, nlow, rounds;     // the vectors' length (zeros behind it), low indices, rounds of this launch
    Fr* sums;                     // round r's q-th sum at sums[(3 r + q) nlow + workgroup]
    const Fr* prev; Fr* prev_out; // the sums of a launch before: prev_count times prev_nb of them
    uint32_t prev_nb, prev_count;
    uint32_t a_parts;             // a is the sum of so many vectors, one behind the other
    const Fr* ev; const int32_t* ev_E; Fr* ev_out;      // for a workgroup more than nlow: sum_i ev_E[i] ev[i], i < ev_n
    uint32_t ev_n;
};
__device__ __forceinline__ void ip_evaluate(uint32_t (&red)[3][9], const IpArgs& a) {      // 256 lanes, at most 64 terms each
    const uint32_t t = threadIdx.x;
    Wide29 acc = wide29_zero();
    uint32_t term = 0;
    if (t < 256u)
        for (uint32_t i = t; i < a.ev_n; i += 256u) {
            wide29_mac(acc, EqAos{a.ev_E}(i), fr29_repack(a.ev[i]));
            if ((++term & 3u) == 0) wide29_carry(acc);
        }
    const Fr29 s = fr29_canon<2>(wide29_redc(acc));
    uint32_t l9[9];
#pragma unroll
    for (int l = 0; l < 9; ++l) l9[l] = (uint32_t)s.l[l];
    fr29_wave_sum(l9);
    if ((t & 63u) == 63u && t < 255u) {
#pragma unroll
        for (int l = 0; l < 9; ++l) red[t >> 6][l] = l9[l];
    }
    __syncthreads();
    if (t != 255u) return;
#pragma unroll
    for (int l = 0; l < 9; ++l) l9[l] += red[0][l] + red[1][l] + red[2][l];
    fr29_carry_u(l9);
    Fr29 x;
#pragma unroll
    for (int l = 0; l < 9; ++l) x.l[l] = (int32_t)l9[l];
    *a.ev_out = fr29_canon_pack<5>(fr29_mul(x, fr29_2_261()));
}
__global__ void __launch_bounds__(1024) k_ip_rounds(const IpArgs a) {
    __shared__ int32_t X0[2][IP_P][IP_W], X1[2][IP_P / 2][IP_W];
    __shared__ uint32_t raw[IP_ROUNDS][IP_GROUPS][3][9];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), kind = wave & 1u, group = wave >> 1;
    const uint32_t row = (threadIdx.x >> 4) & 3u, ln = threadIdx.x & 15u;
    const uint32_t P = 1u << a.rounds;
    if (blockIdx.x == a.nlow) { ip_evaluate(raw[0][0], a); return; }
    for (uint32_t i = threadIdx.x; i < 2 * P; i += 1024u) {
        const uint32_t s = i & (P - 1u), g = s * a.nlow + blockIdx.x;
        Fr x = big_zero<8>();
        if (g < a.n) {
            x = (i >> a.rounds ? a.b : a.a)[g];
            if (!(i >> a.rounds))
#pragma unroll 4
                for (uint32_t k = 1; k < a.a_parts; ++k) x = add(x, a.a[(size_t)k * a.n + g]);
        }
        rm_put(X0[i >> a.rounds][s], fr29_repack(x));
    }
    // the sums of the launch before, on waves that have no pairs here (it has at most 24 of them, of at most 32 parts each)
    if (a.prev && wave >= 2u && (wave - 2u) * 4u < a.prev_count) {
        const uint32_t j = (wave - 2u) * 4u + row, jc = j < a.prev_count ? j : 0u;
        uint32_t l9[9];
#pragma unroll
        for (int l = 0; l < 9; ++l) l9[l] = 0;
        for (uint32_t i = ln; i < a.prev_nb; i += 16u) {
            const Fr29 x = fr29_repack(a.prev[(size_t)jc * a.prev_nb + i]);
#pragma unroll
            for (int l = 0; l < 9; ++l) l9[l] += (uint32_t)x.l[l];
        }
        fr29_carry_u(l9);
        fr29_row_sum(l9);
        if (ln == 15u && j < a.prev_count) {
            Fr29 x;
#pragma unroll
            for (int l = 0; l < 9; ++l) x.l[l] = (int32_t)l9[l];
            a.prev_out[j] = fr29_canon_pack<2>(fr29_mul(x, fr29_2_261()));
        }
    }
    __syncthreads();
    for (uint32_t r = 0; r < a.rounds; ++r) {
        const bool odd = (r & 1u) != 0;
        const uint32_t half = P >> (r + 1);
        int32_t* const src = odd ? &X1[0][0][0] : &X0[0][0][0];
        int32_t* const dst = odd ? &X0[0][0][0] : &X1[0][0][0];
        const uint32_t ss = (odd ? IP_P / 2 : IP_P) * IP_W, ds = (odd ? IP_P : IP_P / 2) * IP_W;
        const uint32_t t = group * 16u + ln;
        if (group * 16u < half) {
            const bool live = t < half;
            const uint32_t ta = live ? t : 0u, tb = ta + half;
            auto rd = [&](uint32_t k, uint32_t slot) { return rm_get(src + k * ss + slot * IP_W); };
            if (kind == 0) {
                const Fr29 a0 = rd(0, ta), a1 = rd(0, tb), b0 = rd(1, ta), b1 = rd(1, tb);
                const Fr29 x = fr29_mul(fr29_select(row == 0, a0, fr29_select(row == 1, a1, fr29_sub_plus_r(a1, a0))),
                                        fr29_select(row == 0, b0, fr29_select(row == 1, b1, fr29_sub_plus_r(b1, b0))));
                uint32_t l9[9];
#pragma unroll
                for (int l = 0; l < 9; ++l) l9[l] = live ? (uint32_t)x.l[l] : 0u;
                fr29_row_sum(l9);
                if (ln == 15u && row < 3u) {
#pragma unroll
                    for (int l = 0; l < 9; ++l) raw[r][group][row][l] = l9[l];
                }
            } else {
                const Fr29 x0 = rd(row & 1u, ta), x1 = rd(row & 1u, tb);
                const Fr29 f = fr29_canon<2>(fr29_add(x0, fr29_mul(a.v[r], fr29_sub_plus_r(x1, x0))));
                if (live && row < 2u) rm_put(dst + row * ds + t * IP_W, f);
            }
        }
        __syncthreads();
    }
    // a product of two elements carries 2^-261 here.  Lane 3 r + q adds up round r's q-th sum; the middle coefficient takes its neighbours'
    if (threadIdx.x < 64u) {
        const uint32_t i = threadIdx.x < 3u * a.rounds ? threadIdx.x : 0u, r = i / 3u, q = i - 3u * r, half = P >> (r + 1), ng = (half + 15u) / 16u;
        uint32_t l9[9];
#pragma unroll
        for (int l = 0; l < 9; ++l) {
            l9[l] = 0;
            for (uint32_t g = 0; g < ng; ++g) l9[l] += raw[r][g][q][l];
        }
        fr29_carry_u(l9);
        Fr29 x;
#pragma unroll
        for (int l = 0; l < 9; ++l) x.l[l] = (int32_t)l9[l];
        Fr o = fr29_canon_pack<5>(fr29_mul(x, fr29_2_522()));
        Fr before, behind;
#pragma unroll
        for (int l = 0; l < 8; ++l) {
            before.v[l] = (uint32_t)__shfl_up((int)o.v[l], 1, 64);
            behind.v[l] = (uint32_t)__shfl_down((int)o.v[l], 1, 64);
        }
        if (q == 1) o = sub(sub(o, before), behind);
        if (threadIdx.x < 3u * a.rounds) a.sums[(size_t)threadIdx.x * a.nlow + blockIdx.x] = o;
    }
    const int32_t* const fin = (a.rounds & 1u) ? &X1[0][0][0] : &X0[0][0][0];
    const uint32_t fs = ((a.rounds & 1u) ? IP_P / 2 : IP_P) * IP_W;
    if (threadIdx.x >= 64u && threadIdx.x < 66u) {
        const uint32_t k = threadIdx.x - 64u;
        (k ? a.nb : a.na)[blockIdx.x] = fr29_pack(rm_get(fin + k * fs));
    }
}

// ------------------------------------------------------------------------------------------------
// host side of the C ABI
// ------------------------------------------------------------------------------------------------
static inline Fr load_fr(const uint32_t* p) { Fr r; memcpy(&r, p, 32); return r; }

#define LAUNCH1D(kernel, n, st, ...)                                                         \
    do {                                                                                     \
        if ((n) > 0) {                                                                       \
            hipLaunchKernelGGL(kernel, dim3(cdiv((n), TPB)), dim3(TPB), 0, (hipStream_t)(st), __VA_ARGS__); \
            ZK_LAUNCH_CHECK();                                                               \
        }                                                                                    \
    } while (0)

// out[r] = sum_j (x_rj / scale)^2 in double precision, the terms added one after the other from j = 0 (the order a plain
// host loop uses, so the rounding is the same).  One wave per row: the lanes form 64 terms at a time -- conversion,
// division and square are exactly rounded operations -- and lane 0 adds them in order.
__global__ void __launch_bounds__(64) k_row_sumsq_f64(double* __restrict__ out, const Fr* __restrict__ X, uint32_t cols, double scale) {
    __shared__ double term[64];
    const uint32_t r = blockIdx.x, t = threadIdx.x;
    const Fr* row = X + (size_t)r * cols;
    double acc = 0.0;
    for (uint32_t j0 = 0; j0 < cols; j0 += 64) {
        const uint32_t j = j0 + t;
        double v = 0.0;
        if (j < cols) {
            const double x = (double)fr_to_i64(row[j]) / scale;
            v = x * x;
        }
        term[t] = v;
        __syncthreads();
        if (t == 0) {
            const uint32_t cnt = cols - j0 < 64u ? cols - j0 : 64u;
            for (uint32_t q = 0; q < cnt; ++q) acc += term[q];
        }
        __syncthreads();
    }
    if (t == 0) out[r] = acc;
}

// ------------------------------------------------------------------------------------------------
// FrTensor::sum for callers that cannot allocate (code under stream capture, serving loops, harnesses that forbid
// hipMalloc).  The block partials of k_sum live in a file-scope device array instead of a pool block; the result goes
// to a device element of the caller's.  The array is one per GPU and is shared by every call on that GPU: calls that
// overlap on one GPU (two streams, two threads) race on it.  k_sum writes every partial that k_finish_sums reads, so
// nothing has to be cleared between calls.
// ------------------------------------------------------------------------------------------------
static constexpr unsigned SUM_STATIC_MAX_BLOCKS = 2048;                 // reduce_grid's cap
static constexpr int SUM_STATIC_MAX_DEVICES = 64;
static __device__ __align__(256) uint32_t scratch[SUM_STATIC_MAX_BLOCKS * 8];   // 64 KiB of block partials

static std::mutex g_scratch_mu;
static Fr* g_scratch_ptr[SUM_STATIC_MAX_DEVICES] = {};

// Address of this device's copy of `scratch` (the array's name is only a host-side handle), resolved once per device.
static int scratch_address(Fr** out) {
    int dev = -1;
    ZK_HIP(hipGetDevice(&dev));
    ZK_ARG(dev >= 0 && dev < SUM_STATIC_MAX_DEVICES, "zk_fr_sum_static: device index over 63");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        ZK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        ZK_ARG(p != nullptr, "zk_fr_sum_static: the scratch array has no device address");
        g_scratch_ptr[dev] = (Fr*)p;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}
namespace zk {
int fr_static_scratch_setup() { Fr* p = nullptr; return scratch_address(&p); }
}

extern "C" {

int zk_fr_add(void* out, const void* a, const void* b, size_t n, void* st) { LAUNCH1D(k_ew<EW_ADD>, n, st, (Fr*)out, (const Fr*)a, (const Fr*)b, n); return 0; }
int zk_fr_sub(void* out, const void* a, const void* b, size_t n, void* st) { LAUNCH1D(k_ew<EW_SUB>, n, st, (Fr*)out, (const Fr*)a, (const Fr*)b, n); return 0; }
int zk_fr_mul(void* out, const void* a, const void* b, size_t n, void* st) { LAUNCH1D(k_ew<EW_MUL>, n, st, (Fr*)out, (const Fr*)a, (const Fr*)b, n); return 0; }
int zk_fr_montmul(void* out, const void* a, const void* b, size_t n, void* st) { LAUNCH1D(k_ew<EW_MONTMUL>, n, st, (Fr*)out, (const Fr*)a, (const Fr*)b, n); return 0; }
int zk_fr_neg(void* out, const void* a, size_t n, void* st) { LAUNCH1D(k_neg, n, st, (Fr*)out, (const Fr*)a, n); return 0; }
int zk_fr_add_s(void* out, const void* a, const uint32_t* s, size_t n, void* st) { LAUNCH1D(k_ew_s<EW_ADD>, n, st, (Fr*)out, (const Fr*)a, load_fr(s), n); return 0; }
int zk_fr_sub_s(void* out, const void* a, const uint32_t* s, size_t n, void* st) { LAUNCH1D(k_ew_s<EW_SUB>, n, st, (Fr*)out, (const Fr*)a, load_fr(s), n); return 0; }
int zk_fr_mul_s(void* out, const void* a, const uint32_t* s, size_t n, void* st) {
    const Fr sm = to_mont(load_fr(s));
    LAUNCH1D(k_ew_s<EW_MUL>, n, st, (Fr*)out, (const Fr*)a, sm, n);
    return 0;
}
int zk_fr_add_mul_s(void* out, const void* a, const void* b, const uint32_t* s, size_t n, void* st) {
    LAUNCH1D(k_add_mul_s, n, st, (Fr*)out, (const Fr*)a, (const Fr*)b, to_mont(load_fr(s)), n);
    return 0;
}
// a*R (Scalar_mont) is a Montgomery product with R^2; a*R^-1 (Scalar_unmont) one with 1.
int zk_fr_mont(void* out, const void* a, size_t n, void* st) { LAUNCH1D(k_ew_s<EW_MUL>, n, st, (Fr*)out, (const Fr*)a, big_r2<8>(), n); return 0; }
int zk_fr_unmont(void* out, const void* a, size_t n, void* st) {
    Fr one = big_zero<8>(); one.v[0] = 1;
    LAUNCH1D(k_ew_s<EW_MUL>, n, st, (Fr*)out, (const Fr*)a, one, n);
    return 0;
}
int zk_fr_fill(void* out, const uint32_t* s, size_t n, void* st) { LAUNCH1D(k_fill, n, st, (Fr*)out, load_fr(s), n); return 0; }
int zk_fr_bias_add(void* z, const void* bias, size_t rows, uint32_t cols, void* st) {
    ZK_ARG(cols > 0, "zk_fr_bias_add: cols == 0");
    LAUNCH1D(k_bias, rows * cols, st, (Fr*)z, (const Fr*)bias, rows * cols, cols);
    return 0;
}

int zk_fr_from_i32(void* out, const void* in, size_t n, void* st) { LAUNCH1D(k_from_i32, n, st, (Fr*)out, (const int32_t*)in, n); return 0; }
int zk_fr_from_i64(void* out, const void* in, size_t n, void* st) { LAUNCH1D(k_from_i64, n, st, (Fr*)out, (const int64_t*)in, n); return 0; }
int zk_fr_from_u32(void* out, const void* in, size_t n, void* st) { LAUNCH1D(k_from_u32, n, st, (Fr*)out, (const uint32_t*)in, n); return 0; }
int zk_fr_from_f32(void* out, const void* in, uint64_t sf, size_t n, void* st) { LAUNCH1D(k_from_f32, n, st, (Fr*)out, (const float*)in, sf, n); return 0; }
int zk_fr_from_f64(void* out, const void* in, uint64_t sf, size_t n, void* st) { LAUNCH1D(k_from_f64, n, st, (Fr*)out, (const double*)in, sf, n); return 0; }
int zk_fr_to_i32(void* out, const void* in, size_t n, void* st) { LAUNCH1D(k_to_i32, n, st, (int32_t*)out, (const Fr*)in, n); return 0; }
// sums of squares of the rows of a rows x cols tensor of small signed integers, each divided by `scale` first, in double
// precision with the terms added in index order (the mean square of RMSNorm as a host loop would compute it;
// llama-rmsnorm.py:38-39 computes it with torch before the prover runs).  out_f64: rows doubles on the device.
int zk_row_sumsq_f64(void* out_f64, const void* X, uint32_t rows, uint32_t cols, double scale, void* st) {
    if (rows == 0) return 0;
    ZK_ARG(cols >= 1 && scale != 0.0, "zk_row_sumsq_f64: empty rows or zero scale");
    hipLaunchKernelGGL(k_row_sumsq_f64, dim3(rows), dim3(64), 0, (hipStream_t)st, (double*)out_f64, (const Fr*)X, cols, scale);
    ZK_LAUNCH_CHECK();
    return 0;
}
int zk_fr_to_i64(void* out, const void* in, size_t n, void* st) { LAUNCH1D(k_to_i64, n, st, (int64_t*)out, (const Fr*)in, n); return 0; }

int zk_fr_pad(void* out, const void* in, size_t rows, uint32_t last_in, uint32_t last_out, const uint32_t* pad, void* st) {
    ZK_ARG(last_in > 0 && last_out >= last_in, "zk_fr_pad: need 0 < last_in <= last_out");
    const size_t n_out = rows * last_out;
    LAUNCH1D(k_pad, n_out, st, (Fr*)out, (const Fr*)in, n_out, last_in, last_out, load_fr(pad));
    return 0;
}
int zk_fr_transpose_batched(void* out, const void* in, uint32_t batch, uint32_t M, uint32_t N, void* st) {
    if (batch == 0 || M == 0 || N == 0) return 0;
    ZK_ARG(out != in, "zk_fr_transpose: in-place transpose is not supported");
    ZK_ARG(batch <= 65535 && cdiv(M, 32) <= 65535, "zk_fr_transpose: too many matrices or rows for one launch");
    hipLaunchKernelGGL(k_transpose, dim3(cdiv(N, 32), cdiv(M, 32), batch), dim3(TPB), 0, (hipStream_t)st, (Fr*)out, (const Fr*)in, M, N);
    ZK_LAUNCH_CHECK();
    return 0;
}
int zk_fr_transpose(void* out, const void* in, uint32_t M, uint32_t N, void* st) { return zk_fr_transpose_batched(out, in, 1, M, N, st); }
// out[b][a][c] = in[a][b][c]: the leading two axes of a three-axis tensor swapped, rows of C elements moved whole (what two
// transposes do to bring [token][head][k] to [head][token][k] and back, in one pass)
// a workgroup per output row (b, a): the row's position is worked out once, by the scalar unit, and the lanes move its 16-byte words
__global__ void __launch_bounds__(TPB) k_swap_axes(uint4* __restrict__ out, const uint4* __restrict__ in, uint32_t A, uint32_t B, uint32_t Cw) {
    const uint32_t ba = blockIdx.x, a = ba % A, b = ba / A;
    const uint4* __restrict__ src = in + ((size_t)a * B + b) * Cw;
    uint4* __restrict__ dst = out + (size_t)ba * Cw;
    for (uint32_t w = threadIdx.x; w < Cw; w += TPB) dst[w] = src[w];
}
int zk_fr_swap_axes(void* out, const void* in, uint32_t A, uint32_t B, uint32_t C, void* st) {
    if (A == 0 || B == 0 || C == 0) return 0;
    ZK_ARG(out != in && out != nullptr && in != nullptr, "zk_fr_swap_axes: null or in-place");
    ZK_ARG((size_t)A * B <= 0x7FFFFFFFull && C <= 0x7FFFFFFFu, "zk_fr_swap_axes: too many rows for one launch");
    hipLaunchKernelGGL(k_swap_axes, dim3(A * B), dim3(TPB), 0, (hipStream_t)st, (uint4*)out, (const uint4*)in, A, B, C * 2);
    ZK_LAUNCH_CHECK();
    return 0;
}
// dst[i] = src[offset + i * stride] for elements of `words` 16-byte words (a field element 2, a Jacobian point 9)
__global__ void __launch_bounds__(TPB) k_copy_strided(uint4* __restrict__ dst, const uint4* __restrict__ src, uint32_t words, size_t count, size_t stride, size_t offset) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= count * words) return;
    const size_t e = i / words, w = i - e * words;
    dst[i] = src[(offset + e * stride) * words + w];
}
int zk_copy_strided(void* dst, const void* src, size_t elem_bytes, size_t count, size_t stride, size_t offset, void* st) {
    ZK_ARG(elem_bytes >= 16 && elem_bytes % 16 == 0 && elem_bytes <= 1024, "zk_copy_strided: elements of 16 to 1024 bytes, a multiple of 16");
    ZK_ARG(dst != src, "zk_copy_strided: in place");
    if (count == 0) return 0;
    const uint32_t words = (uint32_t)(elem_bytes / 16);
    LAUNCH1D(k_copy_strided, count * words, st, (uint4*)dst, (const uint4*)src, words, count, stride, offset);
    return 0;
}
int zk_fr_gather(void* out, const void* table, const void* idx, size_t n, void* st) {
    LAUNCH1D(k_gather, n, st, (Fr*)out, (const Fr*)table, (const uint32_t*)idx, n);
    return 0;
}

int zk_fr_sum(uint32_t* out_host, const void* a, size_t n, void* st) {
    if (n == 0) { memset(out_host, 0, 32); return 0; }
    const unsigned nb = reduce_grid(n);
    Scratch part(sizeof(Fr) * nb, (hipStream_t)st);
    if (part.rc) return part.rc;
    hipLaunchKernelGGL(k_sum, dim3(nb), dim3(TPB), 0, (hipStream_t)st, part.as<Fr>(), (const Fr*)a, n);
    ZK_LAUNCH_CHECK();
    return finish_to_host<1>(part.as<Fr>(), nb, (Fr*)out_host, (hipStream_t)st);
}
// sum_i a_i * b_i in standard form
int zk_fr_dot(uint32_t* out_host, const void* a, const void* b, size_t n, void* st) {
    if (n == 0) { memset(out_host, 0, 32); return 0; }
    const unsigned nb = reduce_grid(n);
    Scratch part(sizeof(Fr) * nb, (hipStream_t)st);
    if (part.rc) return part.rc;
    hipLaunchKernelGGL(k_dot, dim3(nb), dim3(TPB), 0, (hipStream_t)st, part.as<Fr>(), (const Fr*)a, (const Fr*)b, n);
    ZK_LAUNCH_CHECK();
    Fr s;
    int rc = finish_to_host<1>(part.as<Fr>(), nb, &s, (hipStream_t)st);
    if (rc) return rc;
    s = to_mont(s);
    memcpy(out_host, &s, 32);
    return 0;
}

// One or more levels of the middle-axis fold; u[0..levels) are standard-form challenges.
// out has other * ceil(cur / 2^levels) * window elements.  levels <= 3 per call.
int zk_fr_fold_axis(void* out, const void* in, const uint32_t* u, int levels, size_t other, uint32_t cur, size_t window, void* st) {
    ZK_ARG(levels >= 1 && levels <= 3, "zk_fr_fold_axis: levels must be 1..3");
    ZK_ARG(cur >= 1 && window >= 1, "zk_fr_fold_axis: empty axis");
    ZK_ARG(out != in, "zk_fr_fold_axis: out must differ from in");
    const uint32_t cur_out = (uint32_t)(((uint64_t)cur + (1u << levels) - 1) >> levels);
    const size_t n_out = other * cur_out * window;
    if (n_out == 0) return 0;
    if (levels == 1) {
        FrPack<1> p; p.x[0] = to_mont(load_fr(u));
        LAUNCH1D(k_fold_axis<1>, n_out, st, (Fr*)out, (const Fr*)in, p, n_out, cur, cur_out, window);
    } else {
        // weights of the 2^levels inputs of one output, Montgomery form
        Fr x[3], w[8];
        for (int i = 0; i < levels; ++i) x[i] = to_mont(load_fr(u + 8 * i));
        const Fr one = big_one_mont<8>();
        for (int j = 0; j < (1 << levels); ++j) {
            Fr p = (j & 1) ? x[0] : sub(one, x[0]);
            for (int l = 1; l < levels; ++l) p = mont_mul(p, ((j >> l) & 1) ? x[l] : sub(one, x[l]));
            w[j] = p;
        }
        if (levels == 2) {
            FrPack<4> p; for (int j = 0; j < 4; ++j) p.x[j] = w[j];
            LAUNCH1D(k_fold_axis_dot<2>, n_out, st, (Fr*)out, (const Fr*)in, p, n_out, cur, cur_out, window);
        } else {
            FrPack<8> p; for (int j = 0; j < 8; ++j) p.x[j] = w[j];
            LAUNCH1D(k_fold_axis_dot<3>, n_out, st, (Fr*)out, (const Fr*)in, p, n_out, cur, cur_out, window);
        }
    }
    return 0;
}

// All `levels` of the axis: out has other * ceil(cur / 2^levels) * window elements.  The whole axis in one pass where it is long enough for the table of
// weights to pay (a launch of its own) and the tensor large enough that its passes and not their launches count (2^15 elements, 1 MB);
// else three levels a launch.
int zk_fr_fold_axis_all(void* out, const void* in, const uint32_t* u, int levels, size_t other, uint32_t cur, size_t window, void* stv) {
    hipStream_t st = (hipStream_t)stv;
    ZK_ARG(levels >= 1 && levels <= 32 && cur >= 1 && window >= 1, "zk_fr_fold_axis_all: bad axis");
    ZK_ARG(out != in, "zk_fr_fold_axis_all: out must differ from in");
    if (other == 0) return 0;
    if (levels < 32 && cur % (1u << levels) == 0) { other *= cur >> levels; cur = 1u << levels; }      // fewer levels than the axis has: as many axes of 2^levels
    const bool whole = (uint64_t)cur <= ((uint64_t)1 << levels), rows = window == 1 && cur >= 128, cols = window >= 32 && cur >= 16 && other <= 65535;
    if (whole && levels <= EQ29_MAX && (rows || cols) && other * cur * window >= ((size_t)1 << 15) && cdiv(other, 2) <= 0x7FFFFFFFu) {
        Eq29Tabs tabs;
        const int bits[3] = {(levels + 2) / 3, (levels + 1) / 3, levels / 3};
        int at = 0;
        for (int f = 0; f < 3; ++f) {
            Fr t[32];
            t[0] = fr29_pack(fr29_2_261());
            for (int b = 0; b < bits[f]; ++b, ++at) {
                const Fr x = to_mont(load_fr(u + 8 * at));
                for (int i = 0; i < (1 << b); ++i) {
                    t[i + (1 << b)] = mont_mul(t[i], x);
                    t[i] = sub(t[i], t[i + (1 << b)]);
                }
            }
            for (int i = 0; i < (1 << bits[f]); ++i) tabs.t[32 * f + i] = fr29_repack(t[i]);
        }
        Scratch eq(sizeof(int32_t) * 9 * (size_t)cur, st);
        if (eq.rc) return eq.rc;
        if (rows) {
            hipLaunchKernelGGL(k_eq29<true>, dim3(cdiv(cur, TPB)), dim3(TPB), 0, st, eq.as<int32_t>(), tabs, cur, bits[0], bits[1]);
            // a wave for two rows where that fills the chip (four waves a SIMD) or the rows are short, four waves else
            if (cur < 512 || (other >= 8192 && cur <= 4096)) hipLaunchKernelGGL(k_fold_rows<1>, dim3(cdiv(other, 8)), dim3(TPB), 0, st, (Fr*)out, (const Fr*)in, eq.as<int32_t>(), other, cur);
            else hipLaunchKernelGGL(k_fold_rows<4>, dim3(cdiv(other, 2)), dim3(TPB), 0, st, (Fr*)out, (const Fr*)in, eq.as<int32_t>(), other, cur);
            ZK_LAUNCH_CHECK();
            return 0;
        }
        hipLaunchKernelGGL(k_eq29<false>, dim3(cdiv(cur, TPB)), dim3(TPB), 0, st, eq.as<int32_t>(), tabs, cur, bits[0], bits[1]);
        // terms of a lane: as many as leave 8192 waves, between 8 and 64 (the reduction at a lane's end costs as much as three terms)
        const size_t groups = (window + 63) / 64, n_out = other * window;
        uint32_t J = 64;
        while (J > 8 && other * groups * ((cur + J - 1) / J) < 8192) J >>= 1;
        const uint32_t chunks = (cur + 4 * J - 1) / (4 * J);
        Scratch part(chunks > 1 ? sizeof(Fr) * n_out * chunks : 1, st);
        if (part.rc) return part.rc;
        hipLaunchKernelGGL(k_fold_cols, dim3((unsigned)groups, chunks, (unsigned)other), dim3(TPB), 0, st, chunks > 1 ? part.as<Fr>() : (Fr*)out, (const Fr*)in, eq.as<int32_t>(), cur, window, J);
        ZK_LAUNCH_CHECK();
        if (chunks > 1) {
            hipLaunchKernelGGL(k_sum_partials, dim3(cdiv(n_out, 16)), dim3(TPB), 0, st, (Fr*)out, part.as<Fr>(), n_out, chunks);
            ZK_LAUNCH_CHECK();
        }
        return 0;
    }
    if (whole && cur <= FOLD_SMALL_CUR && levels <= 10 && other * cur * window <= FOLD_SMALL_MAX) {
        Fr um[10];
        for (int i = 0; i < levels; ++i) um[i] = to_mont(load_fr(u + 8 * i));
        EqSmall eq;
        eq_small_tables(eq, um, levels);
        return fold_small_queue((Fr*)out, (const Fr*)in, eq, (uint32_t)(other * window), (uint32_t)(other * cur * window), cur, (uint32_t)window, st);
    }
    std::unique_ptr<Scratch> keep[2];
    const void* src = in;
    for (int done = 0, which = 0; done < levels; which ^= 1) {
        const int L = std::min(3, levels - done);
        const uint32_t cur_out = (uint32_t)(((uint64_t)cur + (1u << L) - 1) >> L);
        void* dst = out;
        if (done + L < levels) {
            keep[which].reset(new Scratch(sizeof(Fr) * other * cur_out * window, st));
            if (keep[which]->rc) return keep[which]->rc;
            dst = keep[which]->p;
        }
        const int rc = zk_fr_fold_axis(dst, src, u + 8 * done, L, other, cur, window, stv);
        if (rc) return rc;
        src = dst;
        cur = cur_out;
        done += L;
    }
    return 0;
}

// Multilinear extension of a (n elements, zero-extended to 2^k) at u[0..k): index bit j is bound
// to u[j].  Requires 2^(k-1) < n <= 2^k (k = 0 allowed for n == 1).
int zk_fr_me(uint32_t* out_host, const void* a, size_t n, const uint32_t* u, int k, void* stv) {
    hipStream_t st = (hipStream_t)stv;
    ZK_ARG(n >= 1 && k >= 0 && k <= 32, "zk_fr_me: bad size");
    ZK_ARG(n <= ((size_t)1 << k) && (k == 0 || n > ((size_t)1 << (k - 1))), "zk_fr_me: need 2^(k-1) < n <= 2^k");
    const Fr* cur_ptr = (const Fr*)a;
    size_t cur = n;
    int done = 0;
    void* bufs[2] = {nullptr, nullptr};
    int which = 0, rc = 0;
    while (cur > FOLD_SMALL_CUR && rc == 0) {
        const int L = 3;
        const size_t next = (cur + 7) >> 3;
        if (!bufs[which]) rc = pool_alloc(&bufs[which], next * sizeof(Fr), st);
        if (rc) break;
        rc = zk_fr_fold_axis(bufs[which], cur_ptr, u + 8 * done, L, 1, (uint32_t)cur, 1, stv);
        cur_ptr = (const Fr*)bufs[which];
        which ^= 1;
        cur = next;
        done += L;
    }
    if (rc == 0) {
        const int rest = k - done;
        Fr um[10];
        for (int i = 0; i < rest; ++i) um[i] = to_mont(load_fr(u + 8 * (done + i)));
        EqSmall eq;
        eq_small_tables(eq, um, rest);
        Delivery d;
        rc = deliver_begin(d, 1, 0);
        if (!rc) {
            rc = fold_small_queue((Fr*)d.dst, cur_ptr, eq, 1u, (uint32_t)cur, (uint32_t)cur, 1u, st);
            if (!rc) rc = deliver_end(d, st, out_host);
        }
    }
    for (int i = 0; i < 2; ++i) if (bufs[i]) pool_free(bufs[i], st);
    return rc;
}

int zk_fr_fold_halves(void* out, const void* a, const uint32_t* v, size_t n_in, size_t n_out, void* st) {
    ZK_ARG(out != a, "zk_fr_fold_halves: out must differ from in");
    LAUNCH1D(k_fold_halves, n_out, st, (Fr*)out, (const Fr*)a, to_mont(load_fr(v)), n_in, n_out);
    return 0;
}

// One round of the inner-product sumcheck: poly3_host = [sum a0 b0, sum a0 db + b0 da, sum da db].
int zk_ip_round(uint32_t* poly3_host, const void* a, const void* b, size_t n_in, size_t n_out, void* stv) {
    ZK_ARG(n_out >= 1 && n_in >= 1 && n_in <= 2 * n_out, "zk_ip_round: need n_in <= 2*n_out");
    const unsigned nb = reduce_grid(n_out);
    Scratch part(sizeof(Fr) * 3 * nb, (hipStream_t)stv);
    if (part.rc) return part.rc;
    hipLaunchKernelGGL(k_ip_round, dim3(nb), dim3(TPB), 0, (hipStream_t)stv, part.as<Fr>(), (const Fr*)a, (const Fr*)b, n_in, n_out);
    ZK_LAUNCH_CHECK();
    Delivery d;
    const int rc = deliver_begin(d, 3, 3);
    if (rc) return rc;
    hipLaunchKernelGGL(k_finish_sums, dim3(3), dim3(TPB), 0, (hipStream_t)stv, (Fr*)d.dst, part.as<Fr>(), nb);
    ZK_LAUNCH_CHECK();
    return deliver_end(d, (hipStream_t)stv, poly3_host);
}

// Stacked round over [N][D] tensors: rows_in = N, rows_out = 2^ceil(log2 N) / 2, E = eq table over the
// remaining stacking challenges (rows_out entries, Montgomery form).
int zk_ip_round_stacked(uint32_t* poly3_host, const void* a, const void* b, const void* E, size_t D, size_t rows_in, size_t rows_out, void* stv) {
    ZK_ARG(D >= 1 && rows_out >= 1 && rows_in >= 1 && rows_in <= 2 * rows_out, "zk_ip_round_stacked: bad shape");
    const size_t n_in = rows_in * D, n_out = rows_out * D;
    const unsigned nb = reduce_grid(n_out);
    Scratch part(sizeof(Fr) * 3 * nb, (hipStream_t)stv);
    if (part.rc) return part.rc;
    hipLaunchKernelGGL(k_ip_round_w, dim3(nb), dim3(TPB), 0, (hipStream_t)stv, part.as<Fr>(), (const Fr*)a, (const Fr*)b, (const Fr*)E, D, n_in, n_out);
    ZK_LAUNCH_CHECK();
    Fr s[3];
    int rc = finish_to_host<3>(part.as<Fr>(), nb, s, (hipStream_t)stv);
    if (rc) return rc;
    for (int i = 0; i < 3; ++i) s[i] = to_mont(s[i]);
    memcpy(poly3_host, s, 96);
    return 0;
}

// The launches of a complete inner-product sumcheck for n <= 8192.  work: ip_work(k) elements; out: 3 k sums, then the folded a and b.
struct IpEval { const Fr* v; const int32_t* E; uint32_t n; Fr* out; };
static size_t ip_work(int k) { return k <= IP_ROUNDS ? 0 : (3 * (size_t)IP_ROUNDS + 2) << (k - IP_ROUNDS); }
static int ip_rounds_queue(Fr* work, Fr* out, const Fr* a, uint32_t a_parts, const Fr* b, uint32_t n, const uint32_t* u, int k, const IpEval* ev, hipStream_t st) {
    // work: what passes from the first launch to the second
    const int r1 = k <= IP_ROUNDS ? 0 : IP_ROUNDS, r2 = k - r1;
    const uint32_t nb1 = r1 ? 1u << (k - r1) : 0u;
    Fr* part = work;
    Fr* mid = part + 3 * (size_t)r1 * nb1;
    IpArgs q;
    memset(&q, 0, sizeof(q));
    q.a = a; q.b = b; q.n = n; q.a_parts = a_parts;
    if (ev) { q.ev = ev->v; q.ev_E = ev->E; q.ev_n = ev->n; q.ev_out = ev->out; }
    auto challenges = [&](int from, int count) {
        for (int i = 0; i < count; ++i) q.v[i] = fr29_repack(mont_mul(to_mont(load_fr(u + 8 * (size_t)(k - 1 - from - i))), fr29_pack(fr29_2_261())));
    };
    uint32_t extra = ev ? 1u : 0u;
    if (r1) {
        challenges(0, r1);
        q.rounds = (uint32_t)r1; q.nlow = nb1; q.sums = part; q.na = mid; q.nb = mid + nb1;
        hipLaunchKernelGGL(k_ip_rounds, dim3(nb1 + extra), dim3(1024), 0, st, q);
        ZK_LAUNCH_CHECK();
        q.a = mid; q.b = mid + nb1; q.n = nb1; q.a_parts = 1;
        q.prev = part; q.prev_out = out; q.prev_nb = nb1; q.prev_count = 3u * (uint32_t)r1;
        extra = 0;
    }
    challenges(r1, r2);
    q.rounds = (uint32_t)r2; q.nlow = 1; q.sums = out + 3 * r1; q.na = out + 3 * k; q.nb = q.na + 1;
    hipLaunchKernelGGL(k_ip_rounds, dim3(1 + extra), dim3(1024), 0, st, q);
    ZK_LAUNCH_CHECK();
    return 0;
}
// Complete inner-product sumcheck for n <= 8192 in one or two launches.  u[0..k) standard form, consumed
// from the back; polys_host gets 3*k coefficients, fin_host the folded a and b.
int zk_ip_sumcheck_small(uint32_t* polys_host, uint32_t* fin_host, const void* a, const void* b, uint32_t n, const uint32_t* u, int k, void* stv) {
    hipStream_t st = (hipStream_t)stv;
    ZK_ARG(k >= 1 && k <= 13, "zk_ip_sumcheck_small: k must be 1..13");
    ZK_ARG(n >= 1 && n <= (1u << k) && n > ((1u << k) >> 1), "zk_ip_sumcheck_small: need 2^(k-1) < n <= 2^k");
    Scratch work(sizeof(Fr) * ip_work(k), st);
    if (work.rc) return work.rc;
    // one delivery of 3k + 2 values: the round polynomials, then the two fully folded values
    Delivery d;
    int rc = deliver_begin(d, 3 * (size_t)k + 2, 0);
    if (rc) return rc;
    rc = ip_rounds_queue(work.as<Fr>(), (Fr*)d.dst, (const Fr*)a, 1u, (const Fr*)b, n, u, k, nullptr, st);
    if (rc) return rc;
    Fr both[3 * 13 + 2];
    rc = deliver_end(d, st, both);
    if (rc) return rc;
    memcpy(polys_host, both, sizeof(Fr) * 3 * k);           // (while results are deferred these two are not what the kernel wrote: see zk_defer_begin)
    memcpy(fin_host, both + 3 * k, sizeof(Fr) * 2);
    return 0;
}
// the factors of an eq table, with the factor 2^261: entry i = t_0[low bits of i] t_1[the next] ..., factor f with bits[f] bits
static void eq_factors(Fr29* out, const uint32_t* u, const int* bits, int nf) {
    for (int f = 0; f < nf; ++f) {
        Fr t[32];
        t[0] = fr29_pack(fr29_2_261());
        for (int b = 0; b < bits[f]; ++b, u += 8) {
            const Fr x = to_mont(load_fr(u));
            for (int i = 0; i < (1 << b); ++i) {
                t[i + (1 << b)] = mont_mul(t[i], x);
                t[i] = sub(t[i], t[i + (1 << b)]);
            }
        }
        for (int i = 0; i < (1 << bits[f]); ++i) *out++ = fr29_repack(t[i]);
    }
}
int zk_matmul_sumcheck(uint32_t* claim_host, uint32_t* polys_host, uint32_t* fin_host, const void* X, const void* W, const void* Y, uint32_t B, uint32_t D, uint32_t O,
                       const uint32_t* u_batch, int kb, const uint32_t* u_input, int kd, const uint32_t* u_output, int ko, void* stv) {
    hipStream_t st = (hipStream_t)stv;
    auto fits = [](uint32_t n, int k, int most) { return k >= 0 && k <= most && n >= 1 && n <= (1u << k) && n > ((1u << k) >> 1); };
    ZK_ARG(kd >= 1 && fits(D, kd, 13), "zk_matmul_sumcheck: inner axis: 1 to 13 challenges, 2^(k-1) < D <= 2^k");
    ZK_ARG(fits(B, kb, EQ29_MAX) && fits(O, ko, EQ29_MAX), "zk_matmul_sumcheck: outer axes: at most 14 challenges, 2^(k-1) < n <= 2^k");
    ZK_ARG(X != nullptr && W != nullptr && Y != nullptr, "zk_matmul_sumcheck: null operand or result");
    ZK_ARG(u_input != nullptr && (kb == 0 || u_batch != nullptr) && (ko == 0 || u_output != nullptr), "zk_matmul_sumcheck: null challenges");
    ZK_ARG(deferring() || (claim_host != nullptr && polys_host != nullptr && fin_host != nullptr), "zk_matmul_sumcheck: null output");      // (deferred: delivered elsewhere)
    FcFolds a;
    a.X = (const Fr*)X; a.W = (const Fr*)W; a.Y = (const Fr*)Y;
    a.B = B; a.D = D; a.O = O;
    // X: sixteen terms a lane, fewer where the axis is that short, more where there would be more than eight parts to add up
    a.J = B < 64 ? (B + 15) / 16 * 4 : 16;
    while (a.J < 64 && B > 32 * a.J) a.J *= 2;
    a.xgroups = (D + 63) / 64; a.xchunks = (B + 4 * a.J - 1) / (4 * a.J);
    auto waves = [&](uint32_t rows) { return O < 512 || (rows >= 8192 && O <= 4096) ? 1u : 4u; };      // as zk_fr_fold_axis_all
    a.wwaves = waves(D); a.ywaves = waves(B);
    a.wblocks = a.wwaves == 1 ? cdiv(D, 8) : cdiv(D, 2);
    a.yblocks = a.ywaves == 1 ? cdiv(B, 8) : cdiv(B, 2);
    const size_t words = 9 * ((size_t)B + O), elems = (size_t)a.xchunks * D + D + B + ip_work(kd);
    Scratch work(sizeof(Fr) * elems + sizeof(int32_t) * words, st);
    if (work.rc) return work.rc;
    a.Xf = work.as<Fr>(); a.Wf = a.Xf + (size_t)a.xchunks * D; a.Yf = a.Wf + D;
    Fr* ip = a.Yf + B;
    a.Eb = (int32_t*)(ip + ip_work(kd)); a.Eo = a.Eb + 9 * (size_t)B;
    Delivery d;
    int rc = deliver_begin(d, 3 * (size_t)kd + 3, 0);
    if (rc) return rc;
    if (kb <= FC_SMALL_BITS && ko <= FC_SMALL_BITS) {
        FcEq<true> eq;
        const int bb[2] = {std::min(kb, 5), std::max(kb - 5, 0)}, bo[2] = {std::min(ko, 5), std::max(ko - 5, 0)};
        auto factors = [](EqArgs& e, const uint32_t* u, const int* bits) {
            eq_factors(e.lo, u, bits, 1);
            eq_factors(e.hi, u + 8 * bits[0], bits + 1, 1);
        };
        factors(eq.batch, u_batch, bb);
        factors(eq.output, u_output, bo);
        hipLaunchKernelGGL(k_fc_folds<true>, dim3(a.wblocks + a.yblocks + a.xgroups * a.xchunks + 1), dim3(TPB), 0, st, a, eq);
    } else {
        EqTwoTabs t;
        auto split = [](int* bits, int k) { for (int f = 0; f < 4; ++f) bits[f] = (k + 3 - f) / 4; };
        split(t.bits[0], kb); split(t.bits[1], ko);
        t.n[0] = B; t.n[1] = O;
        eq_factors(t.t[0], u_batch, t.bits[0], 4);
        eq_factors(t.t[1], u_output, t.bits[1], 4);
        const uint32_t first = cdiv(B, TPB);
        hipLaunchKernelGGL(k_eq29_two, dim3(first + cdiv(O, TPB)), dim3(TPB), 0, st, a.Eb, a.Eo, t, first);
        hipLaunchKernelGGL(k_fc_folds<false>, dim3(a.wblocks + a.yblocks + a.xgroups * a.xchunks), dim3(TPB), 0, st, a, FcEq<false>{});
    }
    ZK_LAUNCH_CHECK();
    const IpEval ev{a.Yf, a.Eb, B, (Fr*)d.dst};
    rc = ip_rounds_queue(ip, (Fr*)d.dst + 1, a.Xf, a.xchunks, a.Wf, D, u_input, kd, &ev, st);
    if (rc) return rc;
    Fr all[3 * 13 + 3];
    rc = deliver_end(d, st, all);
    if (rc) return rc;
    memcpy(claim_host, all, sizeof(Fr));
    memcpy(polys_host, all + 1, sizeof(Fr) * 3 * kd);
    memcpy(fin_host, all + 1 + 3 * kd, sizeof(Fr) * 2);
    return 0;
}

int zk_fr_sum_static(void* out_dev, const void* a, size_t n, void* st) {
    ZK_ARG(out_dev != nullptr, "zk_fr_sum_static: null output");
    ZK_ARG(n <= ZK_FR_SUM_STATIC_MAX_N, "zk_fr_sum_static: more than 2^32 - 1 elements (ZK_FR_SUM_STATIC_MAX_N)");
    ZK_ARG(n == 0 || a != nullptr, "zk_fr_sum_static: null input");
    Fr* part = nullptr;
    int rc = scratch_address(&part);
    if (rc) return rc;
    const unsigned nb = n ? reduce_grid(n) : 1;       // n == 0: one block that writes a zero partial
    hipLaunchKernelGGL(k_sum, dim3(nb), dim3(TPB), 0, (hipStream_t)st, part, (const Fr*)a, n);
    ZK_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_finish_sums, dim3(1), dim3(TPB), 0, (hipStream_t)st, (Fr*)out_dev, (const Fr*)part, nb);
    ZK_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
