// G1 tensor kernels and the Pedersen commitment for gfx950.
//
// Points are Jacobian (x,y,z) over Fp in Montgomery form, 144 B each -- the reference's
// G1Jacobian_t layout (bls12-381.cuh:429-433).  Replaces g1-tensor.cu:61-625 (elementwise ops,
// sum, row-wise sum, scalar multiplication, G1 multilinear fold) and commitment.cu:22-129
// (commit, commit_int, me_open_step).
//
// commit_int is a fixed-base windowed multi-scalar multiplication: the generators are shared by
// every row of the committed matrix, so their signed-window multiples d*2^(cw)*G_j are built once
// (affine, batch-normalised) and each row is a run of mixed additions out of that table -- no
// per-pair doublings and no materialised m*n temporary (the reference writes 144 B per pair).
// All of it is VALU integer work on 12-limb Fp; results equal the reference's as group elements
// (a Jacobian triple depends on the order of additions, so bytes are compared after normalising).
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>
#include "fq29.hpp"
#include "rt.hpp"
#include "../../include/zkllm_hip.h"

using namespace zk;

static constexpr int GT = 64;   // threads per workgroup for point kernels (one wave; ~200 VGPRs per lane)

// ---- elementwise -------------------------------------------------------------------------------------
// For kernels of a few waves that a chain of launches waits for: their instructions go before those of the wide kernels of other streams that
// share their SIMDs: an opening of 128 x 131072, with the workgroups of one wave that k_tail_levels explains, 9.13 -> 8.70 ms
__device__ __forceinline__ void urgent() { __builtin_amdgcn_s_setprio(3); }
__global__ void __launch_bounds__(GT) k_g1_fill(G1Jac* __restrict__ out, const G1Jac p, size_t n) {
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    if (i < n) out[i] = p;
}
__global__ void __launch_bounds__(GT) k_g1_neg(G1Jac* __restrict__ out, const G1Jac* __restrict__ a, size_t n) {
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    if (i < n) out[i] = g1_neg(a[i]);
}
__global__ void __launch_bounds__(GT) k_g1aff_neg(G1Affine* __restrict__ out, const G1Affine* __restrict__ a, size_t n) {
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    if (i < n) out[i] = g1_neg(a[i]);
}
__global__ void __launch_bounds__(GT) k_g1aff_to_jac(G1Jac* __restrict__ out, const G1Affine* __restrict__ a, size_t n) {
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    if (i >= n) return;
    G1Jac r; r.x = a[i].x; r.y = a[i].y; r.z = big_one_mont<12>();
    out[i] = r;
}
// out = a (+/-) b ; nb == n elementwise, nb == 1 broadcast
__global__ void __launch_bounds__(GT) k_g1_add(G1Jac* __restrict__ out, const G1Jac* __restrict__ a, const G1Jac* __restrict__ b, size_t n, size_t nb, int negate) {
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    if (i >= n) return;
    G1Jac q = b[nb == 1 ? 0 : i];
    if (negate) q = g1_neg(q);
    out[i] = g1_add(a[i], q);
}
__global__ void __launch_bounds__(GT) k_g1_madd(G1Jac* __restrict__ out, const G1Jac* __restrict__ a, const G1Affine* __restrict__ b, size_t n, size_t nb, int negate) {
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    if (i >= n) return;
    G1Affine q = b[nb == 1 ? 0 : i];
    if (negate) q = g1_neg(q);
    out[i] = g1_add_mixed(a[i], q);
}
// out[i] = [s[i]] g[i % ng]   (G1_jacobian_elementwise_mul / _mul_broadcast, g1-tensor.cu:456-482)
__global__ void __launch_bounds__(GT) k_g1_scalar_mul(G1Jac* __restrict__ out, const G1Jac* __restrict__ g, const Fr* __restrict__ s, size_t ng, size_t n) {
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    if (i < n) out[i] = g1_mul(g[i % ng], s[i]);
}

// ---- reductions ------------------------------------------------------------------------------------------
// LDS tree over the GT lanes of a workgroup; lane 0 returns the total
__device__ __forceinline__ G1Jac block_sum_g1(G1Jac v) {
    __shared__ uint32_t lds[36][GT];
    const uint32_t t = threadIdx.x;
    const uint32_t* src = reinterpret_cast<const uint32_t*>(&v);
#pragma unroll
    for (int l = 0; l < 36; ++l) lds[l][t] = src[l];
    __syncthreads();
    for (uint32_t s = GT / 2; s > 0; s >>= 1) {
        if (t < s) {
            G1Jac x, y;
            uint32_t* px = reinterpret_cast<uint32_t*>(&x);
            uint32_t* py = reinterpret_cast<uint32_t*>(&y);
#pragma unroll
            for (int l = 0; l < 36; ++l) { px[l] = lds[l][t]; py[l] = lds[l][t + s]; }
            x = g1_add(x, y);
#pragma unroll
            for (int l = 0; l < 36; ++l) lds[l][t] = px[l];
        }
        __syncthreads();
    }
    G1Jac r;
    uint32_t* pr = reinterpret_cast<uint32_t*>(&r);
#pragma unroll
    for (int l = 0; l < 36; ++l) pr[l] = lds[l][0];
    __syncthreads();
    return r;
}
// rows of length ncol: out[row] = sum_j in[row*ncol + j]; gridDim.y splits a row into segments
__global__ void __launch_bounds__(GT) k_g1_rowsum(G1Jac* __restrict__ out, const G1Jac* __restrict__ in, size_t ncol, uint32_t nseg) {
    const size_t row = blockIdx.x;
    const uint32_t seg = blockIdx.y;
    const size_t per = (ncol + nseg - 1) / nseg;
    const size_t j0 = seg * per, j1 = (j0 + per < ncol) ? j0 + per : ncol;
    G1Jac acc = g1_infinity();
    for (size_t j = j0 + threadIdx.x; j < j1; j += GT) acc = g1_add(acc, in[row * ncol + j]);
    acc = block_sum_g1(acc);
    if (threadIdx.x == 0) out[row * nseg + seg] = acc;
}

// ---- G1 multilinear fold step (G1_me_step, g1-tensor.cu:486-498); x is already "unmont"-ed ----------------
__global__ void __launch_bounds__(GT) k_g1_me_step(G1Jac* __restrict__ out, const G1Jac* __restrict__ in, const Fr x, size_t in_size, size_t out_size) {
    const size_t g = (size_t)blockIdx.x * GT + threadIdx.x;
    if (g >= out_size) return;
    const size_t g0 = 2 * g, g1 = 2 * g + 1;
    G1Jac r;
    if (g1 < in_size) r = g1_add(in[g0], g1_mul(g1_add(in[g1], g1_neg(in[g0])), x));
    else if (g0 < in_size) r = g1_add(in[g0], g1_neg(g1_mul(in[g0], x)));
    else r = g1_infinity();
    out[g] = r;
}

// ---- batch normalisation to z = 1 -------------------------------------------------------------------------
// Each lane owns CH points, GT apart: prefix products of z, one inversion, back-substitution.
// Infinity (z == 0) is skipped in the product and written as all-zero limbs.
template <bool AFFINE_OUT, int CH> __global__ void __launch_bounds__(GT) k_g1_normalize(void* outv, const G1Jac* in, size_t n) {
    urgent();
    const size_t base = (size_t)blockIdx.x * GT * CH + threadIdx.x;
    if (base >= n) return;
    Fp pre[CH];
    Fp run = big_one_mont<12>();
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        pre[c] = run;
        if (base + (size_t)c * GT < n) {
            const Fp z = in[base + (size_t)c * GT].z;
            if (!is_zero(z)) run = fp_mul(run, z);
        }
    }
    Fp inv = mont_inverse(run);
#pragma unroll
    for (int c = CH - 1; c >= 0; --c) {
        if (base + (size_t)c * GT >= n) continue;
        const G1Jac p = in[base + (size_t)c * GT];
        Fp ox = big_zero<12>(), oy = big_zero<12>(), oz = big_zero<12>();
        if (!is_zero(p.z)) {
            const Fp zi = fp_mul(inv, pre[c]);
            inv = fp_mul(inv, p.z);
            const Fp zi2 = fp_sqr(zi);
            ox = fp_mul(p.x, zi2);
            oy = fp_mul(fp_mul(p.y, zi2), zi);
            oz = big_one_mont<12>();
        }
        if (AFFINE_OUT) {
            G1Affine* out = reinterpret_cast<G1Affine*>(outv);
            out[base + (size_t)c * GT].x = ox; out[base + (size_t)c * GT].y = oy;
        } else {
            G1Jac* out = reinterpret_cast<G1Jac*>(outv);
            out[base + (size_t)c * GT].x = ox; out[base + (size_t)c * GT].y = oy; out[base + (size_t)c * GT].z = oz;
        }
    }
}

// An inversion costs a lane about ten products and a point's own part eight: one point a lane while the launch is two waves a SIMD
// or less (its time is then about one lane's: 131072 generators took 408 us with eight a lane and the binary inverse), four a lane above.
template <bool AFFINE_OUT> static void g1_normalize_queue(void* out, const G1Jac* in, size_t n, hipStream_t st) {
    if (n <= (size_t)1 << 17) hipLaunchKernelGGL((k_g1_normalize<AFFINE_OUT, 1>), dim3(cdiv(n, (size_t)GT)), dim3(GT), 0, st, out, in, n);
    else hipLaunchKernelGGL((k_g1_normalize<AFFINE_OUT, 4>), dim3(cdiv(n, (size_t)GT * 4)), dim3(GT), 0, st, out, in, n);
}

// the normalised points once more in the 29-bit-limb form that the bucket kernels add in (infinity stays all-zero)
__global__ void __launch_bounds__(256) k_g1aff_to_a29(A29* __restrict__ out, const G1Affine* __restrict__ in, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = a29_from_affine(in[i]);
}

// ---- fixed-base table for commit_int -------------------------------------------------------------------------
// table (Jacobian, before normalisation): tab[(w * ngen + j) * half + (d-1)] = d * 2^(c*w) * G_j, d = 1..half.
// Bases first, one lane per generator walking up the windows by c doublings each (7 us each, in 29-bit limbs; 14 in 32-bit ones); then the multiples by doubling the
// filled part of every row, row[k + i] = row[i] + row[k - 1] for i < k, k = 1, 2, 4, ...: one launch per k with one lane
// per new entry, so every launch is dense whatever the row length (rows are as short as 4 entries when few tensor rows
// share the generators) and the chain of additions is log2(half) deep.
__global__ void __launch_bounds__(GT) k_msm_table_bases(G1Jac* __restrict__ tab, const G1Jac* __restrict__ gens, size_t ngen, uint32_t c, uint32_t nwin, uint32_t half) {
    const size_t j = (size_t)blockIdx.x * GT + threadIdx.x;
    if (j >= ngen) return;
    J29 base = j29_from_jac(gens[j]);
    for (uint32_t w = 0; w < nwin; ++w) {
        tab[((size_t)w * ngen + j) * half] = w ? j29_to_jac(base) : gens[j];
        if (w + 1 < nwin) for (uint32_t k = 0; k < c; ++k) j29_double_walk(base);
    }
}
__global__ void __launch_bounds__(GT) k_msm_table_fill(G1Jac* __restrict__ tab, size_t nrows, uint32_t logh, uint32_t logk) {
    const size_t t = (size_t)blockIdx.x * GT + threadIdx.x;
    if ((t >> logk) >= nrows) return;
    const uint32_t k = 1u << logk, i = (uint32_t)(t & (k - 1));
    G1Jac* row = tab + ((t >> logk) << logh);
    row[k + i] = g1_add(row[i], row[k - 1]);
}
// ---- commit_int: the table in affine 29-bit limbs, and the sums over rows -----------------------------------------------------------
// Window w of generator j: the multiples d 2^(c w) G_j, d = 1 .. E_w at tab[off_w + j E_w + d - 1].  E_w is 2^(c-1), in the highest window
// what the largest scalar needs (a power of two).
struct MsmTable { A29* tab; size_t ngen; uint32_t c, nwin, half, top; };
__device__ __forceinline__ size_t msm_slot(const MsmTable& T, uint32_t w, size_t j, uint32_t d) {
    const bool last = w + 1 == T.nwin;
    return (size_t)w * T.ngen * T.half + j * (last ? T.top : T.half) + (d - 1);
}
__device__ __forceinline__ Fq29 fq29_inverse(const Fq29& v) { return fq29_from_fp(mont_inverse(fq29_to_fp(v))); }
// How the entries of a window grow from h to t: entries c + i and c - i out of entry c, the centre, and entry i <= h, which share the slope's denominator
// x_c - x_i.  With c halfway between h and t <= 3 h that is every entry above h but the centre itself; np: pairs.
struct GrowSpec { uint32_t h, c, t, np; };
static constexpr int GROW_MAX = 12;
struct GrowCentres { uint32_t full_n, top_n; uint16_t full[GROW_MAX], top[GROW_MAX]; };
// The first entries of every window (those that it has) and the centres of its growth out of the normalised bases (window-major), a lane an entry: doublings and additions
// of the base along the bits of the multiple, and an inversion.  A step of k_msm_table_grow takes what one lane's inversion and
// its launch take however few its entries are: the first sixteen of 8192 rows took 330 us in four steps that doubled them, and take 170 here, 200 with the five centres.
// The centres come first: a wave of them, all of one multiple, takes longest.
__global__ void __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2))) k_msm_table_first(const MsmTable T, const G1Affine* __restrict__ bases, uint32_t first, const GrowCentres gc) {
    const size_t rows_full = (size_t)(T.nwin - 1) * T.ngen, n_full = rows_full * gc.full_n, n_centres = n_full + T.ngen * gc.top_n;
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    size_t r;
    uint32_t d;
    if (i < n_full) { r = i % rows_full; d = gc.full[i / rows_full]; }
    else if (i < n_centres) { r = rows_full + (i - n_full) % T.ngen; d = gc.top[(i - n_full) / T.ngen]; }
    else { r = (i - n_centres) / first; d = (uint32_t)((i - n_centres) % first) + 1u; }
    const bool full = r < rows_full;
    if (r >= T.ngen * T.nwin || d > (full ? T.half : T.top)) return;
    const A29 base = a29_from_affine(bases[r]);
    A29 out = base;
    if (d > 1u && !a29_is_inf(base)) {
        J29 p;
        p.x = base.x; p.y = base.y; p.z = fq29_one(); p.inf = 0u;
        for (int b = 30 - __clz((int)d); b >= 0; --b) {
            j29_double_walk(p);
            if ((d >> b) & 1u) j29_add_mixed_walk(p, base);
        }
        const Fq29 zi = fq29_inverse(p.z), zi2 = fq29_sqr(zi);
        out.x = fq29_mul(p.x, zi2);
        out.y = fq29_mul(p.y, fq29_mul(zi2, zi));
        if (p.inf) { out.x = fq29_zero(); out.y = fq29_zero(); }
    }
    (full ? T.tab + r * T.half : T.tab + rows_full * T.half + (r - rows_full) * T.top)[d - 1u] = out;
}
// A step of the windows' growth (GrowSpec: of the full windows, and of the highest): a lane's pairs share one inversion (about 26 products), and a pair takes nine products for its two entries
// and 320 bytes an entry (1419 MB fetched and 1267 written for 8.4 M).  Equal and opposite points and infinity are told apart from the coordinates, whatever the generators are.
// The products before a pair wait in the slot of one of its entries.  Entry by entry, each with a denominator of its own and the windows doubled from launch to launch, 8.4 M entries took 2.0 ms
// at 56 % of the issue slots (526 bytes an entry); three entries for one
// from launch to launch this way they take 1.3 to 1.4 ms, the large launches at 60 to 64 % (11008 x 4096 of 13 bits; the whole commitment 10.68 -> 10.18 ms).  Sending for the next pair's points early spills and gains nothing.
__global__ void __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2))) k_msm_table_grow(const MsmTable T, const GrowSpec full, const GrowSpec top, uint32_t n, uint32_t per_lane) {
    const uint32_t base = blockIdx.x * GT * per_lane + threadIdx.x;
    if (base >= n) return;
    const size_t rows_full = (size_t)(T.nwin - 1) * T.ngen;
    const uint32_t n_full = (uint32_t)rows_full * full.np;
    struct At { A29* row; uint32_t i, c, h, t; };
    auto at = [&](uint32_t q) {
        if (q < n_full) return At{T.tab + (size_t)(q / full.np) * T.half, q % full.np + 1u, full.c, full.h, full.t};
        q -= n_full;
        return At{T.tab + rows_full * T.half + (size_t)(q / top.np) * T.top, q % top.np + 1u, top.c, top.h, top.t};
    };
    // 0: slopes over dx; 1: equal points (their sum is a doubling, their difference infinity); 2: opposite ones; 3: the centre is infinity; 4: entry i is; 5: both results are infinity
    auto kind_of = [&](const A29& a, const A29& b, Fq29& den) {
        den = fq29_one();
        if (a29_is_inf(a)) return 4u;
        if (a29_is_inf(b)) return 3u;
        const Fq29 dx = fq29_sub(a.x, b.x);
        if (!fq29_is_zero_mod_p(dx)) { den = dx; return 0u; }
        const Fq29 y2 = fq29_dbl(b.y);
        if (fq29_is_zero_mod_p(y2)) return 5u;
        den = y2;
        return fq29_is_zero_mod_p(fq29_sub(a.y, b.y)) ? 1u : 2u;
    };
    Fq29 run = fq29_one();
    uint32_t count = 0;
    for (uint32_t q = base; count < per_lane && q < n; q += GT, ++count) {
        const At p = at(q);
        Fq29 den;
        (void)kind_of(p.row[p.i - 1], p.row[p.c - 1], den);
        p.row[(p.c + p.i <= p.t ? p.c + p.i : p.c - p.i) - 1].x = run;
        run = fq29_mul_inline(run, den);
    }
    Fq29 inv = fq29_inverse(run);
    while (count-- > 0) {
        const At p = at(base + count * GT);
        const A29 a = p.row[p.i - 1], b = p.row[p.c - 1];
        const bool up = p.c + p.i <= p.t, down = p.c - p.i > p.h;
        Fq29 den;
        const uint32_t kind = kind_of(a, b, den);
        const Fq29 di = fq29_mul_inline(inv, p.row[(up ? p.c + p.i : p.c - p.i) - 1].x);
        inv = fq29_mul_inline(inv, den);
        // coordinates back to (-eps, p + eps): they must not grow with the table
        auto x_of = [&](const Fq29& l) { return fq29_lift(fq29_lift(fq29_sub(fq29_sub(fq29_sqr_inline(l), a.x), b.x))); };
        A29 twice = b;                                      // of equal or opposite points: twice the centre
        if (kind == 1u || kind == 2u) {
            const Fq29 xx = fq29_sqr(b.x), l = fq29_mul(fq29_add(fq29_dbl(xx), xx), di);
            twice.x = x_of(l);
            twice.y = fq29_lift(fq29_sub(fq29_mul(l, fq29_sub_raw(b.x, twice.x)), b.y));
        }
        if (up) {
            const Fq29 l = fq29_mul_inline(fq29_sub_raw(a.y, b.y), di);
            A29 r;
            r.x = x_of(l);
            r.y = fq29_lift(fq29_sub(fq29_mul_inline(l, fq29_sub_raw(a.x, r.x)), a.y));
            if (kind == 1u) r = twice;
            if (kind == 3u) r = a;
            if (kind == 4u) r = b;
            if (kind == 2u || kind == 5u) { r.x = fq29_zero(); r.y = fq29_zero(); }
            p.row[p.c + p.i - 1] = r;
        }
        if (down) {          // the centre and entry i's opposite
            const Fq29 l = fq29_mul_inline(fq29_add(a.y, b.y), di);
            A29 r;
            r.x = x_of(l);
            r.y = fq29_lift(fq29_add(fq29_mul_inline(l, fq29_sub_raw(r.x, a.x)), a.y));
            if (kind == 2u) r = twice;
            if (kind == 3u) { r.x = a.x; r.y = fq29_lift(fq29_neg(a.y)); }
            if (kind == 4u) r = b;
            if (kind == 1u || kind == 5u) { r.x = fq29_zero(); r.y = fq29_zero(); }
            p.row[p.c - p.i - 1] = r;
        }
    }
}
static constexpr int P29_WORDS = 42;
static_assert(sizeof(P29) == 4 * P29_WORDS, "a point is its coordinates");
__device__ __forceinline__ P29 p29_shfl(const P29& a, int lane) {
    P29 r;
    const int32_t* src = reinterpret_cast<const int32_t*>(&a);
    int32_t* dst = reinterpret_cast<int32_t*>(&r);
#pragma unroll
    for (int l = 0; l < P29_WORDS; ++l) dst[l] = __shfl(src[l], lane, 64);
    return r;
}
// Sums of [s_j] G_j over segments of the rows (item = segment * m + row, so that a wave's items use the same part of the table), to
// out[row], or to part[row * nseg + segment] where rows have several.  Sixteen lanes take an item, four items a wave.
// The scalars' non-zero digits go through a list in LDS, sixteen scalars at a time, and an addition starts when every item of the wave
// has sixteen: where the second digit of most scalars is zero, lanes that each walked their own scalar's digits would wait for the one
// in sixty-four that is not.  Sixteen lanes and not the whole wave, because a sum over the lanes of one row is serial: five additions on four lanes
// (four levels of Jacobian additions on a lane: 300 rows of 4096 generators 1.67 ms, with k_msm_parts as it is now 1.24).
// Instruction issue binds it (two waves a SIMD).  11008 rows of 4096 14-bit scalars: 7-bit signed digits of the whole wave's lanes, in
// Jacobian coordinates, took 17.7 ms; 12-bit digits this way take less than half.
static constexpr uint32_t MSM_CAP = 256;
__global__ void __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_msm_rows(G1Jac* __restrict__ out, P29* __restrict__ part, const MsmTable T, const int32_t* __restrict__ scalars, size_t m_rows, uint32_t nseg, uint32_t per) {
    __shared__ uint32_t list[4][MSM_CAP];
    __shared__ int32_t sums[P29_WORDS][GT];
    const uint32_t t = threadIdx.x, grp = t >> 4, ln = t & 15u;
    const size_t item = (size_t)blockIdx.x * 4 + grp;
    const bool valid = item < m_rows * nseg;
    const size_t seg = valid ? item / m_rows : 0, row = valid ? item - seg * m_rows : 0, j0 = valid ? seg * per : 0;
    const size_t j1 = valid ? (j0 + per < T.ngen ? j0 + per : T.ngen) : 0;
    const int32_t* src = scalars + row * T.ngen;
    uint32_t cnt = 0;
    X29 acc = x29_infinity();
    const uint32_t room = MSM_CAP - 16u * T.nwin, steps = (per + 15u) / 16u;
    auto least = [&] {
        const int v = valid ? (int)cnt : 0x7fffffff;
        return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)), min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
    };
    auto most = [&] {
        const int v = (int)cnt;
        return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)), max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
    };
    int32_t s_next = j0 + ln < j1 ? src[j0 + ln] : 0;
    for (uint32_t step = 0; step <= steps; ++step) {
        if (step < steps) {
            const size_t j = j0 + (size_t)step * 16u + ln;
            const int32_t s = s_next;
            s_next = j + 16u < j1 ? src[j + 16u] : 0;
            const bool negs = s < 0;
            uint64_t x = negs ? (uint64_t)(-(int64_t)s) : (uint64_t)s;
            for (uint32_t w = 0; w < T.nwin; ++w) {
                if (__ballot(x != 0) == 0ull) break;
                int32_t d = (int32_t)(x & (((uint64_t)1 << T.c) - 1));
                x >>= T.c;
                if (d > (int32_t)T.half && w + 1 < T.nwin) { d -= (int32_t)(1u << T.c); x += 1; }
                const uint32_t m = (uint32_t)(__ballot(d != 0) >> (16u * grp)) & 0xFFFFu;
                if (d != 0) list[grp][cnt + __popc(m & ((1u << ln) - 1u))] = (uint32_t)msm_slot(T, w, j, (uint32_t)(d < 0 ? -d : d)) | ((d < 0) != negs ? 0x80000000u : 0u);
                cnt += __popc(m);
            }
        }
        __syncthreads();
        const bool drain = step == steps;
        for (;;) {
            const int mx = most();
            if (drain ? mx == 0 : !(least() >= 16 || mx > (int)room)) break;
            const uint32_t take = cnt < 16u ? cnt : 16u;
            cnt -= take;
            if (ln < take) {
                const uint32_t e = list[grp][cnt + ln];
                A29 p = T.tab[e & 0x7FFFFFFFu];
                if (!a29_is_inf(p)) {
                    if (e >> 31) p.y = fq29_neg(p.y);
                    x29_add_mixed(acc, p);
                }
            }
        }
        __syncthreads();
    }
    P29 r = p29_from_x29(acc);
    {
        const int32_t* w = reinterpret_cast<const int32_t*>(&r);
#pragma unroll
        for (int l = 0; l < P29_WORDS; ++l) sums[l][t] = w[l];
    }
    __syncthreads();
    auto get = [&](uint32_t lane) {
        P29 o;
        int32_t* w = reinterpret_cast<int32_t*>(&o);
#pragma unroll
        for (int l = 0; l < P29_WORDS; ++l) w[l] = sums[l][lane];
        return o;
    };
    r = get(t & 60u);
    for (uint32_t step = 0; step < 5; ++step) {             // a quad's other three lanes, then the item's other quads
        const P29 o = step < 3 ? get((t & 60u) + step + 1) : p29_shfl(r, (int)(t ^ (step == 3 ? 4u : 8u)));
        p29_quad_add(r, o, t & 3u);
    }
    if (valid && ln == 0) {
        if (nseg > 1) part[row * nseg + seg] = r;
        else out[row] = p29_to_jac(r);
    }
}
// out[row] = the sum of row's nseg parts, 2^lg <= nseg groups of four lanes a row.  A chain of additions that nothing else runs beside: one after another
// on one lane, sixteen parts took 410 us of the 880 that
// committing 20 rows of 512 generators took; now the whole of it takes 454.
__global__ void __launch_bounds__(GT) k_msm_parts(G1Jac* __restrict__ out, const P29* __restrict__ part, size_t m_rows, uint32_t nseg, uint32_t lg) {
    const uint32_t t = threadIdx.x, groups = 1u << lg;
    const size_t at = (size_t)blockIdx.x * (GT / 4) + (t >> 2), row = at >> lg;
    const uint32_t g = (uint32_t)at & (groups - 1u), own = nseg >> lg;
    const P29* __restrict__ P = part + (row < m_rows ? row : 0) * nseg + g;
    P29 r = P[0];
    for (uint32_t step = 1; step < own + lg; ++step) {
        const P29 o = step < own ? P[(size_t)step << lg] : p29_shfl(r, (int)(t ^ (4u << (step - own))));
        p29_quad_add(r, o, t & 3u);
    }
    if (row < m_rows && g == 0 && (t & 3u) == 0) out[row] = p29_to_jac(r);
}
// out[i] = [s_i] B for one base point B: additions out of the table of B's multiples d * 2^(8w) B, d = 1..128, w = 0..32
// (signed 8-bit digits of the 256-bit integer s_i; window 32 only ever holds the last carry).  33 mixed additions at
// most instead of 255 doublings and ~128 additions.
static constexpr uint32_t FB_WIN = 33;
__global__ void __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_g1_fixed_base_mul(G1Jac* __restrict__ out, const A29* __restrict__ tab, const Fr* __restrict__ scalars, size_t n) {
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    if (i >= n) return;
    const Fr x = scalars[i];
    X29 acc29 = x29_infinity();
    uint32_t carry = 0;
    for (uint32_t w = 0; w < FB_WIN; ++w) {
        const uint32_t b = (w < 32 ? ((x.v[w >> 2] >> (8 * (w & 3))) & 255u) : 0u) + carry;
        carry = b > 128u ? 1u : 0u;
        const uint32_t mag = carry ? 256u - b : b;
        if (mag == 0) continue;
        A29 p = tab[w * 128u + (mag - 1)];
        if (a29_is_inf(p)) continue;
        if (carry) p.y = fq29_neg(p.y);
        x29_add_mixed(acc29, p);
    }
    out[i] = j29_to_jac(j29_from_x29(acc29));
}
// stats[0]: raised when an element is not the embedding of an int32, [1]: largest magnitude, [2 + b]: of the elements looked at (one in
// CONV_SAMPLE), those whose magnitude has b bits.  Eight elements a lane in flight: one a lane and an atomic a workgroup ran at 0.8 TB/s; the words looked at
// instead of the embedding formed again, and one round of workgroups at four waves a SIMD: 45 million elements 425 -> 338 us, 4.8 TB/s
static constexpr int CONV_SAMPLE = 8, CONV_STATS = 35, CONV_GRID = 1024;
__global__ void __launch_bounds__(256) k_fr_to_i32_checked(int32_t* __restrict__ out, uint32_t* __restrict__ stats, const Fr* __restrict__ in, size_t n) {
    __shared__ uint32_t wmax[4], wbad[4], hist[33];
    if (threadIdx.x < 33u) hist[threadIdx.x] = 0u;
    __syncthreads();
    uint32_t a = 0, bad = 0;
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i0 = (size_t)blockIdx.x * 256 + threadIdx.x; i0 < n; i0 += CONV_SAMPLE * stride) {
        Fr x[CONV_SAMPLE];
#pragma unroll
        for (int q = 0; q < CONV_SAMPLE; ++q) x[q] = i0 + q * stride < n ? in[i0 + q * stride] : big_zero<8>();
#pragma unroll
        for (int q = 0; q < CONV_SAMPLE; ++q) {
            // x itself, or r - |x|: the words from the third on are zero or r's (r's two low words leave 2^31 room, so nothing borrows from above)
            uint32_t high = 0, high_neg = 0;
#pragma unroll
            for (int l = 2; l < 8; ++l) { high |= x[q].v[l]; high_neg |= x[q].v[l] ^ FrK::P(l); }
            const uint64_t low = (uint64_t)x[q].v[1] << 32 | x[q].v[0], r_low = (uint64_t)FrK::P(1) << 32 | FrK::P(0);
            const uint64_t mag = high ? r_low - low : low;
            if (i0 + q * stride < n) out[i0 + q * stride] = (int32_t)(high ? 0u - (uint32_t)mag : (uint32_t)mag);
            bad |= (high ? high_neg == 0 && mag - 1 < 0x80000000ull : mag < 0x80000000ull) ? 0u : 1u;
            const uint32_t m = (uint32_t)mag;
            a = m > a ? m : a;
            if (q == 0) atomicAdd(&hist[m ? 32 - __clz((int)m) : 0], 1u);
        }
    }
    for (int off = 32; off >= 1; off >>= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)a, off, 64);
        a = o > a ? o : a;
        bad |= (uint32_t)__shfl_xor((int)bad, off, 64);
    }
    if ((threadIdx.x & 63u) == 0) { wmax[threadIdx.x >> 6] = a; wbad[threadIdx.x >> 6] = bad; }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t m = wmax[0];
        for (int k = 1; k < 4; ++k) { m = wmax[k] > m ? wmax[k] : m; bad |= wbad[k]; }
        if (m > __atomic_load_n(&stats[1], __ATOMIC_RELAXED)) atomicMax(&stats[1], m);
        if (bad | wbad[0]) atomicOr(&stats[0], 1u);
    }
    if (threadIdx.x < 33u && hist[threadIdx.x]) atomicAdd(&stats[2 + threadIdx.x], hist[threadIdx.x]);
}

// ---- opening (Commitment::me_open, commitment.cu:79-129) -------------------------------------------------------------
// A round of the opening halves the scalars s and the generators g with the challenge u,
//   s'_i = s_2i + u (s_2i+1 - s_2i),   g'_i = g_2i+1 + [u](g_2i - g_2i+1),
// and publishes T = sum [s_j] g_j, T0 = sum [s_2i] g_2i+1, T1 = sum [s_2i+1] g_2i.  The reference spends five
// 255-bit scalar multiplications per pair on this.  Here
//  * T0 and T1 (and T of the first round) are bucket multi-scalar multiplications over the affine-normalised
//    generators: signed windows of 8 to 12 bits, the elements sorted by bucket, one bucket per lane;
//  * T of every later round follows from the previous round's three points, because <s', g'> expands to
//    u(1-u) T + (1-u)^2 T0 + u^2 T1, or all T from the last round's result the other way round;
//  * the one remaining scalar multiplication per pair, by the round's common challenge u, uses the curve
//    endomorphism (x, y) -> (beta x, y) = [lambda](x, y): u = k1 + k2 lambda with k1, k2 < 2^128 (r = lambda^2 +
//    lambda + 1, so this is one integer division on the host), then 128 doublings instead of 255.
// The endomorphism and the expansion of T hold for points of the order-r subgroup, which is where the
// generators live (Commitment::random draws multiples of the group generator, commitment.cu:9-20).
// All rounds are queued without a host round trip; the proof points come back in one copy, normalised to z = 1.
static constexpr int MW = 32;        // bytes of a scalar split as k1 + k2 lambda: 16 of each half
static constexpr int MWH = MW / 2;
static constexpr int MT = 128;       // buckets that a wave of k_msm_windows reduces
static constexpr int MSL = 64;       // lanes of a bucket-accumulation workgroup (one wave)
static constexpr int MHB = 2048;     // most buckets of a window
static constexpr int MPIECE = 128;   // most elements of a bucket that one lane adds up
static constexpr int MFEWP = 8;      // most pieces that one lane puts together
// element i: recoded scalar i*s_mul+s_off of dstride, point base[i*b_mul+b_off]; list_at: the counts of the sums before this one
struct MsmDesc { const void* digits; const A29* base; uint32_t dstride, count, s_mul, s_off, b_mul, b_off, list_at, pad; };
// How scalars are written for their sums: nwh windows a half, the first 128 % nwh of them one bit wider than the rest (bias: a half of every
// window's range), or (nwh = 0) the bytes that k_msm_few reads
struct DigitPlan { uint32_t nwh, bias[4]; };
static inline size_t digit_bytes(const DigitPlan& p) { return p.nwh ? 4 * (size_t)p.nwh : (size_t)MW + 1; }       // of a scalar
static constexpr int OB_MAX = 8;           // openings of equal size that share their rounds' launches
static constexpr int TABLE_MIN_N = 1024;   // results of a fold below which no fold tables are made for it
static constexpr int LAST_N = 16384;       // generators of a job (all its openings together) at which the remaining rounds are computed in one batch
static constexpr int TAIL_LEVELS = 20;     // most rounds the batch takes
static constexpr int T_SUM_MAX_N = 8192;    // generators of a job's last batch up to which it sums its rounds' T itself
static constexpr int SPAN_MAX_N = 1 << 17; // generators of a job up to which three rounds are taken as a batch of sums beside one fold
struct GlvK { uint32_t k1[4], k2[4]; };

__device__ __forceinline__ bool aff_is_inf(const G1Affine& p) { return is_zero(p.x) && is_zero(p.y); }   // normalised infinity: all-zero limbs
__device__ __forceinline__ G1Jac aff_to_jac(const G1Affine& p) {
    G1Jac r;
    if (aff_is_inf(p)) return g1_infinity();
    r.x = p.x; r.y = p.y; r.z = big_one_mont<12>();
    return r;
}
// beta (Montgomery form): the cube root of unity in Fp with (beta x, y) = [lambda](x, y), lambda = 0xac45a4010001a40200000000ffffffff
__device__ __forceinline__ Fp glv_beta() {
    Fp b;
    constexpr uint32_t t[12] = {2255614065u, 3439577572u, 533571026u, 1571496518u, 3548715925u, 1483752111u, 29019038u, 2394295998u, 2211467474u, 66682222u, 1415808833u, 418390117u};
#pragma unroll
    for (int i = 0; i < 12; ++i) b.v[i] = t[i];
    return b;
}
__device__ __forceinline__ Fp glv_beta2() {   // beta^2 = -1 - beta
    Fp b;
    constexpr uint32_t t[12] = {2039112936u, 821114395u, 2127452714u, 4088978859u, 3323295735u, 380160570u, 1962738331u, 3261739000u, 1617960046u, 909555558u, 605774176u, 85697707u};
#pragma unroll
    for (int i = 0; i < 12; ++i) b.v[i] = t[i];
    return b;
}
__device__ __forceinline__ Fp glv_minus2_over_beta_minus_1() {   // -2 / (beta - 1), Montgomery form
    Fp b;
    constexpr uint32_t t[12] = {72385493u, 4027593027u, 4077721914u, 4036542869u, 1636888181u, 235204061u, 17598343u, 35324347u, 360752738u, 1434563812u, 3508079257u, 43087383u};
#pragma unroll
    for (int i = 0; i < 12; ++i) b.v[i] = t[i];
    return b;
}
// joint sparse form of (k1, k2): position i holds (d1 + 1) | (d2 + 1) << 2 in 4 bits, d in {-1, 0, 1}; len <= 129
struct JsfK { uint32_t dig[17]; uint32_t len; };
// [k1]P + [k2]phi(P); every lane of a wave must carry the same k (the add pattern is uniform)
static __device__ __attribute__((noinline)) G1Jac g1_mul_glv(const G1Jac& P, const GlvK& k) {
    if (is_zero(P.z)) return P;
    G1Jac Q = P;
    Q.x = fp_mul(P.x, glv_beta());
    const G1Jac PQ = g1_add(P, Q);
    int top = -1;
    for (int i = 3; i >= 0 && top < 0; --i) {
        const uint32_t x = k.k1[i] | k.k2[i];
        if (x) top = i * 32 + 31 - __builtin_clz(x);
    }
    G1Jac out = g1_infinity();
    for (int i = top; i >= 0; --i) {
        out = g1_double(out);
        const uint32_t b = ((k.k1[i >> 5] >> (i & 31)) & 1u) | (((k.k2[i >> 5] >> (i & 31)) & 1u) << 1);
        if (b == 1) out = g1_add(out, P);
        else if (b == 2) out = g1_add(out, Q);
        else if (b == 3) out = g1_add(out, PQ);
    }
    return out;
}

// Signed digits of every scalar, written window-major: the scalar is split as +-k1 +-k2 lambda with |k1|, |k2| < 2^127
// ([lambda](x, y) = (beta x, y), see glv_beta).  The halves share the points they are summed over;
// what the split buys is the end of a sum, whose Horner walk over the windows is about 117 doublings instead of 248.
// The smaller of s and r - s is split (weights are embedded as small values of either sign: a value below lambda / 2 is its own k1,
// and its high windows are empty).
// A plan of nwh windows a half: D (int16) [w*n + i] is digit w of +-k1 for w < nwh and digit w - nwh of +-k2 above.  With half of every
// window's range added to |k| beforehand, the digits are bits of that sum less the half range, without carries from window to window:
// |k| is at most 2^126.44 and the halves together below 2^127.02, so the sum has 128 bits.
// The bytes of k_msm_few: D[w*n + i] in [-128, 127] is digit w of |k1| for w < MWH and digit w - MWH of |k2| above, and D[MW*n + i] says
// which halves are subtracted (bit 0: k1, bit 1: k2).  A window byte above 127 becomes byte - 256 and carries one into the next window; the
// top byte of a half is at most 0x57, so the carry ends there.
struct RecodeBatch { void* D[OB_MAX]; const Fr* S[OB_MAX]; };      // blockIdx.y names the pair
// a = round(x / lambda) and k1 = x - a lambda for x < 2^254: the quotient's estimate is the high half of x times 2^256 / lambda, at
// most one short, and the remainder's comparison with lambda / 2 mends it.  k1 comes as magnitude and sign.
__device__ __forceinline__ void glv_split_centred(const uint32_t* x, uint32_t (&k1)[4], bool& k1_neg, uint32_t (&a)[4]) {
    constexpr uint32_t MU[5] = {0xf6cfee30u, 0x63f6e522u, 0xe01faaddu, 0x7c6becf1u, 1u};          // floor(2^256 / lambda)
    constexpr uint32_t LAM[4] = {0xffffffffu, 0u, 0x0001a402u, 0xac45a401u};
    uint32_t p[13];
#pragma unroll
    for (int i = 0; i < 13; ++i) p[i] = 0;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        uint64_t c = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            c += (uint64_t)MU[i] * x[j] + p[i + j];
            p[i + j] = (uint32_t)c;
            c >>= 32;
        }
        p[i + 8] = (uint32_t)c;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = p[8 + i];
    // rem = x - a lambda, in [0, 2 lambda): five limbs hold it
    uint32_t q[5], rem[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) q[i] = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint64_t c = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (i + j > 4) break;
            c += (uint64_t)a[i] * LAM[j] + q[i + j];
            q[i + j] = (uint32_t)c;
            c >>= 32;
        }
        if (i == 0) q[4] = (uint32_t)c;
    }
    uint32_t br = 0;
#pragma unroll
    for (int i = 0; i < 5; ++i) rem[i] = subb32(x[i], q[i], br);
    // above lambda / 2 (0x5622d200.8000d201.00000000.7fffffff): one more lambda off; twice when the estimate was short
    constexpr uint32_t HALF[5] = {0x7fffffffu, 0u, 0x8000d201u, 0x5622d200u, 0u};
    bool negative = false;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        uint32_t lt = 0, b2 = 0, c = 0;
#pragma unroll
        for (int i = 0; i < 5; ++i) (void)subb32(HALF[i], rem[i], lt);
        const bool more = lt != 0 && !negative;                     // rem > lambda / 2
#pragma unroll
        for (int i = 0; i < 5; ++i) rem[i] = subb32(rem[i], more && i < 4 ? LAM[i] : 0u, b2);
        a[0] = addc32(a[0], more ? 1u : 0u, c);
#pragma unroll
        for (int i = 1; i < 4; ++i) a[i] = addc32(a[i], 0u, c);
        negative = (rem[4] >> 31) != 0;
    }
    k1_neg = negative;
    uint32_t b3 = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t n = subb32(0u, rem[i], b3);
        k1[i] = negative ? n : rem[i];
    }
}
// the digits of scalar i of n (standard form)
__device__ __forceinline__ void msm_recode_store(void* __restrict__ Dv, size_t n, size_t i, const Fr& sv, const DigitPlan& plan) {
    Fr ng;
    uint32_t br = 0;
#pragma unroll
    for (int l = 0; l < 8; ++l) ng.v[l] = subb32(FrK::P(l), sv.v[l], br);
    uint32_t lt = 0;    // borrow of (r - s) - s: r - s is the smaller one
#pragma unroll
    for (int l = 0; l < 8; ++l) (void)subb32(ng.v[l], sv.v[l], lt);
    const bool flip = lt != 0;
    uint32_t x[8], k1[4], k2[4];
    bool neg1;
#pragma unroll
    for (int l = 0; l < 8; ++l) x[l] = flip ? ng.v[l] : sv.v[l];
    glv_split_centred(x, k1, neg1, k2);
    if (plan.nwh) {
        int16_t* __restrict__ D = reinterpret_cast<int16_t*>(Dv);
        const uint32_t q = 128u / plan.nwh, rem = 128u % plan.nwh;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool neg = h ? flip : flip != neg1;
            uint32_t v[4], c = 0;
#pragma unroll
            for (int l = 0; l < 4; ++l) v[l] = addc32(h ? k2[l] : k1[l], plan.bias[l], c);
            for (uint32_t w = 0; w < plan.nwh; ++w) {
                const uint32_t width = q + (w < rem ? 1u : 0u), range = 1u << width;
                const int dg = (int)(v[0] & (range - 1u)) - (int)(range >> 1);
                D[(size_t)(h * plan.nwh + w) * n + i] = (int16_t)(neg ? -dg : dg);
#pragma unroll
                for (int l = 0; l < 3; ++l) v[l] = v[l] >> width | v[l + 1] << (32u - width);
                v[3] >>= width;
            }
        }
        return;
    }
    int8_t* __restrict__ D = reinterpret_cast<int8_t*>(Dv);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t carry = 0;
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const uint32_t word = h ? k2[l] : k1[l];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t raw = ((word >> (8 * q)) & 0xFFu) + carry;
                carry = raw > 127u ? 1u : 0u;
                D[(size_t)(h * MWH + 4 * l + q) * n + i] = (int8_t)(raw > 127u ? (int)raw - 256 : (int)raw);
            }
        }
    }
    D[(size_t)MW * n + i] = (int8_t)((flip != neg1 ? 1 : 0) | (flip ? 2 : 0));
}
// What the sums behind a recoding count with (SortState), cleared by its first workgroup
__device__ __forceinline__ void clear_state(uint32_t* __restrict__ state, uint32_t words) {
    if (blockIdx.x == 0 && blockIdx.y == 0)
        for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) state[i] = 0u;
}
__global__ void __launch_bounds__(GT) k_msm_recode(const RecodeBatch rb, size_t n, const DigitPlan plan, uint32_t* __restrict__ state, uint32_t state_words) {      // one wave a workgroup: as k_tail_levels
    urgent();
    clear_state(state, state_words);
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    if (i >= n) return;
    msm_recode_store(rb.D[blockIdx.y], n, i, rb.S[blockIdx.y][i], plan);
}

// The end of a list of points in bucket order that a wave's lanes have divided evenly (lane t the t-th share).  x: the sum of the last part of
// the lane's share, which belongs to bucket b; begun: the bucket begins in this share (or the share is empty); whole: it ends with this
// share; lacks: bucket `split`, the first part's, went out already without the shares before this one.  A segmented inclusive scan, as
// long as a bucket spans further lanes, then the sums to `out`.  All lanes call it; pool: 42 x 64 words.
__device__ __forceinline__ void bucket_shares_merge(uint32_t* pool, P29 x, bool begun, bool whole, uint32_t b, bool lacks, uint32_t split, P29* __restrict__ out, uint32_t t) {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(&x);
    for (uint32_t sd = 1; sd < (uint32_t)MSL && !__all(begun); sd <<= 1) {
        __syncthreads();
#pragma unroll
        for (int l = 0; l < P29_WORDS; ++l) pool[l * MSL + t] = src[l];
        __syncthreads();
        const bool before = __shfl_up(begun ? 1 : 0, sd) != 0;
        if (t >= sd && !begun) {
            P29 y;
            uint32_t* py = reinterpret_cast<uint32_t*>(&y);
#pragma unroll
            for (int l = 0; l < P29_WORDS; ++l) py[l] = pool[l * MSL + t - sd];
            x = p29_add<false>(x, y);
            begun = before;
        }
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < P29_WORDS; ++l) pool[l * MSL + t] = src[l];
    __syncthreads();
    if (whole) out[b] = x;
    if (lacks) {
        P29 y;
        uint32_t* py = reinterpret_cast<uint32_t*>(&y);
#pragma unroll
        for (int l = 0; l < P29_WORDS; ++l) py[l] = pool[l * MSL + t - 1];
        out[split] = p29_add<false>(out[split], y);
    }
}

// Bucket sums, [(sum * 2 nwh + w) * hb + b] for magnitude b + 1 of window w of a sum, in four launches over the windows w0 .. w0 + gridDim.x - 1:
//  1. k_msm_sort: a workgroup a window sorts the sum's elements by bucket (counting sort in LDS) into one list in memory, the point's index and
//     the digit's sign an entry, and counts the buckets by size.  A bucket above `most` elements (scalars that share a digit: equal values,
//     small integers) is cut into pieces of equal size.
//  2. k_msm_tasks: the buckets and pieces of ALL sums and windows ordered by size, the longest first.
//  3. k_msm_lists: a lane adds up the points of one bucket or piece.  The 64 of a wave are of one size, so its lanes are busy to the end, and
//     the waves get shorter towards the end of the launch, so that the chip empties at once.
//  4. k_msm_merge: a lane puts the pieces of a bucket together, a wave those of a bucket in many.
// Bound by the instructions of 3.  That the lists lie in memory is what lets windows be wider than 8 bits (22 additions an element with 11 windows a half instead
// of 32).  The sums of an opening of 128 x 131072 alone: 0.20 ms of sorting and 2.3 ms of k_msm_lists at 76 % of the issue slots; with 8-bit windows, a wave for the 128 buckets of a chunk and
// a window sorted in LDS, and the chunks' buckets added up, 5.5 + 0.3 ms at 66 %: the whole opening 8.7 -> 6.8 ms, of 16 x 4096 2.19 -> 1.45 ms.
static constexpr uint32_t SORT_CURSOR = MPIECE + 1, SORT_PARTS = 2 * (MPIECE + 1), SORT_CUT = SORT_PARTS + 1, SORT_HEAVY = SORT_CUT + 1, SORT_WORDS = SORT_HEAVY + 1;
// what the four launches share; state: tasks of each size, how many of a size are placed, pieces, cut buckets
// heavy: buckets of few pieces from the front, those of more than MFEWP from the back of `cuts` entries
struct SortSpace { uint32_t* state; uint4* info; uint32_t* lists; uint4* heavy; uint4* tasks; P29* buckets; uint32_t nwh, hb, w0, total, most, parts_at, cuts; };
__device__ __forceinline__ uint32_t sort_wave_scan(uint32_t v, uint32_t lane) {      // inclusive
    for (int sd = 1; sd < 64; sd <<= 1) {
        const uint32_t a = __shfl_up(v, sd);
        if (lane >= (uint32_t)sd) v += a;
    }
    return v;
}
template <int BT> __global__ void __launch_bounds__(BT) k_msm_sort(const SortSpace sp, const MsmDesc* __restrict__ descs) {
    urgent();
    __shared__ uint32_t cursor[MHB], sizes[MPIECE + 1], wave_sum[3][BT / 64], at_part, at_cut, at_heavy;
    constexpr int AHEAD = 8;
    const MsmDesc d = descs[blockIdx.y];
    const uint32_t t = threadIdx.x, w = sp.w0 + blockIdx.x, row = blockIdx.y * 2 * sp.nwh + w, list0 = blockIdx.x * sp.total + d.list_at;
    const int16_t* __restrict__ Dw = reinterpret_cast<const int16_t*>(d.digits) + (size_t)w * d.dstride + d.s_off;
    for (uint32_t b = t; b < sp.hb; b += BT) cursor[b] = 0;
    for (uint32_t b = t; b <= (uint32_t)MPIECE; b += BT) sizes[b] = 0;
    __syncthreads();
    for (uint32_t e = t; e < d.count; e += BT * AHEAD) {
        int dg[AHEAD];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) dg[k] = e + k * BT < d.count ? (int)Dw[(size_t)(e + k * BT) * d.s_mul] : 0;
#pragma unroll
        for (int k = 0; k < AHEAD; ++k)
            if (dg[k] != 0) atomicAdd(&cursor[(dg[k] < 0 ? -dg[k] : dg[k]) - 1], 1u);
    }
    __syncthreads();
    const uint32_t per = (sp.hb + BT - 1) / BT, b0 = min(t * per, sp.hb), b1 = min(b0 + per, sp.hb);
    uint32_t mine = 0, parts = 0, cuts = 0;                 // elements, pieces, cut buckets and above bit 16 those of more than MFEWP pieces
    for (uint32_t b = b0; b < b1; ++b) {
        const uint32_t c = cursor[b], np = (c + sp.most - 1) / sp.most;
        mine += c;
        if (np > 1) { parts += np; cuts += np > (uint32_t)MFEWP ? 0x10000u : 1u; }
    }
    uint32_t run = sort_wave_scan(mine, t & 63u), run_parts = sort_wave_scan(parts, t & 63u), run_cuts = sort_wave_scan(cuts, t & 63u);
    if ((t & 63u) == 63u) { wave_sum[0][t >> 6] = run; wave_sum[1][t >> 6] = run_parts; wave_sum[2][t >> 6] = run_cuts; }
    __syncthreads();
    run -= mine; run_parts -= parts; run_cuts -= cuts;
    for (uint32_t k = 0; k < t >> 6; ++k) { run += wave_sum[0][k]; run_parts += wave_sum[1][k]; run_cuts += wave_sum[2][k]; }
    if (t == BT - 1 && run_parts + parts) {
        const uint32_t c = run_cuts + cuts;
        at_part = atomicAdd(&sp.state[SORT_PARTS], run_parts + parts);
        at_cut = atomicAdd(&sp.state[SORT_CUT], c & 0xFFFFu);
        at_heavy = atomicAdd(&sp.state[SORT_HEAVY], c >> 16);
    }
    __syncthreads();
    for (uint32_t b = b0; b < b1; ++b) {
        const uint32_t c = cursor[b], np = (c + sp.most - 1) / sp.most, at = row * sp.hb + b;
        uint32_t slot = 0;
        cursor[b] = run;
        if (np == 1) atomicAdd(&sizes[c], 1u);
        else if (np > 1) {
            const uint32_t len = c / np, more = c % np;
            if (more) atomicAdd(&sizes[len + 1], more);
            atomicAdd(&sizes[len], np - more);
            const bool many = np > (uint32_t)MFEWP;
            slot = at_part + run_parts;
            sp.heavy[many ? sp.cuts - 1 - (at_heavy + (run_cuts >> 16)) : at_cut + (run_cuts & 0xFFFFu)] = make_uint4(at, sp.parts_at + slot, np, 0u);
            run_parts += np;
            run_cuts += many ? 0x10000u : 1u;
        } else sp.buckets[at] = p29_infinity();
        sp.info[at] = make_uint4(list0 + run, c, sp.parts_at + slot, 0u);
        run += c;
    }
    __syncthreads();
    if (t <= (uint32_t)MPIECE && sizes[t]) atomicAdd(&sp.state[t], sizes[t]);
    for (uint32_t e = t; e < d.count; e += BT * AHEAD) {
        int dg[AHEAD];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) dg[k] = e + k * BT < d.count ? (int)Dw[(size_t)(e + k * BT) * d.s_mul] : 0;
#pragma unroll
        for (int k = 0; k < AHEAD; ++k)
            if (dg[k] != 0) sp.lists[list0 + atomicAdd(&cursor[(dg[k] < 0 ? -dg[k] : dg[k]) - 1], 1u)] = ((e + k * BT) * d.b_mul + d.b_off) | (dg[k] < 0 ? 0x80000000u : 0u);
    }
}
static constexpr int TASK_T = 256;
static_assert(TASK_T > MPIECE, "a lane for every size");
__global__ void __launch_bounds__(TASK_T) k_msm_tasks(const SortSpace sp) {
    urgent();
    __shared__ uint32_t all[MPIECE + 1], at[MPIECE + 1], own[MPIECE + 1];
    const uint32_t t = threadIdx.x, row = blockIdx.y * 2 * sp.nwh + sp.w0 + blockIdx.x;
    const uint4* __restrict__ info = sp.info + (size_t)row * sp.hb;
    if (t <= (uint32_t)MPIECE) { all[t] = sp.state[t]; own[t] = 0; }
    __syncthreads();
    for (uint32_t b = t; b < sp.hb; b += TASK_T) {
        const uint32_t c = info[b].y, np = (c + sp.most - 1) / sp.most;
        if (np == 0) continue;
        const uint32_t len = c / np, more = c % np;
        if (more) atomicAdd(&own[len + 1], more);
        atomicAdd(&own[len], np - more);
    }
    __syncthreads();
    if (t <= (uint32_t)MPIECE && own[t]) {
        uint32_t before = 0;
        for (uint32_t l = t + 1; l <= (uint32_t)MPIECE; ++l) before += all[l];
        at[t] = before + atomicAdd(&sp.state[SORT_CURSOR + t], own[t]);
        own[t] = 0;
    }
    __syncthreads();
    for (uint32_t b = t; b < sp.hb; b += TASK_T) {
        const uint4 in = info[b];
        const uint32_t np = (in.y + sp.most - 1) / sp.most;
        if (np == 0) continue;
        const uint32_t len = in.y / np, more = in.y % np;
        uint32_t from = in.x;
        for (uint32_t p = 0; p < np; ++p) {
            const uint32_t l = len + (p < more ? 1u : 0u);
            sp.tasks[at[l] + atomicAdd(&own[l], 1u)] = make_uint4(from, l, np == 1 ? row * sp.hb + b : in.z + p, blockIdx.y);
            from += l;
        }
    }
}
__global__ void __launch_bounds__(MSL) __attribute__((amdgpu_waves_per_eu(2, 2))) k_msm_lists(const SortSpace sp, const MsmDesc* __restrict__ descs) {
    const uint32_t t = threadIdx.x, id = blockIdx.x * MSL + t;
    uint32_t n = 0;                                         // tasks
    for (uint32_t l = t; l <= (uint32_t)MPIECE; l += MSL) n += sp.state[l];
    for (int sd = 1; sd < MSL; sd <<= 1) n += __shfl_xor(n, sd);
    if (id >= n) return;
    const uint4 task = sp.tasks[id];
    const A29* __restrict__ A = descs[task.w].base;
    const uint32_t* __restrict__ list = sp.lists + task.x;
    // an entry is sent for two additions ahead, its point one
    uint32_t en = list[0], en2 = list[min(1u, task.y - 1)];
    A29 next = A[en & 0x7FFFFFFFu];
    X29 acc;
    for (uint32_t i = 0; i < task.y; ++i) {
        A29 pt = next;
        if (en >> 31) pt.y = fq29_neg(pt.y);
        if (i + 1 < task.y) {
            en = en2;
            next = A[en & 0x7FFFFFFFu];
            en2 = list[min(i + 2, task.y - 1)];
        }
        if (i == 0) {
            acc.x = pt.x; acc.y = pt.y;
            acc.zz = acc.zzz = fq29_one();
            acc.inf = a29_is_inf(pt) ? 1u : 0u;             // infinity stays infinity when its sign is changed
        } else if (!a29_is_inf(pt)) x29_add_mixed(acc, pt);
    }
    sp.buckets[task.z] = p29_from_x29(acc);
}
__global__ void __launch_bounds__(MSL) k_msm_merge(const SortSpace sp) {
    urgent();
    __shared__ uint32_t pool[P29_WORDS * MSL];
    const uint32_t t = threadIdx.x, n = sp.state[SORT_HEAVY], few = sp.state[SORT_CUT];
    for (uint32_t k = blockIdx.x * MSL + t; k < few; k += gridDim.x * MSL) {
        const uint4 h = sp.heavy[k];
        P29 x = sp.buckets[h.y];
        for (uint32_t p = 1; p < h.z; ++p) x = p29_add<false>(x, sp.buckets[h.y + p]);
        sp.buckets[h.x] = x;
    }
    for (uint32_t k = blockIdx.x; k < n; k += gridDim.x) {
        const uint4 h = sp.heavy[sp.cuts - 1 - k];
        const P29* __restrict__ part = sp.buckets + h.y;
        P29 x = t < h.z ? part[t] : p29_infinity();
        for (uint32_t p = t + MSL; p < h.z; p += MSL) x = p29_add<false>(x, part[p]);
        uint32_t* src = reinterpret_cast<uint32_t*>(&x);
        uint32_t sd = 1;
        while (sd < (uint32_t)MSL / 2 && 2 * sd < h.z) sd <<= 1;
        for (; sd > 0; sd >>= 1) {                          // lanes sd .. 2 sd - 1 to those below
            __syncthreads();
#pragma unroll
            for (int l = 0; l < P29_WORDS; ++l) pool[l * MSL + t] = src[l];
            __syncthreads();
            if (t < sd) {
                P29 y;
                uint32_t* py = reinterpret_cast<uint32_t*>(&y);
#pragma unroll
                for (int l = 0; l < P29_WORDS; ++l) py[l] = pool[l * MSL + t + sd];
                x = p29_add<false>(x, y);
            }
        }
        if (t == 0) sp.buckets[h.x] = x;
    }
}
// Bucket sums of few elements: the 8-bit digits taken as two signed 4-bit digits each, so that a sum has 512 buckets (64 windows
// of 8) instead of 4096 and the walk over its buckets, which is most of such a sum's work, fits two waves instead of sixteen.  A wave
// takes nw windows, sorts their elements by bucket in LDS and divides that list evenly over its lanes, whatever the digits are.
// nw (8 up to 64 elements, 4 up to 128, else 2) gives a lane about eight elements, so that the scan behind them costs less than they do.
// FEW_MAX: an element costs 64 additions here and 32 there, a sum 512 buckets here and 4096 there; an opening of 8 x 512 alone takes
// 1.00 ms here, 0.93 sorted, one of 4 x 256 0.91 here.
static constexpr int FEW_MAX = 256, FEW_WINDOWS = 2 * MW, FEW_T = 8, FEW_BUCKETS = FEW_WINDOWS * FEW_T;
// grid (64 / nw, sums); buckets[(sum * 64 + window) * 8 + magnitude - 1]
__global__ void __launch_bounds__(MSL) __attribute__((amdgpu_waves_per_eu(2, 2))) k_msm_few(P29* __restrict__ buckets, const MsmDesc* __restrict__ descs, uint32_t nw) {
    __shared__ uint32_t cnt[MSL], off[MSL], cursor[MSL];
    __shared__ uint32_t pool[P29_WORDS * MSL];      // the sorted list (u16), then the points of the shares' scan
    static_assert(FEW_MAX <= 4096 && 8 * MSL * 2 <= P29_WORDS * MSL * 4 && 8 * FEW_T == MSL, "list entries, the pool and a lane for each bucket");
    uint16_t* list = reinterpret_cast<uint16_t*>(pool);
    const MsmDesc d = descs[blockIdx.y];
    const A29* __restrict__ A = d.base;
    const uint32_t t = threadIdx.x, v0 = blockIdx.x * nw, half = v0 / (FEW_WINDOWS / 2);
    const int8_t* __restrict__ D8 = reinterpret_cast<const int8_t*>(d.digits);
    const int8_t* __restrict__ Df = D8 + (size_t)MW * d.dstride;
    P29* __restrict__ out = buckets + ((size_t)blockIdx.y * FEW_WINDOWS + v0) * FEW_T;
    cnt[t] = 0;
    if (t < nw * FEW_T) out[t] = p29_infinity();
    __syncthreads();
    auto digit = [&](uint32_t v, size_t si) {
        const int dg = D8[(size_t)(v >> 1) * d.dstride + si], hi = (dg + 8) >> 4;
        return (v & 1u) ? hi : dg - 16 * hi;
    };
    for (uint32_t j = 0; j < nw; ++j)
        for (uint32_t e = t; e < d.count; e += MSL) {
            const int g = digit(v0 + j, (size_t)e * d.s_mul + d.s_off);
            if (g != 0) atomicAdd(&cnt[j * FEW_T + (g < 0 ? -g : g) - 1], 1u);
        }
    __syncthreads();
    uint32_t run = cnt[t];
    for (int sd = 1; sd < MSL; sd <<= 1) {
        const uint32_t a = __shfl_up(run, sd);
        if (t >= (uint32_t)sd) run += a;
    }
    off[t] = cursor[t] = run - cnt[t];
    const uint32_t total = __shfl(run, MSL - 1);
    __syncthreads();
    for (uint32_t j = 0; j < nw; ++j)
        for (uint32_t e = t; e < d.count; e += MSL) {
            const size_t si = (size_t)e * d.s_mul + d.s_off;
            const int g = digit(v0 + j, si);
            if (g == 0) continue;
            const uint32_t pos = atomicAdd(&cursor[j * FEW_T + (g < 0 ? -g : g) - 1], 1u);
            list[pos] = (uint16_t)(e | (((g < 0) != (((Df[si] >> half) & 1) != 0)) ? 0x8000u : 0u));
        }
    __threadfence_block();
    __syncthreads();
    if (total == 0) return;                                 // the same for every lane
    const uint32_t share = (total + MSL - 1) / MSL, p0 = min(t * share, total), p1 = min(p0 + share, total);
    uint32_t b = 0;                                         // the last bucket that begins at p0 or before: it holds entry p0, if there is one
    for (uint32_t sd = MSL / 2; sd > 0; sd >>= 1)
        if (off[b + sd] <= p0) b += sd;
    uint32_t b_end = off[b] + cnt[b], split = 0;
    bool start = p0 >= total || p0 == off[b], lacks = false;
    X29 acc29 = x29_infinity();
    for (uint32_t pos = p0; pos < p1; ++pos) {
        if (pos == b_end) {
            out[b] = p29_from_x29(acc29);
            if (!start) { split = b; lacks = true; start = true; }
            acc29 = x29_infinity();
            do ++b; while (cnt[b] == 0);
            b_end = off[b] + cnt[b];
        }
        const uint32_t en = list[pos];
        A29 pt = A[(size_t)(en & 0x7FFFu) * d.b_mul + d.b_off];
        if (a29_is_inf(pt)) continue;
        if (en & 0x8000u) pt.y = fq29_neg(pt.y);
        x29_add_mixed(acc29, pt);
    }
    bucket_shares_merge(pool, p29_from_x29(acc29), start, p1 > p0 && p1 == b_end, b, lacks, split, out, t);
}
// The sums of a list from the raw buckets of all their windows, in two launches, three for windows of more than 128 buckets.  k_msm_windows: a wave takes 128 buckets,
// sum_b (b + 1) B[b]: each four lanes the running sums over eight neighbouring buckets (fourteen additions), then a tree over the sixteen of them in which one
// of four lanes carries the weighted sum and one the plain sum times the buckets below it (eight additions).
// Wider windows: the weighted sums and 128 times the plain sums of their blocks of 128 (BLOCKS), then the same tree over those.  A sum of few elements has two sets of 8
// buckets a window, weighted 1 .. 8 and 16 .. 128: a wave takes eight of its windows.  k_msm_horner: four lanes walk the windows of a
// half, 128 doublings less the top window's width, and the halves are added, the endomorphism on the second.
// All of a job's sums that nothing waits for go into one launch each.  Both are chains of one wave's
// instructions; the windows are summed before the walk so that 32 waves and two walks of four lanes do what took 256 walks a sum.
// The list: sums of one number of windows stand together and begin at a multiple of eight (a wave of k_msm_horner; gaps: out = null), those of few elements last.
struct PointDesc { P29* buckets; P29* blocks; G1Jac* out; uint32_t few, nwh, hb, pad; };
// win[sum * MW + w]: the windows' sums.  grid: MW workgroups for each of the first `full` sums, then MW / 8 for each from first_few on, of few elements
// BLOCKS: grid (blocks of a sum, sums), the first of the list; blocks[2 (w * hb / MT + block)]: the two sums of a block
template <bool BLOCKS> __global__ void __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2))) k_msm_windows(P29* __restrict__ win, const PointDesc* __restrict__ list, uint32_t full, uint32_t first_few) {
    urgent();
    __shared__ int32_t pool[3][16][44];                     // of each four lanes: S, V, T below
    const uint32_t q = threadIdx.x & 3u, g = threadIdx.x >> 2;
    const bool few = !BLOCKS && blockIdx.x >= MW * full;               // the same for the workgroup
    const uint32_t at = few ? blockIdx.x - MW * full : blockIdx.x, per = few ? MW / 8 : MW;
    const uint32_t sum = BLOCKS ? blockIdx.y : (few ? first_few : 0u) + at / per;
    const PointDesc& desc = list[sum];
    const uint32_t w = BLOCKS ? blockIdx.x : (few ? at % per * 8 + g / 2 : at % per);      // BLOCKS: the block's number among all
    const uint32_t nblk = desc.hb / MT;
    if (desc.out == nullptr || (!few && w >= 2 * desc.nwh * (BLOCKS ? nblk : 1u))) return;
    const bool tree = !BLOCKS && !few && nblk > 1;
    const P29* __restrict__ B = desc.buckets + (few ? w * (2 * FEW_T) + (g & 1u) * FEW_T : w * MT + g * 8);
    enum : uint32_t { S = 0, V = 1, T = 2 };                // the running sum, the sum of the running sums, half a step of the tree
    auto get = [&](uint32_t slot, uint32_t of) {
        P29 r;
        int32_t* dst = reinterpret_cast<int32_t*>(&r);
#pragma unroll
        for (int l = 0; l < P29_WORDS; ++l) dst[l] = pool[slot][of & 15u][l];
        return r;
    };
    auto put = [&](uint32_t slot, const P29& v) {
        const int32_t* src = reinterpret_cast<const int32_t*>(&v);
        if (q == 0) {
#pragma unroll
            for (int l = 0; l < P29_WORDS; ++l) pool[slot][g][l] = src[l];
        }
    };
    P29 nxt = p29_infinity();
    if (tree) {
        const P29* __restrict__ b2 = desc.blocks + 2 * (size_t)(w * nblk + (g < nblk ? g : 0u));
        put(V, g < nblk ? b2[0] : nxt);
        put(S, g < nblk ? b2[1] : nxt);
    } else {
        const P29 top = B[7];
        put(S, top);
        put(V, top);
        nxt = B[6];
    }
    const uint32_t steps = few ? 19 : (tree ? 17 + 2 * (31 - __builtin_clz(nblk)) : 25);
    for (uint32_t step = tree ? 17 : 0; step < steps; ++step) {         // one addition, whatever it is for, so that its instructions are there once
        uint32_t xs, ys, yg = g, to;
        const bool odd = (g & 1u) != 0;
        bool bucket = false;
        if (step < 14) {
            bucket = !(step & 1u);
            xs = (step & 1u) ? V : S; ys = S; to = xs;
        } else if (step < (few ? 18u : 17u)) {              // eight times the plain sum; of few elements sixteen times the weighted one
            xs = ys = few && step == 14 ? V : S; to = S;
        } else if (few) {                                   // the upper set's to the lower's
            xs = V; ys = S; yg = g ^ 1u; to = V;
        } else {                                            // level k of the tree: the left half's first four lanes carry the weighted sum, its second the plain one
            const uint32_t k = (step - 17) >> 1;
            if (step & 1u) {
                xs = ys = k == 0 && odd ? S : V; yg = k == 0 ? g ^ 1u : g + (1u << k); to = T;
            } else {                                        // and the right half's plain sum to the weighted; the plain sum doubled
                xs = T; ys = odd ? T : (k == 0 ? S : V); yg = odd ? g : (k == 0 ? g ^ 1u : g + (1u << k) + 1u); to = V;
            }
        }
        __syncthreads();
        P29 x = get(xs, g), y;
        if (bucket) y = nxt;
        else {
            y = get(ys, yg);
            if (step < 13) nxt = B[5 - (step >> 1)];
        }
        p29_quad_add(x, y, q);
        put(to, x);
        if (step + 1 == steps && q == 0) {
            if constexpr (BLOCKS) {
                if (g < 2) desc.blocks[2 * (size_t)w + g] = x;
            } else if (few ? !odd : g == 0) win[(size_t)sum * MW + w] = x;
        }
    }
}
// The same for windows of 128 buckets of lists that fill the chip: a lane has eight neighbouring buckets and a wave four windows.  An addition takes
// 2700 instructions on four lanes and 5700 on one, so this takes half of them, but 340 to 390 us where a wave a window takes 150 alone: the proof of a small layer, with lists of 66 and 155 sums,
// takes 5.45 ms instead of 5.76 (medians of six).  Blocks of wider windows (2112 and 3016 waves of an opening of 131072 columns) gain nothing by it.
// grid: (windows of a sum / 4, sums from `first` on)
static constexpr uint32_t WIN_LANES = 4;                   // windows a wave
__global__ void __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2))) k_msm_windows_lanes(P29* __restrict__ win, const PointDesc* __restrict__ list, uint32_t first) {
    urgent();
    __shared__ int32_t pool[2][P29_WORDS][GT];              // of each lane: S, V below
    const uint32_t t = threadIdx.x, g = t & 15u, sum = first + blockIdx.y, w = blockIdx.x * WIN_LANES + (t >> 4);
    const PointDesc& desc = list[sum];
    if (desc.out == nullptr) return;
    const bool mine = w < 2 * desc.nwh;
    const P29* __restrict__ B = desc.buckets + (mine ? w : 0u) * MT + g * 8;
    enum : uint32_t { S = 0, V = 1 };                       // the running sum, the sum of the running sums
    auto get = [&](uint32_t slot, uint32_t of) {
        P29 r;
        int32_t* dst = reinterpret_cast<int32_t*>(&r);
#pragma unroll
        for (int l = 0; l < P29_WORDS; ++l) dst[l] = pool[slot][l][(t & 48u) | (of & 15u)];
        return r;
    };
    auto put = [&](uint32_t slot, const P29& v) {
        const int32_t* src = reinterpret_cast<const int32_t*>(&v);
#pragma unroll
        for (int l = 0; l < P29_WORDS; ++l) pool[slot][l][t] = src[l];
    };
    const bool odd = (g & 1u) != 0;
    P29 x = B[7];
    put(V, x);
    for (uint32_t step = 0; step < 25; ++step) {            // as above; x: the last step's result
        P29 y;
        uint32_t to = S;
        if (step < 14) {                                    // S and its bucket, V and S
            if (step & 1u) { y = x; x = get(V, g); to = V; }
            else { if (step) x = get(S, g); y = B[6 - (step >> 1)]; }
        } else if (step < 17) {
            if (step == 14) x = get(S, g);
            y = x;
        } else {
            const uint32_t k = (step - 17) >> 1;
            to = V;
            if (step & 1u) { x = get(k == 0 && odd ? S : V, g); y = k == 0 ? get(odd ? S : V, g ^ 1u) : get(V, g + (1u << k)); }
            else if (!odd) y = k == 0 ? get(S, g ^ 1u) : get(V, g + (1u << k) + 1u);
            else y = x;
        }
        x = p29_add<true>(x, y);
        if (step < 17 || !(step & 1u)) { __syncthreads(); put(to, x); __syncthreads(); }
    }
    if (mine && g == 0) win[(size_t)sum * MW + w] = x;
}
// grid: eight sums a wave
__global__ void __launch_bounds__(GT) k_msm_horner(const P29* __restrict__ win, const PointDesc* __restrict__ list, uint32_t n) {
    urgent();
    const uint32_t q = threadIdx.x & 3u, sum = (blockIdx.x * GT + threadIdx.x) >> 3, half = (threadIdx.x >> 2) & 1u;
    const uint32_t nwh = list[blockIdx.x * (GT / 8)].nwh, width = 128u / nwh, wider = 128u % nwh;      // of the wave's sums
    G1Jac* __restrict__ out = sum < n ? list[sum].out : nullptr;
    const P29* __restrict__ W = win + (size_t)(out ? sum : blockIdx.x * (GT / 8)) * MW + half * nwh;
    P29 r = W[nwh - 1];
    for (int w = (int)nwh - 2; w >= -1; --w) {
        P29 p;
        if (w >= 0) {
            p = W[w];                                       // on its way during the doublings
            for (uint32_t k = width + ((uint32_t)w < wider ? 1u : 0u); k > 0; --k) p29_quad_double(r, q);
        } else {                                            // the halves: [lambda] of the second
            if (half) r.x = fq29_mul(r.x, fq29_from_fp(glv_beta()));
            p = p29_shfl(r, (int)(threadIdx.x ^ 4u));
        }
        p29_quad_add(r, p, q);
    }
    if (out && half == 0 && q == 0) *out = p29_to_jac(r);
}

// Sums of an opening's first rounds from commitments of the opened tensor's rows.  The opened vector is the row fold of a
// tensor W, s = sum_r e_r W[r] with e_r = prod_j (bit_j(r) ? v_j : 1 - v_j) over the row challenges v, so every sum of the
// form  sum_j s_(L j + x) g_(L j + y)  equals  sum_r e_r X[r]  with  X[r] = sum_j W[r][L j + x] g_(L j + y),  a point that
// depends on the tensor and the generators alone and can be made in advance (a commitment of a strided part of the row
// under a strided part of the generators).  T0 and T1 of round q are combinations of 4^q such sums each: with u_0 .. u_(q-1)
// the challenges of the rounds before,
//   s^(q)_m = sum_{a < 2^q} s_(2^q m + a) prod_k (bit_k(a) ? u_k : 1 - u_k),   g^(q)_m = sum_{b < 2^q} g_(2^q m + b) prod_k (bit_k(b) ? 1 - u_k : u_k),
//   T0_q = sum_j s^(q)_(2j) g^(q)_(2j+1) = sum_{a,b} c(a,b) sum_j s_(2^(q+1) j + a) g_(2^(q+1) j + 2^q + b),   T1_q likewise with the halves exchanged,
// and T of round 0 is the same combination of the row commitments themselves.  `pts`: [pattern][row] points, pattern 0 the row
// commitments, then for q = 0 .. cross_rounds - 1 the 4^q patterns (a 2^q + b) of T0_q followed by those of T1_q.
// Target t of an opening with `full` rounds: 0 = T of round 0, 1 + 2q + side = T0_q / T1_q.  The sums equal the sums over all generators
// exactly when `pts` are such commitments of the opened tensor -- what the caller states by passing them.
__host__ __device__ __forceinline__ uint32_t cross_patterns(uint32_t rounds) { return 1u + 2u * (((1u << (2 * rounds)) - 1u) / 3u); }
// first_pattern, npat: the points of target t; slot: its place in the proof
__host__ __device__ __forceinline__ void cross_target(uint32_t t, uint32_t& first_pattern, uint32_t& npat, uint32_t& slot) {
    if (t == 0) { first_pattern = 0; npat = 1; slot = 0; return; }
    const uint32_t q = (t - 1) >> 1, side = (t - 1) & 1u;
    npat = 1u << (2 * q);
    first_pattern = cross_patterns(q) + side * npat;
    slot = 3 * q + 1 + side;
}
// These sums are bucket multi-scalar multiplications.  Term g = pattern * nrows + row of an opening, in the order `pts`
// lays the points out, has the coefficient eq(u_rows, row) * c(pattern) -- c = 1 for the row commitments, the product of the
// earlier rounds' challenges for a cross pattern -- and a target is the sum over a contiguous range of terms: one bucket sum per target over the normalised points, with the digits of all
// terms written once, as k_msm_recode writes them.  A term costs at most 32 mixed additions (a scalar
// multiplication of its own would cost a 129-step walk).
struct CrossDigitItem { void* D; const Fr* u_rows; const Fr* u; uint32_t nrows, k_rows; };
struct CrossDigitBatch { CrossDigitItem it[OB_MAX]; };
// grid (ceil(most terms / 256), openings)
__global__ void __launch_bounds__(256) k_open_cross_digits(const CrossDigitBatch cb, uint32_t npatterns, const DigitPlan plan, uint32_t* __restrict__ state, uint32_t state_words) {
    clear_state(state, state_words);
    const CrossDigitItem& it = cb.it[blockIdx.y];
    const size_t terms = (size_t)npatterns * it.nrows, i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= terms) return;
    const uint32_t p = (uint32_t)(i / it.nrows), row = (uint32_t)(i - (size_t)p * it.nrows);
    const Fr one = big_one_mont<8>();
    Fr coef = one;
    for (uint32_t j = 0; j < it.k_rows; ++j) coef = mont_mul(coef, ((row >> j) & 1u) ? it.u_rows[j] : sub(one, it.u_rows[j]));
    if (p != 0) {
        uint32_t q = 0;                                 // the patterns of round q: T0's 4^q, then T1's
        while (p >= cross_patterns(q + 1)) ++q;
        const uint32_t pl = (p - cross_patterns(q)) & ((1u << (2 * q)) - 1u), a = pl >> q, b = pl & ((1u << q) - 1u);
        for (uint32_t k = 0; k < q; ++k) {
            const Fr uk = it.u[k], nk = sub(one, uk);
            coef = mont_mul(coef, mont_mul(((a >> k) & 1u) ? uk : nk, ((b >> k) & 1u) ? nk : uk));
        }
    }
    msm_recode_store(it.D, terms, i, from_mont(coef), plan);
}
// T of the rounds behind the first follows from T of round 0 and from T0, T1 of the rounds before:
//   T_r = u(1-u) T_(r-1) + (1-u)^2 T0_(r-1) + u^2 T1_(r-1)   (u = the challenge of round r-1)
// unrolled down to round 0, with the products of those coefficients.  Those points lie in the proof itself: the digits of T_1 .. T_(R-1) as
// bucket sums over an opening's first 3 (R - 1) proof points (T, T0, T1 a round; the T of later rounds take no part: zeros).  A round's T
// is a sum over as many generators as its T0 and T1 together, so this halves what is summed.  T of the rounds above `again` (0: none) is unrolled
// from T of round `again`.  U: the challenges, opening y's at U + y * ustride
__global__ void __launch_bounds__(256) k_open_unroll_digits(int8_t* __restrict__ D0, const Fr* __restrict__ U, uint32_t ustride, uint32_t R, uint32_t again) {
    urgent();
    const uint32_t np = 3 * (R - 1), terms = (R - 1) * np, i = blockIdx.x * 256 + threadIdx.x;
    if (i >= terms) return;
    const Fr* __restrict__ u = U + (size_t)blockIdx.y * ustride;
    const uint32_t r = 1 + i / np, m = i % np, k = m / 3, j = m % 3, from = again && r > again ? again : 0u;
    const Fr one = big_one_mont<8>();
    Fr c = big_zero<8>();
    if (k >= from && k < r && (j != 0 || k == from)) {
        c = one;
        if (j != 0) {
            const Fr f = j == 2 ? u[k] : sub(one, u[k]);
            c = mont_mul(f, f);
        }
        for (uint32_t q = j == 0 ? k : k + 1; q < r; ++q) c = mont_mul(c, mont_mul(u[q], sub(one, u[q])));
    }
    msm_recode_store(D0 + (size_t)blockIdx.y * (MW + 1) * terms, terms, i, from_mont(c), DigitPlan{});
}
// The same the other way round, for openings whose T is not given for any round: behind the last round T_R = [s] g of the final scalar and generator, and
//   T_r = (T_(r+1) - (1-u)^2 T0_r - u^2 T1_r) / (u(1-u))   (u = the challenge of round r, neither 0 nor 1)
// so no round's T is summed at all: the sum over all generators in the first round was a quarter of the sums of an opening of 128 x 131072.
// The digits of T_0 .. T_(R-1) over the 3 R + 1 proof points (T's: zeros).  V: 1 / (u(1-u)) of every round, as U
struct FinalScalars { const Fr* s[OB_MAX]; };
__global__ void __launch_bounds__(256) k_open_back_digits(int8_t* __restrict__ D0, const Fr* __restrict__ U, const Fr* __restrict__ V, const FinalScalars fs, uint32_t R) {
    urgent();
    const uint32_t np = 3 * R + 1, terms = R * np, i = blockIdx.x * 256 + threadIdx.x;
    if (i >= terms) return;
    const Fr* __restrict__ u = U + (size_t)blockIdx.y * R;
    const Fr* __restrict__ v = V + (size_t)blockIdx.y * R;
    const uint32_t r = i / np, m = i % np, k = m / 3, j = m % 3;
    const Fr one = big_one_mont<8>();
    Fr c = big_zero<8>();
    if (m == 3 * R || (j != 0 && k >= r)) {
        if (m == 3 * R) c = to_mont(*fs.s[blockIdx.y]);
        else {
            const Fr f = j == 2 ? u[k] : sub(one, u[k]);
            c = sub(c, mont_mul(f, f));
        }
        for (uint32_t q = r; q < (m == 3 * R ? R : k + 1); ++q) c = mont_mul(c, v[q]);
    }
    msm_recode_store(D0 + (size_t)blockIdx.y * (MW + 1) * terms, terms, i, from_mont(c), DigitPlan{});
}
// ---- the fold on 29-bit-limb affine points ----------------------------------------------------------------------------------
// The rounds of an opening keep the generators in ONE form: affine, 29-bit limbs (A29; all-zero limbs = infinity), canonical
// limbs.  The bucket sums add out of it, the fold reads it and writes the next round's generators in it -- no
// normalisation or conversion pass between two rounds.
// 1 / v, every lane its own: all lanes of a wave execute the inversion's instructions in any case, so a product tree over the
// lanes around one inversion only adds to them.  v must not be 0 mod p (lanes with nothing to invert pass one).
// w as an affine point with canonical limbs (infinity: all zero)
__device__ __forceinline__ A29 a29_from_j29(const J29& w) {
    A29 o;
    o.x = o.y = fq29_zero();
    const Fq29 zi = fq29_inverse(w.inf ? fq29_one() : w.z);
    if (!w.inf) {
        const Fq29 zi2 = fq29_sqr(zi);
        o.x = fq29_canon(fq29_mul(w.x, zi2));
        o.y = fq29_canon(fq29_mul(fq29_mul(w.y, zi2), zi));
    }
    return o;
}
__device__ __forceinline__ A29 a29_from_p29(const P29& w) {
    A29 o;
    o.x = o.y = fq29_zero();
    const bool inf = fq29_is_zero_mod_p(w.z);
    const Fq29 zi = fq29_inverse(inf ? fq29_one() : w.z);
    if (!inf) {
        o.x = fq29_canon(fq29_mul(w.x, zi));
        o.y = fq29_canon(fq29_mul(w.y, zi));
    }
    return o;
}
struct FoldItem { Fr* ns; A29* ng; const Fr* s; const A29* g; uint32_t* special; Fr u_mont; JsfK jsf; };
struct FoldBatch { FoldItem it[OB_MAX]; };          // blockIdx.y names the opening; all of one size
// Pair g of the round: s' and g' = a1 + [u](a0 - a1), all in 29-bit limbs.  The scalar multiplication walks the joint
// sparse form of the split challenge over the all-affine table {D, phi(D), D + phi(D), D - phi(D)}, D = a0 - a1, and the
// result is brought back to affine form in the kernel.  Pairs whose inputs
// are special (a0 at infinity, equal abscissae, an abscissa of zero) are not computed here: their indices go to
// `special` ([0] = count, then the indices) and k_open_fold_special takes them.
__global__ void __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_open_fold29(const FoldBatch fb, size_t old_size, size_t new_size) {
    Fr* __restrict__ new_scalars = fb.it[blockIdx.y].ns;
    A29* __restrict__ new_gens = fb.it[blockIdx.y].ng;
    const Fr* __restrict__ scalars = fb.it[blockIdx.y].s;
    const A29* __restrict__ A = fb.it[blockIdx.y].g;
    uint32_t* __restrict__ special = fb.it[blockIdx.y].special;
    const Fr u_mont = fb.it[blockIdx.y].u_mont;
    const JsfK& jsf = fb.it[blockIdx.y].jsf;
    __shared__ int32_t tab[4][14][GT];
    const size_t g = (size_t)blockIdx.x * GT + threadIdx.x;
    const bool live = g < new_size;
    const size_t g0 = 2 * g, g1 = 2 * g + 1;
    const bool has1 = live && g1 < old_size;
    A29 a0, a1;
    a0.x = a0.y = a1.x = a1.y = fq29_zero();
    if (live) a0 = A[g0];
    if (has1) a1 = A[g1];
    if (live) {
        if (has1) new_scalars[g] = add(scalars[g0], mont_mul(u_mont, sub(scalars[g1], scalars[g0])));
        else new_scalars[g] = sub(scalars[g0], mont_mul(u_mont, scalars[g0]));
    }
    const bool inf0 = a29_is_inf(a0), inf1 = !has1 || a29_is_inf(a1);
    const Fq29 one29 = fq29_one();
    bool general = live && inf0;
    Fq29 den = one29;
    if (live && !general && !inf1) {
        den = fq29_sub(a0.x, a1.x);
        if (fq29_is_zero_mod_p(den)) { general = true; den = one29; }
    }
    const bool need_sub = live && !general && !inf1;          // D = a0 - a1 needs 1 / (x0 - x1)
    Fq29 inv = fq29_inverse(den);
    Fq29 xD = a0.x, yD = a0.y;
    if (need_sub) {
        const Fq29 lam = fq29_mul(fq29_add(a0.y, a1.y), inv);          // -a1 = (x1, -y1)
        const Fq29 x3 = fq29_sub(fq29_sub(fq29_sqr(lam), a0.x), a1.x);
        yD = fq29_mul(fq29_sub(fq29_mul(lam, fq29_sub(a0.x, x3)), a0.y), one29);      // the products by one bring the sums back into (-eps, p + eps)
        xD = fq29_mul(x3, one29);
    }
    if (live && !general && fq29_is_zero_mod_p(xD)) general = true;       // x = 0: not in the subgroup; the table below would divide by it
    const bool fast = live && !general;
    inv = fq29_inverse(fast ? xD : one29);
    J29 w = j29_infinity();
    if (fast) {
        {
            const Fq29 xQ = fq29_mul(xD, fq29_from_fp(glv_beta())), xPQ = fq29_mul(xD, fq29_from_fp(glv_beta2()));
            const Fq29 lam = fq29_mul(fq29_mul(fq29_from_fp(glv_minus2_over_beta_minus_1()), yD), inv);   // slope of D + (beta x, -y)
            const Fq29 xPmQ = fq29_mul(fq29_add(fq29_sqr(lam), xPQ), one29);
            const Fq29 yPmQ = fq29_mul(fq29_sub(fq29_mul(lam, fq29_sub(xD, xPmQ)), yD), one29);
            // D stays in registers; the other three abscissae and the second ordinate wait in LDS (word-interleaved over the
            // lanes) and negations are formed when a point is taken: the walk then fits 256 registers without spilling.
#pragma unroll
            for (int l = 0; l < 14; ++l) {
                tab[0][l][threadIdx.x] = xQ.l[l];
                tab[1][l][threadIdx.x] = xPQ.l[l];
                tab[2][l][threadIdx.x] = xPmQ.l[l];
                tab[3][l][threadIdx.x] = yPmQ.l[l];
            }
        }
        for (int i = (int)jsf.len - 1; i >= 0; --i) {
            j29_double_walk(w);
            const uint32_t dg = (jsf.dig[i >> 3] >> ((i & 7) * 4)) & 0xFu;    // (d1 + 1) | (d2 + 1) << 2, the same for every lane
            const int d1 = (int)(dg & 3u) - 1, d2 = (int)(dg >> 2) - 1;
            if (d1 == 0 && d2 == 0) continue;
            A29 t;
            bool negate;
            if (d2 == 0) { t.x = xD; t.y = yD; negate = d1 < 0; }
            else {
                const int xi = d1 == 0 ? 0 : (d1 == d2 ? 1 : 2);
#pragma unroll
                for (int l = 0; l < 14; ++l) t.x.l[l] = tab[xi][l][threadIdx.x];
                if (xi == 2) {
#pragma unroll
                    for (int l = 0; l < 14; ++l) t.y.l[l] = tab[3][l][threadIdx.x];
                    negate = d1 < 0;
                } else {
                    t.y = yD;
                    negate = xi == 0 ? d2 < 0 : d1 > 0;                          // D + phi(D) = (beta^2 x, -y)
                }
            }
            if (negate) t.y = fq29_neg(t.y);
            j29_add_mixed_walk(w, t);
        }
        if (!inf1) j29_add_mixed_walk(w, a1);
    }
    const A29 o = a29_from_j29(w);
    if (fast) {
        new_gens[g] = o;
    } else if (general) {
        const uint32_t slot = atomicAdd(&special[0], 1u);
        special[1 + slot] = (uint32_t)g;
    }
}
// ---- the first round over prepared generators: a fixed-base comb per pair ----------------------------------------------------------
// The generators of an opening are public and fixed, so D_i = g_2i - g_2i+1 is known before any challenge is.  For each
// pair the prepared form holds the COMB_N = 2^COMB_A - 1 sums  E[m] = sum_{j : bit j of m} 2^(j COMB_W) D_i  as affine
// points.  With u = k1 + k2 lambda (k1, k2 < 2^128 <= 2^(COMB_A COMB_W)), position b of the comb takes bit j COMB_W + b
// of k1 for every tooth j as the index m1(b), likewise m2(b) from k2, and
//     [u] D = sum_b 2^b ( E[m1(b)] + phi(E[m2(b)]) ),   phi(x, y) = (beta x, y):
// COMB_W doublings and at most 2 COMB_W mixed additions instead of 129 doublings and ~65 additions, and no inversion for a
// table.  Every lane of the launch uses the same indices, so the table is laid out entry-major ([m][pair]): the lanes of a
// wave read consecutive points.
static constexpr int COMB_A = 8, COMB_W = 16, COMB_N = (1 << COMB_A) - 1;
static_assert(COMB_A * COMB_W >= 128, "the comb must cover 128-bit half scalars");
struct CombK { uint8_t m1[COMB_W + 2], m2[COMB_W + 2]; };
// No pair is special here: the table holds multiples of D whatever D is (infinity when the two generators are equal, a
// doubling when they are opposite), an entry at infinity is skipped, and the mixed addition itself handles a sum that
// meets its own operand.
// NT = 2 (the second round): the pair difference of that round is itself a fixed combination of prepared points,
//     g'_2j - g'_2j+1 = F_j + [u1] H_j,   F_j = g_4j+1 - g_4j+3,  H_j = (g_4j - g_4j+1) - (g_4j+2 - g_4j+3)
// (g'_i = g_2i+1 + [u1](g_2i - g_2i+1) are the first round's results, a missing generator is the point at infinity), so
//     g''_j = g'_2j+1 + [u2] F_j + [u1 u2] H_j:
// two combs that share their doublings, COMB_W doublings and at most 4 COMB_W additions instead of the 129-step walk.
struct CombItem { Fr* ns; A29* ng; const Fr* s; const A29* g; const A29* tab; const A29* tab2; Fr u_mont; CombK ck, ck2; };
struct CombBatch { CombItem it[OB_MAX]; };
template <int NT>
__global__ void __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_open_fold_comb(const CombBatch cb, size_t old_size, size_t new_size) {
    Fr* __restrict__ new_scalars = cb.it[blockIdx.y].ns;
    A29* __restrict__ new_gens = cb.it[blockIdx.y].ng;
    const Fr* __restrict__ scalars = cb.it[blockIdx.y].s;
    const A29* __restrict__ A = cb.it[blockIdx.y].g;
    const A29* __restrict__ tab = cb.it[blockIdx.y].tab;
    const A29* __restrict__ tab2 = cb.it[blockIdx.y].tab2;
    const Fr u_mont = cb.it[blockIdx.y].u_mont;
    const CombK& ck = cb.it[blockIdx.y].ck;
    const CombK& ck2 = cb.it[blockIdx.y].ck2;
    const size_t g = (size_t)blockIdx.x * GT + threadIdx.x;
    const bool live = g < new_size;
    const size_t g0 = 2 * g, g1 = 2 * g + 1;
    const bool has1 = live && g1 < old_size;
    A29 a1;
    a1.x = a1.y = fq29_zero();
    if (has1) a1 = A[g1];
    if (live) {
        if (has1) new_scalars[g] = add(scalars[g0], mont_mul(u_mont, sub(scalars[g1], scalars[g0])));
        else new_scalars[g] = sub(scalars[g0], mont_mul(u_mont, scalars[g0]));
    }
    const bool inf1 = !has1 || a29_is_inf(a1);
    const bool fast = live;
    J29 w = j29_infinity();
    if (fast) {
        const Fq29 beta = fq29_from_fp(glv_beta());
        for (int b = COMB_W - 1; b >= 0; --b) {
            j29_double_walk(w);
#pragma unroll
            for (int ti = 0; ti < NT; ++ti) {
                const A29* __restrict__ tb = ti ? tab2 : tab;
                const uint32_t m1 = ti ? ck2.m1[b] : ck.m1[b], m2 = ti ? ck2.m2[b] : ck.m2[b];          // the same for every lane
                if (m1) {
                    const A29 t = tb[(size_t)(m1 - 1) * new_size + g];
                    if (!a29_is_inf(t)) j29_add_mixed_walk(w, t);
                }
                if (m2) {
                    A29 t = tb[(size_t)(m2 - 1) * new_size + g];
                    if (!a29_is_inf(t)) {
                        t.x = fq29_mul(t.x, beta);
                        j29_add_mixed_walk(w, t);
                    }
                }
            }
        }
        if (!inf1) j29_add_mixed_walk(w, a1);
    }
    const A29 o = a29_from_j29(w);
    if (fast) new_gens[g] = o;
}
// ---- three rounds in one: the generators after the third fold straight from the prepared ones -------------------------------------
// When T0 and T1 of the first three rounds come from cross commitments of the opened tensor, nothing reads the generators of
// the second and third round but the next fold.  With c_b = prod_{k<3} (bit_k(b) ? 1 - u_k : u_k) (u_0 .. u_2 the three
// challenges; the c_b sum to one) the generators after three folds are
//     g^(3)_m = sum_{b<8} c_b g_(8m+b) = g_(8m+7) + sum_{b<7} [c_b] P_b,m,     P_b,m = g_(8m+b) - g_(8m+7),
// seven fixed-base combs that share their COMB_W doublings: at most 14 COMB_W additions per eight generators, where the
// three rounds one after the other take a comb per pair, a double comb per four and a 129-step walk per eight.
// Tables: [b][entry][m], built like the first round's.  The scalars are folded three times on the way.
static constexpr int JUMP_ROUNDS = 3, JUMP_SPAN = 1 << JUMP_ROUNDS, JUMP_TABS = JUMP_SPAN - 1;
struct JumpItem { Fr* ns; A29* ng; const Fr* s; const A29* g; const A29* tab; Fr u_mont[JUMP_ROUNDS]; CombK ck[JUMP_TABS]; };
struct JumpBatch { JumpItem it[OB_MAX]; };
__global__ void __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_open_fold_jump(const JumpBatch jb, size_t new_size) {
    const JumpItem& it = jb.it[blockIdx.y];
    const size_t g = (size_t)blockIdx.x * GT + threadIdx.x;
    const bool live = g < new_size;
    A29 a1;
    a1.x = a1.y = fq29_zero();
    if (live) {
        a1 = it.g[JUMP_SPAN * g + JUMP_SPAN - 1];
        // the scalars, level by level as the rounds would fold them
        Fr v[JUMP_SPAN];
#pragma unroll
        for (int i = 0; i < JUMP_SPAN; ++i) v[i] = it.s[JUMP_SPAN * g + i];
#pragma unroll
        for (int k = 0; k < JUMP_ROUNDS; ++k)
#pragma unroll
            for (int i = 0; i < (JUMP_SPAN >> (k + 1)); ++i) v[i] = add(v[2 * i], mont_mul(it.u_mont[k], sub(v[2 * i + 1], v[2 * i])));
        it.ns[g] = v[0];
    }
    const bool inf1 = !live || a29_is_inf(a1);
    J29 w = j29_infinity();
    if (live) {
        const Fq29 beta = fq29_from_fp(glv_beta());
        for (int b = COMB_W - 1; b >= 0; --b) {
            j29_double_walk(w);
            for (int ti = 0; ti < JUMP_TABS; ++ti) {
                const A29* __restrict__ tb = it.tab + (size_t)ti * COMB_N * new_size;
                const uint32_t m1 = it.ck[ti].m1[b], m2 = it.ck[ti].m2[b];          // the same for every lane
                if (m1) {
                    const A29 t = tb[(size_t)(m1 - 1) * new_size + g];
                    if (!a29_is_inf(t)) j29_add_mixed_walk(w, t);
                }
                if (m2) {
                    A29 t = tb[(size_t)(m2 - 1) * new_size + g];
                    if (!a29_is_inf(t)) {
                        t.x = fq29_mul(t.x, beta);
                        j29_add_mixed_walk(w, t);
                    }
                }
            }
        }
        if (!inf1) j29_add_mixed_walk(w, a1);
    }
    const A29 o = a29_from_j29(w);
    if (live) it.ng[g] = o;
}
// ---- three rounds in one without tables ------------------------------------------------------------------------------------------
// The same combination g^(3)_m = sum_{b<8} c_b g_(8m+b) with nothing prepared, in two launches.  The joint sparse forms of the eight split
// c_b are cut into eight slices of `slice` positions.  k_open_span_slices: wave b of a workgroup makes the table of the b-th
// generator of 64 results (P, phi(P), P - phi(P); P + phi(P) is their x's sum negated), then sums slice b over all eight generators --
// a walk of `slice` doublings, every digit the same for the wave.  k_open_span_walk: four lanes a result put the slices together, seven
// times `slice` doublings.  An eighth of the doublings that eight walks beside each other take, and the second launch, whose chain
// hardly fills the chip, leaves it to the bucket sums.
struct SpanBatch { A29* ng[OB_MAX]; const A29* g[OB_MAX]; P29* part; };
__global__ void __launch_bounds__(8 * GT) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_open_span_slices(const SpanBatch sb, const JsfK* __restrict__ jsfs, size_t old_size, size_t new_size, uint32_t slice) {
    __shared__ int32_t tab[8][5][14][GT];      // x, y of P, x of phi(P), x and y of P - phi(P)
    __shared__ uint8_t flags[8][GT];
    const uint32_t b = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / GT)), t = threadIdx.x % GT;
    const size_t m = (size_t)blockIdx.x * GT + t;
    {
        A29 p;
        p.x = p.y = fq29_zero();
        if (m < new_size && 8 * m + b < old_size) p = sb.g[blockIdx.y][8 * m + b];
        const bool inf = a29_is_inf(p), x0 = !inf && fq29_is_zero_mod_p(p.x);
        const Fq29 inv = fq29_inverse((inf || x0) ? fq29_one() : p.x), one29 = fq29_one();
        const Fq29 xQ = fq29_mul(p.x, fq29_from_fp(glv_beta())), xPQ = fq29_mul(p.x, fq29_from_fp(glv_beta2()));
        const Fq29 lam = fq29_mul(fq29_mul(fq29_from_fp(glv_minus2_over_beta_minus_1()), p.y), inv);   // slope of P + (beta x, -y)
        const Fq29 xPmQ = fq29_mul(fq29_add(fq29_sqr(lam), xPQ), one29);
        const Fq29 yPmQ = fq29_mul(fq29_sub(fq29_mul(lam, fq29_sub(p.x, xPmQ)), p.y), one29);
#pragma unroll
        for (int l = 0; l < 14; ++l) {
            tab[b][0][l][t] = p.x.l[l];
            tab[b][1][l][t] = p.y.l[l];
            tab[b][2][l][t] = xQ.l[l];
            tab[b][3][l][t] = xPmQ.l[l];
            tab[b][4][l][t] = yPmQ.l[l];
        }
        flags[b][t] = (uint8_t)((inf ? 1 : 0) | (x0 ? 2 : 0));
    }
    __syncthreads();
    const JsfK* const jsf = jsfs + blockIdx.y * 8;
    J29 w = j29_infinity();
    for (int i = (int)slice - 1; i >= 0; --i) {
        if (__any(!w.inf)) j29_double_walk(w);
        const uint32_t at = b * slice + (uint32_t)i;
        for (uint32_t k = 0; k < 8; ++k) {
            if (at >= jsf[k].len) continue;
            const uint32_t dg = (jsf[k].dig[at >> 3] >> ((at & 7) * 4)) & 0xFu;    // (d1 + 1) | (d2 + 1) << 2, the same for every lane
            const int d1 = (int)(dg & 3u) - 1, d2 = (int)(dg >> 2) - 1;
            if (d1 == 0 && d2 == 0) continue;
            A29 q;
            bool negate;
            const bool diff = d1 * d2 < 0;
            const uint32_t xi = diff ? 3u : (d1 == 0 ? 2u : 0u), yi = diff ? 4u : 1u;
#pragma unroll
            for (int l = 0; l < 14; ++l) { q.x.l[l] = tab[k][xi][l][t]; q.y.l[l] = tab[k][yi][l][t]; }
            if (d1 == d2) {                                                      // P + phi(P) = (beta^2 x, -y), beta^2 = -1 - beta
                Fq29 s;
#pragma unroll
                for (int l = 0; l < 14; ++l) s.l[l] = tab[k][2][l][t];
                q.x = fq29_neg(fq29_add(q.x, s));
                negate = d1 > 0;
            } else negate = d1 == 0 ? d2 < 0 : d1 < 0;
            if (negate) q.y = fq29_neg(q.y);
            // a point of abscissa zero is its own image under phi (outside the prime-order subgroup): P - phi(P) is infinity
            const uint32_t fl = flags[k][t];
            if (!(fl & 1u) && !((fl & 2u) && diff)) j29_add_mixed_walk(w, q);
        }
    }
    if (m < new_size) {
        int32_t* out = reinterpret_cast<int32_t*>(sb.part) + ((size_t)blockIdx.y * 8 + b) * P29_WORDS * new_size + m;
        const P29 v = p29_from_j29(w);
        const int32_t* src = reinterpret_cast<const int32_t*>(&v);
#pragma unroll
        for (int l = 0; l < P29_WORDS; ++l) out[(size_t)l * new_size] = src[l];
    }
}
__global__ void __launch_bounds__(GT) k_open_span_walk(const SpanBatch sb, size_t new_size, uint32_t slice) {
    urgent();
    const size_t m = ((size_t)blockIdx.x * GT + threadIdx.x) >> 2;
    const uint32_t q = threadIdx.x & 3u;
    if (m >= new_size) return;
    const int32_t* part = reinterpret_cast<const int32_t*>(sb.part) + (size_t)blockIdx.y * 8 * P29_WORDS * new_size + m;
    P29 w = p29_infinity();
    for (int b = 7; b >= 0; --b) {
        if (b != 7)
            for (uint32_t i = 0; i < slice; ++i) p29_quad_double(w, q);
        P29 s;
        int32_t* dst = reinterpret_cast<int32_t*>(&s);
#pragma unroll
        for (int l = 0; l < P29_WORDS; ++l) dst[l] = part[((size_t)b * P29_WORDS + l) * new_size];
        p29_quad_add(w, s, q);
    }
    const A29 o = a29_from_p29(w);
    if (q == 0) sb.ng[blockIdx.y][m] = o;
}
// the pairs k_open_fold29 left out, by the general Jacobian route in 32-bit limbs (one lane per pair, an inversion each)
__device__ __forceinline__ G1Affine a29_to_affine(const A29& p) {
    G1Affine r;
    r.x = fq29_to_fp(p.x); r.y = fq29_to_fp(p.y);
    return r;
}
struct SpecialBatch { A29* ng[OB_MAX]; const A29* g[OB_MAX]; const uint32_t* special[OB_MAX]; GlvK ku[OB_MAX]; };
__global__ void __launch_bounds__(GT) k_open_fold_special(const SpecialBatch sb, size_t old_size) {
    A29* __restrict__ new_gens = sb.ng[blockIdx.y];
    const A29* __restrict__ A = sb.g[blockIdx.y];
    const uint32_t* __restrict__ special = sb.special[blockIdx.y];
    const GlvK ku = sb.ku[blockIdx.y];
    const uint32_t count = special[0];
    for (uint32_t i = blockIdx.x * GT + threadIdx.x; i < count; i += gridDim.x * GT) {
        const size_t g = special[1 + i];
        const G1Affine a0 = a29_to_affine(A[2 * g]);
        const bool has1 = 2 * g + 1 < old_size;
        G1Affine a1;
        a1.x = a1.y = big_zero<12>();
        if (has1) a1 = a29_to_affine(A[2 * g + 1]);
        const bool inf1 = !has1 || aff_is_inf(a1);
        G1Jac diff = aff_to_jac(a0);
        if (!inf1) diff = g1_add_mixed(diff, g1_neg(a1));
        G1Jac r = g1_mul_glv(diff, ku);
        if (!inf1) r = g1_add_mixed(r, a1);
        A29 o;
        o.x = o.y = fq29_zero();
        if (!is_zero(r.z)) {
            const Fp zi = mont_inverse(r.z), zi2 = fp_sqr(zi);
            G1Affine af;
            af.x = fp_mul(r.x, zi2);
            af.y = fp_mul(fp_mul(r.y, zi2), zi);
            o = a29_from_affine(af);
            o.x = fq29_canon(o.x); o.y = fq29_canon(o.y);
        }
        new_gens[g] = o;
    }
}
// the generator pairs' differences g_2i - g_2i+1 (an odd last element alone): what the first round's comb is built on
__global__ void __launch_bounds__(GT) k_open_pair_points(G1Jac* __restrict__ pj, const G1Affine* __restrict__ A, size_t old_size, size_t half_up) {
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    if (i >= half_up) return;
    G1Jac p = aff_to_jac(A[2 * i]);
    if (2 * i + 1 < old_size) {
        const G1Affine b = g1_neg(A[2 * i + 1]);
        if (!aff_is_inf(b)) p = g1_add_mixed(p, b);
    }
    pj[i] = p;
}
// out[j] = V[2j] - V[2j+1] over the points V[i] = A[off + i * stride], i < cnt (a missing one is the point at infinity)
__global__ void __launch_bounds__(GT) k_open_pair_diff(G1Jac* __restrict__ out, const G1Affine* __restrict__ A, size_t off, size_t stride, size_t cnt, size_t n_out) {
    const size_t j = (size_t)blockIdx.x * GT + threadIdx.x;
    if (j >= n_out) return;
    G1Jac p = g1_infinity();
    if (2 * j < cnt) p = aff_to_jac(A[off + 2 * j * stride]);
    if (2 * j + 1 < cnt) {
        const G1Affine b = g1_neg(A[off + (2 * j + 1) * stride]);
        if (!aff_is_inf(b)) p = g1_add_mixed(p, b);
    }
    out[j] = p;
}
// out[m] = A[m * span + b] - A[m * span + span - 1], m < n_out (the points of k_open_fold_jump's tables)
__global__ void __launch_bounds__(GT) k_open_span_diff(G1Jac* __restrict__ out, const G1Affine* __restrict__ A, uint32_t span, uint32_t b, size_t n_out) {
    const size_t m = (size_t)blockIdx.x * GT + threadIdx.x;
    if (m >= n_out) return;
    G1Jac p = aff_to_jac(A[m * span + b]);
    const G1Affine last = g1_neg(A[m * span + span - 1]);
    if (!aff_is_inf(last)) p = g1_add_mixed(p, last);
    out[m] = p;
}
__global__ void __launch_bounds__(GT) k_a29_to_jac(G1Jac* __restrict__ out, const A29* __restrict__ in, size_t n) {
    const size_t i = (size_t)blockIdx.x * GT + threadIdx.x;
    if (i >= n) return;
    out[i] = a29_is_inf(in[i]) ? g1_infinity() : aff_to_jac(a29_to_affine(in[i]));
}
// ---- rounds in one batch ------------------------------------------------------------------------------------------------
// Over n0 generators, every later round's generators are fixed linear combinations of these n0 points: g at level j, block i, is
// sum over k in block i of W_j(k) g_k with W_j(k) = prod_{b<j} (bit_b(k) ? 1-u_b : u_b).  So T, T0, T1 of any number of rounds and the
// final generator are multi-scalar multiplications over the same n0 affine points with coefficients that are plain field
// arithmetic; they run as one launch instead of a chain of rounds that each wait for a scalar multiplication.
// Folded scalars of all levels: level 0 is S itself, level j >= 1 sits at SL + sum_{1<=i<j} n_i, n_i = ceil(n0 / 2^i).
struct TailPtrs { Fr* SL[OB_MAX]; const Fr* S[OB_MAX]; };      // per opening of a batch (blockIdx.x of k_tail_scalars, blockIdx.y of k_tail_levels and k_tail_coeffs)
// One wave a workgroup: beside a kernel of many single waves that hold every SIMD's registers, four waves at once found no room on a compute unit until
// that kernel's queue had drained (in an opening of 128 x 131072: 670 to 1370 us for 16384 scalars, 13 alone and 56 so).
static constexpr int TAIL_T = 64;
// L levels at once, a lane for every 2^L scalars
template <int L> __global__ void __launch_bounds__(TAIL_T) k_tail_levels(const TailPtrs tp, const Fr* __restrict__ U, uint32_t ustride, uint32_t n0) {
    urgent();
    uint32_t n[L + 1];
    n[0] = n0;
#pragma unroll
    for (int k = 0; k < L; ++k) n[k + 1] = (n[k] + 1) / 2;
    const uint32_t g = blockIdx.x * TAIL_T + threadIdx.x;
    if (g >= n[L]) return;
    const Fr* __restrict__ usu = U + (size_t)blockIdx.y * ustride;
    const Fr* __restrict__ S = tp.S[blockIdx.y];
    Fr* __restrict__ out = tp.SL[blockIdx.y];
    Fr v[1 << L];
#pragma unroll
    for (int i = 0; i < (1 << L); ++i) v[i] = (g << L) + i < n0 ? S[(g << L) + i] : big_zero<8>();      // a missing scalar counts as zero: s0 - u s0
#pragma unroll
    for (int k = 0; k < L; ++k) {
        const Fr u = usu[k];
#pragma unroll
        for (int i = 0; i < (1 << (L - 1 - k)); ++i) {
            const uint32_t at = (g << (L - 1 - k)) + i;
            v[i] = add(v[2 * i], mont_mul(u, sub(v[2 * i + 1], v[2 * i])));
            if (at < n[k + 1]) out[at] = v[i];
        }
        out += n[k + 1];
    }
}
// U: the tail's challenges (Montgomery form), opening y's at U + y * ustride
// the last levels, of at most TAIL_SHORT scalars: one wave per opening
static constexpr size_t TAIL_SHORT = 512;
__global__ void __launch_bounds__(TAIL_T) k_tail_scalars(const TailPtrs tp, const Fr* __restrict__ U, uint32_t ustride, uint32_t n0, uint32_t levels) {
    urgent();
    const Fr* __restrict__ usu = U + (size_t)blockIdx.x * ustride;
    const Fr* cur = tp.S[blockIdx.x];
    Fr* nxt = tp.SL[blockIdx.x];
    uint32_t n = n0;
    for (uint32_t j = 0; j < levels; ++j) {
        const uint32_t ns = (n + 1) / 2;
        for (uint32_t g = threadIdx.x; g < ns; g += TAIL_T) {
            const Fr s0 = cur[2 * g];
            nxt[g] = (2 * g + 1 < n) ? add(s0, mont_mul(usu[j], sub(cur[2 * g + 1], s0))) : sub(s0, mont_mul(usu[j], s0));
        }
        __syncthreads();
        cur = nxt;
        nxt += ns;
        n = ns;
    }
}
// The digits (k_msm_recode) of C[(3j+0)*n0 + k] = s_j[k>>j] W_j(k); C[(3j+1)*n0 + k] = s_j[(k>>j)-1] W_j(k) for odd k>>j; C[(3j+2)*n0 + k] = s_j[(k>>j)+1] W_j(k)
// for even k>>j with a partner; zero elsewhere.  C[3*levels*n0 + k] = W_levels(k), the final generator's.  A lane forms its own W: the products cost less than a chain of
// all levels' recodings on one lane.  blockIdx.z: which of these; given: the levels whose first is not wanted.  An opening's coefficients stand behind those
// of the one before, ncoef of all of them.
__global__ void __launch_bounds__(TAIL_T) k_tail_coeffs(void* __restrict__ D, size_t ncoef, const TailPtrs tp, const Fr* __restrict__ U, uint32_t ustride, uint32_t n0, uint32_t levels, uint32_t given,
                                                        const DigitPlan plan, uint32_t* __restrict__ state, uint32_t state_words) {
    urgent();
    if (blockIdx.z == 0) clear_state(state, state_words);
    const uint32_t k = blockIdx.x * TAIL_T + threadIdx.x, j = blockIdx.z / 3, kind = blockIdx.z % 3;
    if (k >= n0 || (j < levels && kind == 0 && (given >> j & 1u))) return;
    const Fr* __restrict__ usu = U + (size_t)blockIdx.y * ustride;
    const Fr one_m = big_one_mont<8>();
    Fr W = one_m;                 // Montgomery form
    const Fr* sj = tp.S[blockIdx.y];
    uint32_t n = n0;
    for (uint32_t i = 0; i < j; ++i) {
        const Fr f = (k >> i & 1u) ? sub(one_m, usu[i]) : usu[i];
        W = i == 0 ? f : mont_mul(W, f);
        sj = i == 0 ? tp.SL[blockIdx.y] : sj + n;
        n = (n + 1) / 2;
    }
    const uint32_t i = k >> j;
    Fr c = big_zero<8>();
    if (j == levels) c = from_mont(W);
    else if (kind == 0 || (kind == 1 ? (i & 1u) != 0 : !(i & 1u) && i + 1 < n))
        c = mont_mul(W, sj[kind == 0 ? i : (kind == 1 ? i - 1 : i + 1)]);      // Montgomery W times standard s: the product's standard form
    msm_recode_store(D, ncoef, ((size_t)blockIdx.y * gridDim.z + blockIdx.z) * n0 + k, c, plan);
}
__global__ void __launch_bounds__(64) k_u32_zero(uint32_t* __restrict__ p, uint32_t n, size_t stride) {      // p[i * stride] = 0, i < n
    for (uint32_t i = threadIdx.x; i < n; i += 64) p[(size_t)i * stride] = 0u;
}
// after the last round of an opening without a batched tail: the folded generator is the last proof point
__global__ void __launch_bounds__(GT) k_open_finish(G1Jac* __restrict__ pts, const A29* __restrict__ last_gen, uint32_t rounds) {
    if (blockIdx.x == 0 && threadIdx.x == 0) pts[3 * rounds] = a29_is_inf(last_gen[0]) ? g1_infinity() : aff_to_jac(a29_to_affine(last_gen[0]));
}

// ---- host side ----------------------------------------------------------------------------------------------------------
static inline Fr load_fr(const uint32_t* p) { Fr r; memcpy(&r, p, 32); return r; }
static inline G1Jac load_g1(const uint32_t* p) { G1Jac r; memcpy(&r, p, 144); return r; }

#define GLAUNCH(kernel, n, st, ...)                                                                          \
    do {                                                                                                     \
        if ((n) > 0) {                                                                                       \
            hipLaunchKernelGGL(kernel, dim3(cdiv((n), GT)), dim3(GT), 0, (hipStream_t)(st), __VA_ARGS__);     \
            ZK_LAUNCH_CHECK();                                                                               \
        }                                                                                                    \
    } while (0)

// sum of n points at `in` into one point at `out` (device); `in` is not modified
static int g1_sum_device(G1Jac* out, const G1Jac* in, size_t n, hipStream_t st) {
    if (n == 0) {
        G1Jac inf = g1_infinity();
        hipLaunchKernelGGL(k_g1_fill, dim3(1), dim3(GT), 0, st, out, inf, (size_t)1);
        ZK_LAUNCH_CHECK();
        return 0;
    }
    uint32_t nseg = (uint32_t)((n + 4 * GT - 1) / (4 * GT));
    if (nseg > 1024) nseg = 1024;
    if (nseg <= 1) {
        hipLaunchKernelGGL(k_g1_rowsum, dim3(1, 1), dim3(GT), 0, st, out, in, n, 1u);
        ZK_LAUNCH_CHECK();
        return 0;
    }
    Scratch part(sizeof(G1Jac) * nseg, st);
    if (part.rc) return part.rc;
    hipLaunchKernelGGL(k_g1_rowsum, dim3(1, nseg), dim3(GT), 0, st, part.as<G1Jac>(), in, n, nseg);
    hipLaunchKernelGGL(k_g1_rowsum, dim3(1, 1), dim3(GT), 0, st, out, part.as<G1Jac>(), (size_t)nseg, 1u);
    ZK_LAUNCH_CHECK();
    return 0;
}

// Optional timing of the fold kernel's launches with events on its own stream (measurement only).
struct FoldTimer {
    std::mutex mu;
    bool on = false;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> ev;
    double fp_mults = 0;      // Fp multiplications the timed launches perform by the formulas' count
    unsigned long long pairs = 0;
    // the same per method: 0 the walk (k_open_fold29), 1 the one- and two-table combs (k_open_fold_comb), 2 the three-round fold (k_open_fold_jump)
    std::vector<int> method;
    double m_mults[3] = {0, 0, 0};
    unsigned long long m_pairs[3] = {0, 0, 0};
};
static FoldTimer g_fold_timer;
static const int g_fold_timer_hook = (at_shutdown([] {
    std::lock_guard<std::mutex> lk(g_fold_timer.mu);
    for (auto& e : g_fold_timer.ev) { (void)hipEventDestroy(e.first); (void)hipEventDestroy(e.second); }
    g_fold_timer.ev.clear();
    g_fold_timer.on = false;
}), 0);
struct FoldTimed {
    hipEvent_t t0 = nullptr;
    hipStream_t st;
    explicit FoldTimed(hipStream_t st) : st(st) {
        if (g_fold_timer.on && hipEventCreate(&t0) == hipSuccess) (void)hipEventRecord(t0, st);
    }
    void end(int method, double fp_mults, unsigned long long pairs) {
        hipEvent_t t1 = nullptr;
        if (!t0 || hipEventCreate(&t1) != hipSuccess) return;
        (void)hipEventRecord(t1, st);
        std::lock_guard<std::mutex> lk(g_fold_timer.mu);
        g_fold_timer.ev.emplace_back(t0, t1);
        g_fold_timer.fp_mults += fp_mults;
        g_fold_timer.pairs += pairs;
        g_fold_timer.method.push_back(method);
        g_fold_timer.m_mults[method] += fp_mults;
        g_fold_timer.m_pairs[method] += pairs;
    }
};
// Fp multiplications of one pair of the fold by the formulas' count (two 8-limb products aside)
static double fold_fp_mults_per_pair(const JsfK& j) {
    int adds = 0;
    for (uint32_t i = 0; i < j.len; ++i) adds += (((j.dig[i >> 3] >> ((i & 7) * 4)) & 0xFu) != 5u) ? 1 : 0;    // 5 = both digits zero
    // difference (4), its share of two batched inversions (6), table (7), doublings (7 each), mixed additions (11 each), final addition (11)
    return 4.0 + 6.0 + 7.0 + 7.0 * j.len + 11.0 * adds + 11.0;
}

// u = k1 + k2 * lambda with 0 <= k1 < lambda and k2 <= lambda + 1 (r = lambda^2 + lambda + 1): one long division
static GlvK glv_split(const Fr& u) {
    const unsigned __int128 lam = ((unsigned __int128)0xac45a4010001a402ull << 64) | 0x00000000ffffffffull;
    unsigned __int128 rem = 0, q = 0;
    for (int i = 255; i >= 0; --i) {
        const bool top = (rem >> 127) != 0;
        rem = (rem << 1) | ((u.v[i >> 5] >> (i & 31)) & 1u);
        q <<= 1;
        if (top || rem >= lam) { rem -= lam; q |= 1; }
    }
    GlvK k;
    for (int i = 0; i < 4; ++i) { k.k1[i] = (uint32_t)(rem >> (32 * i)); k.k2[i] = (uint32_t)(q >> (32 * i)); }
    return k;
}
// joint sparse form of the two halves of a split scalar (Solinas): the fewest non-zero digit pairs among signed binary forms
static JsfK jsf_of(const GlvK& k) {
    unsigned __int128 a = 0, b = 0;
    for (int i = 3; i >= 0; --i) { a = (a << 32) | k.k1[i]; b = (b << 32) | k.k2[i]; }
    JsfK out;
    memset(&out, 0, sizeof(out));
    unsigned d1 = 0, d2 = 0, len = 0;
    while (a + d1 > 0 || b + d2 > 0) {
        const unsigned l1 = (unsigned)((a & 7) + d1) & 7u, l2 = (unsigned)((b & 7) + d2) & 7u;
        int u1 = 0, u2 = 0;
        if (l1 & 1u) { u1 = 2 - (int)(l1 & 3u); if ((l1 == 3 || l1 == 5) && (l2 & 3u) == 2) u1 = -u1; }
        if (l2 & 1u) { u2 = 2 - (int)(l2 & 3u); if ((l2 == 3 || l2 == 5) && (l1 & 3u) == 2) u2 = -u2; }
        if (2 * (int)d1 == 1 + u1) d1 = 1 - d1;
        if (2 * (int)d2 == 1 + u2) d2 = 1 - d2;
        a >>= 1;
        b >>= 1;
        out.dig[len >> 3] |= (uint32_t)((u1 + 1) | ((u2 + 1) << 2)) << ((len & 7) * 4);
        ++len;
    }
    out.len = len;
    return out;
}

// The generators of an opening in the form its rounds work on: A29 points.  Nothing in it depends on what is opened, so a
// caller that opens against the same generators again keeps it (zk_g1_open_prepare).
static int open_prep_build(A29* out, const G1Jac* gens, size_t n, Arena& arena, hipStream_t st) {
    Scratch& aff = arena.add(sizeof(G1Affine) * n);
    if (aff.rc) return aff.rc;
    g1_normalize_queue<true>(aff.p, gens, n, st);
    hipLaunchKernelGGL(k_g1aff_to_a29, dim3(cdiv(n, 256)), dim3(256), 0, st, out, aff.as<G1Affine>(), n);
    ZK_LAUNCH_CHECK();
    return 0;
}

// One opening of the batch: its scalars, its challenges (rounds x 8 limbs) and its generators -- Jacobian, or null when
// `prep` (their prepared form, open_prep_build) is given
struct OpenItem { const void* scalars; const void* gens; const A29* prep; const uint32_t* u; const A29* comb = nullptr; const A29* comb2 = nullptr;
                  const void* rows = nullptr; uint32_t nrows = 0; const uint32_t* u_rows = nullptr; int k_rows = 0; int cross_rounds = 0;
                  const A29* comb3 = nullptr; };
// One round of `count` openings of equal size (count <= OB_MAX): one launch of each kernel covers all of them.
// comb: the first round's table; comb2 (second round): the tables of F and H one after the other, u_prev the first round's challenge
struct RoundItem { Fr* new_scalars; A29* new_gens; const Fr* scalars; const A29* gens; Fr u; const A29* comb = nullptr; const A29* comb2 = nullptr; Fr u_prev = Fr(); };
// Fp multiplications of one pair of the comb fold by the formulas' count
static double comb_fp_mults_per_pair(const CombK& ck, const CombK* ck2 = nullptr) {
    int adds = 0, phis = 0;
    for (int b = 0; b < COMB_W; ++b) { adds += (ck.m1[b] ? 1 : 0) + (ck.m2[b] ? 1 : 0); phis += ck.m2[b] ? 1 : 0; }
    if (ck2) for (int b = 0; b < COMB_W; ++b) { adds += (ck2->m1[b] ? 1 : 0) + (ck2->m2[b] ? 1 : 0); phis += ck2->m2[b] ? 1 : 0; }
    // doublings (7 each), mixed additions (11 each), the endomorphism's product, final addition (11), its share of one batched inversion (3) and the way back to affine (5)
    return 7.0 * COMB_W + 11.0 * adds + phis + 11.0 + 3.0 + 5.0;
}
static CombK comb_of(const GlvK& k) {
    CombK ck;
    memset(&ck, 0, sizeof(ck));
    for (int b = 0; b < COMB_W; ++b)
        for (int j = 0; j < COMB_A; ++j) {
            const int bit = j * COMB_W + b;
            if (bit >= 128) continue;
            ck.m1[b] |= (uint8_t)(((k.k1[bit >> 5] >> (bit & 31)) & 1u) << j);
            ck.m2[b] |= (uint8_t)(((k.k2[bit >> 5] >> (bit & 31)) & 1u) << j);
        }
    return ck;
}
// c_b = prod_q (bit_q(b) ? 1 - u_q : u_q) over three rounds' challenges (standard form in and out)
static void fold_span_coefficients(Fr* c, const uint32_t* u) {
    const Fr one = big_one_mont<8>();
    for (int b = 0; b < JUMP_SPAN; ++b) {
        Fr m = one;
        for (int q = 0; q < JUMP_ROUNDS; ++q) {
            const Fr um = to_mont(load_fr(u + 8 * (size_t)q));
            m = mont_mul(m, ((b >> q) & 1) ? sub(one, um) : um);
        }
        c[b] = from_mont(m);
    }
}
// Small host arrays of a job (challenges, descriptors) on their way to the device: copied through pinned buffers of 64 KiB that are
// held until the job ends, into device blocks of the job's arena.
struct JobUploads {
    Arena* arena = nullptr;
    std::vector<void*> pins;
    std::vector<char*> devs;
    size_t used = 0;
    static constexpr size_t CAP = 64 << 10;
    int put(const void* src, size_t bytes, hipStream_t st, const void** dev) {
        ZK_ARG(bytes <= CAP, "opening: too many sums");
        if (pins.empty() || used + bytes > CAP) {
            Scratch& d = arena->add(CAP);
            if (d.rc) return d.rc;
            void* h = nullptr;
            const int rc = pinned_acquire(&h);
            if (rc) return rc;
            pins.push_back(h);
            devs.push_back(d.as<char>());
            used = 0;
        }
        memcpy((char*)pins.back() + used, src, bytes);
        ZK_HIP(hipMemcpyAsync(devs.back() + used, (char*)pins.back() + used, bytes, hipMemcpyHostToDevice, st));
        *dev = devs.back() + used;
        used = (used + bytes + 255) / 256 * 256;
        return 0;
    }
    ~JobUploads() { for (void* h : pins) pinned_release(h); }
};
// `aux` waits for what `st` holds so far
static int join_streams(hipStream_t st, hipStream_t aux, std::vector<hipEvent_t>& events) {
    if (aux == st) return 0;
    hipEvent_t ev;
    ZK_HIP(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
    events.push_back(ev);
    ZK_HIP(hipEventRecord(ev, st));
    ZK_HIP(hipStreamWaitEvent(aux, ev, 0));
    return 0;
}
// How some sums are taken, decided before their scalars' digits are written.  n: the sums; count_max, terms: elements of the longest, and about how many of
// them have a scalar other than zero; total: elements of all of them.
struct SumsPlan { DigitPlan digits{}; uint32_t hb = 0, most = 0, group = 0, state_words = 0; size_t total = 0; uint32_t* state = nullptr; };
// Windows of a half, and the longest list of one lane: two and a half times the mean of the wide windows' buckets, which cuts outliers alone; buckets a bit narrower have twice the mean,
// start first and leave the shorter ones to fill up.  Nothing below 32 is cut, or below 12 where all lists run at once (two waves a SIMD) and the launch takes what its longest list does: opened without a
// fold of rows, small integers share the few digits that they have, and 512 of them take 1.00 ms where lists of 32 take 1.11 (1.01 as k_msm_few), 2048 1.33 and 1.41; 16 x 1024 0.95 and 1.01.  With 8 some of these
// are 3 % faster and 1 x 512 4 % slower; from 4096 generators on nothing changes.
// In instructions of a lane: an element costs an addition of 4700 a window (the first of a list none), a list 1700 and a bucket about 1350 for each step
// of its wave in k_msm_windows.  The time of these on the whole chip at three quarters of its issue slots, half a list of the last waves, and the launch that
// windows of more than 128 buckets add.
static uint32_t msm_windows_of_half(size_t terms, uint32_t n, uint32_t* most) {
    uint32_t best = 0;
    double best_us = 0;
    for (uint32_t nwh : {16u, 13u, 12u, 11u}) {
        const uint32_t q = 128u / nwh, rem = 128u % nwh, hb = 1u << (q - 1 + (rem ? 1u : 0u));
        const double buckets = 2.0 * ((double)rem * (1u << q) + (double)(nwh - rem) * (1u << (q - 1))), mean = std::min((double)terms / hb, (double)MPIECE);
        const double all = (double)n * (std::max(0.0, (double)terms * 2.0 * nwh - buckets) * 4700.0 + buckets * (1700.0 + 1350.0 * (hb > 128 ? 29.0 : 25.0)));
        const double us = all * 4.0 / 64.0 / (1024.0 * 2400.0) / 0.75 + 6.0 * mean + (hb > 128u ? 80.0 : 0.0);
        if (best == 0 || us < best_us) {
            best = nwh; best_us = us;
            *most = (uint32_t)std::min(std::max(2.5 * mean, (double)n * buckets <= 2048.0 * MSL ? 12.0 : 32.0), (double)MPIECE);
        }
    }
    return best;
}
static int sums_plan(SumsPlan& p, uint32_t n, size_t count_max, size_t terms, size_t total, Arena& arena) {
    if (n == 0 || count_max <= (size_t)FEW_MAX) return 0;
    ZK_ARG(total < (1ull << 32), "opening: too many elements");
    const uint32_t nwh = msm_windows_of_half(terms, n, &p.most), q = 128u / nwh, rem = 128u % nwh;
    p.total = total;
    p.digits.nwh = nwh;
    for (uint32_t w = 0, off = 0; w < nwh; ++w) {
        off += q + (w < rem ? 1u : 0u);
        p.digits.bias[(off - 1) / 32] |= 1u << ((off - 1) % 32);
    }
    p.hb = 1u << (q - 1 + (rem ? 1u : 0u));
    // windows at a time, equally many: lists of at most 256 MiB (or one window's), which 1.5 M generators in a round alone exceed
    const uint32_t most_windows = (uint32_t)std::min<size_t>(std::max<size_t>((1ull << 26) / std::max<size_t>(total, 1), 1), 2 * nwh);
    p.group = (uint32_t)cdiv(2 * nwh, cdiv(2 * nwh, most_windows));
    p.state_words = (uint32_t)cdiv(2 * nwh, p.group) * SORT_WORDS;
    Scratch& st = arena.add(sizeof(uint32_t) * p.state_words);
    p.state = st.as<uint32_t>();
    return st.rc;
}
// The bucket accumulation of some sums of at most count_max elements on aux, which waits for st; their reductions, sum z into out[z], are appended to `later`.
// The sorting goes on st: what st holds next and the sums fill the chip together, and in front of both the short launches find room.
static int bucket_sums_queue(std::vector<MsmDesc> d, const std::vector<G1Jac*>& out, size_t count_max, const SumsPlan& plan, Arena& arena, JobUploads& up, hipStream_t st, hipStream_t aux,
                             std::vector<hipEvent_t>& events, std::vector<PointDesc>& later) {
    const uint32_t n_msm = (uint32_t)d.size();
    if (n_msm == 0) return 0;
    size_t total = 0;
    for (MsmDesc& m : d) { m.list_at = (uint32_t)total; total += m.count; }
    const void* dd = nullptr;
    int rc = up.put(d.data(), sizeof(MsmDesc) * n_msm, st, &dd);
    if (rc) return rc;
    if (plan.digits.nwh == 0) {
        uint32_t nw = 8;
        while (nw * count_max > 8 * MSL) nw /= 2;            // 2 at FEW_MAX
        Scratch& buckets = arena.add(sizeof(P29) * (size_t)n_msm * FEW_BUCKETS);
        if (buckets.rc) return buckets.rc;
        rc = join_streams(st, aux, events);
        if (rc) return rc;
        hipLaunchKernelGGL(k_msm_few, dim3(FEW_WINDOWS / nw, n_msm), dim3(MSL), 0, aux, buckets.as<P29>(), (const MsmDesc*)dd, nw);
        ZK_LAUNCH_CHECK();
        for (uint32_t z = 0; z < n_msm; ++z) later.push_back(PointDesc{buckets.as<P29>() + (size_t)z * FEW_BUCKETS, nullptr, out[z], 1u, (uint32_t)MWH, (uint32_t)MT, 0u});
        return 0;
    }
    ZK_ARG(total <= plan.total, "opening: more elements than planned");
    const uint32_t nw = 2 * plan.digits.nwh;
    const size_t entries = (size_t)plan.group * total, cut = entries / plan.most + 1;               // of a launch; buckets above `most` at most
    const size_t rows = (size_t)n_msm * nw, nb = rows * plan.hb, max_tasks = std::min((size_t)n_msm * plan.group * plan.hb + 2 * cut, entries);
    ZK_ARG(nb + 2 * cut < (1ull << 32), "opening: too many sums");
    Scratch& info = arena.add(sizeof(uint4) * nb);
    Scratch& lists = arena.add(sizeof(uint32_t) * entries);
    Scratch& heavy = arena.add(sizeof(uint4) * cut);
    Scratch& tasks = arena.add(sizeof(uint4) * max_tasks);
    Scratch& buckets = arena.add(sizeof(P29) * (nb + 2 * cut));                                      // a cut bucket has less than twice as many pieces as it is longer than `most`
    if (info.rc || lists.rc || heavy.rc || tasks.rc || buckets.rc) return info.rc ? info.rc : (lists.rc ? lists.rc : (heavy.rc ? heavy.rc : (tasks.rc ? tasks.rc : buckets.rc)));
    SortSpace sp{plan.state, info.as<uint4>(), lists.as<uint32_t>(), heavy.as<uint4>(), tasks.as<uint4>(), buckets.as<P29>(), plan.digits.nwh, plan.hb, 0u, (uint32_t)total, plan.most, (uint32_t)nb, (uint32_t)cut};
    for (sp.w0 = 0; sp.w0 < nw; sp.w0 += plan.group, sp.state += SORT_WORDS) {
        const dim3 grid(std::min(plan.group, nw - sp.w0), n_msm);
        const hipStream_t sort_on = sp.w0 ? aux : st;
        // a workgroup passes over its sum's digits twice: more lanes for long ones
        if (count_max > 8192) hipLaunchKernelGGL(k_msm_sort<1024>, grid, dim3(1024), 0, sort_on, sp, (const MsmDesc*)dd);
        else hipLaunchKernelGGL(k_msm_sort<256>, grid, dim3(256), 0, sort_on, sp, (const MsmDesc*)dd);
        hipLaunchKernelGGL(k_msm_tasks, grid, dim3(TASK_T), 0, sort_on, sp);
        if (sp.w0 == 0) rc = join_streams(st, aux, events);
        if (rc) return rc;
        hipLaunchKernelGGL(k_msm_lists, dim3(cdiv(max_tasks, MSL)), dim3(MSL), 0, aux, sp, (const MsmDesc*)dd);
        hipLaunchKernelGGL(k_msm_merge, dim3((uint32_t)std::min<size_t>(cut, 256)), dim3(MSL), 0, aux, sp);
        ZK_LAUNCH_CHECK();
    }
    for (uint32_t z = 0; z < n_msm; ++z) later.push_back(PointDesc{buckets.as<P29>() + (size_t)z * nw * plan.hb, nullptr, out[z], 0u, plan.digits.nwh, plan.hb, 0u});
    return 0;
}
static int points_queue(std::vector<PointDesc>& sums, Arena& arena, JobUploads& up, hipStream_t st) {
    if (sums.empty()) return 0;
    // fewer windows (of more buckets) first, few elements last
    std::stable_sort(sums.begin(), sums.end(), [](const PointDesc& a, const PointDesc& b) { return a.few != b.few ? a.few < b.few : a.nwh < b.nwh; });
    std::vector<PointDesc> list;
    size_t blocks_n = 0;
    uint32_t wide = 0, blocks_max = 0;                       // entries up to the last sum of wide windows; most blocks of one
    for (const PointDesc& d : sums) {
        if (!list.empty() && list.back().nwh != d.nwh)
            while (list.size() % (GT / 8)) { PointDesc gap = list.back(); gap.out = nullptr; list.push_back(gap); }
        list.push_back(d);
        if (d.hb > (uint32_t)MT) {
            wide = (uint32_t)list.size();
            blocks_max = std::max(blocks_max, 2 * d.nwh * d.hb / MT);
            blocks_n += 2 * (size_t)(2 * d.nwh * d.hb / MT);
        }
    }
    const uint32_t n = (uint32_t)list.size();
    uint32_t first_few = n;
    while (first_few > 0 && list[first_few - 1].few) --first_few;
    Scratch& win = arena.add(sizeof(P29) * (MW * (size_t)n + blocks_n));
    if (win.rc) return win.rc;
    P29* blocks = win.as<P29>() + MW * (size_t)n;
    for (PointDesc& d : list)
        if (d.hb > (uint32_t)MT && d.out) { d.blocks = blocks; blocks += 2 * (size_t)(2 * d.nwh * d.hb / MT); }
    const void* dl = nullptr;
    int rc = up.put(list.data(), sizeof(PointDesc) * n, st, &dl);
    if (rc) return rc;
    // a wave a window while they fit two a SIMD: sixty-four sums of 16 windows a half, the next would start a second round of waves
    const uint32_t plain = first_few - wide, plain_w = plain ? 2 * list[first_few - 1].nwh : 0;         // (a gap may stand at `wide`)
    const bool plain_lanes = (size_t)plain_w * plain > 2048;
    if (wide) hipLaunchKernelGGL(k_msm_windows<true>, dim3(blocks_max, wide), dim3(GT), 0, st, win.as<P29>(), (const PointDesc*)dl, 0u, 0u);
    if (plain_lanes) hipLaunchKernelGGL(k_msm_windows_lanes, dim3(cdiv(plain_w, WIN_LANES), plain), dim3(GT), 0, st, win.as<P29>(), (const PointDesc*)dl, wide);
    const uint32_t full = plain_lanes ? wide : first_few;
    if (full || first_few < n) hipLaunchKernelGGL(k_msm_windows<false>, dim3(MW * full + MW / 8 * (n - first_few)), dim3(GT), 0, st, win.as<P29>(), (const PointDesc*)dl, full, first_few);
    hipLaunchKernelGGL(k_msm_horner, dim3(cdiv(8 * (size_t)n, (size_t)GT)), dim3(GT), 0, st, (const P29*)win.as<P29>(), (const PointDesc*)dl, n);
    ZK_LAUNCH_CHECK();
    sums.clear();
    return 0;
}
// One halving round: the scalars' digits and the fold on st, the bucket sums on aux (their reductions are appended to `later`).
// pts: where the round's T, T0, T1 of opening 0 go; opening i's npts further.
// given: what of this round's sums comes from commitments of the tensor's rows or from the rounds before (open_cross_sums_queue,
// open_unroll_queue) and is not summed here: 0 nothing, 1 T, 2 T0 and T1 as well (no bucket sums at all: the round is its fold)
// comb_round: 0 the first round (fold table RoundItem::comb, when all items have one), 1 the second (comb2), 2 a later one
static int open_round_launch(const RoundItem* items, int count, size_t old_size, int comb_round, int given, G1Jac* pts, size_t npts, Arena& arena, JobUploads& up,
                             hipStream_t st, hipStream_t aux, std::vector<hipEvent_t>& events, std::vector<PointDesc>& later) {
    ZK_ARG(old_size < (1ull << 31), "opening: more than 2^31 generators");
    ZK_ARG(count >= 1 && count <= OB_MAX, "opening: bad batch size");
    const size_t new_size = (old_size + 1) / 2;
    SumsPlan plan;
    if (given < 2) {
        const char* digits = nullptr;
        size_t dig_bytes = 0;
        const size_t half = old_size / 2;
        int rc = sums_plan(plan, (given == 0 ? 3u : 2u) * (uint32_t)count, given == 0 ? old_size : half, half, count * (2 * half + (given == 0 ? old_size : 0)), arena);
        if (rc) return rc;
        dig_bytes = digit_bytes(plan.digits) * old_size;
        Scratch& dig = arena.add(dig_bytes * count);
        if (dig.rc) return dig.rc;
        digits = dig.as<char>();
        RecodeBatch rb;
        for (int i = 0; i < OB_MAX; ++i) { rb.D[i] = dig.as<char>() + dig_bytes * (i < count ? i : 0); rb.S[i] = items[i < count ? i : 0].scalars; }
        hipLaunchKernelGGL(k_msm_recode, dim3(cdiv(old_size, GT), count), dim3(GT), 0, st, rb, old_size, plan.digits, plan.state, plan.state_words);
        ZK_LAUNCH_CHECK();
        // ---- side chain (aux): nothing here feeds the fold ----
        std::vector<MsmDesc> d;
        std::vector<G1Jac*> out;
        const uint32_t ds = (uint32_t)old_size, dh = (uint32_t)half;
        for (int i = 0; i < count; ++i) {
            const char* dg = digits + dig_bytes * i;
            G1Jac* o = pts + npts * i;
            if (given == 0) { d.push_back(MsmDesc{dg, items[i].gens, ds, ds, 1u, 0u, 1u, 0u, 0u, 0u}); out.push_back(o); }
            d.push_back(MsmDesc{dg, items[i].gens, ds, dh, 2u, 0u, 2u, 1u, 0u, 0u}); out.push_back(o + 1);
            d.push_back(MsmDesc{dg, items[i].gens, ds, dh, 2u, 1u, 2u, 0u, 0u, 0u}); out.push_back(o + 2);
        }
        rc = bucket_sums_queue(d, out, given == 0 ? old_size : half, plan, arena, up, st, aux, events, later);
        if (rc) return rc;
    }
    // ---- critical chain (st): the fold ----
    const size_t sp_stride = 1 + new_size;
    Scratch& special = arena.add(sizeof(uint32_t) * sp_stride * count);
    if (special.rc) return special.rc;
    bool use_comb = comb_round == 0, use_comb2 = comb_round == 1;
    for (int i = 0; i < count; ++i) { use_comb = use_comb && items[i].comb != nullptr; use_comb2 = use_comb2 && items[i].comb2 != nullptr; }
    FoldBatch fb;
    CombBatch cbt;
    SpecialBatch sb;
    double fp_mults = 0;
    for (int i = 0; i < OB_MAX; ++i) {
        const int k = i < count ? i : 0;
        const GlvK ku = glv_split(items[k].u);
        uint32_t* sp = special.as<uint32_t>() + sp_stride * k;
        if (use_comb || use_comb2) {
            CombItem& f = cbt.it[i];
            f.ns = items[k].new_scalars; f.ng = items[k].new_gens; f.s = items[k].scalars; f.g = items[k].gens;
            f.u_mont = to_mont(items[k].u);
            f.ck = comb_of(ku);
            if (use_comb) {
                f.tab = items[k].comb; f.tab2 = items[k].comb;
                f.ck2 = f.ck;
                if (i < count) fp_mults += comb_fp_mults_per_pair(f.ck) * (double)new_size;
            } else {
                f.tab = items[k].comb2; f.tab2 = items[k].comb2 + (size_t)COMB_N * new_size;
                // [u2] of [u1] H is [u1 u2 mod r] H: the generators have order r
                f.ck2 = comb_of(glv_split(from_mont(mont_mul(to_mont(items[k].u_prev), to_mont(items[k].u)))));
                if (i < count) fp_mults += comb_fp_mults_per_pair(f.ck, &f.ck2) * (double)new_size;
            }
        } else {
            FoldItem& f = fb.it[i];
            f.ns = items[k].new_scalars; f.ng = items[k].new_gens; f.s = items[k].scalars; f.g = items[k].gens; f.special = sp;
            f.u_mont = to_mont(items[k].u);
            f.jsf = jsf_of(ku);
            if (i < count) fp_mults += fold_fp_mults_per_pair(f.jsf) * (double)new_size;
        }
        sb.ng[i] = items[k].new_gens; sb.g[i] = items[k].gens; sb.special[i] = sp; sb.ku[i] = ku;
    }
    hipLaunchKernelGGL(k_u32_zero, dim3(1), dim3(64), 0, st, special.as<uint32_t>(), (uint32_t)count, sp_stride);
    FoldTimed timed(st);
    if (use_comb) hipLaunchKernelGGL(k_open_fold_comb<1>, dim3(cdiv(new_size, GT), count), dim3(GT), 0, st, cbt, old_size, new_size);
    else if (use_comb2) hipLaunchKernelGGL(k_open_fold_comb<2>, dim3(cdiv(new_size, GT), count), dim3(GT), 0, st, cbt, old_size, new_size);
    else hipLaunchKernelGGL(k_open_fold29, dim3(cdiv(new_size, GT), count), dim3(GT), 0, st, fb, old_size, new_size);
    timed.end((use_comb || use_comb2) ? 1 : 0, fp_mults, new_size * (size_t)count);
    hipLaunchKernelGGL(k_open_fold_special, dim3(16, count), dim3(GT), 0, st, sb, old_size);
    ZK_LAUNCH_CHECK();
    return 0;
}

// `levels` rounds (r0 .. r0 + levels - 1 of `rounds`) in one batch over n0 generators: the scalars of all levels on st, then T, T0, T1 of
// those rounds as bucket sums with formed coefficients on aux.  last: the batch takes all rounds that are left and the final
// generator is one more sum; otherwise (three levels) the generators are folded three times at once on st and *gens names the results.
// *scalars: the folded scalars.  pts: the proof points of opening 0 (npts an opening).  t_given: the rounds whose T is not summed here.
static int open_batch_launch(const Fr** scalars, const A29** gens, int count, size_t n0, int levels, bool last, int r0, int rounds, const std::function<bool(int)>& t_given, const OpenItem* items, G1Jac* pts, size_t npts,
                             const Fr* U_dev, Arena& arena, JobUploads& up, hipStream_t st, hipStream_t aux, std::vector<hipEvent_t>& events, std::vector<PointDesc>& later);
// g^(3) of every opening from its generators (k_open_span_slices, k_open_span_walk); challenges: rounds r0 .. r0 + 2
static int open_span_fold(const A29** gens, int count, size_t n0, int r0, const OpenItem* items, Arena& arena, JobUploads& up, hipStream_t st);

extern "C" {

int zk_g1_fill(void* out, const uint32_t* point, size_t n, void* st) { GLAUNCH(k_g1_fill, n, st, (G1Jac*)out, load_g1(point), n); return 0; }
int zk_g1_neg(void* out, const void* a, size_t n, void* st) { GLAUNCH(k_g1_neg, n, st, (G1Jac*)out, (const G1Jac*)a, n); return 0; }
int zk_g1_affine_neg(void* out, const void* a, size_t n, void* st) { GLAUNCH(k_g1aff_neg, n, st, (G1Affine*)out, (const G1Affine*)a, n); return 0; }
int zk_g1_affine_to_jacobian(void* out, const void* a, size_t n, void* st) { GLAUNCH(k_g1aff_to_jac, n, st, (G1Jac*)out, (const G1Affine*)a, n); return 0; }
// out[i] = a[i] +/- b[i or 0]; b_count is n (elementwise) or 1 (broadcast, b on the device)
int zk_g1_add(void* out, const void* a, const void* b, size_t n, size_t b_count, int subtract, void* st) {
    ZK_ARG(b_count == n || b_count == 1, "zk_g1_add: b_count must be n or 1");
    GLAUNCH(k_g1_add, n, st, (G1Jac*)out, (const G1Jac*)a, (const G1Jac*)b, n, b_count, subtract);
    return 0;
}
int zk_g1_madd(void* out, const void* a, const void* b_affine, size_t n, size_t b_count, int subtract, void* st) {
    ZK_ARG(b_count == n || b_count == 1, "zk_g1_madd: b_count must be n or 1");
    GLAUNCH(k_g1_madd, n, st, (G1Jac*)out, (const G1Jac*)a, (const G1Affine*)b_affine, n, b_count, subtract);
    return 0;
}
int zk_g1_scalar_mul(void* out, const void* g, const void* s, size_t ng, size_t n, void* st) {
    ZK_ARG(ng >= 1 || n == 0, "zk_g1_scalar_mul: no generators");
    GLAUNCH(k_g1_scalar_mul, n, st, (G1Jac*)out, (const G1Jac*)g, (const Fr*)s, ng, n);
    return 0;
}
int zk_g1_sum(uint32_t* out_host, const void* a, size_t n, void* stv) {
    hipStream_t st = (hipStream_t)stv;
    Scratch res(sizeof(G1Jac), st);
    if (res.rc) return res.rc;
    int rc = g1_sum_device(res.as<G1Jac>(), (const G1Jac*)a, n, st);
    if (rc) return rc;
    void* stage = nullptr;
    rc = staging(&stage, sizeof(G1Jac));
    if (rc) return rc;
    ZK_HIP(hipMemcpyAsync(stage, res.p, sizeof(G1Jac), hipMemcpyDeviceToHost, st));
    ZK_HIP(hipStreamSynchronize(st));
    memcpy(out_host, stage, sizeof(G1Jac));
    return 0;
}
int zk_g1_rowwise_sum(void* out, const void* in, size_t nrow, size_t ncol, void* stv) {
    hipStream_t st = (hipStream_t)stv;
    if (nrow == 0) return 0;
    ZK_ARG(ncol >= 1, "zk_g1_rowwise_sum: ncol == 0");
    ZK_ARG(nrow <= 0x7fffffffu, "zk_g1_rowwise_sum: too many rows");
    uint32_t nseg = 1;
    if (nrow < 1024 && ncol > 8 * GT) { nseg = (uint32_t)(ncol / (4 * GT)); if (nseg > 64) nseg = 64; if (nseg < 1) nseg = 1; }
    if (nseg == 1) {
        hipLaunchKernelGGL(k_g1_rowsum, dim3((unsigned)nrow, 1), dim3(GT), 0, st, (G1Jac*)out, (const G1Jac*)in, ncol, 1u);
        ZK_LAUNCH_CHECK();
        return 0;
    }
    Scratch part(sizeof(G1Jac) * nrow * nseg, st);
    if (part.rc) return part.rc;
    hipLaunchKernelGGL(k_g1_rowsum, dim3((unsigned)nrow, nseg), dim3(GT), 0, st, part.as<G1Jac>(), (const G1Jac*)in, ncol, nseg);
    hipLaunchKernelGGL(k_g1_rowsum, dim3((unsigned)nrow, 1), dim3(GT), 0, st, (G1Jac*)out, part.as<G1Jac>(), (size_t)nseg, 1u);
    ZK_LAUNCH_CHECK();
    return 0;
}
// G1TensorJacobian::operator()(u) (g1-tensor.cu:500-514); out_host receives one point
int zk_g1_me(uint32_t* out_host, const void* a, size_t n, const uint32_t* u, int k, void* stv) {
    hipStream_t st = (hipStream_t)stv;
    ZK_ARG(n >= 1, "zk_g1_me: empty tensor");
    const G1Jac* cur = (const G1Jac*)a;
    size_t cur_n = n;
    void* bufs[2] = {nullptr, nullptr};
    int which = 0, rc = 0;
    for (int lvl = 0; lvl < k && rc == 0; ++lvl) {
        const size_t out_n = (cur_n + 1) / 2;
        if (!bufs[which]) rc = pool_alloc(&bufs[which], sizeof(G1Jac) * out_n, st);
        if (rc) break;
        const Fr x = from_mont(load_fr(u + 8 * lvl));   // the reference passes unmont(u) to the scalar multiplication
        hipLaunchKernelGGL(k_g1_me_step, dim3(cdiv(out_n, GT)), dim3(GT), 0, st, (G1Jac*)bufs[which], cur, x, cur_n, out_n);
        if (hipGetLastError() != hipSuccess) { rc = hip_fail(hipErrorLaunchFailure, "k_g1_me_step", __FILE__, __LINE__); break; }
        cur = (const G1Jac*)bufs[which];
        cur_n = out_n;
        which ^= 1;
    }
    if (rc == 0) {
        void* stage = nullptr;
        rc = staging(&stage, sizeof(G1Jac));
        if (rc == 0) {
            hipError_t e = hipMemcpyAsync(stage, cur, sizeof(G1Jac), hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipStreamSynchronize(st);
            if (e != hipSuccess) rc = hip_fail(e, "zk_g1_me copy", __FILE__, __LINE__);
            else memcpy(out_host, stage, sizeof(G1Jac));
        }
    }
    for (int i = 0; i < 2; ++i) if (bufs[i]) pool_free(bufs[i], st);
    return rc;
}
// canonical form: z = ONE (Montgomery), infinity = all-zero limbs.  out may alias in.
int zk_g1_normalize(void* out, const void* in, size_t n, void* st) {
    if (n == 0) return 0;
    g1_normalize_queue<false>(out, (const G1Jac*)in, n, (hipStream_t)st);
    ZK_LAUNCH_CHECK();
    return 0;
}

// the growth of a window from h to `target` entries, at most GROW_MAX steps
static std::vector<GrowSpec> grow_steps(uint32_t h, uint32_t target) {
    std::vector<GrowSpec> v;
    while (h < target) {
        const uint32_t t = std::min(target, 3 * h), c = (h + t + 1) / 2;
        v.push_back(GrowSpec{h, c, t, std::max(c - h - 1, t - c)});
        h = t;
    }
    return v;
}
// The entries of a window that k_msm_table_first makes: as many as leave it, with the growth's centres, the lanes of two waves a SIMD, and no more than the longest has.  rows: the full windows
// of all generators; half, top: entries of a full and of a highest window.  steps: the growth's launches.
static uint32_t msm_first_entries(size_t rows, size_t ngen, uint32_t half, uint32_t top, uint32_t* steps) {
    const uint32_t longest = rows ? std::max(half, top) : top;
    uint32_t first = (uint32_t)std::min<size_t>(longest, std::max<size_t>(1, ((size_t)1 << 17) / (rows + ngen)));
    for (;; --first) {
        const size_t full_n = rows ? grow_steps(first, half).size() : 0, top_n = grow_steps(first, top).size();
        *steps = (uint32_t)std::max(full_n, top_n);
        if (first == 1 || (rows + ngen) * first + rows * full_n + ngen * top_n <= (size_t)1 << 17) return first;
    }
}
// Digit width, windows and segments for m rows of ngen scalars.  seen[b]: how many of the sampled scalars have b bits.  Estimated times in us:
// a step of the table's growth counts 75 us (one lane's inversion), its first entries 50 and 30 for each doubling of their number, an entry 0.115 ns,
// a base's doubling 7 us of latency, an addition 0.17 ns; a digit beyond the first is an addition where the scalar reaches it.
// These are weights for the choice and not the kernels' times: in the large steps of k_msm_table_grow an entry takes 0.14 ns and an
// addition 0.18 (11008 x 4096 of 13 bits).  With them no size from 1 to 11008 rows of 64 to 4096 generators
// is slower than with a table that doubles, and 5000 x 2048 takes 3.43 ms instead of 3.75.  Every width timed against a table that doubles, 1 to 11008 rows of 64 to 4096 generators and scalars of 13 and of 28 bits (48 shapes):
// the one chosen here takes 4 % longer than the best on average.  The furthest off are 28-bit scalars in few rows of 64 generators, 14 % (3 bits chosen,
// 7 are best), 512 rows of 4096, 12 % (9, 7), and many rows of 28 bits, 7 % (13, 9); the same model fitted to those times chooses no better (5 %).
struct MsmShape { uint32_t c, nwin, top, nseg; };
static MsmShape msm_shape(size_t m, size_t ngen, uint32_t bits, uint32_t maxabs, const uint32_t* seen) {
    MsmShape best{0, 0, 0, 1};
    double best_us = 0, total = 0;
    for (int b = 0; b <= 32; ++b) total += seen[b];
    if (total < 1) total = 1;
    for (uint32_t c = 3; c <= 13; ++c) {
        const uint32_t nwin = bits == 0 ? 1u : (bits + 1 + c - 1) / c, half = 1u << (c - 1);      // a spare bit for the carry of the signed digits
        uint64_t most = nwin == 1 ? std::max(1u, maxabs) : ((uint64_t)maxabs >> (c * (nwin - 1))) + 1;
        uint32_t top = 1;
        while (top < most) top <<= 1;
        double digits = 0;
        for (uint32_t w = 0; w < nwin; ++w) {
            double reach = 0;
            for (uint32_t b = w ? c * w : 1; b <= 32; ++b) reach += seen[b];
            digits += reach / total;
        }
        double entries = (double)ngen * ((nwin - 1) * (double)half + top);
        if (entries * sizeof(A29) > 8e9) continue;
        uint32_t steps = 0;
        const uint32_t first = msm_first_entries((size_t)(nwin - 1) * ngen, ngen, half, top, &steps);
        const double us = 7.0 * c * (nwin - 1) + 75.0 * steps + (first > 1 ? 50.0 + 30.0 * std::log2((double)first) : 0.0) + entries * 1.15e-4 + (double)m * ngen * digits * 1.7e-4;
        if (!best.c || us < best_us) { best_us = us; best = MsmShape{c, nwin, top, 1}; }
    }
    if (!best.c) {      // more generators than the budget of the table allows any width for
        best.c = 3; best.nwin = bits == 0 ? 1u : (bits + 3) / 3;
        const uint64_t most = best.nwin == 1 ? std::max(1u, maxabs) : ((uint64_t)maxabs >> (3 * (best.nwin - 1))) + 1;
        for (best.top = 1; best.top < most; best.top <<= 1) {}
    }
    // segments of a row: items (sixteen lanes each) for two waves a SIMD while they keep 32 generators each, and for eight where they keep 512
    // (a launch of 1.3 times the waves that fit leaves the chip half empty at its end; the sum over an item's lanes costs five additions on four lanes).
    // Up to 1536 waves leave most SIMDs one wave or a third of them a second one for all of a launch: twice as many of half the length, where 128 generators are left
    // for each, take 2100 to 2780 rows of 1024 from 1.66 to 1.40 ms, 5500 of 512 from 1.55 to 1.43; from 8000 items on (4000 rows of 1024, 8000 of 512) they lose 3 %.
    while ((m * best.nseg * 2 <= 8192 && ngen / (best.nseg * 2) >= 32) || (m * best.nseg < 32768 && ngen / (best.nseg * 2) >= 512)
           || (m * best.nseg < 6144 && ngen / (best.nseg * 2) >= 128)) best.nseg *= 2;
    return best;
}

// Commitment::commit_int (commitment.cu:50-58): out[row] = sum_j [t[row,j]] gens[j], t = embedded int32 values.
// scalars: Fr tensor of m*ngen elements.  Values outside the int32 embedding are rejected.
int zk_g1_commit_int(void* out, const void* gens, const void* scalars_fr, size_t m, size_t ngen, void* stv) {
    hipStream_t st = (hipStream_t)stv;
    if (m == 0) return 0;
    ZK_ARG(ngen >= 1, "zk_g1_commit_int: no generators");
    ZK_ARG(m <= 0x7fffffffu, "zk_g1_commit_int: too many rows");
    const size_t total = m * ngen;
    Scratch ints(sizeof(int32_t) * total, st), stats(4 * CONV_STATS, st);
    if (ints.rc) return ints.rc;
    if (stats.rc) return stats.rc;
    if (const int crc = clear_words(stats.p, CONV_STATS, st)) return crc;
    hipLaunchKernelGGL(k_fr_to_i32_checked, dim3((unsigned)std::min<size_t>(cdiv(total, 256), CONV_GRID)), dim3(256), 0, st, ints.as<int32_t>(), stats.as<uint32_t>(), (const Fr*)scalars_fr, total);
    ZK_LAUNCH_CHECK();
    void* stage = nullptr;
    int rc = staging(&stage, 4 * CONV_STATS);
    if (rc) return rc;
    ZK_HIP(hipMemcpyAsync(stage, stats.p, 4 * CONV_STATS, hipMemcpyDeviceToHost, st));
    ZK_HIP(hipStreamSynchronize(st));
    uint32_t seen[CONV_STATS];
    memcpy(seen, stage, sizeof(seen));
    const uint32_t maxabs = seen[1];
    ZK_ARG(seen[0] == 0, "zk_g1_commit_int: a scalar is not the embedding of an int32 value");
    uint32_t bits = 0;
    while (bits < 32 && (maxabs >> bits)) ++bits;
    const MsmShape shape = msm_shape(m, ngen, bits, maxabs, seen + 2);
    MsmTable T;
    T.ngen = ngen; T.c = shape.c; T.nwin = shape.nwin; T.half = 1u << (shape.c - 1); T.top = shape.top;
    const size_t nbase = (size_t)T.nwin * ngen, tab_n = (size_t)(T.nwin - 1) * ngen * T.half + ngen * T.top;
    ZK_ARG(tab_n < ((size_t)1 << 31), "zk_g1_commit_int: too many generators");
    Scratch tab(sizeof(A29) * tab_n, st), basej(sizeof(G1Jac) * nbase, st), basea(sizeof(G1Affine) * nbase, st);
    if (tab.rc) return tab.rc;
    if (basej.rc) return basej.rc;
    if (basea.rc) return basea.rc;
    T.tab = tab.as<A29>();
    hipLaunchKernelGGL(k_msm_table_bases, dim3(cdiv(ngen, GT)), dim3(GT), 0, st, basej.as<G1Jac>(), (const G1Jac*)gens, ngen, T.c, T.nwin, 1u);
    g1_normalize_queue<true>(basea.p, basej.as<G1Jac>(), nbase, st);
    const size_t rows_full = (size_t)(T.nwin - 1) * ngen;
    uint32_t steps = 0;
    const uint32_t first = msm_first_entries(rows_full, ngen, T.half, T.top, &steps);
    const std::vector<GrowSpec> full = T.nwin > 1 ? grow_steps(first, T.half) : std::vector<GrowSpec>(), top = grow_steps(first, T.top);
    GrowCentres gc;
    gc.full_n = (uint32_t)full.size(); gc.top_n = (uint32_t)top.size();
    ZK_ARG(gc.full_n <= (uint32_t)GROW_MAX && gc.top_n <= (uint32_t)GROW_MAX, "zk_g1_commit_int: too many generators");
    for (int i = 0; i < GROW_MAX; ++i) { gc.full[i] = i < (int)gc.full_n ? (uint16_t)full[i].c : 1; gc.top[i] = i < (int)gc.top_n ? (uint16_t)top[i].c : 1; }
    const size_t first_n = rows_full * gc.full_n + ngen * gc.top_n + nbase * first;
    hipLaunchKernelGGL(k_msm_table_first, dim3(cdiv(first_n, GT)), dim3(GT), 0, st, T, basea.as<G1Affine>(), first, gc);
    for (size_t i = 0; i < std::max(full.size(), top.size()); ++i) {
        const GrowSpec none{1u, 1u, 1u, 0u}, f = i < full.size() ? full[i] : none, p = i < top.size() ? top[i] : none;
        const size_t n = rows_full * f.np + ngen * p.np;
        if (n == 0) continue;
        // pairs a lane: whole rounds of the lanes of two waves a SIMD, of at most 32 pairs each
        const size_t lanes = (size_t)1 << 17, rounds = (n + 32 * lanes - 1) / (32 * lanes);
        const uint32_t per_lane = (uint32_t)((n + rounds * lanes - 1) / (rounds * lanes));
        hipLaunchKernelGGL(k_msm_table_grow, dim3(cdiv(n, (size_t)GT * per_lane)), dim3(GT), 0, st, T, f, p, (uint32_t)n, per_lane);
    }
    ZK_LAUNCH_CHECK();
    const size_t per = (ngen + shape.nseg - 1) / shape.nseg, items = m * shape.nseg;
    Scratch part(shape.nseg > 1 ? sizeof(P29) * items : 1, st);
    if (part.rc) return part.rc;
    hipLaunchKernelGGL(k_msm_rows, dim3(cdiv(items, 4)), dim3(GT), 0, st, (G1Jac*)out, part.as<P29>(), T, ints.as<int32_t>(), m, shape.nseg, (uint32_t)per);
    if (shape.nseg > 1) {           // a power of two: half as many groups as parts are as fast as all
        uint32_t lg = 0;
        while (lg < 4 && (4u << lg) <= shape.nseg) ++lg;
        hipLaunchKernelGGL(k_msm_parts, dim3(cdiv(m << lg, (size_t)GT / 4)), dim3(GT), 0, st, (G1Jac*)out, part.as<P29>(), m, shape.nseg, lg);
    }
    ZK_LAUNCH_CHECK();
    return 0;
}

// out[i] = [s_i] B for a base point B given on the host (Jacobian, Montgomery form) and n scalars in standard form: what
// Commitment::random does with the group generator (commitment.cu:3-8, a broadcast G1Jacobian_mul).  The table of B's
// multiples is kept on the device from one call to the next with the same base (one table per process, 4224 points).
int zk_g1_fixed_base_mul(void* out, const uint32_t* base_host, const void* scalars_fr, size_t n, void* stv) {
    hipStream_t st = (hipStream_t)stv;
    if (n == 0) return 0;
    static std::mutex mu;
    static void* tab = nullptr;
    static int tab_dev = -1;
    static uint32_t tab_base[36];
    std::lock_guard<std::mutex> lk(mu);
    int dev = 0;
    ZK_HIP(hipGetDevice(&dev));
    if (!tab || tab_dev != dev || std::memcmp(tab_base, base_host, sizeof(tab_base)) != 0) {
        const size_t tab_n = (size_t)FB_WIN * 128;
        if (tab && tab_dev != dev) { int cur = dev; ZK_HIP(hipSetDevice(tab_dev)); ZK_HIP(hipFree(tab)); ZK_HIP(hipSetDevice(cur)); tab = nullptr; }
        if (!tab) ZK_HIP(hipMalloc(&tab, sizeof(A29) * tab_n));
        tab_dev = -1;                                   // not valid until the build below has finished
        Scratch b(sizeof(G1Jac), st), tabj(sizeof(G1Jac) * tab_n, st), taba(sizeof(G1Affine) * tab_n, st);
        if (b.rc) return b.rc;
        if (tabj.rc) return tabj.rc;
        if (taba.rc) return taba.rc;
        ZK_HIP(hipMemcpyAsync(b.p, base_host, sizeof(G1Jac), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(k_msm_table_bases, dim3(1), dim3(GT), 0, st, tabj.as<G1Jac>(), b.as<G1Jac>(), (size_t)1, 8u, FB_WIN, 128u);
        for (uint32_t logk = 0; logk < 7; ++logk)
            hipLaunchKernelGGL(k_msm_table_fill, dim3(cdiv((size_t)FB_WIN << logk, GT)), dim3(GT), 0, st, tabj.as<G1Jac>(), (size_t)FB_WIN, 7u, logk);
        g1_normalize_queue<true>(taba.p, tabj.as<G1Jac>(), tab_n, st);
        hipLaunchKernelGGL(k_g1aff_to_a29, dim3(cdiv(tab_n, 256)), dim3(256), 0, st, (A29*)tab, taba.as<G1Affine>(), tab_n);
        ZK_LAUNCH_CHECK();
        ZK_HIP(hipStreamSynchronize(st));               // later calls may come on other streams
        std::memcpy(tab_base, base_host, sizeof(tab_base));
        tab_dev = dev;
    }
    hipLaunchKernelGGL(k_g1_fixed_base_mul, dim3(cdiv(n, GT)), dim3(GT), 0, st, (G1Jac*)out, (const A29*)tab, (const Fr*)scalars_fr, n);
    ZK_LAUNCH_CHECK();
    return 0;
}

// One round of Commitment::me_open (commitment.cu:79-129) with all three sums computed directly.  u: standard-form
// challenge (the field scalar of the fold and the integer of the scalar multiplications, as in the reference).
// new_scalars / new_gens: (old_size+1)/2 elements.  sums_host: 3 points (T, T0, T1), normalised to z = 1.
int zk_g1_open_round(void* new_scalars, void* new_gens, uint32_t* sums_host, const void* scalars, const void* gens, const uint32_t* u, size_t old_size, void* stv) {
    hipStream_t st = (hipStream_t)stv;
    ZK_ARG(old_size >= 1, "zk_g1_open_round: empty input");
    const size_t new_size = (old_size + 1) / 2;
    Scratch pts(sizeof(G1Jac) * 3, st);
    if (pts.rc) return pts.rc;
    Arena arena(st);
    JobUploads up;
    up.arena = &arena;
    Scratch& g29 = arena.add(sizeof(A29) * old_size);
    Scratch& n29 = arena.add(sizeof(A29) * new_size);
    if (g29.rc || n29.rc) return g29.rc ? g29.rc : n29.rc;
    int rc = open_prep_build(g29.as<A29>(), (const G1Jac*)gens, old_size, arena, st);
    if (rc) return rc;
    std::vector<hipEvent_t> evs;          // one stream: none is made
    std::vector<PointDesc> later;
    const RoundItem item{(Fr*)new_scalars, n29.as<A29>(), (const Fr*)scalars, g29.as<A29>(), load_fr(u), nullptr};
    rc = open_round_launch(&item, 1, old_size, 0, 0, pts.as<G1Jac>(), 3, arena, up, st, st, evs, later);
    if (rc == 0) rc = points_queue(later, arena, up, st);
    if (rc) { (void)hipStreamSynchronize(st); return rc; }
    hipLaunchKernelGGL(k_a29_to_jac, dim3(cdiv(new_size, GT)), dim3(GT), 0, st, (G1Jac*)new_gens, n29.as<A29>(), new_size);
    g1_normalize_queue<false>(pts.p, pts.as<G1Jac>(), (size_t)3, st);
    ZK_LAUNCH_CHECK();
    void* stage = nullptr;
    rc = staging(&stage, sizeof(G1Jac) * 3);
    if (rc) return rc;
    ZK_HIP(hipMemcpyAsync(stage, pts.p, sizeof(G1Jac) * 3, hipMemcpyDeviceToHost, st));
    ZK_HIP(hipStreamSynchronize(st));          // (the uploads' pinned buffers go back when this returns)
    memcpy(sums_host, stage, sizeof(G1Jac) * 3);
    return 0;
}

// The whole recursion of Commitment::me_open (commitment.cu:109-129): `rounds` halvings of (scalars, gens) of length n
// with the challenges u[0..rounds).  An OpenJob queues all of it on one stream and keeps every buffer until the
// result has been fetched.
struct OpenJob {
    Arena arena;
    hipStream_t st = nullptr;
    int rounds = 0, count = 0;
    G1Jac* pts = nullptr;                      // count x (3 rounds + 1) points
    const Fr* final_scalar[OB_MAX] = {};
    hipEvent_t ready = nullptr;    // only for jobs on a side stream
    hipStream_t aux = nullptr;     // second stream of the job (bucket sums beside the folds); equals st when the job has one stream
    std::vector<hipEvent_t> events;
    JobUploads up;                 // challenges, descriptors
    uint64_t ticket = 0;           // the launch thread's ticket while it queues the job's kernels
    int queue_rc = 0;              // what queuing returned, and its message
    std::string queue_err;
    OpenJob() { up.arena = &arena; }
};
// The targets of every opening of a batch (T of round 0; T0, T1 of the first `full` rounds) as bucket sums over the openings' [pattern][row] points, on aux.
static int open_cross_sums_queue(const OpenItem* items, int count, uint32_t full, G1Jac* pts, size_t npts, const Fr* const* urow_dev, const Fr* U_dev, int rounds, Arena& arena,
                                 JobUploads& up, hipStream_t aux, std::vector<hipEvent_t>& events, std::vector<PointDesc>& later) {
    const uint32_t ntargets = 1u + 2u * full, npatterns = cross_patterns(full);
    CrossDigitBatch db;
    const A29* base[OB_MAX];
    const void* digs[OB_MAX];
    size_t most_terms = 0, most_count = 0, all_terms = 0;
    for (int i = 0; i < count; ++i) {
        all_terms += (size_t)npatterns * items[i].nrows;
        for (uint32_t t = 0; t < ntargets; ++t) {
            uint32_t p0, npat, slot;
            cross_target(t, p0, npat, slot);
            most_count = std::max(most_count, (size_t)npat * items[i].nrows);
        }
    }
    SumsPlan plan;
    int rc = sums_plan(plan, ntargets * (uint32_t)count, most_count, all_terms / (ntargets * (uint32_t)count), all_terms, arena);
    if (rc) return rc;
    for (int i = 0; i < count; ++i) {
        const size_t points = (size_t)npatterns * items[i].nrows;          // and as many terms
        ZK_ARG(items[i].nrows >= 1 && points < (1ull << 31), "zk_g1_open: bad row count");
        most_terms = std::max(most_terms, points);
        Scratch& aff = arena.add(sizeof(G1Affine) * points);
        Scratch& a29 = arena.add(sizeof(A29) * points);
        Scratch& dg = arena.add(digit_bytes(plan.digits) * points);
        if (aff.rc || a29.rc || dg.rc) return aff.rc ? aff.rc : (a29.rc ? a29.rc : dg.rc);
        g1_normalize_queue<true>(aff.p, (const G1Jac*)items[i].rows, points, aux);
        hipLaunchKernelGGL(k_g1aff_to_a29, dim3(cdiv(points, 256)), dim3(256), 0, aux, a29.as<A29>(), aff.as<G1Affine>(), points);
        base[i] = a29.as<A29>();
        digs[i] = dg.p;
        db.it[i] = CrossDigitItem{dg.p, urow_dev[i], U_dev + (size_t)i * rounds, items[i].nrows, (uint32_t)items[i].k_rows};
    }
    for (int i = count; i < OB_MAX; ++i) db.it[i] = db.it[0];
    hipLaunchKernelGGL(k_open_cross_digits, dim3(cdiv(most_terms, 256), count), dim3(256), 0, aux, db, npatterns, plan.digits, plan.state, plan.state_words);
    ZK_LAUNCH_CHECK();
    std::vector<MsmDesc> d;
    std::vector<G1Jac*> out;
    for (int i = 0; i < count; ++i)
        for (uint32_t t = 0; t < ntargets; ++t) {
            uint32_t p0, npat, slot;
            cross_target(t, p0, npat, slot);
            const uint32_t nr = items[i].nrows;
            d.push_back(MsmDesc{digs[i], base[i], npatterns * nr, npat * nr, 1u, p0 * nr, 1u, p0 * nr, 0u, 0u});
            out.push_back(pts + npts * i + slot);
        }
    return bucket_sums_queue(d, out, most_count, plan, arena, up, aux, aux, events, later);
}
static int open_span_fold(const A29** gens, int count, size_t n0, int r0, const OpenItem* items, Arena& arena, JobUploads& up, hipStream_t st) {
    const size_t ns = (((n0 + 1) / 2 + 1) / 2 + 1) / 2;
    Scratch& g2 = arena.add(sizeof(A29) * ns * count);
    if (g2.rc) return g2.rc;
    Scratch& part = arena.add(sizeof(P29) * 8 * ns * count);
    if (part.rc) return part.rc;
    std::vector<JsfK> jsf((size_t)count * JUMP_SPAN);
    SpanBatch sb;
    sb.part = part.as<P29>();
    double fp_mults = 0;
    uint32_t longest = 1;
    for (int i = 0; i < OB_MAX; ++i) { const int k = i < count ? i : 0; sb.ng[i] = g2.as<A29>() + ns * k; sb.g[i] = gens[k]; }
    for (int i = 0; i < count; ++i) {
        Fr c[JUMP_SPAN];
        fold_span_coefficients(c, items[i].u + 8 * (size_t)r0);
        for (int b = 0; b < JUMP_SPAN; ++b) {
            jsf[(size_t)i * JUMP_SPAN + b] = jsf_of(glv_split(c[b]));
            longest = std::max(longest, jsf[(size_t)i * JUMP_SPAN + b].len);
            fp_mults += (fold_fp_mults_per_pair(jsf[(size_t)i * JUMP_SPAN + b]) + 2.0 - (b ? 7.0 * jsf[(size_t)i * JUMP_SPAN + b].len : 0.0)) * (double)ns;      // about: one of the eight doubles
        }
    }
    const void* dj = nullptr;
    int rc = up.put(jsf.data(), sizeof(JsfK) * jsf.size(), st, &dj);
    if (rc) return rc;
    FoldTimed timed(st);
    const uint32_t slice = (longest + 7) / 8;
    hipLaunchKernelGGL(k_open_span_slices, dim3(cdiv(ns, GT), count), dim3(8 * GT), 0, st, sb, (const JsfK*)dj, n0, ns, slice);
    hipLaunchKernelGGL(k_open_span_walk, dim3(cdiv(4 * ns, (size_t)GT), count), dim3(GT), 0, st, sb, ns, slice);
    ZK_LAUNCH_CHECK();
    timed.end(0, fp_mults, ns * (size_t)count * (JUMP_SPAN - 1));
    for (int i = 0; i < count; ++i) gens[i] = g2.as<A29>() + ns * i;
    return 0;
}
static int open_batch_launch(const Fr** scalars, const A29** gens, int count, size_t n0, int levels, bool last, int r0, int rounds, const std::function<bool(int)>& t_given, const OpenItem* items, G1Jac* pts, size_t npts,
                             const Fr* U_dev, Arena& arena, JobUploads& up, hipStream_t st, hipStream_t aux, std::vector<hipEvent_t>& events, std::vector<PointDesc>& later) {
    const uint32_t fin = last ? 1u : 0u, n_msm = 3 * (uint32_t)levels + fin;
    const size_t sl_n = n0 + (size_t)levels + 1;
    Scratch& sl = arena.add(sizeof(Fr) * sl_n * count);
    const size_t ncoef = (size_t)n_msm * n0 * count;
    ZK_ARG(ncoef < (1ull << 32), "opening: batched rounds too large");
    uint32_t given = 0, summed = fin;                          // levels whose T is not summed; sums of an opening
    for (int j = 0; j < levels; ++j) {
        if (t_given(r0 + j)) given |= 1u << j;
        summed += t_given(r0 + j) ? 2 : 3;
    }
    SumsPlan plan;
    int rc = sums_plan(plan, summed * (uint32_t)count, n0, (n0 + 1) / 2, (size_t)summed * count * n0, arena);
    if (rc) return rc;
    Scratch& dig = arena.add(digit_bytes(plan.digits) * ncoef);
    if (sl.rc || dig.rc) return sl.rc ? sl.rc : dig.rc;
    TailPtrs tp;
    for (int i = 0; i < OB_MAX; ++i) { const int k = i < count ? i : 0; tp.SL[i] = sl.as<Fr>() + sl_n * k; tp.S[i] = scalars[k]; }
    const TailPtrs all = tp;
    size_t n = n0, off = 0;               // off: where the level just formed starts
    for (int j = 0; j < levels;) {
        if (n > TAIL_SHORT) {
            const int L = std::min(3, levels - j);
            const dim3 grid(cdiv((n + (1u << L) - 1) >> L, TAIL_T), count);
            const Fr* u = U_dev + r0 + j;
            if (L == 3) hipLaunchKernelGGL(k_tail_levels<3>, grid, dim3(TAIL_T), 0, st, tp, u, (uint32_t)rounds, (uint32_t)n);
            else if (L == 2) hipLaunchKernelGGL(k_tail_levels<2>, grid, dim3(TAIL_T), 0, st, tp, u, (uint32_t)rounds, (uint32_t)n);
            else hipLaunchKernelGGL(k_tail_levels<1>, grid, dim3(TAIL_T), 0, st, tp, u, (uint32_t)rounds, (uint32_t)n);
            size_t before = 0;            // the levels in front of the last one
            for (int k = 0; k < L; ++k) { n = (n + 1) / 2; if (k + 1 < L) before += n; }
            for (int i = 0; i < OB_MAX; ++i) { tp.S[i] = tp.SL[i] + before; tp.SL[i] += before + n; }
            off = (size_t)(tp.S[0] - sl.as<Fr>());
            j += L;
        } else {
            hipLaunchKernelGGL(k_tail_scalars, dim3(count), dim3(TAIL_T), 0, st, tp, U_dev + r0 + j, (uint32_t)rounds, (uint32_t)n, (uint32_t)(levels - j));
            off = (size_t)(tp.SL[0] - sl.as<Fr>());
            for (; j < levels; ++j) { n = (n + 1) / 2; if (j + 1 < levels) off += n; }
        }
    }
    ZK_LAUNCH_CHECK();
    const A29* before[OB_MAX];
    for (int i = 0; i < count; ++i) before[i] = gens[i];
    hipLaunchKernelGGL(k_tail_coeffs, dim3(cdiv(n0, TAIL_T), count, n_msm), dim3(TAIL_T), 0, st, dig.p, ncoef, all, U_dev + r0, (uint32_t)rounds, (uint32_t)n0, (uint32_t)levels, given, plan.digits,
                       plan.state, plan.state_words);
    ZK_LAUNCH_CHECK();
    std::vector<MsmDesc> d;
    std::vector<G1Jac*> out;
    for (int it = 0; it < count; ++it)
        for (uint32_t i = 0; i < n_msm; ++i) {
            if (i < 3 * (uint32_t)levels && i % 3 == 0 && (given >> (i / 3) & 1u)) continue;
            d.push_back(MsmDesc{dig.p, before[it], (uint32_t)ncoef, (uint32_t)n0, 1u, (uint32_t)(((size_t)it * n_msm + i) * n0), 1u, 0u, 0u, 0u});
            out.push_back(pts + npts * it + (i == 3 * (uint32_t)levels ? 3 * (size_t)rounds : 3 * (size_t)r0 + i));
        }
    rc = bucket_sums_queue(d, out, n0, plan, arena, up, st, aux, events, later);
    if (rc) return rc;
    if (!last) {
        rc = open_span_fold(gens, count, n0, r0, items, arena, up, st);
        if (rc) return rc;
    }
    for (int it = 0; it < count; ++it) scalars[it] = sl.as<Fr>() + sl_n * it + off;
    return 0;
}
// T of the rounds 1 .. rounds_t - 1 but `again` of every opening from its T of round 0 (above `again`, of that round) and T0, T1 of the rounds below, on st;
// with V_dev of all rounds from the final generators, the final scalars and T0, T1
static int open_unroll_queue(G1Jac* pts, size_t npts, int count, int rounds_t, int again, const Fr* U_dev, const Fr* V_dev, const Fr* const* finals, int rounds, Arena& arena, JobUploads& up, hipStream_t st) {
    if (!V_dev && (rounds_t <= 1 || (rounds_t == 2 && again == 1))) return 0;
    const uint32_t R = (uint32_t)rounds_t, first = V_dev ? 0u : 1u, np = V_dev ? 3 * R + 1 : 3 * (R - 1), terms = (R - first) * np;
    Scratch& aff = arena.add(sizeof(G1Affine) * np);
    Scratch& a29 = arena.add(sizeof(A29) * np * count);
    Scratch& dg = arena.add((size_t)(MW + 1) * terms * count);
    if (aff.rc || a29.rc || dg.rc) return aff.rc ? aff.rc : (a29.rc ? a29.rc : dg.rc);
    std::vector<MsmDesc> d;
    std::vector<G1Jac*> out;
    for (int i = 0; i < count; ++i) {
        g1_normalize_queue<true>(aff.p, pts + npts * i, np, st);
        hipLaunchKernelGGL(k_g1aff_to_a29, dim3(cdiv(np, 256)), dim3(256), 0, st, a29.as<A29>() + (size_t)np * i, aff.as<G1Affine>(), (size_t)np);
        for (uint32_t q = first; q < R; ++q) {
            if (!V_dev && (int)q == again) continue;
            d.push_back(MsmDesc{dg.as<int8_t>() + (size_t)(MW + 1) * terms * i, a29.as<A29>() + (size_t)np * i, terms, np, 1u, (q - first) * np, 1u, 0u, 0u, 0u});
            out.push_back(pts + npts * i + 3 * q);
        }
    }
    if (V_dev) {
        FinalScalars fs;
        for (int i = 0; i < OB_MAX; ++i) fs.s[i] = finals[i < count ? i : 0];
        hipLaunchKernelGGL(k_open_back_digits, dim3(cdiv(terms, 256), count), dim3(256), 0, st, dg.as<int8_t>(), U_dev, V_dev, fs, R);
    } else hipLaunchKernelGGL(k_open_unroll_digits, dim3(cdiv(terms, 256), count), dim3(256), 0, st, dg.as<int8_t>(), U_dev, (uint32_t)rounds, R, (uint32_t)again);
    ZK_LAUNCH_CHECK();
    static_assert(3 * 64 + 1 <= FEW_MAX, "the points of a proof are few");
    std::vector<PointDesc> mine;
    std::vector<hipEvent_t> none;                             // one stream
    int rc = bucket_sums_queue(d, out, np, SumsPlan{}, arena, up, st, st, none, mine);
    if (rc == 0) rc = points_queue(mine, arena, up, st);
    return rc;
}
// rows (optional): commitments of the opened tensor's rows, [pattern][row] as open_cross_sums_queue takes them -- the row
// commitments alone (cross_rounds = 0) or with the cross patterns of the first cross_rounds rounds
static int open_queue(OpenJob& job, const OpenItem* items, int count, size_t n, int rounds, hipStream_t st, hipStream_t aux) {
    ZK_ARG(n >= 1, "zk_g1_open: empty input");
    ZK_ARG(count >= 1 && count <= OB_MAX, "zk_g1_open: a batch holds 1 to 8 openings");
    ZK_ARG(rounds >= 0 && rounds <= 64, "zk_g1_open: bad round count");
    ZK_ARG(sizeof(G1Jac) * (3 * (size_t)rounds + 1) + sizeof(Fr) <= 65536, "zk_g1_open: proof larger than the staging buffer");
    job.st = st;
    job.aux = aux;
    job.arena.streams(st, aux);      // blocks serve kernels of both streams; aux joins st before the job ends
    job.rounds = rounds;
    job.count = count;
    const size_t npts = 3 * (size_t)rounds + 1;
    Scratch& pts = job.arena.add(sizeof(G1Jac) * npts * count);
    if (pts.rc) return pts.rc;
    job.pts = pts.as<G1Jac>();
    std::vector<Fr> hu;           // the challenges, Montgomery form, `rounds` an opening; the row challenges follow
    for (int i = 0; i < count; ++i)
        for (int r = 0; r < rounds; ++r) hu.push_back(to_mont(load_fr(items[i].u + 8 * r)));
    for (int i = 0; i < count; ++i)
        if (items[i].rows)
            for (int j = 0; j < items[i].k_rows; ++j) hu.push_back(to_mont(load_fr(items[i].u_rows + 8 * j)));
    const void* ud = nullptr;
    if (!hu.empty()) {
        int rc = job.up.put(hu.data(), sizeof(Fr) * hu.size(), st, &ud);
        if (rc) return rc;
    }
    const Fr* U_dev = (const Fr*)ud;
    const Fr* urow_dev[OB_MAX];
    {
        size_t at = (size_t)rounds * count;
        for (int i = 0; i < count; ++i) { urow_dev[i] = U_dev + at; if (items[i].rows) at += (size_t)items[i].k_rows; }
    }
    const Fr* cs[OB_MAX];
    const A29* cg[OB_MAX];
    for (int i = 0; i < count; ++i) {
        cs[i] = (const Fr*)items[i].scalars;
        cg[i] = items[i].prep;
        if (!cg[i]) {
            Scratch& g29 = job.arena.add(sizeof(A29) * n);
            if (g29.rc) return g29.rc;
            int rc = open_prep_build(g29.as<A29>(), (const G1Jac*)items[i].gens, n, job.arena, st);
            if (rc) return rc;
            cg[i] = g29.as<A29>();
        }
    }
    auto last_batch = [&](size_t size, int r) { return size * (size_t)count <= (size_t)LAST_N && rounds - r <= TAIL_LEVELS; };
    // commitments of the tensors' rows: which sums they replace (all openings of the batch must bring them)
    bool with_rows = rounds > 0 && n > (size_t)TABLE_MIN_N, comb3 = true, comb1 = true, comb2 = true;
    int cross_r = 64;
    for (int i = 0; i < count; ++i) {
        with_rows = with_rows && items[i].rows != nullptr;
        cross_r = std::min(cross_r, items[i].cross_rounds);
        comb1 = comb1 && items[i].comb != nullptr;
        comb2 = comb2 && items[i].comb2 != nullptr;
        comb3 = comb3 && items[i].comb3 != nullptr;
    }
    int halving = 0;
    {
        size_t sz = n;
        for (int r = 0; r < rounds && !last_batch(sz, r); ++r) { ++halving; sz = (sz + 1) / 2; }
    }
    if (!with_rows || halving == 0) cross_r = 0;
    // three rounds as one fold: their sums all come from cross commitments
    const bool jump = halving > 0 && with_rows && cross_r >= JUMP_ROUNDS && rounds >= JUMP_ROUNDS && !(n & (n - 1)) && n >= (size_t)JUMP_SPAN;
    if (jump) cross_r = JUMP_ROUNDS;
    else cross_r = std::min(cross_r, halving);
    // What round r over `size` generators begins.  Three rounds as a batch of sums beside one fold where a round's fold would leave the chip
    // half empty and take one walk's latency all the same; above that a round at a time, which sums over fewer points.  Openings of 128 x 2^17,
    // the first round alone / in a span: 9.9 / 9.2 ms; of 16 x 2^18, two rounds alone / one and a span: 14.7 / 14.9.  One opening with the line at 2^16, 2^17
    // and 2^18 generators of a job, in ms: of 147456 generators 11.0, 10.4, 11.3; 163840 11.2, 10.8, 11.8; 196608 12.8, 11.8, 12.8; 229376 14.0, 13.4,
    // 14.0; 2^18 14.9, 14.2, 15.3; of 2^17 9.0, 8.9.  Three of 65536 at once 12.8, 12.4, 12.4; five of 32768 11.5, 11.0, 12.0; six 13.5, 12.7, 13.3.
    enum Step { LAST, SPAN, ROUND };
    auto step_of = [&](size_t size, int r) {
        if (last_batch(size, r)) return LAST;
        const bool comb = r == 0 ? comb1 : (r == 1 && comb2);
        return !comb && r >= cross_r && rounds - r >= JUMP_ROUNDS && size * (size_t)count <= (size_t)SPAN_MAX_N ? SPAN : ROUND;
    };
    // T of round 0 from the row commitments or summed; T of the rounds from 1 to t_rounds - 1 unrolled from it.  The tensor's commitments say what
    // T is for the rounds they have cross patterns for, or else while a round has more than TABLE_MIN_N generators: the first round behind those,
    // t_again, has its T summed, and the rounds behind it follow from that.  A last batch that is so small that its own T cost less than the
    // unrolling's chain of launches behind it sums them, and the unrolling of the rounds before it runs beside it: openings of 8192
    // generators 2.15 ms by sums, 2.68 unrolled, of 16384 3.20 and 2.83.
    // An opening without row commitments whose last batch is larger has all T from its final generator and scalar, behind the last batch as well.
    int t_rounds = rounds, t_again = 0;
    bool unroll_early = false, back = false;
    {
        if (cross_r > 0) t_again = cross_r;
        else if (with_rows)
            for (size_t sz = n; t_again < rounds && sz > (size_t)TABLE_MIN_N; sz = (sz + 1) / 2) ++t_again;
        size_t sz = n;
        int r = 0;
        if (jump) { sz = n >> JUMP_ROUNDS; r = JUMP_ROUNDS; }
        while (r < rounds && step_of(sz, r) != LAST)
            for (int q = step_of(sz, r) == SPAN ? JUMP_ROUNDS : 1; q > 0; --q) { sz = (sz + 1) / 2; ++r; }
        if (r < rounds && sz * (size_t)count <= (size_t)T_SUM_MAX_N) {
            t_rounds = std::min(std::max(r + 1, t_again), rounds);
            unroll_early = t_rounds == r + 1;
        }
        if (t_again >= t_rounds) t_again = 0;
        size_t left = n;
        for (int q = 0; q < rounds && left > 1; ++q) left = (left + 1) / 2;
        back = !with_rows && !unroll_early && r < rounds && left == 1;
    }
    const Fr* V_dev = nullptr;
    if (back) {                                              // 1 / (u (1 - u)), all by one inversion
        const size_t m = (size_t)rounds * count;
        std::vector<Fr> w(m), v(m);
        Fr run = big_one_mont<8>();
        for (size_t i = 0; i < m; ++i) {
            w[i] = mont_mul(hu[i], sub(big_one_mont<8>(), hu[i]));
            v[i] = run;
            run = mont_mul(run, w[i]);
        }
        back = !is_zero(run);
        if (back) {
            run = mont_inverse(run);
            for (size_t i = m; i-- > 0;) { v[i] = mont_mul(v[i], run); run = mont_mul(run, w[i]); }
            const void* vd = nullptr;
            int rc = job.up.put(v.data(), sizeof(Fr) * m, st, &vd);
            if (rc) return rc;
            V_dev = (const Fr*)vd;
        }
    }
    auto t_given = [&](int r) { return back || (r == 0 ? with_rows : r < t_rounds && r != t_again); };
    std::vector<PointDesc> later;        // bucket reductions that nothing waits for before the end: one launch behind the last round
    if (t_rounds > 1 || back) GLAUNCH(k_g1_fill, npts * count, st, job.pts, g1_infinity(), npts * count);
    if (with_rows) {
        int rc = join_streams(st, aux, job.events);          // the challenges travel on st
        if (rc == 0) rc = open_cross_sums_queue(items, count, (uint32_t)cross_r, job.pts, npts, urow_dev, U_dev, rounds, job.arena, job.up, aux, job.events, later);
        if (rc) return rc;
    }
    size_t size = n;
    int r = 0;
    bool tail_done = false;
    if (jump) {
        const size_t ns = n >> JUMP_ROUNDS;
        if (comb3) {
            Scratch& s2 = job.arena.add(sizeof(Fr) * ns * count);
            Scratch& g2 = job.arena.add(sizeof(A29) * ns * count);
            if (s2.rc) return s2.rc;
            if (g2.rc) return g2.rc;
            JumpBatch jb;
            double fp_mults = 0;
            for (int i = 0; i < OB_MAX; ++i) {
                const int k = i < count ? i : 0;
                JumpItem& f = jb.it[i];
                f.ns = s2.as<Fr>() + ns * k; f.ng = g2.as<A29>() + ns * k; f.s = cs[k]; f.g = cg[k]; f.tab = items[k].comb3;
                for (int q = 0; q < JUMP_ROUNDS; ++q) f.u_mont[q] = to_mont(load_fr(items[k].u + 8 * q));
                Fr c[JUMP_SPAN];
                fold_span_coefficients(c, items[k].u);
                for (int b = 0; b < JUMP_TABS; ++b) {
                    f.ck[b] = comb_of(glv_split(c[b]));
                    if (i < count) fp_mults += (comb_fp_mults_per_pair(f.ck[b]) - 7.0 * COMB_W - 19.0) * (double)ns;
                }
                if (i < count) fp_mults += (7.0 * COMB_W + 19.0) * (double)ns;
            }
            FoldTimed timed(st);
            hipLaunchKernelGGL(k_open_fold_jump, dim3(cdiv(ns, GT), count), dim3(GT), 0, st, jb, ns);
            ZK_LAUNCH_CHECK();
            timed.end(2, fp_mults, ns * (size_t)count * (JUMP_SPAN - 1));       // pairs the three rounds fold: 4 + 2 + 1 per result
            for (int i = 0; i < count; ++i) { cs[i] = s2.as<Fr>() + ns * i; cg[i] = g2.as<A29>() + ns * i; }
        } else {
            const size_t sl_n = n;          // levels 1 to 3 of the scalars
            Scratch& sl = job.arena.add(sizeof(Fr) * sl_n * count);
            if (sl.rc) return sl.rc;
            TailPtrs tp;
            for (int i = 0; i < OB_MAX; ++i) { const int k = i < count ? i : 0; tp.SL[i] = sl.as<Fr>() + sl_n * k; tp.S[i] = cs[k]; }
            hipLaunchKernelGGL(k_tail_levels<3>, dim3(cdiv(ns, TAIL_T), count), dim3(TAIL_T), 0, st, tp, U_dev, (uint32_t)rounds, (uint32_t)n);
            ZK_LAUNCH_CHECK();
            int rc = open_span_fold(cg, count, n, 0, items, job.arena, job.up, st);
            if (rc) return rc;
            for (int i = 0; i < count; ++i) cs[i] = sl.as<Fr>() + sl_n * i + n / 2 + n / 4;
        }
        size = ns;
        r = JUMP_ROUNDS;
    }
    auto reductions = [&]() {            // on aux: the sums that nothing waited for, and T of the rounds that follow from them
        int rc = points_queue(later, job.arena, job.up, aux);
        if (rc == 0 && unroll_early) rc = open_unroll_queue(job.pts, npts, count, t_rounds, t_again, U_dev, nullptr, nullptr, rounds, job.arena, job.up, aux);
        return rc;
    };
    while (r < rounds) {
        const Step step = step_of(size, r);
        if (step == LAST) {
            if (unroll_early && aux != st) {
                int rc = reductions();
                if (rc) return rc;
            }
            std::vector<PointDesc> mine;
            int rc = open_batch_launch(cs, cg, count, size, rounds - r, true, r, rounds, t_given, items, job.pts, npts, U_dev, job.arena, job.up, st, st, job.events, mine);
            if (rc == 0) rc = points_queue(mine, job.arena, job.up, st);
            if (rc) return rc;
            tail_done = true;
            break;
        }
        if (step == SPAN) {
            int rc = open_batch_launch(cs, cg, count, size, JUMP_ROUNDS, false, r, rounds, t_given, items, job.pts, npts, U_dev, job.arena, job.up, st, aux, job.events, later);
            if (rc) return rc;
            size = (((size + 1) / 2 + 1) / 2 + 1) / 2;
            r += JUMP_ROUNDS;
            continue;
        }
        const size_t ns = (size + 1) / 2;
        Scratch& s2 = job.arena.add(sizeof(Fr) * ns * count);
        Scratch& g2 = job.arena.add(sizeof(A29) * ns * count);
        if (s2.rc) return s2.rc;
        if (g2.rc) return g2.rc;
        RoundItem ri[OB_MAX];
        for (int i = 0; i < count; ++i) {
            ri[i] = RoundItem{s2.as<Fr>() + ns * i, g2.as<A29>() + ns * i, cs[i], cg[i], load_fr(items[i].u + 8 * r)};
            if (r == 0) ri[i].comb = items[i].comb;
            if (r == 1) { ri[i].comb2 = items[i].comb2; ri[i].u_prev = load_fr(items[i].u + 8 * (r - 1)); }
        }
        const int given = r < cross_r ? 2 : (t_given(r) ? 1 : 0);
        int rc = open_round_launch(ri, count, size, std::min(r, 2), given, job.pts + 3 * (size_t)r, npts, job.arena, job.up, st, aux, job.events, later);
        if (rc) return rc;
        for (int i = 0; i < count; ++i) { cs[i] = ri[i].new_scalars; cg[i] = ri[i].new_gens; }
        size = ns;
        ++r;
    }
    {
        int rc = unroll_early && aux != st && tail_done ? 0 : reductions();
        if (rc == 0) rc = join_streams(aux, st, job.events);
        if (rc == 0 && !unroll_early) rc = open_unroll_queue(job.pts, npts, count, t_rounds, t_again, U_dev, V_dev, cs, rounds, job.arena, job.up, st);
        if (rc) return rc;
    }
    if (!tail_done)
        for (int i = 0; i < count; ++i) hipLaunchKernelGGL(k_open_finish, dim3(1), dim3(GT), 0, st, job.pts + npts * i, cg[i], (uint32_t)rounds);
    g1_normalize_queue<false>(pts.p, job.pts, npts * count, st);
    ZK_LAUNCH_CHECK();
    for (int i = 0; i < count; ++i) job.final_scalar[i] = cs[i];
    return 0;
}
// waits for the job's stream and copies the proof points and the folded scalars out: opening i's points at
// proof_host + i * (3 rounds + 1) * 36, its scalar at final_scalar_host + i * 8
static int open_collect(OpenJob& job, uint32_t* proof_host, uint32_t* final_scalar_host) {
    const size_t npts = 3 * (size_t)job.rounds + 1;
    void* stage = nullptr;
    int rc = staging(&stage, sizeof(G1Jac) * npts + sizeof(Fr));
    if (rc) return rc;
    for (int i = 0; i < job.count; ++i) {
        ZK_HIP(hipMemcpyAsync(stage, job.pts + npts * i, sizeof(G1Jac) * npts, hipMemcpyDeviceToHost, job.st));
        ZK_HIP(hipMemcpyAsync((char*)stage + sizeof(G1Jac) * npts, job.final_scalar[i], sizeof(Fr), hipMemcpyDeviceToHost, job.st));
        ZK_HIP(hipStreamSynchronize(job.st));
        memcpy(proof_host + 36 * npts * i, stage, sizeof(G1Jac) * npts);
        memcpy(final_scalar_host + 8 * (size_t)i, (char*)stage + sizeof(G1Jac) * npts, sizeof(Fr));
    }
    return 0;
}
// proof_host receives 3*rounds + 1 points: T, T0, T1 of every round, then the folded generator; all normalised to
// z = 1 (infinity: all-zero limbs).  final_scalar_host: the folded scalar.
int zk_g1_open(uint32_t* proof_host, uint32_t* final_scalar_host, const void* scalars, const void* gens, size_t n, const uint32_t* u, int rounds, void* stv) {
    if (n > (size_t)LAST_N) {          // folds and bucket sums beside each other, on two streams
        void* h = nullptr;
        int rc = zk_g1_open_begin(&h, scalars, gens, n, u, rounds, stv);
        return rc ? rc : zk_g1_open_end(h, proof_host, final_scalar_host);
    }
    OpenJob job;
    const OpenItem item{scalars, gens, nullptr, u};
    int rc = open_queue(job, &item, 1, n, rounds, (hipStream_t)stv, (hipStream_t)stv);
    if (rc) { (void)hipStreamSynchronize((hipStream_t)stv); return rc; }
    return open_collect(job, proof_host, final_scalar_host);
}
// The same in two halves.  begin queues the recursion on a stream of the library's own, ordered after everything queued
// on `stream` so far, and returns at once; the caller goes on using `stream`, and both run side by side.  scalars and gens
// must stay alive and unmodified until end, which waits for the opening, delivers its results and releases its buffers.
static int open_begin_impl(void** handle, const OpenItem* items, int count, size_t n, int rounds, void* stv) {
    ZK_ARG(handle != nullptr, "zk_g1_open_begin: null handle");
    // The folds on one stream, the bucket sums on another.  A job whose rounds are one batch has no folds: one stream, so that the others
    // (and their hardware queues) are left to other jobs.
    hipStream_t side = nullptr, aux = nullptr;
    if (n * (size_t)count <= (size_t)LAST_N && rounds <= TAIL_LEVELS) aux = side = side_stream(0);
    else opening_streams(&side, &aux);
    ZK_ARG(side != nullptr && aux != nullptr, "zk_g1_open_begin: could not create a stream");
    // what open_queue refuses is refused here, before anything is handed to the launch thread
    ZK_ARG(n >= 1, "zk_g1_open: empty input");
    ZK_ARG(count >= 1 && count <= OB_MAX, "zk_g1_open: a batch holds 1 to 8 openings");
    ZK_ARG(rounds >= 0 && rounds <= 64, "zk_g1_open: bad round count");
    ZK_ARG(sizeof(G1Jac) * (3 * (size_t)rounds + 1) + sizeof(Fr) <= 65536, "zk_g1_open: proof larger than the staging buffer");
    std::unique_ptr<OpenJob> job(new OpenJob);
    ZK_HIP(hipEventCreateWithFlags(&job->ready, hipEventDisableTiming));
    ZK_HIP(hipEventRecord(job->ready, (hipStream_t)stv));
    ZK_HIP(hipStreamWaitEvent(side, job->ready, 0));
    pool_note_wait((hipStream_t)stv, side);
    if (!launcher_enabled()) {
        int rc = open_queue(*job, items, count, n, rounds, side, aux);
        if (rc) {
            (void)hipStreamSynchronize(side);
            (void)hipStreamSynchronize(aux);
            for (hipEvent_t e : job->events) (void)hipEventDestroy(e);
            (void)hipEventDestroy(job->ready);
            return rc;
        }
        *handle = job.release();
        return 0;
    }
    // The launch thread queues the job's few hundred launches (a millisecond of host time an opening) while the caller
    // goes on; zk_g1_open_end waits for the ticket and reports what queuing returned.  The challenge arrays are the
    // caller's and only valid during this call: the job takes copies.
    struct Owned { OpenItem items[OB_MAX]; std::vector<uint32_t> u[OB_MAX], u_rows[OB_MAX]; };
    std::shared_ptr<Owned> own(new Owned);
    for (int i = 0; i < count; ++i) {
        own->items[i] = items[i];
        own->u[i].assign(items[i].u, items[i].u + 8 * (size_t)rounds);
        own->items[i].u = own->u[i].data();
        if (items[i].rows && items[i].k_rows > 0) {
            own->u_rows[i].assign(items[i].u_rows, items[i].u_rows + 8 * (size_t)items[i].k_rows);
            own->items[i].u_rows = own->u_rows[i].data();
        }
    }
    OpenJob* j = job.get();
    j->st = side;
    j->aux = aux;
    j->ticket = launcher_submit([j, own, count, n, rounds, side, aux] {
        j->queue_rc = open_queue(*j, own->items, count, n, rounds, side, aux);
        if (j->queue_rc) j->queue_err = last_error_text();
    });
    *handle = job.release();
    return 0;
}
int zk_g1_open_begin(void** handle, const void* scalars, const void* gens, size_t n, const uint32_t* u, int rounds, void* stv) {
    const OpenItem item{scalars, gens, nullptr, u};
    return open_begin_impl(handle, &item, 1, n, rounds, stv);
}
// Generators prepared once for any number of openings against them: their affine 29-bit-limb form
// (weight-independent; n points of 112 bytes).  The handle is freed with zk_g1_open_prepared_free
// once no opening that uses it is pending.
struct OpenPrepared { void* a29 = nullptr; size_t n = 0; void* comb = nullptr; void* comb2 = nullptr; void* comb3 = nullptr; size_t table_bytes = 0; };      // comb3: k_open_fold_jump's tables (instead of the other two)
static int open_prepare_impl(void** prepared, const void* gens, size_t n, int table_mode, void* stv);
int zk_g1_open_prepare(void** prepared, const void* gens, size_t n, void* stv) { return open_prepare_impl(prepared, gens, n, 2, stv); }
int zk_g1_open_prepare_tables(void** prepared, const void* gens, size_t n, int tables, void* stv) {
    ZK_ARG(tables >= 0 && tables <= 3, "zk_g1_open_prepare_tables: tables 0 to 3");
    return open_prepare_impl(prepared, gens, n, tables, stv);
}
// bytes of fold tables that zk_g1_open_prepare_tables(.., tables) keeps for n generators (0 where that mode makes none for this n)
static size_t open_table_bytes(size_t n, int tables) {
    if (tables >= 3 && !(n & (n - 1)) && (n >> JUMP_ROUNDS) >= (size_t)TABLE_MIN_N) return sizeof(A29) * (n >> JUMP_ROUNDS) * COMB_N * JUMP_TABS;
    if (tables < 1 || n <= (size_t)TABLE_MIN_N) return 0;
    const size_t np = (n + 1) / 2, nq = (np + 1) / 2;
    size_t b = sizeof(A29) * np * COMB_N;
    if (tables >= 2 && np > (size_t)TABLE_MIN_N) b += sizeof(A29) * 2 * nq * COMB_N;
    return b;
}
size_t zk_g1_open_table_bytes(size_t n, int tables) { return open_table_bytes(n, tables < 0 ? 0 : (tables > 3 ? 3 : tables)); }
// The richest tables that fit `max_table_bytes`: mode `want` (0..3) if its tables fit, else the next smaller mode, down to none.
int zk_g1_open_prepare_budget(void** prepared, const void* gens, size_t n, int want, size_t max_table_bytes, int* tables_made, void* stv) {
    ZK_ARG(want >= 0 && want <= 3, "zk_g1_open_prepare_budget: tables 0 to 3");
    int mode = want;
    while (mode > 0 && open_table_bytes(n, mode) > max_table_bytes) --mode;
    if (tables_made) *tables_made = mode;
    return open_prepare_impl(prepared, gens, n, mode, stv);
}
size_t zk_g1_open_prepared_table_bytes(const void* prepared) { return prepared ? ((const OpenPrepared*)prepared)->table_bytes : 0; }
static int open_prepare_impl(void** prepared, const void* gens, size_t n, int table_mode, void* stv) {
    hipStream_t st = (hipStream_t)stv;
    ZK_ARG(prepared != nullptr && n >= 1, "zk_g1_open_prepare: null handle or no generators");
    std::unique_ptr<OpenPrepared> pr(new OpenPrepared);
    int rc = pool_alloc(&pr->a29, sizeof(A29) * n, st);
    if (rc) return rc;
    pr->n = n;
    {
        Arena arena(st);
        rc = open_prep_build((A29*)pr->a29, (const G1Jac*)gens, n, arena, st);
        // The combs of the first two rounds, for each round over more than TABLE_MIN_N generators: how many openings share a job is not known
        // here, and a job of more than LAST_N generators in all folds these rounds.  Entry-major tables of the subset sums of
        // 2^(j COMB_W) P over the round's prepared points P (the pair differences D; for the second round F and H, see k_open_fold_comb), built from elementwise point kernels -- the
        // teeth by repeated doubling (an addition of an array to itself), entry m = entry (m without its lowest bit) + entry
        // (that bit).
        // The tables only make the folds cheaper: ZKLLM_OPEN_TABLES = 0 or 1 keeps none or the first round's alone (28 KB
        // per generator pair and round), and when the device has no room for them or for their construction the handle
        // is made without them -- those rounds then walk (k_open_fold29), the results are the same.
        static const int env_rounds = [] { const char* e = getenv("ZKLLM_OPEN_TABLES"); return e ? atoi(e) : -1; }();
        const int table_rounds = env_rounds >= 0 ? env_rounds : table_mode;
        // mode 3: the seven tables of k_open_fold_jump in place of those two (as large as both together); only for a power of
        // two of generators that leaves at least TABLE_MIN_N after three folds
        const bool jump = table_rounds >= 3 && !(n & (n - 1)) && (n >> JUMP_ROUNDS) >= (size_t)TABLE_MIN_N;
        if (rc == 0 && jump) {
            const size_t no = n >> JUMP_ROUNDS, ne = no * COMB_N * JUMP_TABS;
            int trc = pool_alloc(&pr->comb3, sizeof(A29) * ne, st);
            Scratch& aff = arena.add(sizeof(G1Affine) * n);
            Scratch& tj = arena.add(sizeof(G1Jac) * ne);
            Scratch& ta = arena.add(sizeof(G1Affine) * ne);
            Scratch& tmp = arena.add(sizeof(G1Jac) * no);
            if (trc == 0) trc = aff.rc ? aff.rc : (tj.rc ? tj.rc : (ta.rc ? ta.rc : tmp.rc));
            if (trc) {
                if (pr->comb3) (void)pool_free(pr->comb3, st, true);
                pr->comb3 = nullptr;
            } else {
                static_assert(COMB_W % 2 == 0, "the doublings alternate between two buffers and must end in the table");
                g1_normalize_queue<true>(aff.p, (const G1Jac*)gens, n, st);
                for (int b = 0; b < JUMP_TABS; ++b) {
                    G1Jac* T = tj.as<G1Jac>() + (size_t)b * COMB_N * no;
                    auto entry = [&](int m) { return T + (size_t)(m - 1) * no; };
                    hipLaunchKernelGGL(k_open_span_diff, dim3(cdiv(no, GT)), dim3(GT), 0, st, T, aff.as<G1Affine>(), (uint32_t)JUMP_SPAN, (uint32_t)b, no);
                    for (int t = 1; t < COMB_A; ++t) {
                        const G1Jac* src = entry(1 << (t - 1));
                        for (int k = 0; k < COMB_W; ++k) {          // no launch writes what it reads
                            G1Jac* dst = (k & 1) ? entry(1 << t) : tmp.as<G1Jac>();
                            hipLaunchKernelGGL(k_g1_add, dim3(cdiv(no, GT)), dim3(GT), 0, st, dst, src, src, no, no, 0);
                            src = dst;
                        }
                    }
                    for (int m = 3; m <= COMB_N; ++m) {
                        const int prev = m & (m - 1);
                        if (!prev) continue;
                        hipLaunchKernelGGL(k_g1_add, dim3(cdiv(no, GT)), dim3(GT), 0, st, entry(m), entry(prev), entry(m ^ prev), no, no, 0);
                    }
                }
                g1_normalize_queue<true>(ta.p, tj.as<G1Jac>(), ne, st);
                hipLaunchKernelGGL(k_g1aff_to_a29, dim3(cdiv(ne, 256)), dim3(256), 0, st, (A29*)pr->comb3, ta.as<G1Affine>(), ne);
                if (hipGetLastError() != hipSuccess) rc = hip_fail(hipErrorLaunchFailure, "jump table build", __FILE__, __LINE__);
            }
        }
        if (rc == 0 && n > (size_t)TABLE_MIN_N && table_rounds >= 1 && !pr->comb3) {
            const size_t np = (n + 1) / 2, ne = np * COMB_N;
            const size_t nq = (np + 1) / 2, ne2 = nq * COMB_N;        // second round: two tables over the pairs of pairs
            bool second = np > (size_t)TABLE_MIN_N && table_rounds >= 2;   // that round is a fold too
            int trc = pool_alloc(&pr->comb, sizeof(A29) * ne, st);
            if (trc == 0 && second && pool_alloc(&pr->comb2, sizeof(A29) * 2 * ne2, st) != 0) { pr->comb2 = nullptr; second = false; }
            const size_t nt = second ? std::max(ne, 2 * ne2) : ne;
            Scratch& aff = arena.add(sizeof(G1Affine) * n);
            Scratch& tj = arena.add(sizeof(G1Jac) * nt);
            Scratch& ta = arena.add(sizeof(G1Affine) * nt);
            Scratch& tmp = arena.add(sizeof(G1Jac) * np);
            if (trc == 0) trc = aff.rc ? aff.rc : (tj.rc ? tj.rc : (ta.rc ? ta.rc : tmp.rc));
            if (trc) {                                                // nothing has been queued on the tables yet
                if (pr->comb) (void)pool_free(pr->comb, st, true);
                if (pr->comb2) (void)pool_free(pr->comb2, st, true);
                pr->comb = pr->comb2 = nullptr;
            } else {
                static_assert(COMB_W % 2 == 0, "the doublings alternate between two buffers and must end in the table");
                // T[0 .. cnt) holds entry 1 (the points themselves); fills the other COMB_N - 1 entries, cnt points each
                auto fill = [&](G1Jac* T, size_t cnt) {
                    auto entry = [&](int m) { return T + (size_t)(m - 1) * cnt; };
                    for (int t = 1; t < COMB_A; ++t) {
                        const G1Jac* src = entry(1 << (t - 1));
                        for (int k = 0; k < COMB_W; ++k) {          // no launch writes what it reads
                            G1Jac* dst = (k & 1) ? entry(1 << t) : tmp.as<G1Jac>();
                            hipLaunchKernelGGL(k_g1_add, dim3(cdiv(cnt, GT)), dim3(GT), 0, st, dst, src, src, cnt, cnt, 0);
                            src = dst;
                        }
                    }
                    for (int m = 3; m <= COMB_N; ++m) {
                        const int prev = m & (m - 1);
                        if (!prev) continue;
                        hipLaunchKernelGGL(k_g1_add, dim3(cdiv(cnt, GT)), dim3(GT), 0, st, entry(m), entry(prev), entry(m ^ prev), cnt, cnt, 0);
                    }
                };
                G1Jac* T = tj.as<G1Jac>();
                g1_normalize_queue<true>(aff.p, (const G1Jac*)gens, n, st);
                hipLaunchKernelGGL(k_open_pair_points, dim3(cdiv(np, GT)), dim3(GT), 0, st, T, aff.as<G1Affine>(), n, np);
                fill(T, np);
                g1_normalize_queue<true>(ta.p, tj.as<G1Jac>(), ne, st);
                hipLaunchKernelGGL(k_g1aff_to_a29, dim3(cdiv(ne, 256)), dim3(256), 0, st, (A29*)pr->comb, ta.as<G1Affine>(), ne);
                if (second) {
                    // F from the odd-numbered generators, H from the first round's differences (entry 1 of its table, affine in ta);
                    // both are read before the buffers they sit in are written again
                    hipLaunchKernelGGL(k_open_pair_diff, dim3(cdiv(nq, GT)), dim3(GT), 0, st, T, aff.as<G1Affine>(), (size_t)1, (size_t)2, n / 2, nq);
                    hipLaunchKernelGGL(k_open_pair_diff, dim3(cdiv(nq, GT)), dim3(GT), 0, st, T + ne2, ta.as<G1Affine>(), (size_t)0, (size_t)1, np, nq);
                    fill(T, nq);
                    fill(T + ne2, nq);
                    g1_normalize_queue<true>(ta.p, tj.as<G1Jac>(), 2 * ne2, st);
                    hipLaunchKernelGGL(k_g1aff_to_a29, dim3(cdiv(2 * ne2, 256)), dim3(256), 0, st, (A29*)pr->comb2, ta.as<G1Affine>(), 2 * ne2);
                }
                if (rc == 0 && hipGetLastError() != hipSuccess) rc = hip_fail(hipErrorLaunchFailure, "comb build", __FILE__, __LINE__);
            }
        }
        // the temporaries go back to the allocator only when the stream has drained
        if (hipStreamSynchronize(st) != hipSuccess && rc == 0) rc = hip_fail(hipGetLastError(), "zk_g1_open_prepare sync", __FILE__, __LINE__);
        arena.mark_idle();
    }
    // (openings read the prepared form on the library's own streams: it is complete before the handle is handed out)
    if (rc) {
        (void)hipStreamSynchronize(st);
        pool_free(pr->a29, st, true);
        if (pr->comb) pool_free(pr->comb, st, true);
        if (pr->comb2) pool_free(pr->comb2, st, true);
        if (pr->comb3) pool_free(pr->comb3, st, true);
        return rc;
    }
    if (pr->comb3) pr->table_bytes += sizeof(A29) * (n >> JUMP_ROUNDS) * COMB_N * JUMP_TABS;
    if (pr->comb) pr->table_bytes += sizeof(A29) * ((n + 1) / 2) * COMB_N;
    if (pr->comb2) pr->table_bytes += sizeof(A29) * 2 * (((n + 1) / 2 + 1) / 2) * COMB_N;
    *prepared = pr.release();
    return 0;
}
int zk_g1_open_prepared_free(void* prepared) {
    if (!prepared) return 0;
    OpenPrepared* pr = (OpenPrepared*)prepared;
    int rc = pool_free(pr->a29, nullptr);
    if (pr->comb) (void)pool_free(pr->comb, nullptr);
    if (pr->comb2) (void)pool_free(pr->comb2, nullptr);
    if (pr->comb3) (void)pool_free(pr->comb3, nullptr);
    delete pr;
    return rc;
}
int zk_g1_open_begin_prepared(void** handle, const void* scalars, const void* prepared, const uint32_t* u, int rounds, void* stv) {
    ZK_ARG(prepared != nullptr, "zk_g1_open_begin_prepared: null generators");
    const OpenPrepared* pr = (const OpenPrepared*)prepared;
    OpenItem item{scalars, nullptr, (const A29*)pr->a29, u, (const A29*)pr->comb, (const A29*)pr->comb2};
    item.comb3 = (const A29*)pr->comb3;
    return open_begin_impl(handle, &item, 1, pr->n, rounds, stv);
}
// `count` (1 to 8) openings against prepared generator sets of one size and with one round count, as ONE job: every
// kernel of a round is launched once for all of them, so the late rounds have count times the waves.  u: opening i's
// challenges at u + i * rounds * 8.  zk_g1_open_end_batch delivers opening i's points at proof_host + i * (3 rounds + 1) * 36
// and its folded scalar at final_scalar_host + i * 8.
int zk_g1_open_begin_batch(void** handle, int count, const void* const* scalars, const void* const* prepared, const uint32_t* u, int rounds, void* stv) {
    ZK_ARG(count >= 1 && count <= OB_MAX, "zk_g1_open_begin_batch: 1 to 8 openings");
    ZK_ARG(scalars != nullptr && prepared != nullptr && u != nullptr, "zk_g1_open_begin_batch: null argument");
    OpenItem items[OB_MAX];
    size_t n = 0;
    for (int i = 0; i < count; ++i) {
        ZK_ARG(prepared[i] != nullptr && scalars[i] != nullptr, "zk_g1_open_begin_batch: null opening");
        const OpenPrepared* pr = (const OpenPrepared*)prepared[i];
        if (i == 0) n = pr->n;
        ZK_ARG(pr->n == n, "zk_g1_open_begin_batch: the generator sets differ in size");
        items[i] = OpenItem{scalars[i], nullptr, (const A29*)pr->a29, u + (size_t)i * rounds * 8, (const A29*)pr->comb, (const A29*)pr->comb2};
    }
    return open_begin_impl(handle, items, count, n, rounds, stv);
}
// zk_g1_open_begin_batch for vectors that are row folds of committed tensors: rows[i] holds tensor i's nrows[i] row
// commitments under the same generators, u_rows[i] the k_rows[i] challenges its rows were folded with (lowest row bit
// first, 2^k_rows >= nrows).  T of the first round is then the same combination of the row commitments -- equal as a group
// element to the sum over all generators that zk_g1_open_begin_batch computes, provided the commitments are the tensor's.
int zk_g1_open_begin_batch_rows(void** handle, int count, const void* const* scalars, const void* const* prepared, const uint32_t* u, int rounds,
                                const void* const* rows, const uint32_t* nrows, const uint32_t* const* u_rows, const int* k_rows, int cross_rounds, void* stv) {
    ZK_ARG(cross_rounds >= 0 && cross_rounds <= 4, "zk_g1_open_begin_batch_rows: 0 to 4 rounds of cross commitments");
    ZK_ARG(count >= 1 && count <= OB_MAX, "zk_g1_open_begin_batch_rows: 1 to 8 openings");
    ZK_ARG(scalars != nullptr && prepared != nullptr && u != nullptr && rows != nullptr && nrows != nullptr && u_rows != nullptr && k_rows != nullptr, "zk_g1_open_begin_batch_rows: null argument");
    OpenItem items[OB_MAX];
    size_t n = 0;
    for (int i = 0; i < count; ++i) {
        ZK_ARG(prepared[i] != nullptr && scalars[i] != nullptr && rows[i] != nullptr, "zk_g1_open_begin_batch_rows: null opening");
        ZK_ARG(nrows[i] >= 1 && k_rows[i] >= 0 && k_rows[i] <= 31 && ((uint64_t)1 << k_rows[i]) >= nrows[i] && (k_rows[i] == 0 || u_rows[i] != nullptr), "zk_g1_open_begin_batch_rows: rows and row challenges do not fit");
        const OpenPrepared* pr = (const OpenPrepared*)prepared[i];
        if (i == 0) n = pr->n;
        ZK_ARG(pr->n == n, "zk_g1_open_begin_batch_rows: the generator sets differ in size");
        items[i] = OpenItem{scalars[i], nullptr, (const A29*)pr->a29, u + (size_t)i * rounds * 8, (const A29*)pr->comb, (const A29*)pr->comb2, rows[i], nrows[i], u_rows[i], k_rows[i], cross_rounds,
                            (const A29*)pr->comb3};
    }
    return open_begin_impl(handle, items, count, n, rounds, stv);
}
int zk_g1_open_end_batch(void* handle, uint32_t* proof_host, uint32_t* final_scalar_host) { return zk_g1_open_end(handle, proof_host, final_scalar_host); }
int zk_g1_open_end(void* handle, uint32_t* proof_host, uint32_t* final_scalar_host) {
    ZK_ARG(handle != nullptr, "zk_g1_open_end: null handle");
    std::unique_ptr<OpenJob> job((OpenJob*)handle);
    launcher_wait(job->ticket);
    job->ticket = 0;
    int rc = job->queue_rc;
    if (rc) set_error(rc, job->queue_err);
    else rc = open_collect(*job, proof_host, final_scalar_host);
    if (rc) { (void)hipStreamSynchronize(job->st); (void)hipStreamSynchronize(job->aux); }
    job->arena.mark_idle();          // both streams have drained behind the job's last kernel
    (void)hipEventDestroy(job->ready);
    for (hipEvent_t e : job->events) (void)hipEventDestroy(e);
    return rc;
}

// Measurement: time every launch of the opening's fold kernel between begin and read with events on the launch stream.
static double g_fold_method_ms[3] = {0, 0, 0};
static unsigned long long g_fold_method_launches[3] = {0, 0, 0}, g_fold_method_pairs[3] = {0, 0, 0};
static double g_fold_method_mults[3] = {0, 0, 0};
int zk_prof_fold_begin(void) {
    for (auto& e : g_fold_timer.ev) { (void)hipEventDestroy(e.first); (void)hipEventDestroy(e.second); }
    g_fold_timer.ev.clear();
    g_fold_timer.method.clear();
    g_fold_timer.fp_mults = 0;
    g_fold_timer.pairs = 0;
    for (int m = 0; m < 3; ++m) { g_fold_timer.m_mults[m] = 0; g_fold_timer.m_pairs[m] = 0; }
    g_fold_timer.on = true;
    return 0;
}
// total_ms / launches: summed durations and number of timed launches; fp_mults: Fp multiplications they performed; pairs: pairs folded
int zk_prof_fold_read(double* total_ms, unsigned long long* launches, double* fp_mults, unsigned long long* pairs) {
    g_fold_timer.on = false;
    double tot = 0;
    for (int m = 0; m < 3; ++m) { g_fold_method_ms[m] = 0; g_fold_method_launches[m] = 0; }
    for (size_t i = 0; i < g_fold_timer.ev.size(); ++i) {
        auto& e = g_fold_timer.ev[i];
        ZK_HIP(hipEventSynchronize(e.second));
        float ms = 0;
        ZK_HIP(hipEventElapsedTime(&ms, e.first, e.second));
        tot += ms;
        const int m = i < g_fold_timer.method.size() ? g_fold_timer.method[i] : 0;
        g_fold_method_ms[m] += ms;
        g_fold_method_launches[m] += 1;
    }
    for (int m = 0; m < 3; ++m) { g_fold_method_mults[m] = g_fold_timer.m_mults[m]; g_fold_method_pairs[m] = g_fold_timer.m_pairs[m]; }
    *total_ms = tot;
    *launches = g_fold_timer.ev.size();
    *fp_mults = g_fold_timer.fp_mults;
    *pairs = g_fold_timer.pairs;
    for (auto& e : g_fold_timer.ev) { (void)hipEventDestroy(e.first); (void)hipEventDestroy(e.second); }
    g_fold_timer.ev.clear();
    g_fold_timer.method.clear();
    return 0;
}
// what the last zk_prof_fold_read counted, by method (0 walk, 1 comb, 2 three-round fold): ms, launches, pairs, Fp multiplications
int zk_prof_fold_methods(double* ms3, unsigned long long* launches3, unsigned long long* pairs3, double* fp_mults3) {
    for (int m = 0; m < 3; ++m) { ms3[m] = g_fold_method_ms[m]; launches3[m] = g_fold_method_launches[m]; pairs3[m] = g_fold_method_pairs[m]; fp_mults3[m] = g_fold_method_mults[m]; }
    return 0;
}

}  // extern "C"
