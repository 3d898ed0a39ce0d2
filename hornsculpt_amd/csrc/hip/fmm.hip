// Far field of the wideband FMM operator (low-frequency spherical form), FP64.
//
// Replaces the device side of SupportLeafOperator and the LF translations of
// SupportFmmOperator (modules/bem/cuda/wideband_leaf.cu:14-903,
// wideband_rotation.cu, wideband_axial.cu, support_fmm_operator.cu:1103-1296):
//   * leaf moments   per (leaf, support panel): the panel rule's samples of the
//                    regular waves R_lm(y - c) = Jhat_l(k r) (r/a)^l Y_lm and their
//                    gradients, reduced over a 16-lane group per panel, give the
//                    emission rows conj(n . grad R_lm) phi_j and the testing rows
//                    (-R_lm - alpha n . grad R_lm) phi_i / m_i of the leaf's P1 DOFs;
//   * emission       multipole of a leaf = E_leaf p (one block per leaf);
//   * translation    every M2M / M2L / L2L link is rotate-to-axis, coaxial m-block
//                    translation, rotate-back (O(p^3)): three passes per chunk of up to
//                    16 links that share a direction and a coaxial plan, as products on
//                    the matrix cores with operands straight from memory, and one block per
//                    destination sums its links (no atomics);
//   * testing        y_i += T_leaf L_leaf (one wavefront per DOF).
#include "fmm_kernels.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <stdexcept>

namespace hsbem::dev {
namespace {

constexpr int kGroupSmall = 16; // lanes per (leaf, panel) item: rules of at most 16 points
constexpr int kGroupLarge = 64; // one wavefront per item: rules of at most 64 points (degrees 12, 14)
constexpr int kMillerMax = 256; // Miller recurrence start bound (z <= 96 at the leaves)

struct C2 {
    double re, im;
};
__device__ __forceinline__ C2 operator+(C2 a, C2 b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ C2 operator-(C2 a, C2 b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ C2 operator*(C2 a, C2 b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ C2 operator*(double s, C2 a) { return {s * a.re, s * a.im}; }
__device__ __forceinline__ C2 conj(C2 a) { return {a.re, -a.im}; }

// FP32 complex (the FP32-bulk form's expansions and translation workspaces)
struct C2f {
    float re, im;
};
__device__ __forceinline__ C2f operator+(C2f a, C2f b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ C2f operator*(C2f a, C2f b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ C2f operator*(float s, C2f a) { return {s * a.re, s * a.im}; }
__device__ __forceinline__ C2f conj(C2f a) { return {a.re, -a.im}; }
// complex type of an expansion scalar E (double: C2, float: C2f)
template <class E> struct CplxOf {
    using type = C2;
};
template <> struct CplxOf<float> {
    using type = C2f;
};
template <class E> using Cx = typename CplxOf<E>::type;
template <class E> __device__ __forceinline__ Cx<E> to_cx(C2 v) { return {static_cast<E>(v.re), static_cast<E>(v.im)}; }

// value and gradient of one solid harmonic
struct Wave {
    C2 v, g[3];
};

__device__ __forceinline__ Wave product(const Wave &a, const Wave &b) {
    Wave r;
    r.v = a.v * b.v;
#pragma unroll
    for (int i = 0; i < 3; ++i)
        r.g[i] = a.g[i] * b.v + a.v * b.g[i];
    return r;
}

__device__ __forceinline__ Wave scaled(Wave a, double s) {
    a.v = s * a.v;
#pragma unroll
    for (int i = 0; i < 3; ++i)
        a.g[i] = s * a.g[i];
    return a;
}

// Jhat_l(z) = (2l+1)!! j_l(z) / z^l for l = 0..top (top <= kMaxBigOrder + 1): the
// power series while its first correction z^2 / (2 (2l+3)) is at most one, else
// j_l by normalised Miller recursion (downward from past the turning point,
// normalised by the larger of j0 and j1) divided by z^l / (2l+1)!!.
__device__ bool normalized_regular(int top, double z, double *J) {
    int split = 0; // l < split use the j_l table
    if (z > 1)
        while (split <= top && z * z > 2 * (2.0 * split + 3))
            ++split;
    if (split) {
        const int start = max(split + 48, static_cast<int>(ceil(z + 48 + 8 * cbrt(z))));
        if (start + 2 > kMillerMax)
            return false;
        double mil[kMillerMax];
        mil[start + 1] = 0;
        mil[start] = 1;
        for (int l = start; l > 0; --l) {
            mil[l - 1] = ((2.0 * l + 1) / z) * mil[l] - mil[l + 1];
            if (fabs(mil[l - 1]) > 1e200)
                for (int j = l - 1; j <= start + 1; ++j)
                    mil[j] *= 1e-200;
        }
        double s, c;
        sincos(z, &s, &c);
        const double j0 = s / z, j1 = (j0 - c) / z;
        const double norm = fabs(j0) > fabs(j1) ? j0 / mil[0] : j1 / mil[1];
        double lead = 1;
        for (int l = 0; l < split; ++l) {
            if (l)
                lead *= z / (2.0 * l + 1);
            J[l] = norm * mil[l] / lead;
        }
    }
    for (int l = split; l <= top; ++l) {
        double term = 1, sum = 1;
        for (int n = 1; n < 128; ++n) {
            term *= -z * z / (2.0 * n * (2.0 * l + 2 * n + 1));
            sum += term;
            if (fabs(term) < 2.220446049250313e-16 * fabs(sum))
                break;
        }
        J[l] = sum;
    }
    return true;
}

template <int kGroup> __device__ __forceinline__ double group_sum(double v) {
#pragma unroll
    for (int off = kGroup / 2; off > 0; off >>= 1)
        v += __shfl_xor(v, off, kGroup);
    return v;
}

__device__ __forceinline__ void atomic_add_c(double *p, C2 v) {
    atomicAdd(p, v.re);
    atomicAdd(p + 1, v.im);
}

// One kGroup-lane group per (leaf, support panel) item, lane = rule point.
template <int kGroup, int kTop> __global__ __launch_bounds__(64) void leaf_moments(FmmLeafMomentsLaunch L) {
    const int lane = threadIdx.x % kGroup;
    const std::uint32_t item = blockIdx.x * (64 / kGroup) + threadIdx.x / kGroup;
    const bool live_item = item < L.item_count;
    const FmmLeafItem it = live_item ? L.items[item] : FmmLeafItem{};
    const FmmLeaf leaf = L.leaves[live_item ? it.leaf : 0];
    const std::uint32_t nt = L.nt, t = it.panel;
    const bool live = live_item && lane < L.rule_points;
    const double *rp = L.rule + 4 * (live ? lane : 0);
    const double b0 = rp[0], b1 = rp[1], b2 = rp[2];
    const double *g = L.geo;
    const double area = g[static_cast<std::size_t>(G_AREA) * nt + t];
    const double w = live ? rp[3] * 2 * area : 0.0; // rule weights sum to 1/2
    double y[3], n[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const double v0 = g[static_cast<std::size_t>(G_V0 + i) * nt + t];
        y[i] = v0 + b1 * g[static_cast<std::size_t>(G_E1 + i) * nt + t] + b2 * g[static_cast<std::size_t>(G_E2 + i) * nt + t];
        n[i] = g[static_cast<std::size_t>(G_N + i) * nt + t];
    }
    const double a = leaf.radius, k = L.k;
    const double x[3] = {y[0] - leaf.center[0], y[1] - leaf.center[1], y[2] - leaf.center[2]};
    const double u[3] = {x[0] / a, x[1] / a, x[2] / a};
    const int p = static_cast<int>(leaf.order);
    double J[kTop + 2];
    const bool ok = normalized_regular(p + 1, k * sqrt(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]), J);
    if (!ok && live && L.error)
        atomicMax(L.error, 1);
    const double bc[3] = {b0, b1, b2};
    const C2 alpha{L.alpha_re, L.alpha_im};
    const std::size_t nc = static_cast<std::size_t>(p + 1) * (p + 1);
    // solid harmonics |u|^l Y_lm(u) as polynomials in x + iy, z, r^2 with gradients in u
    const Wave xy{{u[0], u[1]}, {{1, 0}, {0, 1}, {0, 0}}}, zz{{u[2], 0}, {{0, 0}, {0, 0}, {1, 0}}},
        r2{{u[0] * u[0] + u[1] * u[1] + u[2] * u[2], 0}, {{2 * u[0], 0}, {2 * u[1], 0}, {2 * u[2], 0}}};
    Wave diag{{0.28209479177387814, 0}, {{0, 0}, {0, 0}, {0, 0}}}; // 1 / sqrt(4 pi)
    for (int m = 0; m <= p; ++m) {
        if (m)
            diag = scaled(product(xy, diag), -sqrt((2.0 * m + 1) / (2.0 * m)));
        Wave prev{}, cur = diag;
        for (int l = m; l <= p; ++l) {
            if (l == m + 1) {
                prev = cur;
                cur = scaled(product(zz, diag), sqrt(2.0 * m + 3));
            } else if (l > m + 1) {
                const double den = static_cast<double>(l) * l - static_cast<double>(m) * m;
                const double ca = sqrt((4.0 * l * l - 1) / den),
                             cb = sqrt((2.0 * l + 1) * ((l - 1.0) * (l - 1.0) - static_cast<double>(m) * m) /
                                       ((2.0 * l - 3) * den));
                const Wave za = scaled(product(zz, cur), ca), rb = scaled(product(r2, prev), cb);
                Wave nx;
                nx.v = za.v - rb.v;
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    nx.g[i] = za.g[i] - rb.g[i];
                prev = cur;
                cur = nx;
            }
            // R_lm and n . grad R_lm
            const double jl = J[l], jl1 = J[l + 1];
            const C2 R = jl * cur.v;
            C2 dn{0, 0};
#pragma unroll
            for (int i = 0; i < 3; ++i)
                dn = dn + n[i] * ((jl / a) * cur.g[i] - (k * k * x[i] / (2.0 * l + 3) * jl1) * cur.v);
            // emission conj(dn) w, testing (-R - alpha dn) w; the -m partners follow from
            // R_{l,-m} = (-1)^m conj(R_lm) (real n and Jhat)
            const C2 e = w * conj(dn), tt = w * (C2{-R.re, -R.im} - alpha * dn);
            const C2 em = (m % 2 ? -w : w) * dn,
                     tm = (m % 2 ? -w : w) * (C2{-R.re, R.im} - alpha * conj(dn));
            const std::size_t jp = static_cast<std::size_t>(l) * l + l + m, jm = static_cast<std::size_t>(l) * l + l - m;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const double s = bc[c];
                const C2 sums[4] = {{group_sum<kGroup>(s * e.re), group_sum<kGroup>(s * e.im)},
                                    {group_sum<kGroup>(s * tt.re), group_sum<kGroup>(s * tt.im)},
                                    {group_sum<kGroup>(s * em.re), group_sum<kGroup>(s * em.im)},
                                    {group_sum<kGroup>(s * tm.re), group_sum<kGroup>(s * tm.im)}};
                const std::int32_t j = it.corner[c];
                if (live_item && lane == 0 && j >= 0) {
                    const std::size_t row = static_cast<std::size_t>(j) * nc;
                    const double scale = L.row_scale[L.leaf_dofs[leaf.first_dof + j]];
                    atomic_add_c(L.emission + 2 * (leaf.emission + row + jp), sums[0]);
                    atomic_add_c(L.testing + 2 * (leaf.emission + row + jp), scale * sums[1]);
                    if (m) {
                        atomic_add_c(L.emission + 2 * (leaf.emission + row + jm), sums[2]);
                        atomic_add_c(L.testing + 2 * (leaf.emission + row + jm), scale * sums[3]);
                    }
                }
            }
        }
    }
}

// M_leaf = E_leaf p: one block per leaf, thread per coefficient; the expansions are
// stored as S (the sums run in FP64).
template <class S>
__global__ __launch_bounds__(256) void leaf_emit(const FmmLeaf *leaves, const std::uint32_t *leaf_dofs,
                                                 const double *emission, const double *p, S *expansions) {
    __shared__ double sp[2 * kMaxLeafDofs];
    const FmmLeaf leaf = leaves[blockIdx.x];
    for (std::uint32_t j = threadIdx.x; j < leaf.dof_count; j += blockDim.x) {
        const std::uint32_t d = leaf_dofs[leaf.first_dof + j];
        sp[2 * j] = p[2 * d];
        sp[2 * j + 1] = p[2 * d + 1];
    }
    __syncthreads();
    const std::size_t nc = static_cast<std::size_t>(leaf.order + 1) * (leaf.order + 1);
    const double2 *E = reinterpret_cast<const double2 *>(emission) + leaf.emission;
    for (std::size_t c = threadIdx.x; c < nc; c += blockDim.x) {
        double re = 0, im = 0;
        for (std::uint32_t j = 0; j < leaf.dof_count; ++j) {
            const double2 e = E[j * nc + c];
            re += e.x * sp[2 * j] - e.y * sp[2 * j + 1];
            im += e.x * sp[2 * j + 1] + e.y * sp[2 * j];
        }
        expansions[2 * (leaf.multipole + c)] = static_cast<S>(re);
        expansions[2 * (leaf.multipole + c) + 1] = static_cast<S>(im);
    }
}

// y_i += T_leaf[i] . L_leaf: one wavefront per DOF; the expansions are read as S.
template <class S>
__global__ __launch_bounds__(256) void leaf_test(const FmmLeaf *leaves, const std::uint32_t *leaf_dofs,
                                                 const double *testing, const S *expansions, double *y) {
    const FmmLeaf leaf = leaves[blockIdx.x];
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const std::size_t nc = static_cast<std::size_t>(leaf.order + 1) * (leaf.order + 1);
    const double2 *T = reinterpret_cast<const double2 *>(testing) + leaf.emission;
    const Cx<S> *Lc = reinterpret_cast<const Cx<S> *>(expansions) + leaf.local;
    for (std::uint32_t j = wave; j < leaf.dof_count; j += blockDim.x / 64) {
        double re = 0, im = 0;
        for (std::size_t c = lane; c < nc; c += 64) {
            const double2 t = T[j * nc + c];
            const double lr = Lc[c].re, li = Lc[c].im;
            re += t.x * lr - t.y * li;
            im += t.x * li + t.y * lr;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            re += __shfl_xor(re, off, 64);
            im += __shfl_xor(im, off, 64);
        }
        if (lane == 0) {
            const std::uint32_t d = leaf_dofs[leaf.first_dof + j];
            y[2 * d] += re;
            y[2 * d + 1] += im;
        }
    }
}

__device__ __forceinline__ void split_index(int e, int &l, int &t) {
    l = static_cast<int>(sqrt(static_cast<double>(e)));
    while (l * l > e)
        --l;
    while ((l + 1) * (l + 1) <= e)
        ++l;
    t = e - l * l;
}

// Offset of the |m| block of a coaxial plan: sum_{j<m} (pt+1-j)(ps+1-j).
__device__ __forceinline__ std::size_t axial_block(int m, int ps, int pt) {
    const std::size_t j = m, a = pt + 1, b = ps + 1, first = j ? j * (j - 1) / 2 : 0; // sum of the j below m
    return j * a * b - (a + b) * first + (j ? first * (2 * j - 1) / 3 : 0);
}

// Offset of degree l in a rotation's small-d table: sum_{j<l} (2j+1)^2 = l(2l-1)(2l+1)/3.
__device__ __forceinline__ std::size_t degree_block(int l) {
    return static_cast<std::size_t>(l) * (2 * l - 1) * (2 * l + 1) / 3;
}

// Translations run as four passes over the links of one level:
//   rotate    per chunk of links sharing a direction and a coaxial plan: the Wigner blocks
//             d_l applied to every source of the chunk (Y = d^T e^{i m phi} X);
//   coaxial   per-|m| block product Z = T Y;
//   back      W = e^{-i m phi} d Z;
//   gather    one block per destination: the sum of its links' W.
// Y and Z hold a chunk's links interleaved (coefficient (l, m) of link j at
// base + (l^2 + l + m) count + j), W each link's expansion in its slot.
//
// Rotations and coaxial products are small matrix products (a block of 2l + 1 or
// p + 1 - |m| rows against up to 16 links), on the matrix cores in 16 x 16 x 4 steps with
// the operands loaded straight from memory into lanes: a block is read once per chunk by one
// wavefront and a link's values once per wavefront, so nothing is staged, no barrier
// holds wavefronts together and their number per CU hides the latency. (With the blocks and
// slices staged in LDS and FP64 vector products, the products were bound by LDS reads: 12
// reads of 16 bytes for 24 multiply-adds.) Each wavefront takes whole degrees l (orders |m|);
// each step
// reads and writes rows of 16 count bytes, so that no pass touches part of a line in one
// order and the rest in another.
// One level of a 20.7k-triangle horn (41k links of order 26, FP64), forward, coaxial, back:
// 620 + 657 + 551 us before, 275 + 377 + 405 us now (Y, Z and W are 480 MB each: 2.2 to 3.6
// TB/s); the whole operator 3.96 -> 2.72 ms. What gave how much: tiles alone about nothing (the
// |m|-major Y and strided Z wrote 2 to 2.4 times their bytes in parts of lines), the
// interleaved layout and dies that share a direction 4.5 -> 3.5 ms, four wavefronts per SIMD
// and d by rows 3.0 ms, 16-byte stores 2.7 ms.
template <class E> struct Tile16;
template <> struct Tile16<double> {
    typedef double V __attribute__((ext_vector_type(4)));
    // row of a lane's i-th value of D (column lane & 15)
    static __device__ __forceinline__ int row(int lane, int i) { return (lane >> 4) + 4 * i; }
    static __device__ __forceinline__ V mac(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};
template <> struct Tile16<float> {
    typedef float V __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ int row(int lane, int i) { return 4 * (lane >> 4) + i; }
    static __device__ __forceinline__ V mac(float a, float b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};

// The value of the neighbouring lane (lane ^ 1).
__device__ __forceinline__ float neighbour(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xb1, 0xf, 0xf, true));
}
__device__ __forceinline__ double neighbour(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0xb1, 0xf, 0xf, true),
              hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0xb1, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// Two values of a lane pair (lane even: real parts, odd: imaginary parts) as one complex
// value per lane, the first for the even lane and the second for the odd one.
template <class E> __device__ __forceinline__ Cx<E> pair_values(E first, E second, int part) {
    const E other = neighbour(part ? first : second);
    return part ? Cx<E>{other, second} : Cx<E>{first, other};
}

// The two column tiles of a chunk: lane & 15 = 2 (link & 7) + (0 real, 1 imaginary). Where
// coefficient e of the lane's link is: first + e step (complex values).
struct LinkColumns {
    std::uint64_t in[2], out[2];
    std::uint32_t in_step, out_step;
    bool live[2];
};

// RT row tiles from row0 of degree l for CT column tiles. Both directions read the block by
// rows q, a row per 16 lanes: back takes d[t][q] = (-1)^(t - q) d[q][t], because columns of it
// would be 16 separate lines a load (that pass took 1.5 times the forward one).
template <class E, bool BACK, int RT, int CT>
__device__ __forceinline__ void rotate_rows(const double *d, const C2 *phase, int l, int row0, const LinkColumns &at,
                                            const Cx<E> *in, Cx<E> *out) {
    using CE = Cx<E>;
    using T = Tile16<E>;
    const int lane = threadIdx.x & 63, n = 2 * l + 1, part = lane & 1;
    const std::size_t base = static_cast<std::size_t>(l) * l;
    typename T::V acc[RT][CT] = {};
    int row[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
        row[r] = min(row0 + 16 * r + (lane & 15), n - 1); // rows beyond n: results dropped
#pragma unroll 2
    for (int q0 = 0; q0 < n; q0 += 4) {
        const int q = q0 + (lane >> 4), qc = min(q, n - 1); // beyond n: zeros in the other operand
        E a[RT], b[CT];
#pragma unroll
        for (int r = 0; r < RT; ++r)
            a[r] = static_cast<E>(d[qc * n + row[r]]);
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            CE x{0, 0};
            if (q < n && at.live[c])
                x = in[at.in[c] + (base + q) * at.in_step];
            if (!BACK)
                x = to_cx<E>(phase[qc - l]) * x;
            b[c] = part ? x.im : x.re;
            if (BACK && (q & 1))
                b[c] = -b[c];
        }
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int c = 0; c < CT; ++c)
                acc[r][c] = T::mac(a[r], b[c], acc[r][c]);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
            const int t = row0 + 16 * r + T::row(lane, i + part); // the lane's value of the two
            const CE ph = BACK ? to_cx<E>(phase[min(t, n - 1) - l]) : CE{1, 0};
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                CE v = pair_values<E>(acc[r][c][i], acc[r][c][i + 1], part);
                if (BACK) {
                    v = conj(ph) * v;
                    if (t & 1)
                        v = CE{-v.re, -v.im};
                }
                if (t < n && at.live[c])
                    out[at.out[c] + (base + t) * at.out_step] = v;
            }
        }
}

template <class E, bool BACK, int CT>
__device__ __forceinline__ void rotate_degrees(const FmmTranslateLaunch &L, const FmmChunk &ch, int top,
                                               const LinkColumns &at) {
    const FmmRotation rot = L.rotations[ch.rotation];
    const C2 *phase = reinterpret_cast<const C2 *>(L.azimuth) + rot.azimuth + rot.order; // of m = 0
    const Cx<E> *in = reinterpret_cast<const Cx<E> *>(BACK ? L.work_z : L.source_expansions);
    Cx<E> *out = reinterpret_cast<Cx<E> *>(L.work_y);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    for (int l = 4 * blockIdx.y + wave; l <= top; l += 4 * gridDim.y) {
        const double *d = L.small_d + rot.small_d + degree_block(l);
        for (int row0 = 0; row0 < 2 * l + 1; row0 += 64)
            switch (min((2 * l + 1 - row0 + 15) / 16, 4)) {
            case 1: rotate_rows<E, BACK, 1, CT>(d, phase, l, row0, at, in, out); break;
            case 2: rotate_rows<E, BACK, 2, CT>(d, phase, l, row0, at, in, out); break;
            case 3: rotate_rows<E, BACK, 3, CT>(d, phase, l, row0, at, in, out); break;
            default: rotate_rows<E, BACK, 4, CT>(d, phase, l, row0, at, in, out);
            }
    }
}

// Chunk of a workgroup: the chip's 8 dies take workgroups in turn, so each gets a run of
// consecutive chunks, which share their direction's blocks in its L2.
__device__ __forceinline__ std::uint32_t chunk_of(std::uint32_t block, std::uint32_t chunks) {
    const std::uint32_t die = block % 8, per = chunks / 8, more = chunks % 8;
    return die * per + min(die, more) + block / 8;
}

// Workgroup (chunk, y) takes the degrees 4 y .. 4 y + 3, 4 (y + Y) .., (Y = gridDim.y), so a
// level with few chunks spreads its degrees over more workgroups.
template <class E, bool BACK> __global__ __launch_bounds__(256, 3) void rotate_links(FmmTranslateLaunch L) {
    const FmmChunk ch = L.chunks[chunk_of(blockIdx.x, gridDim.x)];
    const FmmLink first = L.links[L.order[ch.first]]; // its orders are the chunk's
    const int top = static_cast<int>(BACK ? first.target_order : first.source_order);
    if (4 * static_cast<int>(blockIdx.y) > top)
        return;
    LinkColumns at;
    at.in_step = BACK ? ch.count : 1;
    at.out_step = BACK ? 1 : ch.count;
#pragma unroll
    for (std::uint32_t c = 0; c < 2; ++c) {
        const std::uint32_t j = 8 * c + (threadIdx.x & 15) / 2;
        at.live[c] = j < ch.count;
        const FmmLink lk = L.links[L.order[ch.first + (at.live[c] ? j : 0)]];
        at.in[c] = BACK ? ch.base + j : lk.source;
        at.out[c] = BACK ? lk.slot : ch.base + j;
    }
    if (ch.count > 8)
        rotate_degrees<E, BACK, 2>(L, ch, top, at);
    else
        rotate_degrees<E, BACK, 1>(L, ch, top, at);
}

// Rows row0 .. row0 + 16 RT of Z = T Y for order |m|, both signs, CT column tiles.
template <class E, int RT, int CT>
__device__ __forceinline__ void axial_rows(const C2 *T, int m, int ps, int pt, int row0, std::uint64_t base, int count,
                                           const Cx<E> *y, Cx<E> *z) {
    using CE = Cx<E>;
    using M = Tile16<E>;
    const int lane = threadIdx.x & 63, rows = pt + 1 - m, cols = ps + 1 - m, part = lane & 1, j0 = (lane & 15) / 2;
    typename M::V acc[RT][CT][2] = {};
    int row[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
        row[r] = min(row0 + 16 * r + (lane & 15), rows - 1);
#pragma unroll 2
    for (int q0 = 0; q0 < cols; q0 += 4) {
        const int q = q0 + (lane >> 4), qc = min(q, cols - 1), l = m + q;
        CE a[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r)
            a[r] = to_cx<E>(T[row[r] * cols + qc]);
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int sgn = 0; sgn < 2; ++sgn) {
                if (sgn && m == 0)
                    continue;
                CE v{0, 0};
                if (q < cols && j0 + 8 * c < count)
                    v = y[base + static_cast<std::size_t>(l * (l + 1) + (sgn ? -m : m)) * count + j0 + 8 * c];
                const E direct = part ? v.im : v.re, crossed = part ? v.re : -v.im;
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    acc[r][c][sgn] = M::mac(a[r].re, direct, acc[r][c][sgn]);
                    acc[r][c][sgn] = M::mac(a[r].im, crossed, acc[r][c][sgn]);
                }
            }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
            const int t = row0 + 16 * r + M::row(lane, i + part), l = m + t;
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                const CE plus = pair_values<E>(acc[r][c][0][i], acc[r][c][0][i + 1], part),
                         minus = pair_values<E>(acc[r][c][1][i], acc[r][c][1][i + 1], part);
                if (t < rows && j0 + 8 * c < count) {
                    CE *at = z + base + static_cast<std::size_t>(l * (l + 1)) * count + j0 + 8 * c;
                    at[m * count] = plus;
                    if (m)
                        at[-m * count] = minus;
                }
            }
        }
}

template <class E, int CT>
__device__ __forceinline__ void axial_orders(const FmmTranslateLaunch &L, const C2 *T, int ps, int pt,
                                             const FmmChunk &ch) {
    const Cx<E> *y = reinterpret_cast<const Cx<E> *>(L.work_y);
    Cx<E> *z = reinterpret_cast<Cx<E> *>(L.work_z);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), mm = min(ps, pt);
    for (int m = 4 * blockIdx.y + wave; m <= mm; m += 4 * gridDim.y) {
        const C2 *block = T + axial_block(m, ps, pt);
        const int rows = pt + 1 - m, count = static_cast<int>(ch.count);
        for (int row0 = 0; row0 < rows; row0 += 32)
            if (rows - row0 > 16)
                axial_rows<E, 2, CT>(block, m, ps, pt, row0, ch.base, count, y, z);
            else
                axial_rows<E, 1, CT>(block, m, ps, pt, row0, ch.base, count, y, z);
    }
}

// Z = T Y per |m| block; workgroup (chunk, y) takes the orders 4 y .. 4 y + 3, 4 (y + Y) .. of
// the chunk.
template <class E> __global__ __launch_bounds__(256, 4) void coaxial_links(FmmTranslateLaunch L) {
    const FmmChunk ch = L.chunks[chunk_of(blockIdx.x, gridDim.x)];
    const FmmLink first = L.links[L.order[ch.first]];
    const int ps = static_cast<int>(first.source_order), pt = static_cast<int>(first.target_order), mm = min(ps, pt);
    const C2 *T = reinterpret_cast<const C2 *>(L.axial) + L.axial_offsets[first.axial];
    // orders above min(ps, pt) have no source: those outputs are zero
    if (blockIdx.y == 0 && pt > mm) {
        Cx<E> *z = reinterpret_cast<Cx<E> *>(L.work_z) + ch.base;
        const int count = static_cast<int>(ch.count);
        for (int e = threadIdx.x; e < count * (pt + 1) * (pt + 1); e += blockDim.x) {
            int l, t;
            split_index(e / count, l, t);
            if (abs(t - l) > mm)
                z[e] = {0, 0};
        }
    }
    if (4 * static_cast<int>(blockIdx.y) > mm)
        return;
    if (ch.count > 8)
        axial_orders<E, 2>(L, T, ps, pt, ch);
    else
        axial_orders<E, 1>(L, T, ps, pt, ch);
}

// target = sum of the destination's link results.
template <class E> __global__ __launch_bounds__(256) void gather_links(FmmTranslateLaunch L) {
    using CE = Cx<E>;
    const FmmDestination dst = L.destinations[blockIdx.x];
    const int nct = static_cast<int>((dst.order + 1) * (dst.order + 1));
    const CE *w = reinterpret_cast<const CE *>(L.work_y);
    CE *out = reinterpret_cast<CE *>(L.target_expansions) + dst.target;
    const FmmLink *links = L.links + dst.first_link;
    const std::uint32_t n = dst.link_count;
    for (int e = threadIdx.x; e < nct; e += blockDim.x) {
        // the sum runs in link order; the loads of four links are issued together
        CE s{0, 0};
        std::uint32_t i = 0;
        for (; i + 4 <= n; i += 4) {
            const CE a = w[links[i].slot + e], b = w[links[i + 1].slot + e];
            const CE c = w[links[i + 2].slot + e], d = w[links[i + 3].slot + e];
            s = s + a;
            s = s + b;
            s = s + c;
            s = s + d;
        }
        for (; i < n; ++i)
            s = s + w[links[i].slot + e];
        out[e] = s;
    }
}

// Block-Jacobi blocks of the near operator: block b holds rows and columns
// order[b*W .. b*W+W) (tree order); entries absent from the CSR are zero.
__global__ void gather_blocks(const std::uint32_t *row_offsets, const std::uint32_t *columns, const double *values,
                              const std::uint32_t *order, const std::uint32_t *position, std::uint32_t n,
                              std::uint32_t width, double *blocks) {
    const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const std::uint32_t W = width, row = order[i], blk = i / W, r = i % W;
    double *B = blocks + static_cast<std::size_t>(blk) * W * W * 2;
    for (std::uint32_t e = row_offsets[row]; e < row_offsets[row + 1]; ++e) {
        const std::uint32_t pc = position[columns[e]];
        if (pc / W != blk)
            continue;
        const std::uint32_t c = pc % W;
        B[2 * (static_cast<std::size_t>(c) * W + r)] = values[2 * e];
        B[2 * (static_cast<std::size_t>(c) * W + r) + 1] = values[2 * e + 1];
    }
}

// Far part of B q for the FMM path, by direct pair quadrature (the flux panels
// are the few driven ones): for test panel s and flux panel t, every corner i of
// s whose pressure leaf is not a near leaf pair of t's flux leaf receives
//   (1/m_i) q_t sum_a sum_b w_a w_b phi_i(x_a) (-G - alpha dG/dn_x)(x_a, y_b).
__global__ __launch_bounds__(256) void far_flux(FmmFarFluxLaunch L) {
    const std::uint64_t pair = static_cast<std::uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (pair >= static_cast<std::uint64_t>(L.nt) * L.flux_count)
        return;
    const std::uint32_t s = static_cast<std::uint32_t>(pair / L.flux_count);
    const std::uint32_t t = L.flux_panels[pair % L.flux_count];
    const std::uint32_t fleaf = L.flux_leaf[t];
    bool far[3];
    std::uint32_t node[3];
    bool any = false;
    for (int c = 0; c < 3; ++c) {
        node[c] = L.nodes[static_cast<std::size_t>(c) * L.nt + s];
        const std::uint32_t pl = L.pressure_leaf[node[c]];
        bool near = false;
        for (std::uint32_t e = L.near_offsets[pl]; e < L.near_offsets[pl + 1]; ++e)
            near |= L.near_sources[e] == fleaf;
        far[c] = !near;
        any |= far[c];
    }
    if (!any)
        return;
    const double *g = L.geo;
    const std::size_t nt = L.nt;
    double vs[3], e1s[3], e2s[3], ns[3], vt[3], e1t[3], e2t[3];
    for (int i = 0; i < 3; ++i) {
        vs[i] = g[(G_V0 + i) * nt + s];
        e1s[i] = g[(G_E1 + i) * nt + s];
        e2s[i] = g[(G_E2 + i) * nt + s];
        ns[i] = g[(G_N + i) * nt + s];
        vt[i] = g[(G_V0 + i) * nt + t];
        e1t[i] = g[(G_E1 + i) * nt + t];
        e2t[i] = g[(G_E2 + i) * nt + t];
    }
    const double ws = 2 * g[G_AREA * nt + s], wt = 2 * g[G_AREA * nt + t], k = L.k;
    const C2 alpha{0, -1 / k};
    C2 acc[3] = {{0, 0}, {0, 0}, {0, 0}};
    for (std::uint32_t a = 0; a < L.rule_points; ++a) {
        const double *ra = L.rule + 4 * a;
        double x[3];
        for (int i = 0; i < 3; ++i)
            x[i] = vs[i] + ra[1] * e1s[i] + ra[2] * e2s[i];
        C2 kern{0, 0};
        for (std::uint32_t b = 0; b < L.rule_points; ++b) {
            const double *rb = L.rule + 4 * b;
            double d[3], r2 = 0, nd = 0;
            for (int i = 0; i < 3; ++i) {
                d[i] = x[i] - (vt[i] + rb[1] * e1t[i] + rb[2] * e2t[i]);
                r2 += d[i] * d[i];
                nd += ns[i] * d[i];
            }
            const double r = sqrt(r2);
            double sn, cs;
            sincos(k * r, &sn, &cs);
            const C2 G = (1.0 / (4 * 3.141592653589793 * r)) * C2{cs, -sn};
            const C2 dG = (nd / r) * (C2{-1 / r, -k} * G);
            kern = kern + (rb[3] * wt) * (C2{-G.re, -G.im} - alpha * dG);
        }
        for (int c = 0; c < 3; ++c)
            acc[c] = acc[c] + (ra[3] * ws * ra[c]) * kern;
    }
    for (std::uint32_t e = 0; e < L.excitations; ++e) {
        const C2 q{L.q[2 * (static_cast<std::size_t>(e) * L.nt_all + t)], L.q[2 * (static_cast<std::size_t>(e) * L.nt_all + t) + 1]};
        if (q.re == 0 && q.im == 0)
            continue;
        for (int c = 0; c < 3; ++c)
            if (far[c]) {
                const C2 v = L.row_scale[node[c]] * (q * acc[c]);
                atomic_add_c(L.out + 2 * (static_cast<std::size_t>(e) * L.nv + node[c]), v);
            }
    }
}

// Direct far action of the Burton-Miller pressure operator. For a test panel s and a
// trial panel t the far corner pairs (ci, cj) contribute
//   (1/m_i) x_j int_s int_t phi_i(x) phi_j(y) [-dG/dn_y - alpha d2G/dn_x dn_y] dy dx,
// G = exp(-ikr)/(4 pi r), d = x - y, g' = -(ik + 1/r) G, g'' = G/r^2 + (ik + 1/r)^2 G:
//   dG/dn_y = -g' (d.n_y)/r,
//   d2G/dn_x dn_y = -(d.n_x)(d.n_y)(g''/r^2 - g'/r^3) - (g'/r)(n_x.n_y).
// Block per test panel, threads over trial panels; per-thread row sums reduced in
// the block, one atomic add per test corner.
__global__ __launch_bounds__(256) void direct_far(FmmDirectLaunch L) {
    __shared__ double red[2][3][4];
    const std::uint32_t s = blockIdx.x;
    const std::size_t nt = L.nt;
    const double *g = L.geo;
    double vs[3], e1s[3], e2s[3], ns[3];
    std::uint32_t node_s[3], leaf_s[3];
    for (int i = 0; i < 3; ++i) {
        vs[i] = g[(G_V0 + i) * nt + s];
        e1s[i] = g[(G_E1 + i) * nt + s];
        e2s[i] = g[(G_E2 + i) * nt + s];
        ns[i] = g[(G_N + i) * nt + s];
        node_s[i] = L.nodes[static_cast<std::size_t>(i) * nt + s];
        leaf_s[i] = L.vertex_leaf[node_s[i]];
    }
    const double ws = 2 * g[G_AREA * nt + s], k = L.k;
    const int Q = static_cast<int>(L.rule_points);
    const C2 alpha{0, -1 / k};
    C2 acc[3] = {{0, 0}, {0, 0}, {0, 0}};
    for (std::uint32_t t = threadIdx.x; t < L.nt; t += blockDim.x) {
        std::uint32_t node_t[3];
        bool far[3][3], any = false;
        for (int c = 0; c < 3; ++c)
            node_t[c] = L.nodes[static_cast<std::size_t>(c) * nt + t];
        for (int ci = 0; ci < 3; ++ci)
            for (int cj = 0; cj < 3; ++cj) {
                far[ci][cj] = !L.near[static_cast<std::size_t>(leaf_s[ci]) * L.leaf_count + L.vertex_leaf[node_t[cj]]];
                any |= far[ci][cj];
            }
        if (!any)
            continue;
        double vt[3], e1t[3], e2t[3], nn[3];
        for (int i = 0; i < 3; ++i) {
            vt[i] = g[(G_V0 + i) * nt + t];
            e1t[i] = g[(G_E1 + i) * nt + t];
            e2t[i] = g[(G_E2 + i) * nt + t];
            nn[i] = g[(G_N + i) * nt + t];
        }
        const double wt = 2 * g[G_AREA * nt + t];
        const double nxny = ns[0] * nn[0] + ns[1] * nn[1] + ns[2] * nn[2];
        C2 M[3][3] = {};
        for (int a = 0; a < Q; ++a) {
            const double *ra = L.rule + 4 * a;
            double x[3];
            for (int i = 0; i < 3; ++i)
                x[i] = vs[i] + ra[1] * e1s[i] + ra[2] * e2s[i];
            C2 T[3] = {{0, 0}, {0, 0}, {0, 0}};
            for (int b = 0; b < Q; ++b) {
                const double *rb = L.rule + 4 * b;
                double d[3], r2 = 0, dnx = 0, dny = 0;
                for (int i = 0; i < 3; ++i) {
                    d[i] = x[i] - (vt[i] + rb[1] * e1t[i] + rb[2] * e2t[i]);
                    r2 += d[i] * d[i];
                    dnx += ns[i] * d[i];
                    dny += nn[i] * d[i];
                }
                const double r = sqrt(r2), ir = 1 / r;
                double sn, cs;
                sincos(k * r, &sn, &cs);
                const C2 G = (ir / (4 * 3.141592653589793)) * C2{cs, -sn};
                const C2 ikr{ir, k};                       // ik + 1/r
                const C2 g1 = C2{-1, 0} * (ikr * G);        // g'
                const C2 g2 = (ir * ir) * G + (ikr * ikr) * G; // g''
                const C2 dGy = (-dny * ir) * g1;
                const C2 H = (-dnx * dny) * ((ir * ir) * g2 - (ir * ir * ir) * g1) - (nxny * ir) * g1;
                const C2 K = (rb[3] * wt) * (C2{-dGy.re, -dGy.im} - alpha * H);
                for (int c = 0; c < 3; ++c)
                    T[c] = T[c] + rb[c] * K;
            }
            for (int ci = 0; ci < 3; ++ci)
                for (int cj = 0; cj < 3; ++cj)
                    M[ci][cj] = M[ci][cj] + (ra[3] * ws * ra[ci]) * T[cj];
        }
        for (int cj = 0; cj < 3; ++cj) {
            const C2 xj{L.x[2 * node_t[cj]], L.x[2 * node_t[cj] + 1]};
            for (int ci = 0; ci < 3; ++ci)
                if (far[ci][cj])
                    acc[ci] = acc[ci] + M[ci][cj] * xj;
        }
    }
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    for (int c = 0; c < 3; ++c) {
        double re = acc[c].re, im = acc[c].im;
        for (int off = 32; off > 0; off >>= 1) {
            re += __shfl_xor(re, off, 64);
            im += __shfl_xor(im, off, 64);
        }
        if (lane == 0) {
            red[0][c][wave] = re;
            red[1][c][wave] = im;
        }
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int c = threadIdx.x;
        double re = 0, im = 0;
        for (int w = 0; w < static_cast<int>(blockDim.x) / 64; ++w) {
            re += red[0][c][w];
            im += red[1][c][w];
        }
        const double sc = L.row_scale[node_s[c]];
        atomic_add_c(L.y + 2 * static_cast<std::size_t>(node_s[c]), C2{sc * re, sc * im});
    }
}

// out[:, e] += B_near q_e with B_near the P1 x face-column near CSR.
__global__ void flux_csr_apply(const std::uint32_t *offsets, const std::uint32_t *columns, const double *values,
                               std::uint32_t rows, const double *q, std::uint32_t faces, std::uint32_t excitations,
                               double *out) {
    const std::uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows)
        return;
    for (std::uint32_t e = 0; e < excitations; ++e) {
        C2 s{0, 0};
        for (std::uint32_t j = offsets[r]; j < offsets[r + 1]; ++j) {
            const C2 v{values[2 * j], values[2 * j + 1]};
            const std::size_t f = static_cast<std::size_t>(e) * faces + columns[j];
            s = s + v * C2{q[2 * f], q[2 * f + 1]};
        }
        out[2 * (static_cast<std::size_t>(e) * rows + r)] += s.re;
        out[2 * (static_cast<std::size_t>(e) * rows + r) + 1] += s.im;
    }
}

// out[map[i]] = in[i] (forward) or out[i] = in[map[i]] (backward), per vector.
__global__ void permute_vectors(const double *in, double *out, const std::uint32_t *map, std::uint32_t n,
                                std::uint32_t count, bool forward) {
    const std::uint64_t i = static_cast<std::uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= static_cast<std::uint64_t>(n) * count)
        return;
    const std::uint64_t v = i / n, j = i % n, base = v * n;
    const std::uint64_t src = base + (forward ? j : map[j]), dst = base + (forward ? map[j] : j);
    out[2 * dst] = in[2 * src];
    out[2 * dst + 1] = in[2 * src + 1];
}

} // namespace

void launch_leaf_moments(const FmmLeafMomentsLaunch &launch, hipStream_t stream) {
    if (!launch.item_count)
        return;
    // register table of the radial factors up to the leaves' largest order
    const bool wide = launch.max_order > static_cast<std::uint32_t>(kMaxLeafOrder);
    if (launch.rule_points <= static_cast<std::uint32_t>(kGroupSmall)) {
        const std::uint32_t per_block = 64 / kGroupSmall;
        const dim3 grid((launch.item_count + per_block - 1) / per_block);
        if (wide)
            hipLaunchKernelGGL((leaf_moments<kGroupSmall, kMaxBigOrder>), grid, dim3(64), 0, stream, launch);
        else
            hipLaunchKernelGGL((leaf_moments<kGroupSmall, kMaxLeafOrder>), grid, dim3(64), 0, stream, launch);
    } else if (wide) {
        hipLaunchKernelGGL((leaf_moments<kGroupLarge, kMaxBigOrder>), dim3(launch.item_count), dim3(64), 0, stream,
                           launch);
    } else {
        hipLaunchKernelGGL((leaf_moments<kGroupLarge, kMaxLeafOrder>), dim3(launch.item_count), dim3(64), 0, stream,
                           launch);
    }
}

void launch_leaf_emit(const FmmLeaf *leaves, std::uint32_t leaf_count, const std::uint32_t *leaf_dofs,
                      const double *emission, const double *p, double *expansions, hipStream_t stream, bool fp32) {
    if (!leaf_count)
        return;
    if (fp32)
        hipLaunchKernelGGL(leaf_emit<float>, dim3(leaf_count), dim3(256), 0, stream, leaves, leaf_dofs, emission, p,
                           reinterpret_cast<float *>(expansions));
    else
        hipLaunchKernelGGL(leaf_emit<double>, dim3(leaf_count), dim3(256), 0, stream, leaves, leaf_dofs, emission, p,
                           expansions);
}

void launch_leaf_test(const FmmLeaf *leaves, std::uint32_t leaf_count, const std::uint32_t *leaf_dofs,
                      const double *testing, const double *expansions, double *y, hipStream_t stream, bool fp32) {
    if (!leaf_count)
        return;
    if (fp32)
        hipLaunchKernelGGL(leaf_test<float>, dim3(leaf_count), dim3(256), 0, stream, leaves, leaf_dofs, testing,
                           reinterpret_cast<const float *>(expansions), y);
    else
        hipLaunchKernelGGL(leaf_test<double>, dim3(leaf_count), dim3(256), 0, stream, leaves, leaf_dofs, testing,
                           expansions, y);
}

// The translations of one launch in scalar E.
template <class E> void launch_links(const FmmTranslateLaunch &launch, dim3 grid, hipStream_t stream) {
    hipLaunchKernelGGL((rotate_links<E, false>), grid, dim3(256), 0, stream, launch);
    hipLaunchKernelGGL((coaxial_links<E>), grid, dim3(256), 0, stream, launch);
    hipLaunchKernelGGL((rotate_links<E, true>), grid, dim3(256), 0, stream, launch);
}

void launch_translate(const FmmTranslateLaunch &launch, std::uint32_t destination_count, std::uint32_t link_count,
                      std::uint32_t chunk_count, std::uint32_t max_order, std::uint32_t split_target,
                      hipStream_t stream) {
    if (!destination_count)
        return;
    if (launch.fp32 && link_count && max_order > kMidFmmOrder)
        throw std::invalid_argument("FP32 translations take orders up to 48 only");
    // Levels with few chunks spread each chunk's degrees (orders), four at a time, over up
    // to `splits` workgroups, so that a launch holds about split_target workgroups; 0 = no split.
    const std::uint32_t stages = max_order / 4 + 1,
                        splits = chunk_count && split_target
                                     ? std::max(1u, std::min(stages, (split_target + chunk_count - 1) / chunk_count))
                                     : 1u;
    if (link_count && launch.fp32)
        launch_links<float>(launch, dim3(chunk_count, splits), stream);
    else if (link_count)
        launch_links<double>(launch, dim3(chunk_count, splits), stream);
    if (launch.fp32)
        hipLaunchKernelGGL(gather_links<float>, dim3(destination_count), dim3(256), 0, stream, launch);
    else
        hipLaunchKernelGGL(gather_links<double>, dim3(destination_count), dim3(256), 0, stream, launch);
}

void launch_gather_blocks(const std::uint32_t *row_offsets, const std::uint32_t *columns, const double *values,
                          const std::uint32_t *order, const std::uint32_t *position, std::uint32_t n,
                          std::uint32_t width, double *blocks, hipStream_t stream) {
    hipLaunchKernelGGL(gather_blocks, dim3((n + 255) / 256), dim3(256), 0, stream, row_offsets, columns, values, order,
                       position, n, width, blocks);
}

void launch_direct_far(const FmmDirectLaunch &launch, hipStream_t stream) {
    if (launch.nt)
        hipLaunchKernelGGL(direct_far, dim3(launch.nt), dim3(256), 0, stream, launch);
}

void launch_far_flux(const FmmFarFluxLaunch &launch, hipStream_t stream) {
    const std::uint64_t pairs = static_cast<std::uint64_t>(launch.nt) * launch.flux_count;
    if (pairs)
        hipLaunchKernelGGL(far_flux, dim3(static_cast<std::uint32_t>((pairs + 255) / 256)), dim3(256), 0, stream, launch);
}

void launch_flux_csr_apply(const std::uint32_t *offsets, const std::uint32_t *columns, const double *values,
                           std::uint32_t rows, const double *q, std::uint32_t faces, std::uint32_t excitations,
                           double *out, hipStream_t stream) {
    if (rows && faces)
        hipLaunchKernelGGL(flux_csr_apply, dim3((rows + 255) / 256), dim3(256), 0, stream, offsets, columns, values,
                           rows, q, faces, excitations, out);
}

void launch_permute(const double *in, double *out, const std::uint32_t *map, std::uint32_t n, std::uint32_t count,
                    bool forward, hipStream_t stream) {
    const std::uint64_t total = static_cast<std::uint64_t>(n) * count;
    if (total)
        hipLaunchKernelGGL(permute_vectors, dim3(static_cast<std::uint32_t>((total + 255) / 256)), dim3(256), 0,
                           stream, in, out, map, n, count, forward);
}

} // namespace hsbem::dev
