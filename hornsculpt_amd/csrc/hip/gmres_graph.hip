// Arnoldi steps of GMRES: the fused orthogonalization that every GMRES here runs (one
// system, several at once, host-driven or captured), and the device-resident restart
// cycle of one right-hand side.
//
// Orthogonalization. At the orders of a horn (500 to 20,000 unknowns) the basis is a few
// MB, so a step is bound by its chain of dependent launches and not by bytes. CGS2, the
// norm and v_{j+1} = w / |w| are therefore four launches: each reduction's partials are
// summed by every workgroup of the launch that needs them (`blocks` x (j + 1) values out of
// L2) instead of by a launch of their own, and each workgroup keeps its rows of w in LDS
// from the subtraction to the next projection. Against ten launches a step (two
// projections, two sums, two subtractions, two norm launches, scaling, rotation), whole
// solves with the rest unchanged: mixed form on a horn of edge 20 mm (4 frequencies, about
// 37 steps each) 16.0 -> 12.9 ms; four systems at once on the horn of edge 8 mm
// 45.2 -> 35.8 ms; one system on that of 5.2 mm (10,373 unknowns, 86 steps) 77.4 -> 74.0 ms.
//
// Restart cycle. The Arnoldi step index j, the Hessenberg column, the Givens rotations, the
// rotated right-hand side g and the stop decision live in device memory, so one
// Arnoldi step is a fixed sequence of launches (the operator's input from v_j, the
// product, the orthogonalization, the rotation) whose arguments never change:
// the host captures it once into a HIP graph and replays it once per iteration,
// reading the state back only every few steps. Each kernel reads j from the state
// and returns at once when the cycle has stopped (target met, breakdown or the
// step limit), so replays queued past the stop cost only their launches. The rotation
// publishes the next j and the stop flag while other workgroups of its launch still run:
// they read the copies that the step's first kernel made.
#include "device.hpp"
#include "kernels.hpp"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

namespace hsbem::dev {
namespace {

enum : int { S_J = 0, S_DONE = 1, S_USED = 2, S_LIMIT = 3, S_ERROR = 4, S_STEP_J = 5, S_STEP_DONE = 6 };

constexpr int kThreads = 512, kWaves = kThreads / 64;
constexpr std::uint32_t kColumns = 256; // basis columns whose coefficients are held in LDS at a time
constexpr std::uint32_t kFinishRows = 256;

// Rows per lane of a pass: 64 rows per workgroup up to n = 4096 (at most 64 workgroups),
// 128 up to 16384 (at most 128), else 256, so that the partials that every workgroup sums
// stay near 100 KB at 60 columns while small systems still spread over the chip.
std::uint32_t rows_per_lane(std::uint32_t n) { return n <= 4096 ? 1 : n <= 16384 ? 2 : 4; }
std::uint32_t pass_blocks(std::uint32_t n) { return (n + 64 * rows_per_lane(n) - 1) / (64 * rows_per_lane(n)); }

struct Layout {
    std::uint32_t stride; // restart + 1
    __host__ __device__ std::size_t h1() const { return 0; }
    __host__ __device__ std::size_t h2() const { return 2 * static_cast<std::size_t>(stride); }
    __host__ __device__ std::size_t nrm() const { return 4 * static_cast<std::size_t>(stride); }
    __host__ __device__ std::size_t target() const { return nrm() + 1; }
    __host__ __device__ std::size_t resid() const { return nrm() + 2; }
    __host__ __device__ std::size_t g() const { return nrm() + 4; }
    __host__ __device__ std::size_t cs() const { return g() + 2 * static_cast<std::size_t>(stride); }
    __host__ __device__ std::size_t sn() const { return cs() + stride; }
    __host__ __device__ std::size_t H() const { return sn() + 2 * static_cast<std::size_t>(stride); }
    __host__ __device__ std::size_t total() const { return H() + 2 * static_cast<std::size_t>(stride) * stride; }
};

__global__ void cycle_begin(int *st, double *small, Layout L, double beta, double target, std::uint32_t limit) {
    const std::uint32_t t = threadIdx.x;
    for (std::size_t i = t; i < 2 * static_cast<std::size_t>(L.stride); i += blockDim.x)
        small[L.g() + i] = 0.0;
    __syncthreads();
    if (t == 0) {
        small[L.g()] = beta;
        small[L.target()] = target;
        small[L.resid()] = beta;
        st[S_J] = 0;
        st[S_DONE] = limit == 0 ? 1 : 0;
        st[S_USED] = 0;
        st[S_LIMIT] = static_cast<int>(limit);
        st[S_ERROR] = 0;
        st[S_STEP_J] = 0;
        st[S_STEP_DONE] = st[S_DONE];
    }
}

// The step index of this launch; false when the cycle has stopped.
__device__ __forceinline__ bool step_index(const ArnoldiBatch &B, std::uint32_t &j) {
    j = B.state ? static_cast<std::uint32_t>(B.state[S_STEP_J]) : B.j;
    return !(B.state && B.state[S_STEP_DONE] != 0);
}

// First kernel of a step: j and the stop flag as the last rotation left them, copied for
// the kernels that follow.
__device__ __forceinline__ bool step_begin(const ArnoldiBatch &B, std::uint32_t &j) {
    if (!B.state) {
        j = B.j;
        return true;
    }
    const int done = B.state[S_DONE], at = B.state[S_J];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        B.state[S_STEP_J] = at;
        B.state[S_STEP_DONE] = done;
    }
    j = static_cast<std::uint32_t>(at);
    return done == 0;
}

// in[a] = v_j of the a-th system of the batch.
__global__ __launch_bounds__(256) void load_step(ArnoldiBatch B, double2 *in) {
    std::uint32_t j;
    if (!step_begin(B, j))
        return;
    const std::uint32_t i = blockIdx.x * 256 + threadIdx.x, a = blockIdx.y;
    if (i < B.n)
        in[static_cast<std::size_t>(a) * B.n + i] =
            reinterpret_cast<const double2 *>(B.basis + B.which[a] * B.basis_stride)[static_cast<std::size_t>(j) * B.n + i];
}

// in[a] = M^{-1} v_j with the 64-wide block-Jacobi inverses: one workgroup per block and
// system, each wavefront a quarter of the block's columns.
__global__ __launch_bounds__(256) void jacobi_step(ArnoldiBatch B, const double2 *inverses, double2 *in) {
    __shared__ double2 sv[64], red[4][64];
    std::uint32_t j;
    if (!step_begin(B, j))
        return;
    const std::uint32_t blk = blockIdx.x, r0 = blk * 64, a = blockIdx.y;
    const int i = threadIdx.x & 63, wave = threadIdx.x / 64;
    const double2 *f = inverses + static_cast<std::size_t>(blk) * 4096 + 1024 * wave;
    double2 c[16];
#pragma unroll
    for (int t = 0; t < 16; ++t)
        c[t] = f[t * 64 + i];
    if (wave == 0)
        sv[i] = r0 + i < B.n ? reinterpret_cast<const double2 *>(B.basis + B.which[a] * B.basis_stride)
                                   [static_cast<std::size_t>(j) * B.n + r0 + i]
                             : double2{0, 0};
    __syncthreads();
    double re = 0, im = 0;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        const double2 v = sv[16 * wave + t];
        re += c[t].x * v.x - c[t].y * v.y;
        im += c[t].x * v.y + c[t].y * v.x;
    }
    red[wave][i] = double2{re, im};
    __syncthreads();
    if (wave == 0 && r0 + i < B.n)
        in[static_cast<std::size_t>(a) * B.n + r0 + i] =
            double2{red[0][i].x + red[1][i].x + red[2][i].x + red[3][i].x,
                    red[0][i].y + red[1][i].y + red[2][i].y + red[3][i].y};
}

// Sum over the wavefront of eight values: lane l returns the sum of v[l & 7]. Three
// exchanges halve the values a lane carries and three more add the lanes that carry the
// same one: 10 exchanges where eight separate sums take 48.
__device__ __forceinline__ double wave_sum8(const double *v, int lane) {
    double a[4], b[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bool hi = lane & 4;
        a[i] = (hi ? v[i + 4] : v[i]) + __shfl_xor(hi ? v[i] : v[i + 4], 4, 64);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const bool hi = lane & 2;
        b[i] = (hi ? a[i + 2] : a[i]) + __shfl_xor(hi ? a[i] : a[i + 2], 2, 64);
    }
    const bool hi = lane & 1;
    double s = (hi ? b[1] : b[0]) + __shfl_xor(hi ? b[0] : b[1], 1, 64);
#pragma unroll
    for (int off = 8; off < 64; off <<= 1)
        s += __shfl_xor(s, off, 64);
    return s;
}

// One pass over the rows of w = v_{j+1}'s slot, 64 RK rows per workgroup, blockIdx.y the
// system. kGather: w = the product's column-chunk partials summed, then part1[b][c] = this
// block's share of conj(v_c) w. kFirst: h1 = the sum of part1, w -= V h1, part2 likewise.
// kSecond: h2 = the sum of part2, w -= V h2, part1[b] = this block's |w|^2. (part1 is read
// by kFirst only, so kSecond may write it.) Rows are lanes and the wavefronts share the
// columns in the subtraction; a wavefront takes four columns at a time in the projection.
enum Pass { kGather, kFirst, kSecond };
template <int RK, Pass PASS>
__global__ __launch_bounds__(kThreads) void arnoldi_pass(ArnoldiBatch B, const double2 *y, std::uint32_t chunks) {
    constexpr int R = 64 * RK;
    __shared__ double2 sw[R], red[kWaves * R], sh[kColumns];
    std::uint32_t j;
    if (!step_index(B, j))
        return;
    const std::uint32_t m = j + 1, n = B.n, ld = B.restart + 1, blocks = gridDim.x, a = blockIdx.y, e = B.which[a];
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
    const std::uint32_t r0 = blockIdx.x * R;
    const double2 *V = reinterpret_cast<const double2 *>(B.basis + e * B.basis_stride);
    double2 *w = reinterpret_cast<double2 *>(B.basis + e * B.basis_stride) + static_cast<std::size_t>(m) * n;
    double2 *part1 = reinterpret_cast<double2 *>(B.part) + 2 * static_cast<std::size_t>(a) * blocks * ld;
    double2 *part2 = part1 + static_cast<std::size_t>(blocks) * ld;
    double2 acc[RK] = {};
    if constexpr (PASS == kGather) {
        for (std::uint32_t c = wave; c < chunks; c += kWaves)
#pragma unroll
            for (int k = 0; k < RK; ++k) {
                const std::uint32_t row = r0 + 64 * k + lane;
                if (row < n) {
                    const double2 v = y[(static_cast<std::size_t>(a) * chunks + c) * n + row];
                    acc[k].x += v.x;
                    acc[k].y += v.y;
                }
            }
    } else {
        const double2 *part = PASS == kFirst ? part1 : part2;
        double2 *h = reinterpret_cast<double2 *>(B.small + e * B.small_stride) + (PASS == kFirst ? 0 : ld);
        for (std::uint32_t c0 = 0; c0 < m; c0 += kColumns) {
            const std::uint32_t cn = min(kColumns, m - c0);
            for (std::uint32_t q = 0; q < cn; q += 64) {
                double2 s = {};
                if (q + lane < cn)
#pragma unroll 8
                    for (std::uint32_t b = wave; b < blocks; b += kWaves) {
                        const double2 v = part[static_cast<std::size_t>(b) * ld + c0 + q + lane];
                        s.x += v.x;
                        s.y += v.y;
                    }
                red[wave * 64 + lane] = s;
                __syncthreads();
                if (wave == 0 && q + lane < cn) {
#pragma unroll
                    for (int t = 1; t < kWaves; ++t) {
                        s.x += red[t * 64 + lane].x;
                        s.y += red[t * 64 + lane].y;
                    }
                    sh[q + lane] = s;
                    if (blockIdx.x == 0)
                        h[c0 + q + lane] = s;
                }
                __syncthreads();
            }
#pragma unroll 4
            for (std::uint32_t c = wave; c < cn; c += kWaves) {
                const double2 hc = sh[c];
                const double2 *col = V + static_cast<std::size_t>(c0 + c) * n;
#pragma unroll
                for (int k = 0; k < RK; ++k) {
                    const std::uint32_t row = r0 + 64 * k + lane;
                    const double2 v = row < n ? col[row] : double2{0, 0};
                    acc[k].x += v.x * hc.x - v.y * hc.y;
                    acc[k].y += v.x * hc.y + v.y * hc.x;
                }
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int k = 0; k < RK; ++k)
        red[wave * R + 64 * k + lane] = acc[k];
    __syncthreads();
    for (int t = threadIdx.x; t < R; t += kThreads) {
        double2 s = red[t];
#pragma unroll
        for (int q = 1; q < kWaves; ++q) {
            s.x += red[q * R + t].x;
            s.y += red[q * R + t].y;
        }
        if (r0 + t < n) {
            if (PASS != kGather)
                s = double2{w[r0 + t].x - s.x, w[r0 + t].y - s.y};
            w[r0 + t] = s;
        }
        sw[t] = r0 + t < n ? s : double2{0, 0};
    }
    __syncthreads();
    if constexpr (PASS == kSecond) {
        if (wave == 0) {
            double s = 0;
#pragma unroll
            for (int k = 0; k < RK; ++k)
                s += sw[64 * k + lane].x * sw[64 * k + lane].x + sw[64 * k + lane].y * sw[64 * k + lane].y;
            s = wave_sum(s);
            if (lane == 0)
                reinterpret_cast<double *>(part1)[blockIdx.x] = s;
        }
    } else {
        double *out = reinterpret_cast<double *>((PASS == kGather ? part1 : part2) + static_cast<std::size_t>(blockIdx.x) * ld);
        for (std::uint32_t c = 4 * wave; c < m; c += 4 * kWaves) {
            double v[8] = {};
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int k = 0; k < RK; ++k) {
                    const std::uint32_t row = r0 + 64 * k + lane;
                    const double2 x = row < n && c + u < m ? V[static_cast<std::size_t>(c + u) * n + row] : double2{0, 0};
                    const double2 wr = sw[64 * k + lane];
                    v[2 * u] += x.x * wr.x + x.y * wr.y;
                    v[2 * u + 1] += x.x * wr.y - x.y * wr.x;
                }
            const double s = wave_sum8(v, lane);
            if (lane < 8 && c + lane / 2 < m)
                out[2 * c + lane] = s;
        }
    }
}

struct Cx {
    double re, im;
};
__device__ __forceinline__ Cx cmul(Cx a, Cx b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ Cx cadd(Cx a, Cx b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ Cx cscale(Cx a, double s) { return {a.re * s, a.im * s}; }
__device__ __forceinline__ Cx cconj(Cx a) { return {a.re, -a.im}; }
__device__ __forceinline__ Cx cneg(Cx a) { return {-a.re, -a.im}; }
__device__ __forceinline__ double cabs(Cx a) { return hypot(a.re, a.im); }

// Column j of the Hessenberg matrix from the two CGS passes and |w|, the earlier
// rotations applied to it, the new rotation, g rotated, and the stop decision. The chain
// of rotations is one lane's work on staged values (through global memory the three loads
// of each rotation were its time: about 15 us at 60 columns).
__device__ void rotate_column(int *st, double *small, Layout L, std::uint32_t j, double norm2, Cx *scol, Cx *ssn,
                              double *scs) {
    Cx *col = reinterpret_cast<Cx *>(small + L.H()) + static_cast<std::size_t>(j) * L.stride;
    const Cx *h1 = reinterpret_cast<const Cx *>(small + L.h1()), *h2 = reinterpret_cast<const Cx *>(small + L.h2());
    Cx *g = reinterpret_cast<Cx *>(small + L.g()), *sn = reinterpret_cast<Cx *>(small + L.sn());
    double *cs = small + L.cs();
    const std::uint32_t tid = threadIdx.x;
    const double next = sqrt(norm2);
    Cx cur = cadd(h1[0], h2[0]); // lane 0's: entry i of the column with the rotations before i applied
    for (std::uint32_t i0 = 0; i0 < j; i0 += kColumns) {
        const std::uint32_t in = min(kColumns, j - i0);
        for (std::uint32_t i = tid; i < in; i += blockDim.x) {
            scol[i] = cadd(h1[i0 + i + 1], h2[i0 + i + 1]);
            ssn[i] = sn[i0 + i];
            scs[i] = cs[i0 + i];
        }
        __syncthreads();
        if (tid == 0)
#pragma unroll 4
            for (std::uint32_t i = 0; i < in; ++i) {
                const Cx below = scol[i], s = ssn[i];
                const double c = scs[i];
                scol[i] = cadd(cscale(cur, c), cmul(s, below));
                cur = cadd(cmul(cneg(cconj(s)), cur), cscale(below, c));
            }
        __syncthreads();
        for (std::uint32_t i = tid; i < in; i += blockDim.x)
            col[i0 + i] = scol[i];
        __syncthreads();
    }
    for (std::uint32_t i = j + 2 + tid; i < L.stride; i += blockDim.x)
        col[i] = {0.0, 0.0};
    if (tid != 0)
        return;
    small[L.nrm()] = norm2;
    const Cx a = cur, bb = {next, 0.0};
    const bool breakdown = !(next > 0);
    const double absa = cabs(a), len = hypot(absa, cabs(bb));
    if (!(len > 0) || !isfinite(len)) {
        st[S_ERROR] = 1;
        st[S_DONE] = 1;
        return;
    }
    const Cx phase = absa > 0 ? Cx{a.re / absa, a.im / absa} : Cx{1.0, 0.0};
    const double c = absa / len;
    const Cx sp = cmul(phase, cconj(bb)), sj = {sp.re / len, sp.im / len};
    cs[j] = c;
    sn[j] = sj;
    col[j] = cscale(phase, len);
    col[j + 1] = {0.0, 0.0};
    const Cx gj = g[j], gn = g[j + 1];
    const Cx gr = cadd(cmul(cneg(cconj(sj)), gj), cscale(gn, c));
    g[j] = cadd(cscale(gj, c), cmul(sj, gn));
    g[j + 1] = gr;
    const double resid = cabs(gr);
    small[L.resid()] = resid;
    st[S_USED] = static_cast<int>(j + 1);
    st[S_J] = static_cast<int>(j + 1);
    if (resid <= small[L.target()] || breakdown || static_cast<int>(j + 1) >= st[S_LIMIT])
        st[S_DONE] = 1;
}

// v_{j+1} = w / |w| (0 when |w| = 0) in place; every wavefront sums the norm's partials.
// With a device cycle the last workgroup rotates the column instead, else |w|^2 goes
// behind h1 and h2.
__global__ __launch_bounds__(kFinishRows) void finish_step(ArnoldiBatch B, std::uint32_t blocks) {
    __shared__ Cx scol[kColumns], ssn[kColumns];
    __shared__ double scs[kColumns];
    std::uint32_t j;
    if (!step_index(B, j))
        return;
    const std::uint32_t n = B.n, ld = B.restart + 1, a = blockIdx.y, e = B.which[a], lane = threadIdx.x & 63;
    const double *part = B.part + 4 * static_cast<std::size_t>(a) * blocks * ld;
    double v = 0;
    for (std::uint32_t b = lane; b < blocks; b += 64)
        v += part[b];
    v = wave_sum(v);
    const std::uint32_t i = blockIdx.x * kFinishRows + threadIdx.x;
    if (blockIdx.x * kFinishRows >= n) {
        rotate_column(B.state, B.small, Layout{ld}, j, v, scol, ssn, scs);
        return;
    }
    if (!B.state && i == 0)
        B.small[e * B.small_stride + 4 * ld] = v;
    if (i >= n)
        return;
    double2 *w = reinterpret_cast<double2 *>(B.basis + e * B.basis_stride) + static_cast<std::size_t>(j + 1) * n;
    const double len = sqrt(v);
    w[i] = v > 0 ? double2{w[i].x / len, w[i].y / len} : double2{0, 0};
}

template <int RK>
void launch_passes(const ArnoldiBatch &B, const double *y, std::uint32_t chunks, hipStream_t s) {
    const dim3 grid(pass_blocks(B.n), B.count), block(kThreads);
    const double2 *yv = reinterpret_cast<const double2 *>(y);
    hipLaunchKernelGGL((arnoldi_pass<RK, kGather>), grid, block, 0, s, B, yv, chunks);
    hipLaunchKernelGGL((arnoldi_pass<RK, kFirst>), grid, block, 0, s, B, nullptr, 0u);
    hipLaunchKernelGGL((arnoldi_pass<RK, kSecond>), grid, block, 0, s, B, nullptr, 0u);
}

} // namespace

std::size_t gmres_cycle_small_doubles(std::uint32_t restart) { return Layout{restart + 1}.total(); }
std::size_t arnoldi_part_doubles(std::uint32_t n, std::uint32_t restart) {
    return 4 * static_cast<std::size_t>(pass_blocks(n)) * (restart + 1);
}
std::size_t gmres_cycle_h_offset(std::uint32_t restart) { return Layout{restart + 1}.H(); }
std::size_t gmres_cycle_g_offset(std::uint32_t restart) { return Layout{restart + 1}.g(); }

void gmres_cycle_begin(const ArnoldiBatch &c, double beta, double target, std::uint32_t limit, hipStream_t s) {
    hipLaunchKernelGGL(cycle_begin, dim3(1), dim3(256), 0, s, c.state, c.small, Layout{c.restart + 1}, beta, target,
                       limit);
}

void arnoldi_load(const ArnoldiBatch &B, double *in, hipStream_t s) {
    hipLaunchKernelGGL(load_step, dim3((B.n + 255) / 256, B.count), dim3(256), 0, s, B, reinterpret_cast<double2 *>(in));
}

void arnoldi_precondition(const ArnoldiBatch &B, const double *inverses, double *in, hipStream_t s) {
    hipLaunchKernelGGL(jacobi_step, dim3((B.n + 63) / 64, B.count), dim3(256), 0, s, B,
                       reinterpret_cast<const double2 *>(inverses), reinterpret_cast<double2 *>(in));
}

void arnoldi_orthogonalize(const ArnoldiBatch &B, const double *y, std::uint32_t chunks, hipStream_t s) {
    switch (rows_per_lane(B.n)) {
    case 1: launch_passes<1>(B, y, chunks, s); break;
    case 2: launch_passes<2>(B, y, chunks, s); break;
    default: launch_passes<4>(B, y, chunks, s);
    }
    hipLaunchKernelGGL(finish_step, dim3((B.n + kFinishRows - 1) / kFinishRows + (B.state ? 1 : 0), B.count),
                       dim3(kFinishRows), 0, s, B, pass_blocks(B.n));
}

} // namespace hsbem::dev
