// Dense complex FP64 linear algebra for the Burton-Miller system, gfx950.
//
// Replaces the vendor calls of the reference dense path
// (cublasZgemv/Zaxpy/Dznrm2 in device_gmres.cu:115-157; the LU is in lu.hip) with own kernels:
//   gemv            y = A X for up to 8 vectors (A FP64 or FP32, vectors FP64):
//                   64 rows x 512 columns per workgroup, A streamed once (HBM
//                   bound), deterministic split-K partials reduced in a second pass;
//                   for one vector the column chunk (512, 1024 or 2048) is chosen by
//                   timing the candidates once per (n, precision) on the live stream.
//   project         CGS2 projections V^H w, one wavefront per (basis column, row block).
#include "../autotune.hpp"
#include "device.hpp"

#include <algorithm>
#include <cstdlib>
#include <optional>
#include <string>
#include <utility>
#include <vector>

namespace hsbem::dev {
namespace {

constexpr int kGemvRows = 64;    // rows per workgroup (one per lane)
constexpr int kGemvWaves = 4;    // waves per workgroup, splitting the column chunk
constexpr int kGemvCols = 512;   // columns per workgroup (split-K chunk)
constexpr int kGemvUnroll = 8;   // column loads in flight per lane
constexpr int kMaxVec = 8;

// Split-K partial products: workgroup (row block, column chunk); lane = row, the
// four waves take interleaved columns of the chunk and are summed in LDS, so one
// partial per (chunk, row) reaches HBM.
template <int NV, class T, int COLS = kGemvCols>
__global__ __launch_bounds__(kGemvRows *kGemvWaves) void gemv_partial(const T *__restrict__ A, std::uint32_t n,
                                                                     const double *__restrict__ x,
                                                                     std::uint32_t chunks, double *__restrict__ part,
                                                                     const int *skip) {
    if (skip && *skip) // a device-resident solver loop has already finished
        return;
    __shared__ double sx[NV][2 * COLS];
    __shared__ double red[kGemvWaves - 1][NV][2][kGemvRows];
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
    const std::uint32_t row = blockIdx.x * kGemvRows + lane;
    const std::uint32_t c0 = blockIdx.y * COLS;
    const std::uint32_t cn = min(static_cast<std::uint32_t>(COLS), n - c0);
    for (std::uint32_t e = threadIdx.x; e < NV * 2 * COLS; e += kGemvRows * kGemvWaves) {
        const std::uint32_t v = e / (2 * COLS), c = e % (2 * COLS);
        sx[v][c] = c / 2 < cn ? x[2 * (static_cast<std::size_t>(v) * n + c0) + c] : 0.0;
    }
    __syncthreads();
    double re[NV], im[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v)
        re[v] = im[v] = 0.0;
    if (row < n) {
        const T *col = A + static_cast<std::size_t>(c0) * n + row;
        std::uint32_t c = wave;
        for (; c + kGemvWaves * (kGemvUnroll - 1) < cn; c += kGemvWaves * kGemvUnroll) {
            T a[kGemvUnroll];
#pragma unroll
            for (int u = 0; u < kGemvUnroll; ++u)
                a[u] = col[static_cast<std::size_t>(c + kGemvWaves * u) * n];
#pragma unroll
            for (int u = 0; u < kGemvUnroll; ++u) {
                const double ar = a[u].x, ai = a[u].y;
                const std::uint32_t cc = c + kGemvWaves * u;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const double xr = sx[v][2 * cc], xi = sx[v][2 * cc + 1];
                    re[v] += ar * xr - ai * xi;
                    im[v] += ar * xi + ai * xr;
                }
            }
        }
        for (; c < cn; c += kGemvWaves) {
            const T a = col[static_cast<std::size_t>(c) * n];
            const double ar = a.x, ai = a.y;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const double xr = sx[v][2 * c], xi = sx[v][2 * c + 1];
                re[v] += ar * xr - ai * xi;
                im[v] += ar * xi + ai * xr;
            }
        }
    }
    if (wave > 0)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            red[wave - 1][v][0][lane] = re[v];
            red[wave - 1][v][1][lane] = im[v];
        }
    __syncthreads();
    if (wave == 0 && row < n)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            double sr = re[v], si = im[v];
#pragma unroll
            for (int w = 0; w < kGemvWaves - 1; ++w) {
                sr += red[w][v][0][lane];
                si += red[w][v][1][lane];
            }
            const std::size_t o = (static_cast<std::size_t>(v) * chunks + blockIdx.y) * n + row;
            part[2 * o] = sr;
            part[2 * o + 1] = si;
        }
}

// The same split-K partials for an FP32 matrix and one vector with ROWS (2 or 4)
// consecutive rows per lane: ROWS / 2 adjacent 16-byte loads per column, so a
// wavefront covers 64 ROWS rows with fewer, wider load instructions. Needs n a
// multiple of ROWS (every column then starts on a 16-byte boundary and no lane is
// partly past the last row).
template <int COLS, int ROWS>
__global__ __launch_bounds__(kGemvRows *kGemvWaves) void gemv_partial_rows(const float2 *__restrict__ A,
                                                                          std::uint32_t n,
                                                                          const double *__restrict__ x,
                                                                          std::uint32_t chunks,
                                                                          double *__restrict__ part, const int *skip) {
    static_assert(ROWS == 2 || ROWS == 4, "two or four rows per lane");
    constexpr int kQuads = ROWS / 2;                 // float4 loads per column per lane
    constexpr int kUnroll = kGemvUnroll * 2 / ROWS;  // the same bytes in flight for both widths
    if (skip && *skip)
        return;
    __shared__ double sx[2 * COLS];
    __shared__ double red[kGemvWaves - 1][2 * ROWS][kGemvRows];
    const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
    const std::uint32_t row = ROWS * (blockIdx.x * kGemvRows + lane);
    const std::uint32_t c0 = blockIdx.y * COLS;
    const std::uint32_t cn = min(static_cast<std::uint32_t>(COLS), n - c0);
    for (std::uint32_t c = threadIdx.x; c < 2 * COLS; c += kGemvRows * kGemvWaves)
        sx[c] = c / 2 < cn ? x[2 * static_cast<std::size_t>(c0) + c] : 0.0;
    __syncthreads();
    double acc[2 * ROWS] = {}; // re, im per row
    if (row < n) {
        const std::size_t stride = n / 2; // one column in float4 units
        const float4 *col = reinterpret_cast<const float4 *>(A + static_cast<std::size_t>(c0) * n + row);
        auto mac = [&](const float4 a, int q, std::uint32_t cc) {
            const double xr = sx[2 * cc], xi = sx[2 * cc + 1];
            const double a0 = a.x, b0 = a.y, a1 = a.z, b1 = a.w;
            acc[4 * q] += a0 * xr - b0 * xi;
            acc[4 * q + 1] += a0 * xi + b0 * xr;
            acc[4 * q + 2] += a1 * xr - b1 * xi;
            acc[4 * q + 3] += a1 * xi + b1 * xr;
        };
        std::uint32_t c = wave;
        for (; c + kGemvWaves * (kUnroll - 1) < cn; c += kGemvWaves * kUnroll) {
            float4 a[kUnroll][kQuads];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
#pragma unroll
                for (int q = 0; q < kQuads; ++q)
                    a[u][q] = col[static_cast<std::size_t>(c + kGemvWaves * u) * stride + q];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
#pragma unroll
                for (int q = 0; q < kQuads; ++q)
                    mac(a[u][q], q, c + kGemvWaves * u);
        }
        for (; c < cn; c += kGemvWaves)
#pragma unroll
            for (int q = 0; q < kQuads; ++q)
                mac(col[static_cast<std::size_t>(c) * stride + q], q, c);
    }
    if (wave > 0)
#pragma unroll
        for (int q = 0; q < 2 * ROWS; ++q)
            red[wave - 1][q][lane] = acc[q];
    __syncthreads();
    if (wave == 0 && row < n) {
#pragma unroll
        for (int w = 0; w < kGemvWaves - 1; ++w)
#pragma unroll
            for (int q = 0; q < 2 * ROWS; ++q)
                acc[q] += red[w][q][lane];
        const std::size_t o = static_cast<std::size_t>(blockIdx.y) * n + row;
#pragma unroll
        for (int q = 0; q < 2 * ROWS; ++q)
            part[2 * o + q] = acc[q];
    }
}

__global__ void gemv_reduce(const double *part, std::uint32_t n, std::uint32_t chunks, std::uint32_t nvec, double *y,
                            const int *skip) {
    if (skip && *skip)
        return;
    const std::size_t idx = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= static_cast<std::size_t>(n) * nvec)
        return;
    const std::uint32_t row = idx % n, v = idx / n;
    double re = 0, im = 0;
    for (std::uint32_t c = 0; c < chunks; ++c) {
        const std::size_t o = (static_cast<std::size_t>(v) * chunks + c) * n + row;
        re += part[2 * o];
        im += part[2 * o + 1];
    }
    y[2 * idx] = re;
    y[2 * idx + 1] = im;
}

__global__ void subtract_combination(const double *V, std::uint32_t n, std::uint32_t m, const double *h, double *w) {
    const std::uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n)
        return;
    double re = w[2 * r], im = w[2 * r + 1];
    for (std::uint32_t j = 0; j < m; ++j) {
        const double vr = V[2 * (static_cast<std::size_t>(j) * n + r)], vi = V[2 * (static_cast<std::size_t>(j) * n + r) + 1];
        const double hr = h[2 * j], hi = h[2 * j + 1];
        re -= vr * hr - vi * hi;
        im -= vr * hi + vi * hr;
    }
    w[2 * r] = re;
    w[2 * r + 1] = im;
}

__global__ __launch_bounds__(256) void norm_partial(const double *x, std::uint32_t n, const double *weight,
                                                   double *part) {
    __shared__ double red[4];
    double s = 0;
    for (std::uint32_t r = blockIdx.x * 256 + threadIdx.x; r < n; r += gridDim.x * 256) {
        const double f = weight ? weight[r] : 1.0;
        const double a = x[2 * r] * f, b = x[2 * r + 1] * f;
        s += a * a + b * b;
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0)
        red[threadIdx.x / 64] = s;
    __syncthreads();
    if (threadIdx.x == 0)
        part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

__global__ void norm_finish(const double *part, std::uint32_t blocks, double *out) {
    double s = 0;
    for (std::uint32_t b = threadIdx.x; b < blocks; b += 64)
        s += part[b];
    s = wave_sum(s);
    if (threadIdx.x == 0)
        out[0] = s;
}

__global__ void axpy_kernel(std::uint32_t n, const double *alpha, const double *x, double *y) {
    const std::uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n)
        return;
    const double ar = alpha[0], ai = alpha[1], xr = x[2 * r], xi = x[2 * r + 1];
    y[2 * r] += ar * xr - ai * xi;
    y[2 * r + 1] += ar * xi + ai * xr;
}

__global__ void add_kernel(std::uint32_t n, const double *x, double *y) {
    const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * n)
        return;
    y[i] += x[i];
}

__global__ void subtract_from_kernel(std::uint32_t n, const double *b, double *r) {
    const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * n)
        return;
    r[i] = b[i] - r[i];
}

__global__ void scale_kernel(std::uint32_t n, double s, const double *x, double *y) {
    const std::uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n)
        return;
    y[2 * r] = s * x[2 * r];
    y[2 * r + 1] = s * x[2 * r + 1];
}

__global__ void subtract_vectors(const double *b, const double *ax, std::size_t count, double *r) {
    const std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < count)
        r[i] = b[i] - ax[i];
}

// ---- block-Jacobi preconditioner: explicit inverses of the kJacobi x kJacobi
// diagonal blocks (consecutive internal nodes, i.e. spatial clusters) of the
// row-scaled system, one workgroup per block, with partial pivoting. FP64, column-major
// per block. A block whose pivot vanishes is replaced by the identity. The apply
// is then a block-diagonal matrix-vector product.
constexpr int kJacobi = 64;

// Diagonal block entry (row r, column c of block blk) of a dense column-major matrix.
template <class T> struct DenseBlocks {
    const T *A;
    std::uint32_t n;
    __device__ double2 operator()(std::uint32_t blk, int r, int c) const {
        const T v = A[static_cast<std::size_t>(blk * kJacobi + c) * n + blk * kJacobi + r];
        return {static_cast<double>(v.x), static_cast<double>(v.y)};
    }
};

// ... of gathered blocks (complex FP64, column-major per block).
struct GatheredBlocks {
    const double *B;
    __device__ double2 operator()(std::uint32_t blk, int r, int c) const {
        const double *e = B + 2 * ((static_cast<std::size_t>(blk) * kJacobi + c) * kJacobi + r);
        return {e[0], e[1]};
    }
};

// Largest value over the wavefront, the same in every lane.
__device__ __forceinline__ std::uint64_t wave_max(std::uint64_t v) {
    auto step = [&](auto control) {
        constexpr int kControl = decltype(control)::value;
        const std::uint32_t lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(v), kControl, 0xf, 0xf, true),
                            hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(v >> 32), kControl, 0xf, 0xf, true);
        const std::uint64_t o = static_cast<std::uint64_t>(hi) << 32 | lo;
        v = o > v ? o : v;
    };
    step(std::integral_constant<int, 0x111>{}); // row_shr 1, 2, 4, 8: lane 15 of a row has its maximum
    step(std::integral_constant<int, 0x112>{});
    step(std::integral_constant<int, 0x114>{});
    step(std::integral_constant<int, 0x118>{});
    step(std::integral_constant<int, 0x142>{}); // row_bcast 15, 31: lane 63 the wavefront's
    step(std::integral_constant<int, 0x143>{});
    const std::uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(v), 63),
                        hi = __builtin_amdgcn_readlane(static_cast<int>(v >> 32), 63);
    return static_cast<std::uint64_t>(hi) << 32 | lo;
}

__device__ __forceinline__ double lane_value(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Gauss-Jordan in registers: lane = row, each of the four wavefronts 16 columns. Step j
// takes the largest entry of column j among the rows without a pivot (magnitudes compared
// to 46 bits, then the first row), exchanges it and updates all columns; rows stay where they are and
// the permutation is applied on the way out: inverse(j, p_c) = G(p_j, c) for pivot rows p.
// Bound by the chain of 64 steps, one barrier each: column and pivot through LDS, the
// pivot row out of the registers. (LU in LDS with four barriers a step and one thread per
// column of the inverse took 280 us for any number of blocks up to 256, this 73 us.)
template <class Load>
__global__ __launch_bounds__(256) void jacobi_factor(Load load, std::uint32_t n, double *inverses) {
    __shared__ double2 column[2][kJacobi];
    __shared__ int chosen[2], order[kJacobi], pivot[kJacobi]; // order: step of a row; pivot: row of a step
    const std::uint32_t blk = blockIdx.x, r0 = blk * kJacobi;
    const int m = static_cast<int>(min(static_cast<std::uint32_t>(kJacobi), n - r0));
    const int r = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    double2 g[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int c = 16 * wave + i;
        g[i] = c < m && r < m ? load(blk, r, c) : double2{c == r ? 1.0 : 0.0, 0.0};
    }
    bool open = r < m, singular = false;
    for (int owner = 0; owner < 4; ++owner)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int j = 16 * owner + i, side = i & 1;
            if (j >= m || singular)
                continue;
            if (wave == owner) {
                const double mag = g[i].x * g[i].x + g[i].y * g[i].y;
                const std::uint64_t key =
                    open && mag > 0 ? (static_cast<std::uint64_t>(__double_as_longlong(mag)) & ~63ull) | (63 - r) : 0;
                const std::uint64_t best = wave_max(key);
                column[side][r] = g[i];
                if (r == 0) {
                    const int row = best >> 6 ? 63 - static_cast<int>(best & 63) : -1;
                    chosen[side] = row;
                    if (row >= 0) {
                        order[row] = j;
                        pivot[j] = row;
                    }
                }
            }
            __syncthreads();
            const int row = __builtin_amdgcn_readfirstlane(chosen[side]);
            if (row < 0) {
                singular = true;
                continue;
            }
            const double2 f = column[side][r], d = column[side][row];
            const double inv = 1.0 / (d.x * d.x + d.y * d.y);
            const double2 e = {d.x * inv, -d.y * inv}; // 1 / d
            const bool mine = r == row;
            open = open && !mine;
            // the pivot row times 1 / d, and the others less f times that
            const double2 s = mine ? double2{0, 0} : f;
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                double2 u = {lane_value(g[c].x, row), lane_value(g[c].y, row)};
                if (wave == owner && c == i)
                    u = double2{1, 0}; // the exchanged column
                const double2 t = {u.x * e.x - u.y * e.y, u.x * e.y + u.y * e.x};
                double2 v = mine ? t : wave == owner && c == i ? double2{0, 0} : g[c];
                v.x -= s.x * t.x - s.y * t.y;
                v.y -= s.x * t.y + s.y * t.x;
                g[c] = v;
            }
        }
    __syncthreads();
    double2 *out = reinterpret_cast<double2 *>(inverses) + static_cast<std::size_t>(blk) * kJacobi * kJacobi;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int c = 16 * wave + i;
        if (singular || c >= m || r >= m)
            out[c * kJacobi + r] = double2{c == r ? 1.0 : 0.0, 0.0};
        else
            out[pivot[c] * kJacobi + order[r]] = g[i];
    }
}

// out = M^{-1} v: one wavefront per block, lane = row, columns streamed. Block
// rows are order[r0 .. r0 + 64) when order is given, else consecutive.
__global__ __launch_bounds__(64) void jacobi_apply(const double *inverses, std::uint32_t n, const double *v,
                                                   double *out, const std::uint32_t *order) {
    __shared__ double sv[kJacobi][2];
    const std::uint32_t blk = blockIdx.x, r0 = blk * kJacobi;
    const int m = static_cast<int>(min(static_cast<std::uint32_t>(kJacobi), n - r0));
    const int i = threadIdx.x;
    const std::uint32_t row = i < m ? (order ? order[r0 + i] : r0 + i) : 0;
    sv[i][0] = i < m ? v[2 * row] : 0.0;
    sv[i][1] = i < m ? v[2 * row + 1] : 0.0;
    __syncthreads();
    const double2 *f = reinterpret_cast<const double2 *>(inverses) + static_cast<std::size_t>(blk) * kJacobi * kJacobi;
    double re = 0, im = 0;
#pragma unroll 8
    for (int c = 0; c < kJacobi; ++c) {
        const double2 b = f[c * kJacobi + i];
        re += b.x * sv[c][0] - b.y * sv[c][1];
        im += b.x * sv[c][1] + b.y * sv[c][0];
    }
    if (i < m) {
        out[2 * row] = re;
        out[2 * row + 1] = im;
    }
}

// Block-Jacobi of any block width W (the FMM preconditioner's preconditionerBlockWidth).
// One workgroup per gathered W x W block (complex FP64, column-major a[c * W + r]),
// factored in place in global memory by a right-looking LU with partial pivoting in
// panels of kWidePanel columns: the panel is factored column by column (pivot search,
// full-row interchange, scaling, update of the remaining panel columns), then the
// panel's rows of U are solved against the unit L11 and the trailing matrix takes
// one rank-kWidePanel update, so the trailing matrix is read and written once per panel
// instead of once per column. The inverse X = U^{-1} L^{-1} P is formed the same
// way: X starts as P, a blocked forward sweep with L and a blocked backward sweep
// with U, each a small per-column triangular solve plus a rank-kWidePanel update of the
// rows below (above). A vanishing pivot gives the identity block, as in the LDS kernel.
constexpr int kWidePanel = 16;

// A[r][c] -= sum_t L(r, t) U(t, c) for r in [rb, re), c in [cb, ce), t < kb, with
// L(r, t) = lp[t * W + r], U(t, c) = up[c * W + t]; all column-major with leading
// dimension W. A thread keeps its row of L in registers and streams columns; when
// there are fewer rows than threads, the threads split the columns into groups.
__device__ void rank_update(double2 *A, std::uint32_t W, int rb, int re, int cb, int ce, const double2 *lp,
                            const double2 *up, int kb) {
    const int rows = re - rb;
    if (rows <= 0 || ce <= cb)
        return;
    const int threads = static_cast<int>(blockDim.x);
    const int groups = rows >= threads ? 1 : threads / rows;
    for (int e = static_cast<int>(threadIdx.x); e < rows * groups; e += threads) {
        const int r = rb + e % rows, g = e / rows;
        double2 l[kWidePanel];
#pragma unroll
        for (int t = 0; t < kWidePanel; ++t)
            l[t] = t < kb ? lp[static_cast<std::size_t>(t) * W + r] : double2{0, 0};
        for (int c = cb + g; c < ce; c += groups) {
            double2 acc = A[static_cast<std::size_t>(c) * W + r];
            const double2 *u = up + static_cast<std::size_t>(c) * W;
#pragma unroll
            for (int t = 0; t < kWidePanel; ++t)
                if (t < kb) {
                    const double2 v = u[t];
                    acc.x -= l[t].x * v.x - l[t].y * v.y;
                    acc.y -= l[t].x * v.y + l[t].y * v.x;
                }
            A[static_cast<std::size_t>(c) * W + r] = acc;
        }
    }
}

__global__ __launch_bounds__(256) void jacobi_factor_wide(double *blocks, std::uint32_t n, std::uint32_t width,
                                                          double *inverses, std::int32_t *pivots) {
    __shared__ double red_mag[256];
    __shared__ int red_idx[256];
    __shared__ int singular;
    const std::uint32_t blk = blockIdx.x, W = width, r0 = blk * W;
    const int m = static_cast<int>(min(W, n - r0));
    double2 *a = reinterpret_cast<double2 *>(blocks) + static_cast<std::size_t>(blk) * W * W;
    std::int32_t *p = pivots + static_cast<std::size_t>(blk) * W;
    const int tid = threadIdx.x;
    auto at = [&](int c, int r) -> double2 & { return a[static_cast<std::size_t>(c) * W + r]; };
    for (int r = tid; r < static_cast<int>(W); r += 256)
        p[r] = r;
    if (tid == 0)
        singular = 0;
    __syncthreads();
    for (int j0 = 0; j0 < m; j0 += kWidePanel) {
        const int je = min(j0 + kWidePanel, m);
        for (int j = j0; j < je; ++j) {
            double best = -1.0;
            int bi = j;
            for (int r = j + tid; r < m; r += 256) {
                const double2 v = at(j, r);
                const double mag = v.x * v.x + v.y * v.y;
                if (mag > best) {
                    best = mag;
                    bi = r;
                }
            }
            red_mag[tid] = best;
            red_idx[tid] = bi;
            __syncthreads();
            for (int off = 128; off > 0; off >>= 1) {
                if (tid < off) {
                    const double om = red_mag[tid + off];
                    const int oi = red_idx[tid + off];
                    if (om > red_mag[tid] || (om == red_mag[tid] && oi < red_idx[tid])) {
                        red_mag[tid] = om;
                        red_idx[tid] = oi;
                    }
                }
                __syncthreads();
            }
            if (!(red_mag[0] > 0)) { // uniform: every thread reads the reduced value
                if (tid == 0)
                    singular = 1;
                break;
            }
            const int pr = red_idx[0];
            if (pr != j) {
                for (int c = tid; c < m; c += 256) {
                    const double2 t = at(c, j);
                    at(c, j) = at(c, pr);
                    at(c, pr) = t;
                }
                if (tid == 0) {
                    const int t = p[j];
                    p[j] = p[pr];
                    p[pr] = t;
                }
            }
            __syncthreads();
            const double2 d = at(j, j);
            const double inv = 1.0 / (d.x * d.x + d.y * d.y);
            for (int r = j + 1 + tid; r < m; r += 256) {
                const double2 x = at(j, r);
                at(j, r) = {(x.x * d.x + x.y * d.y) * inv, (x.y * d.x - x.x * d.y) * inv};
            }
            __syncthreads();
            const int rows = m - j - 1, cols = je - j - 1;
            for (int e = tid; e < rows * cols; e += 256) {
                const int c = j + 1 + e / rows, r = j + 1 + e % rows;
                const double2 l = at(j, r), u = at(c, j);
                double2 &t = at(c, r);
                t.x -= l.x * u.x - l.y * u.y;
                t.y -= l.x * u.y + l.y * u.x;
            }
            __syncthreads();
        }
        __syncthreads();
        if (singular)
            break;
        for (int c = je + tid; c < m; c += 256) // U12 = L11^{-1} A12
            for (int j = j0; j < je; ++j) {
                const double2 u = at(c, j);
                for (int i = j + 1; i < je; ++i) {
                    const double2 l = at(j, i);
                    at(c, i).x -= l.x * u.x - l.y * u.y;
                    at(c, i).y -= l.x * u.y + l.y * u.x;
                }
            }
        __syncthreads();
        rank_update(a, W, je, m, je, m, a + static_cast<std::size_t>(j0) * W, a + j0, je - j0);
        __syncthreads();
    }
    double2 *x = reinterpret_cast<double2 *>(inverses) + static_cast<std::size_t>(blk) * W * W; // x[c * W + r]
    const bool identity = singular != 0;
    for (std::size_t e = tid; e < static_cast<std::size_t>(W) * W; e += 256) {
        const int c = static_cast<int>(e / W), r = static_cast<int>(e % W);
        const bool inside = !identity && r < m && c < m;
        x[e] = {inside ? (p[r] == c ? 1.0 : 0.0) : (r == c ? 1.0 : 0.0), 0.0};
    }
    __syncthreads();
    if (identity)
        return;
    auto xt = [&](int c, int r) -> double2 & { return x[static_cast<std::size_t>(c) * W + r]; };
    for (int j0 = 0; j0 < m; j0 += kWidePanel) { // L X = P
        const int je = min(j0 + kWidePanel, m);
        for (int c = tid; c < m; c += 256)
            for (int j = j0; j < je; ++j) {
                const double2 y = xt(c, j);
                for (int i = j + 1; i < je; ++i) {
                    const double2 l = at(j, i);
                    xt(c, i).x -= l.x * y.x - l.y * y.y;
                    xt(c, i).y -= l.x * y.y + l.y * y.x;
                }
            }
        __syncthreads();
        rank_update(x, W, je, m, 0, m, a + static_cast<std::size_t>(j0) * W, x + j0, je - j0);
        __syncthreads();
    }
    const int last = ((m - 1) / kWidePanel) * kWidePanel;
    for (int j0 = last; j0 >= 0; j0 -= kWidePanel) { // U X = Y
        const int je = min(j0 + kWidePanel, m);
        for (int c = tid; c < m; c += 256)
            for (int j = je - 1; j >= j0; --j) {
                const double2 d = at(j, j), y = xt(c, j);
                const double inv = 1.0 / (d.x * d.x + d.y * d.y);
                const double2 v = {(y.x * d.x + y.y * d.y) * inv, (y.y * d.x - y.x * d.y) * inv};
                xt(c, j) = v;
                for (int i = j0; i < j; ++i) {
                    const double2 u = at(j, i);
                    xt(c, i).x -= u.x * v.x - u.y * v.y;
                    xt(c, i).y -= u.x * v.y + u.y * v.x;
                }
            }
        __syncthreads();
        rank_update(x, W, 0, j0, 0, m, a + static_cast<std::size_t>(j0) * W, x + j0, je - j0);
        __syncthreads();
    }
}

// out = M^{-1} v for width W: one workgroup of min(W, 256) threads per block, the
// block's v in LDS, threads stride over the rows (column-major inverse: coalesced
// per column).
__global__ __launch_bounds__(256) void jacobi_apply_wide(const double *inverses, std::uint32_t n, std::uint32_t width,
                                                         const double *v, double *out, const std::uint32_t *order) {
    __shared__ double2 sv[kMaxJacobiWidth];
    const std::uint32_t blk = blockIdx.x, W = width, r0 = blk * W;
    const int m = static_cast<int>(min(W, n - r0)), threads = static_cast<int>(blockDim.x);
    for (int i = threadIdx.x; i < m; i += threads) {
        const std::uint32_t row = order ? order[r0 + i] : r0 + i;
        sv[i] = double2{v[2 * row], v[2 * row + 1]};
    }
    __syncthreads();
    const double2 *f = reinterpret_cast<const double2 *>(inverses) + static_cast<std::size_t>(blk) * W * W;
    for (int r = threadIdx.x; r < m; r += threads) {
        double re = 0, im = 0;
        for (int c = 0; c < m; ++c) {
            const double2 b = f[static_cast<std::size_t>(c) * W + r];
            re += b.x * sv[c].x - b.y * sv[c].y;
            im += b.x * sv[c].y + b.y * sv[c].x;
        }
        const std::uint32_t row = order ? order[r0 + r] : r0 + r;
        out[2 * row] = re;
        out[2 * row + 1] = im;
    }
}

// One thread per entry of the gathered blocks: block b, column c, row r takes
// A[(W b + c) n + W b + r] (complex, widened to FP64).
template <class T>
__global__ __launch_bounds__(256) void jacobi_gather_dense_kernel(const T *A, std::uint32_t n, std::uint32_t width,
                                                                 double *blocks) {
    const std::size_t e = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const std::size_t W = width, blocks_count = (n + W - 1) / W;
    if (e >= blocks_count * W * W)
        return;
    const std::size_t b = e / (W * W), c = (e / W) % W, r = e % W;
    const std::size_t row = b * W + r, col = b * W + c;
    if (row >= n || col >= n)
        return;
    const T a = A[col * n + row];
    blocks[2 * e] = static_cast<double>(a.x);
    blocks[2 * e + 1] = static_cast<double>(a.y);
}

} // namespace

void jacobi_gather_dense(const void *A, bool fp32, std::uint32_t n, std::uint32_t width, double *blocks,
                         hipStream_t stream) {
    const std::size_t count = static_cast<std::size_t>((n + width - 1) / width) * width * width;
    const dim3 grid(static_cast<std::uint32_t>((count + 255) / 256));
    if (fp32)
        hipLaunchKernelGGL(jacobi_gather_dense_kernel<float2>, grid, dim3(256), 0, stream,
                           static_cast<const float2 *>(A), n, width, blocks);
    else
        hipLaunchKernelGGL(jacobi_gather_dense_kernel<double2>, grid, dim3(256), 0, stream,
                           static_cast<const double2 *>(A), n, width, blocks);
}

std::size_t jacobi_wide_doubles(std::uint32_t n, std::uint32_t width) {
    return static_cast<std::size_t>((n + width - 1) / width) * width * width * 2;
}

void jacobi_factor_wide(double *blocks, std::uint32_t n, std::uint32_t width, double *inverses, std::int32_t *pivots,
                        hipStream_t stream) {
    hipLaunchKernelGGL(jacobi_factor_wide, dim3((n + width - 1) / width), dim3(256), 0, stream, blocks, n, width,
                       inverses, pivots);
}

void jacobi_apply_wide(const double *inverses, std::uint32_t n, std::uint32_t width, const double *v, double *out,
                       hipStream_t stream, const std::uint32_t *order) {
    hipLaunchKernelGGL(jacobi_apply_wide, dim3((n + width - 1) / width), dim3(std::min(width, 256u)), 0, stream,
                       inverses, n, width, v, out, order);
}

std::size_t gemv_scratch_doubles(std::uint32_t n, std::uint32_t nvec) {
    const std::size_t chunks = (n + kGemvCols - 1) / kGemvCols;
    return 2 * chunks * n * std::max<std::uint32_t>(nvec, 1);
}

namespace {

// The partial products of the column chunks; returns the number of chunks.
template <int COLS>
std::uint32_t launch_gemv_one(const void *A, bool fp32, std::uint32_t n, const double *x, double *scratch,
                              hipStream_t stream, const int *skip, std::uint32_t rows) {
    const std::uint32_t chunks = (n + COLS - 1) / COLS;
    const dim3 grid((n + kGemvRows - 1) / kGemvRows, chunks);
    if (fp32 && rows == 4 && n % 4 == 0)
        hipLaunchKernelGGL((gemv_partial_rows<COLS, 4>), dim3((n + 4 * kGemvRows - 1) / (4 * kGemvRows), chunks),
                           dim3(kGemvRows * kGemvWaves), 0, stream, static_cast<const float2 *>(A), n, x, chunks,
                           scratch, skip);
    else if (fp32 && rows == 2 && n % 2 == 0)
        hipLaunchKernelGGL((gemv_partial_rows<COLS, 2>), dim3((n + 2 * kGemvRows - 1) / (2 * kGemvRows), chunks),
                           dim3(kGemvRows * kGemvWaves), 0, stream, static_cast<const float2 *>(A), n, x, chunks,
                           scratch, skip);
    else if (fp32)
        hipLaunchKernelGGL((gemv_partial<1, float2, COLS>), grid, dim3(kGemvRows * kGemvWaves), 0, stream,
                           static_cast<const float2 *>(A), n, x, chunks, scratch, skip);
    else
        hipLaunchKernelGGL((gemv_partial<1, double2, COLS>), grid, dim3(kGemvRows * kGemvWaves), 0, stream,
                           static_cast<const double2 *>(A), n, x, chunks, scratch, skip);
    return chunks;
}

// A product shape: the column chunk (512 / 1024 / 2048, low 16 bits) and, for an FP32
// matrix whose order they divide, the rows per lane (1, 2 or 4; bits 16 and up).
constexpr std::uint32_t gemv_shape(std::uint32_t cols, std::uint32_t rows) { return cols | rows << 16; }

std::uint32_t launch_gemv_cols(std::uint32_t shape, const void *A, bool fp32, std::uint32_t n, const double *x,
                               double *scratch, hipStream_t stream, const int *skip = nullptr) {
    const std::uint32_t cols = shape & 0xffffu, rows = std::max(shape >> 16, 1u);
    if (cols == 2048)
        return launch_gemv_one<2048>(A, fp32, n, x, scratch, stream, skip, rows);
    if (cols == 1024)
        return launch_gemv_one<1024>(A, fp32, n, x, scratch, stream, skip, rows);
    return launch_gemv_one<kGemvCols>(A, fp32, n, x, scratch, stream, skip, rows);
}

void launch_gemv_reduce(std::uint32_t n, std::uint32_t chunks, std::uint32_t nvec, const double *scratch, double *y,
                        hipStream_t stream, const int *skip) {
    const std::size_t count = static_cast<std::size_t>(n) * nvec;
    hipLaunchKernelGGL(gemv_reduce, dim3((count + 255) / 256), dim3(256), 0, stream, scratch, n, chunks, nvec, y, skip);
}

// Shape of the one-vector product per (n, precision), chosen by the autotuner among
// the column chunks 512 / 1024 / 2048 and, for an FP32 matrix whose order they
// divide, one, two or four rows per lane: three timed launches (after one warm launch)
// of each on the caller's stream and data; the product it leaves in y is the last
// candidate's, and the caller's own launch follows. The default chunk while the
// stream is being captured; HSBEM_GEMV_COLS = 512 / 1024 / 2048 pins the chunk (one
// row per lane), "COLSx2" / "COLSx4" the chunk and rows per lane (FP32 matrix whose
// order they divide).
std::uint32_t gemv_columns(const void *A, bool fp32, std::uint32_t n, const double *x, double *y, double *scratch,
                           hipStream_t stream) {
    std::optional<std::uint32_t> pinned;
    if (const char *pin = std::getenv("HSBEM_GEMV_COLS")) { // "COLS" or "COLSxROWS"
        char *end = nullptr;
        const unsigned long v = std::strtoul(pin, &end, 10);
        unsigned long rows = 1;
        if (end && *end == 'x')
            rows = std::strtoul(end + 1, nullptr, 10);
        const bool rows_ok = rows == 1 || ((rows == 2 || rows == 4) && fp32 && n % rows == 0);
        if ((v == 512 || v == 1024 || v == 2048) && rows_ok)
            pinned = gemv_shape(static_cast<std::uint32_t>(v), static_cast<std::uint32_t>(rows));
    }
    std::vector<std::uint32_t> shapes;
    for (const std::uint32_t rows : {1u, 2u, 4u})
        if (rows == 1 || (fp32 && n % rows == 0))
            for (const std::uint32_t cols : {512u, 1024u, 2048u})
                shapes.push_back(gemv_shape(cols, rows));
    const std::string key = "n=" + std::to_string(n) + (fp32 ? " fp32" : " fp64");
    return autotune::choose(
        "gemv_shape", key, shapes, kGemvCols, stream,
        [&](std::uint32_t shape) {
            launch_gemv_reduce(n, launch_gemv_cols(shape, A, fp32, n, x, scratch, stream), 1, scratch, y, stream, nullptr);
        },
        3, pinned);
}

} // namespace

std::uint32_t launch_gemv_partials(const void *A, bool fp32, std::uint32_t n, const double *x, double *y,
                                   std::uint32_t nvec, double *scratch, hipStream_t stream, const int *skip) {
    if (nvec == 1)
        return launch_gemv_cols(gemv_columns(A, fp32, n, x, y, scratch, stream), A, fp32, n, x, scratch, stream, skip);
    const std::uint32_t chunks = (n + kGemvCols - 1) / kGemvCols;
    const dim3 grid((n + kGemvRows - 1) / kGemvRows, chunks);
    switch (nvec) {
#define HS_GEMV_CASE(N)                                                                                          \
    case N:                                                                                                      \
        if (fp32)                                                                                                \
            hipLaunchKernelGGL((gemv_partial<N, float2>), grid, dim3(kGemvRows * kGemvWaves), 0, stream,         \
                               static_cast<const float2 *>(A), n, x, chunks, scratch, skip);                     \
        else                                                                                                     \
            hipLaunchKernelGGL((gemv_partial<N, double2>), grid, dim3(kGemvRows * kGemvWaves), 0, stream,        \
                               static_cast<const double2 *>(A), n, x, chunks, scratch, skip);                    \
        break;
        HS_GEMV_CASE(2)
        HS_GEMV_CASE(3)
        HS_GEMV_CASE(4)
        HS_GEMV_CASE(5)
        HS_GEMV_CASE(6)
        HS_GEMV_CASE(7)
        HS_GEMV_CASE(8)
#undef HS_GEMV_CASE
    default: throw std::invalid_argument("a matrix product takes 1 to 8 vectors at a time");
    }
    return chunks;
}

void launch_gemv(const void *A, bool fp32, std::uint32_t n, const double *x, double *y, std::uint32_t nvec,
                 double *scratch, hipStream_t stream) {
    for (std::uint32_t v0 = 0; v0 < nvec; v0 += kMaxVec) {
        const std::uint32_t nv = nvec == 1 ? 1 : std::min<std::uint32_t>(kMaxVec, nvec - v0);
        const std::size_t at = 2 * static_cast<std::size_t>(v0) * n;
        const std::uint32_t chunks = launch_gemv_partials(A, fp32, n, x + at, y + at, nv, scratch, stream);
        launch_gemv_reduce(n, chunks, nv, scratch, y + at, stream, nullptr);
    }
}

void launch_subtract_combination(const double *V, std::uint32_t n, std::uint32_t m, const double *h, double *w,
                                 hipStream_t stream) {
    hipLaunchKernelGGL(subtract_combination, dim3((n + 255) / 256), dim3(256), 0, stream, V, n, m, h, w);
}

void launch_norm2(const double *x, std::uint32_t n, const double *weight, double *out, double *scratch,
                  hipStream_t stream) {
    const std::uint32_t blocks = std::min<std::uint32_t>(1024, (n + 255) / 256);
    hipLaunchKernelGGL(norm_partial, dim3(blocks), dim3(256), 0, stream, x, n, weight, scratch);
    hipLaunchKernelGGL(norm_finish, dim3(1), dim3(64), 0, stream, scratch, blocks, out);
}

void launch_add(std::uint32_t n, const double *x, double *y, hipStream_t stream) {
    hipLaunchKernelGGL(add_kernel, dim3((2 * n + 255) / 256), dim3(256), 0, stream, n, x, y);
}

void launch_subtract_from(std::uint32_t n, const double *b, double *r, hipStream_t stream) {
    hipLaunchKernelGGL(subtract_from_kernel, dim3((2 * n + 255) / 256), dim3(256), 0, stream, n, b, r);
}

void launch_axpy(std::uint32_t n, const double *alpha, const double *x, double *y, hipStream_t stream) {
    hipLaunchKernelGGL(axpy_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, n, alpha, x, y);
}

void launch_scale(std::uint32_t n, double s, const double *x, double *y, hipStream_t stream) {
    hipLaunchKernelGGL(scale_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, n, s, x, y);
}

void launch_residual(const void *A, bool fp32, std::uint32_t n, const double *b, const double *x, std::uint32_t nvec,
                     double *residual, double *scratch, hipStream_t stream) {
    launch_gemv(A, fp32, n, x, residual, nvec, scratch, stream);
    const std::size_t count = 2 * static_cast<std::size_t>(n) * nvec;
    hipLaunchKernelGGL(subtract_vectors, dim3((count + 255) / 256), dim3(256), 0, stream, b, residual, count, residual);
}

std::size_t jacobi_factor_doubles(std::uint32_t n) {
    return static_cast<std::size_t>((n + kJacobi - 1) / kJacobi) * kJacobi * kJacobi * 2;
}

void jacobi_factor(const void *A, bool fp32, std::uint32_t n, double *inverses, hipStream_t stream) {
    const dim3 grid((n + kJacobi - 1) / kJacobi);
    if (fp32)
        hipLaunchKernelGGL(jacobi_factor<DenseBlocks<float2>>, grid, dim3(256), 0, stream,
                           DenseBlocks<float2>{static_cast<const float2 *>(A), n}, n,
                           inverses);
    else
        hipLaunchKernelGGL(jacobi_factor<DenseBlocks<double2>>, grid, dim3(256), 0, stream,
                           DenseBlocks<double2>{static_cast<const double2 *>(A), n}, n,
                           inverses);
}

void jacobi_factor_gathered(const double *blocks, std::uint32_t n, double *inverses, hipStream_t stream) {
    const dim3 grid((n + kJacobi - 1) / kJacobi);
    hipLaunchKernelGGL(jacobi_factor<GatheredBlocks>, grid, dim3(256), 0, stream, GatheredBlocks{blocks}, n, inverses);
}

void jacobi_apply(const double *inverses, std::uint32_t n, const double *v, double *out, hipStream_t stream,
                  const std::uint32_t *order) {
    hipLaunchKernelGGL(jacobi_apply, dim3((n + kJacobi - 1) / kJacobi), dim3(64), 0, stream, inverses, n, v, out,
                       order);
}

} // namespace hsbem::dev
