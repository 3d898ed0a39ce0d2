// Dense complex FP64 LU with partial pivoting and its solves, gfx950.
//
// Replaces cusolverDnCgetrf/Cgetrs of the reference dense path
// (cuda_solver.cu:1485-1513):
//   lu_factor  right-looking, 64-column panels. One launch factors the next panel on
//              a few workgroups (rows in registers, one exchange through memory per
//              column) while the others apply the previous panel to the rest of the
//              matrix on the FP64 matrix cores.
//   lu_solve   64-row blocks, one launch per block and sweep.
#include "../solver.hpp"
#include "device.hpp"

#include <algorithm>
#include <array>
#include <chrono>
#include <condition_variable>
#include <mutex>
#include <stdexcept>
#include <string>

namespace hsbem::dev {
namespace {

using u64 = unsigned long long;

constexpr int kBlock = 64;         // panel columns
constexpr int kStepThreads = 512;
constexpr int kColumns = 8;        // columns a panel wavefront holds
constexpr int kPart = 32;          // columns of L staged at a time in an update
constexpr int kPanelRows = 128;    // rows per panel workgroup: two per lane
// The workgroups of a panel wait for each other, so all of them have to be resident at once:
// each factorization reserves them (PanelGroups below) and takes panels of more rows than it
// got on one workgroup. Most at a time: the whole of a matrix of 15,360 rows, on half of the
// 256 compute units.
constexpr std::uint32_t kMaxPanelGroups = kLuPanelGroups;
constexpr std::uint32_t kRing = 4;                      // exchange slots per workgroup
constexpr std::uint32_t kSlotWords = 4 + 2 * kBlock;     // size, position, 64 complex entries, the pivot's inverse
static_assert(kLuWorkDoubles == kRing * kMaxPanelGroups * kSlotWords + kBlock);
constexpr u64 kEmpty = ~0ull;                           // an exchange word nobody has written
constexpr u64 kWaitTicks = 1000000000ull;               // 10 s of the 100 MHz clock: only other processes can cause it
constexpr int kWaitFailed = -1;                         // info: a panel workgroup waited that long


// ---- exchange between the panel's workgroups ----
// Every word is written once per use and read until it is no longer kEmpty, so no flag
// or fence orders the words of a message among themselves.

__device__ __forceinline__ u64 word_of(double v) {
    const u64 b = __builtin_bit_cast(u64, v);
    return b == kEmpty ? 0x7ff8000000000000ull : b; // the one NaN that means "empty" becomes another NaN
}

__device__ __forceinline__ void put_word(u64 *w, u64 v) {
    __hip_atomic_store(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The word once it is written; 0 and *late after kWaitTicks.
__device__ __forceinline__ u64 wait_word(const u64 *w, int *late) {
    u64 b = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (b == kEmpty) {
        const u64 start = wall_clock64();
        do {
            b = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (b == kEmpty && wall_clock64() - start > kWaitTicks) {
                *late = 1;
                b = 0;
            }
        } while (b == kEmpty);
    }
    return b;
}

// The status word: 0, the first zero pivot's column + 1, or kWaitFailed, which no pivot replaces.
// Workgroups of one launch read and write it at the same time, on several dies.
__device__ __forceinline__ bool gave_up(const int *info) {
    return __hip_atomic_load(info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < 0;
}
__device__ __forceinline__ void report_wait_failed(int *info) {
    __hip_atomic_fetch_min(info, kWaitFailed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void report_zero_pivot(int *info, int column) {
    int expected = 0;
    __hip_atomic_compare_exchange_strong(info, &expected, column, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
}

// Every outstanding access of this wavefront has completed (stores acknowledged, loads in registers).
__device__ __forceinline__ void drain_memory() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// A pivot candidate: the largest squared modulus (-1: not a number, -2: no row), ties to the
// lowest position.
struct Candidate {
    double size;
    std::uint32_t at;
};

template <int kControl, int kRows> __device__ __forceinline__ std::uint32_t dpp_max(std::uint32_t v) {
    return max(v, static_cast<std::uint32_t>(
                      __builtin_amdgcn_update_dpp(0, static_cast<int>(v), kControl, kRows, 0xf, false)));
}

__device__ __forceinline__ std::uint32_t wave_max(std::uint32_t v) {
    v = dpp_max<0xB1, 0xf>(v);  // lanes 1 apart
    v = dpp_max<0x4E, 0xf>(v);  // 2 apart
    v = dpp_max<0x141, 0xf>(v); // mirrored halves of a row of 16
    v = dpp_max<0x140, 0xf>(v); // mirrored rows
    v = dpp_max<0x142, 0xa>(v); // row 0 into 1, 2 into 3
    v = dpp_max<0x143, 0xc>(v); // rows 0-1 into 2-3: lane 63 has all
    return __builtin_amdgcn_readlane(static_cast<int>(v), 63);
}

// The lane of the wavefront's best candidate. Sizes compare as integers, the upper halves
// first: those of two lanes are rarely equal.
__device__ __forceinline__ int wave_best(double size, std::uint32_t at) {
    const u64 b = __builtin_bit_cast(u64, size);
    const auto lo = static_cast<std::uint32_t>(b);
    const std::uint32_t key = size >= 0 ? static_cast<std::uint32_t>(b >> 32) + 2 : size >= -1 ? 1u : 0u;
    const std::uint32_t top = wave_max(key);
    u64 who = __ballot(key == top);
    if (who & (who - 1)) {
        const std::uint32_t low = wave_max(key == top ? lo : 0);
        who = __ballot(key == top && lo == low);
        std::uint32_t first = ~0u;
        for (u64 ties = who; ties; ties &= ties - 1)
            first = min(first, static_cast<std::uint32_t>(
                                   __builtin_amdgcn_readlane(static_cast<int>(at), __builtin_ctzll(ties))));
        who = __ballot(key == top && lo == low && at == first);
    }
    return __builtin_ctzll(who);
}

struct PanelShared {
    double2 row[kBlock];     // the chosen row: each wavefront's entries, rotated as its registers are
    double2 inverse;         // of the pivot
    double2 factor[kPanelRows];
    std::uint32_t at;        // this group's candidate
    std::uint32_t other_at, other_group, singular, late, quit;
    std::uint32_t pivot[kBlock];
};

struct UpdateShared {
    double2 L[kPart][kBlock + 1]; // L[k][q] = A[r0 + q][k0 + kc + k] (padded row: no bank conflicts across k)
    double2 U[kPart][kBlock + 1]; // U[k][q] = A[k0 + kc + k][c0 + q]
};

union StepShared {
    PanelShared panel;
    UpdateShared update;
};

// What the interchanges of a panel come to: block position i receives row inside[i], and the
// row that was at block position i goes to position out[i] (rows outside the block move only
// into it, so those two tables are all of it).
struct PanelMoves {
    std::uint32_t inside[kBlock], out[kBlock];
};

struct PanelArgs {
    std::uint32_t k0, nb, groups; // groups = 0: no panel in this launch
    std::int32_t *piv;
    int *info;
    u64 *exchange; // [ring][group][kSlotWords]
    PanelMoves *moves;
};

// 1 / a = conj(a) / size, size = |a|^2: reciprocal and two Newton steps, the division itself where
// the reciprocal would leave the normal range.
__device__ __forceinline__ double2 inverse_of(double2 a, double size) {
    double r = __builtin_amdgcn_rcp(size);
    r = fma(fma(-size, r, 1.0), r, r);
    r = fma(fma(-size, r, 1.0), r, r);
    if (size > 0 && !(size > 1e-280 && size < 1e280))
        return {a.x / size, -a.y / size};
    return size > 0 ? double2{a.x * r, -a.y * r} : double2{0.0, 0.0};
}

__device__ __forceinline__ double2 minus_product(double2 b, double2 l, double2 q) { // b - l q
    return {fma(l.y, q.y, fma(-l.x, q.x, b.x)), fma(-l.y, q.x, fma(-l.x, q.y, b.y))};
}

// Factors the panel of columns [k0, k0 + nb) over rows [k0, n): group g's 8 wavefronts
// hold 128 rows in registers, wavefront w the columns [8 w, 8 w + 8) of all of them, two
// rows per lane. Interchanges are positions: a row keeps its lane and knows where it
// belongs, and everything is written there at the end. Per column: the wavefront that
// holds it finds the group's candidate (DPP maximum) and publishes it, every wavefront
// publishes its part of that row, all groups read all candidates, pick the same winner
// and read its row; rows that are not pivots yet take l = a / pivot and subtract l * row.
// Registers rotate by one in that update (v[i] = v[i + 1] - l u[i + 1], and l or column 0's
// update into v[7]), so that the column to search is always v[0] and no register is
// indexed; after 8 columns each is back in its place. The next column is updated,
// searched and published before the others, whose update then hides in the exchange.
// Bound by latency, not by work: about 3 us per column with an exchange (two dependent reads
// through the memory that every XCD sees) and 1.3 us without; leaves of 4 columns on one
// workgroup took 9 us (n = 4099 in all: 20.1 against 52.6 ms, n = 10373: 110 against 252 ms,
// where the launches that factor a panel beside the update of the one before take 92.6 ms for
// 2.98 TFLOP, 32 TFLOP/s).
// Ring slots are emptied by their owner one column after use: by then every group has
// published its next candidate, which it does after reading this one, and a slot is
// written again three columns later.
__device__ __forceinline__ void factor_panel(double2 *A, std::uint32_t n, const PanelArgs &P, std::uint32_t g,
                                             PanelShared &S) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const std::uint32_t k0 = P.k0, nb = P.nb, groups = P.groups, first = k0 + g * kPanelRows;
    std::uint32_t pos[2];
    bool open[2];
    double2 v[2][kColumns];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const std::uint32_t r = first + 64 * h + lane;
        open[h] = r < n;
        pos[h] = open[h] ? r : ~0u;
        const double2 *mine = A + static_cast<std::size_t>(k0) * n + min(r, n - 1);
#pragma unroll
        for (int c = 0; c < kColumns; ++c) // beyond n and nb: a valid entry that is never stored
            v[h][c] = mine[static_cast<std::size_t>(min(wave * kColumns + c, static_cast<int>(nb) - 1)) * n];
    }
    if (threadIdx.x == 0) {
        S.late = 0;
        S.quit = gave_up(P.info);
    }
    drain_memory(); // the rows are in registers before anything of this group is published
    __syncthreads();
    if (S.quit) // a group gave up waiting: nothing is valid any more. (One read for all wavefronts: the word
        return; // may change between two, and those that went on would miss what the others publish.)
    auto ring_of = [&](std::uint32_t j) {
        return P.exchange + static_cast<std::size_t>((k0 + j) & (kRing - 1)) * kMaxPanelGroups * kSlotWords;
    };
    double2 inverse = {0.0, 0.0}; // of this lane's candidate, while this wavefront holds the column
    // The group's candidate in column j, v[.][0] of this wavefront.
    auto search = [&](std::uint32_t j) {
        double m[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            m[h] = v[h][0].x * v[h][0].x + v[h][0].y * v[h][0].y;
            m[h] = !open[h] ? -2.0 : m[h] >= 0 ? m[h] : -1.0; // not a number: only if nothing else is left
        }
        const bool second = m[1] > m[0] || (m[1] == m[0] && pos[1] < pos[0]);
        const double mine = second ? m[1] : m[0];
        const std::uint32_t where = second ? pos[1] : pos[0];
        const int best = wave_best(mine, where);
        if (lane == best) {
            S.at = where;
            S.singular = !(mine > 0);
            if (groups > 1) {
                u64 *slot = ring_of(j) + static_cast<std::size_t>(g) * kSlotWords;
                put_word(slot, word_of(mine));
                put_word(slot + 1, where);
            }
        }
        inverse = inverse_of(second ? v[1][0] : v[0][0], mine);
    };
    if (wave == 0)
        search(0);
    std::uint32_t singular = 0;
    for (std::uint32_t j = 0; j < nb; ++j) {
        const int phase = static_cast<int>(j) / kColumns, c = static_cast<int>(j) % kColumns;
        const bool active = wave == phase, works = wave >= phase;
        u64 *ring = ring_of(j);
        __syncthreads();
        std::uint32_t at = S.at;
        if (works) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (open[h] && pos[h] == at) { // the candidate row's part here
                    if (active)
                        S.inverse = inverse;
#pragma unroll
                    for (int i = 0; i < kColumns; ++i)
                        S.row[wave * kColumns + i] = v[h][i];
                }
            if (active && lane < c) // factored columns have rotated to the end: no update there
                S.row[wave * kColumns + kColumns - 1 - lane] = double2{0.0, 0.0};
        }
        if (groups > 1) {
            double *part = reinterpret_cast<double *>(S.row + wave * kColumns);
            const int word = lane < 2 * kColumns ? 2 + wave * 2 * kColumns + lane : 2 + 2 * kBlock + (lane & 1);
            const bool moves = works && (lane < 2 * kColumns || (active && lane < 2 * kColumns + 2));
            double *shared = lane < 2 * kColumns ? part + lane : reinterpret_cast<double *>(&S.inverse) + (lane & 1);
            if (moves)
                put_word(ring + static_cast<std::size_t>(g) * kSlotWords + word, word_of(*shared));
            int late = S.late;
            if (wave == ((phase + 1) & 7)) { // reads every group's candidate, two slots per lane
                double size = -3.0;
                std::uint32_t where = ~0u;
                int group = lane;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const std::uint32_t o = 64 * h + lane;
                    if (o < groups && !late) {
                        const double s = __builtin_bit_cast(double, wait_word(ring + o * kSlotWords, &late));
                        const auto w = static_cast<std::uint32_t>(wait_word(ring + o * kSlotWords + 1, &late));
                        if (s > size || (s == size && w < where)) {
                            size = s;
                            where = w;
                            group = static_cast<int>(o);
                        }
                    }
                }
                const int best = wave_best(size, where);
                if (lane == best) {
                    S.other_at = where;
                    S.other_group = static_cast<std::uint32_t>(group);
                    S.singular = !(size > 0);
                }
            }
            // a matrix that needs few interchanges has its pivot in group 0: its row is read meanwhile
            u64 entry = 0;
            if (moves && !late)
                entry = wait_word(ring + word, &late);
            if (late)
                S.late = 1;
            __syncthreads();
            at = S.other_at;
            late = S.late;
            if (late) { // nothing valid will come: keep this group's positions in range; see lu_rows
                at = k0 + j;
                if (threadIdx.x == 0)
                    report_wait_failed(P.info);
            }
            if (moves) {
                const std::uint32_t winner = S.other_group;
                if (winner != 0 && !late)
                    entry = wait_word(ring + static_cast<std::size_t>(winner) * kSlotWords + word, &late);
                *shared = __builtin_bit_cast(double, entry);
                if (late)
                    S.late = 1;
            }
            drain_memory(); // the slots emptied in the column before have reached memory before the next publication
            u64 *old = ring_of(j - 1) + static_cast<std::size_t>(g) * kSlotWords;
            if (lane < 2 * kColumns)
                put_word(old + 2 + wave * 2 * kColumns + lane, kEmpty);
            else if (wave == 0 && lane < 2 * kColumns + 4)
                put_word(old + (lane & 2 ? 2 * kBlock : 0) + (lane & 3), kEmpty);
        }
        if (active) {
            const double2 inv = S.inverse;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const double2 a = v[h][0];
                const bool below = open[h] && pos[h] != at;
                S.factor[64 * h + lane] =
                    below ? double2{a.x * inv.x - a.y * inv.y, a.x * inv.y + a.y * inv.x} : double2{0.0, 0.0};
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (open[h] && pos[h] == at) {
                open[h] = false;
                pos[h] = k0 + j;
            } else if (pos[h] == k0 + j) {
                pos[h] = at;
            }
        }
        const bool zero = S.singular != 0; // the next search may write it after the barrier
        if (threadIdx.x == 0)
            S.pivot[j] = at;
        __syncthreads();
        if (zero && singular == 0)
            singular = k0 + j + 1;
        if (works) {
            const double2 *u = S.row + wave * kColumns;
            double2 l[2], last[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                l[h] = S.factor[64 * h + lane];
                const double2 a = v[h][0];
                last[h] = !active ? minus_product(a, l[h], u[0]) : open[h] ? l[h] : a;
                v[h][0] = minus_product(v[h][1], l[h], u[1]);
            }
            if (j + 1 < nb && wave == static_cast<int>(j + 1) / kColumns)
                search(j + 1);
#pragma unroll
            for (int i = 1; i + 1 < kColumns; ++i) {
                const double2 q = u[i + 1];
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    v[h][i] = minus_product(v[h][i + 1], l[h], q);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
                v[h][kColumns - 1] = last[h];
        }
    }
    __syncthreads();
    if (threadIdx.x == 0 && S.late) // also where the last column's row did not come
        report_wait_failed(P.info);
    if (g == 0 && threadIdx.x < nb)
        P.piv[k0 + threadIdx.x] = static_cast<std::int32_t>(S.pivot[threadIdx.x]);
    if (g == 0 && threadIdx.x == 0 && singular)
        report_zero_pivot(P.info, static_cast<int>(singular));
    // v[i] is the wavefront's column (i + its active steps) mod 8; every group has read its rows long ago
    const int steps = max(0, min(static_cast<int>(nb) - wave * kColumns, kColumns));
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const std::uint32_t r = first + 64 * h + lane;
        if (pos[h] == ~0u)
            continue;
        double2 *mine = A + static_cast<std::size_t>(k0) * n + pos[h];
#pragma unroll
        for (int i = 0; i < kColumns; ++i) {
            const std::uint32_t q = wave * kColumns + ((i + steps) & (kColumns - 1));
            if (q < nb)
                mine[static_cast<std::size_t>(q) * n] = v[h][i];
        }
        if (wave == 0 && pos[h] < k0 + nb)
            P.moves->inside[pos[h] - k0] = r;
        if (wave == 0 && r < k0 + nb)
            P.moves->out[r - k0] = pos[h];
    }
}

// C -= L U on the 64 x 64 tile at (r0, c0) of rows below r_end and columns below c_end, with
// L = A[rows][k0 .. k0 + nb) and U = A[k0 .. k0 + nb)[columns], nb <= 64 (staged through LDS
// in chunks of 32, the accumulators carried across the chunks), on the FP64 matrix cores: each
// wavefront 32 rows x 16 columns as two blocks of 16 x 16. The product is formed transposed,
// D = U^T L^T (v_mfma_f64_16x16x4f64: A[i][k] from lane i + 16 k, B[k][j] from lane j + 16 k,
// D[i][j] in lane j + 16 (i mod 4), register i / 4), so D's index j runs over rows and each
// 16-lane group writes 16 consecutive rows of one column. A complex MAC is four real MFMAs:
// Re += Ur Lr - Ui Li, Im += Ui Lr + Ur Li. Each chunk's K is padded with zeros to a multiple
// of 4.
typedef double lu_v4d __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void update_tile(double2 *A, std::uint32_t n, std::uint32_t k0, std::uint32_t nb,
                                            std::uint32_t r0, std::uint32_t r_end, std::uint32_t c0,
                                            std::uint32_t c_end, UpdateShared &S) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, kq = lane >> 4;
    const int rh = wave & 1, cq = wave >> 1;
    // this lane's old C values, loaded first so their latency hides behind the staging and the MFMAs
    double2 cold[2][4];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const std::uint32_t r = r0 + rh * 32 + a * 16 + i, c = c0 + cq * 16 + 4 * v + kq;
            cold[a][v] = A[static_cast<std::size_t>(min(c, n - 1)) * n + min(r, n - 1)];
        }
    lu_v4d accr[2], acci[2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
        accr[a] = acci[a] = lu_v4d{0.0, 0.0, 0.0, 0.0};
    for (std::uint32_t kc = 0; kc < nb; kc += kPart) {
        const std::uint32_t kn = min(static_cast<std::uint32_t>(kPart), nb - kc), kpad = (kn + 3) & ~3u;
        if (kc)
            __syncthreads(); // the previous chunk's reads are done
        for (std::uint32_t e = threadIdx.x; e < kpad * 64; e += kStepThreads) {
            const std::uint32_t kk = e / 64, q = e % 64, r = r0 + q, c = c0 + q;
            const std::size_t k = static_cast<std::size_t>(k0) + kc + kk;
            S.L[kk][q] = kk < kn && r < r_end ? A[k * n + r] : double2{0.0, 0.0};
            S.U[kk][q] = kk < kn && c < c_end ? A[static_cast<std::size_t>(c) * n + k] : double2{0.0, 0.0};
        }
        __syncthreads();
        for (std::uint32_t ks = 0; ks < kpad / 4; ++ks) {
            const std::uint32_t kk = 4 * ks + kq;
            const double2 l0 = S.L[kk][rh * 32 + i], l1 = S.L[kk][rh * 32 + 16 + i], u = S.U[kk][cq * 16 + i];
            // two passes over the four independent accumulators: no MFMA waits on the one before it
            accr[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x, l0.x, accr[0], 0, 0, 0);
            acci[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.y, l0.x, acci[0], 0, 0, 0);
            accr[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x, l1.x, accr[1], 0, 0, 0);
            acci[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.y, l1.x, acci[1], 0, 0, 0);
            accr[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(-u.y, l0.y, accr[0], 0, 0, 0);
            acci[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x, l0.y, acci[0], 0, 0, 0);
            accr[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(-u.y, l1.y, accr[1], 0, 0, 0);
            acci[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x, l1.y, acci[1], 0, 0, 0);
        }
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const std::uint32_t r = r0 + rh * 32 + a * 16 + i, c = c0 + cq * 16 + 4 * v + kq;
            if (r < r_end && c < c_end)
                A[static_cast<std::size_t>(c) * n + r] =
                    double2{cold[a][v].x - accr[a][v], cold[a][v].y - acci[a][v]};
        }
}


struct UpdateArgs {
    std::uint32_t k0, nb, r_begin, r_end, c_begin, c_end; // empty when r_begin == r_end or c_begin == c_end
};

// One step of the factorization: the first `groups` workgroups factor a panel whose columns
// are up to date, the others apply an earlier panel to columns that the panel does not touch,
// one 64 x 64 tile each. Panel workgroups come first in the grid, so they are resident before
// the tiles fill the chip.
__global__ __launch_bounds__(kStepThreads, 4) void lu_step(double *A, std::uint32_t n, PanelArgs P, UpdateArgs U) {
    __shared__ StepShared S;
    double2 *A2 = reinterpret_cast<double2 *>(A);
    if (blockIdx.x < P.groups) {
        factor_panel(A2, n, P, blockIdx.x, S.panel);
        return;
    }
    const std::uint32_t t = blockIdx.x - P.groups, rows = (U.r_end - U.r_begin + kBlock - 1) / kBlock;
    update_tile(A2, n, U.k0, U.nb, U.r_begin + t % rows * kBlock, U.r_end, U.c_begin + t / rows * kBlock, U.c_end,
                S.update);
}

// The same product on 32 x 32 tiles (a quarter per wavefront, K <= 64 staged at once) for the
// few columns of the next panel, where 64 x 64 tiles leave most of the chip idle (6 against
// 22 us at n = 4099).
constexpr int kSmall = 32;
__global__ __launch_bounds__(256) void lu_update_small(double *A, std::uint32_t n, UpdateArgs U) {
    __shared__ double2 Ls[kBlock][kSmall + 1], Us[kBlock][kSmall + 1];
    double2 *A2 = reinterpret_cast<double2 *>(A);
    const std::uint32_t r0 = U.r_begin + blockIdx.x * kSmall, c0 = U.c_begin + blockIdx.y * kSmall;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i = lane & 15, kq = lane >> 4;
    const std::uint32_t r = r0 + 16 * (wave & 1) + i, cw = 16 * (wave >> 1);
    double2 cold[4];
#pragma unroll
    for (int v = 0; v < 4; ++v)
        cold[v] = A2[static_cast<std::size_t>(min(c0 + cw + 4 * v + kq, n - 1)) * n + min(r, n - 1)];
#pragma unroll
    for (int m = 0; m < kBlock * kSmall / 256; ++m) { // consecutive threads: 32 rows of L, 64 of U
        const std::uint32_t e = tid + 256 * m, k = e / kSmall, q = e % kSmall;
        const double2 l = A2[static_cast<std::size_t>(U.k0 + min(k, U.nb - 1)) * n + min(r0 + q, n - 1)];
        Ls[k][q] = k < U.nb ? l : double2{0.0, 0.0};
        const std::uint32_t ku = e % kBlock, qu = e / kBlock;
        const double2 u = A2[static_cast<std::size_t>(min(c0 + qu, n - 1)) * n + U.k0 + min(ku, U.nb - 1)];
        Us[ku][qu] = ku < U.nb ? u : double2{0.0, 0.0};
    }
    __syncthreads();
    lu_v4d re = {0.0, 0.0, 0.0, 0.0}, im = re, re2 = re, im2 = re; // two chains of each
#pragma unroll
    for (int s = 0; s < kBlock / 4; ++s) {
        const double2 l = Ls[4 * s + kq][16 * (wave & 1) + i], u = Us[4 * s + kq][cw + i];
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x, l.x, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(u.y, l.x, im, 0, 0, 0);
        re2 = __builtin_amdgcn_mfma_f64_16x16x4f64(-u.y, l.y, re2, 0, 0, 0);
        im2 = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x, l.y, im2, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const std::uint32_t c = c0 + cw + 4 * v + kq;
        if (r < U.r_end && c < U.c_end)
            A2[static_cast<std::size_t>(c) * n + r] = double2{cold[v].x - (re[v] + re2[v]), cold[v].y - (im[v] + im2[v])};
    }
}

__global__ void set_status(int *info, int value) { *info = value; }

__global__ void clear_exchange(u64 *exchange, std::uint32_t words) {
    const std::uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < words)
        exchange[i] = kEmpty;
}

// The net effect of the interchanges (j0 + i <-> p_i), i = 0 .. nb - 1 in order, for one
// wavefront, lane i holding p (its own position when i >= nb). Afterwards position j0 + i
// holds what was at `inside`, and where `owner`, position p holds what was at `outside`.
struct Interchange {
    std::uint32_t inside, outside;
    bool owner;
    u64 moved; // interchanges that do something
};

__device__ __forceinline__ Interchange net_interchange(std::uint32_t p, std::uint32_t j0, std::uint32_t nb) {
    const int lane = threadIdx.x & 63;
    Interchange out{j0 + lane, p, false, __ballot(p != j0 + lane)};
    int slot = lane; // the first lane with the same outside position
    for (u64 m = __ballot(p >= j0 + nb); m; m &= m - 1) {
        const int i = __builtin_ctzll(m);
        if (static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(p), i)) == p && i < slot)
            slot = i;
    }
    out.owner = p >= j0 + nb && slot == lane && static_cast<std::uint32_t>(lane) < nb;
    int inside = static_cast<int>(out.inside), outside = static_cast<int>(p);
    for (u64 m = out.moved; m; m &= m - 1) {
        const int i = __builtin_ctzll(m);
        const std::uint32_t pi = __builtin_amdgcn_readlane(static_cast<int>(p), i);
        const int a = __builtin_amdgcn_readlane(inside, i);
        if (pi < j0 + nb) {
            const int t = static_cast<int>(pi - j0), b = __builtin_amdgcn_readlane(inside, t);
            inside = lane == i ? b : lane == t ? a : inside;
        } else {
            const int o = __builtin_amdgcn_readlane(slot, i), b = __builtin_amdgcn_readlane(outside, o);
            inside = lane == i ? b : inside;
            outside = lane == o ? a : outside;
        }
    }
    out.inside = static_cast<std::uint32_t>(inside);
    out.outside = static_cast<std::uint32_t>(outside);
    return out;
}

// The panel's interchanges applied to 64 other columns per workgroup, and in the columns
// right of it U12 = L11^{-1} A12: rows staged through LDS, L11 as 4 x 4 blocks of 16 whose
// diagonal blocks are inverted (unit lower triangles, one thread per column) so that the
// whole solve is products on the matrix cores, each wavefront 16 columns that stay in
// registers: the D layout of one product is the B layout of the next. 25 us at n = 4099,
// bound by the latency of its dependent loads and of the chain of products.
// Nothing is done once a panel has given up waiting: its groups then disagree about the positions
// of their rows, so some of `moves` may never have been written. (No other kernel takes an index
// from what a panel wrote.)
__global__ __launch_bounds__(256) void lu_rows(double *A, std::uint32_t n, std::uint32_t k0, std::uint32_t nb,
                                               const PanelMoves *moves, const int *info) {
    __shared__ double2 X[kBlock][kBlock + 1];  // X[q][i] = row k0 + i of column c0 + q
    __shared__ double2 L[kBlock][kBlock + 1];  // L[c][r] = A[k0 + r][k0 + c]
    __shared__ double2 inverse[4][16][17];     // [block][c][r]
    __shared__ std::uint32_t inside[kBlock], out[kBlock], moved;
    double2 *A2 = reinterpret_cast<double2 *>(A);
    if (gave_up(info))
        return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const std::uint32_t left = k0 / kBlock;
    const bool right = blockIdx.x >= left;
    const std::uint32_t c0 = right ? k0 + nb + (blockIdx.x - left) * kBlock : blockIdx.x * kBlock;
    const std::uint32_t cols = right ? min(static_cast<std::uint32_t>(kBlock), n - c0) : kBlock;
    if (wave == 0) {
        const bool in = static_cast<std::uint32_t>(lane) < nb;
        inside[lane] = in ? moves->inside[lane] : k0;
        out[lane] = in ? moves->out[lane] : k0;
        const u64 m = __ballot(in && (inside[lane] != k0 + lane || out[lane] != k0 + lane));
        if (lane == 0)
            moved = m != 0;
    }
    if (right)
        for (std::uint32_t e = tid; e < kBlock * kBlock; e += 256) {
            const std::uint32_t r = e % kBlock, c = e / kBlock;
            L[c][r] = c < r ? A2[static_cast<std::size_t>(k0 + c) * n + k0 + r] : double2{0.0, 0.0};
        }
    __syncthreads();
    if (!right && !moved)
        return;
    double2 old[kBlock * kBlock / 256]; // block rows that leave the block
#pragma unroll
    for (int m = 0; m < kBlock * kBlock / 256; ++m) {
        const std::uint32_t e = tid + 256 * m, q = e / kBlock, i = e % kBlock;
        const double2 *column = A2 + static_cast<std::size_t>(c0 + min(q, cols - 1)) * n;
        X[q][i] = column[inside[i]];
        old[m] = out[i] >= k0 + nb ? column[k0 + i] : double2{0.0, 0.0};
    }
    if (right && tid < kBlock) { // thread (block, c): column c of the block's inverse
        const int b = tid / 16, c = tid % 16;
        double2 y[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            double2 s = {r == c ? 1.0 : 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < r; ++k) {
                const double2 l = L[16 * b + k][16 * b + r];
                s.x -= l.x * y[k].x - l.y * y[k].y;
                s.y -= l.x * y[k].y + l.y * y[k].x;
            }
            y[r] = s;
            inverse[b][c][r] = s;
        }
    }
    drain_memory(); // every old entry has been read
    __syncthreads();
#pragma unroll
    for (int m = 0; m < kBlock * kBlock / 256; ++m) {
        const std::uint32_t e = tid + 256 * m, q = e / kBlock, i = e % kBlock;
        if (q < cols && out[i] >= k0 + nb)
            A2[static_cast<std::size_t>(c0 + q) * n + out[i]] = old[m];
    }
    if (right) { // nb == 64 whenever columns follow the panel
        const int q = 16 * wave + (lane & 15), kq = lane >> 4, i = lane & 15;
        lu_v4d xr[4], xi[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            lu_v4d ar, ai;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const double2 x = X[q][16 * b + 4 * v + kq];
                ar[v] = x.x;
                ai[v] = x.y;
            }
#pragma unroll
            for (int c = 0; c < b; ++c)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const double2 l = L[16 * c + 4 * s + kq][16 * b + i];
                    ar = __builtin_amdgcn_mfma_f64_16x16x4f64(-l.x, xr[c][s], ar, 0, 0, 0);
                    ai = __builtin_amdgcn_mfma_f64_16x16x4f64(-l.x, xi[c][s], ai, 0, 0, 0);
                    ar = __builtin_amdgcn_mfma_f64_16x16x4f64(l.y, xi[c][s], ar, 0, 0, 0);
                    ai = __builtin_amdgcn_mfma_f64_16x16x4f64(-l.y, xr[c][s], ai, 0, 0, 0);
                }
            xr[b] = xi[b] = lu_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const double2 l = inverse[b][4 * s + kq][i];
                xr[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(l.x, ar[s], xr[b], 0, 0, 0);
                xi[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(l.x, ai[s], xi[b], 0, 0, 0);
                xr[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(-l.y, ai[s], xr[b], 0, 0, 0);
                xi[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(l.y, ar[s], xi[b], 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v)
                X[q][16 * b + 4 * v + kq] = double2{xr[b][v], xi[b][v]};
        }
    }
    __syncthreads();
    for (std::uint32_t e = tid; e < cols * kBlock; e += 256) {
        const std::uint32_t q = e / kBlock, r = e % kBlock;
        if (r < nb)
            A2[static_cast<std::size_t>(c0 + q) * n + k0 + r] = X[q][r];
    }
}

// ---- panels of more than kMaxPanelGroups * 128 rows: 32 columns in leaves of 4 ----

constexpr int kPanel = 32;
constexpr int kPanelThreads = 1024;

// Factor the leaf columns [j0, j0 + w) of the panel [k0, pe) over rows [j0, n).
// Per column j, three barriers: (1) pivot search (largest squared modulus, ties to
// the lowest row) reduced per wavefront into LDS; (2) every thread finishes the
// reduction itself, a few threads stage the pivot row p's leaf entries in LDS and
// one records the pivot; (3) one pass over the rows r > j writes
// l = a[r][j] / a[p][j] and a[r][c] - l u[c] for the leaf columns c > j, reading
// row j in place of row p (the interchange folded in), while the thread of row p
// also writes the pivot row into row j, and the other panel columns (the leaf's
// factored columns before j included) swap rows j and p. One workgroup; pivot rows
// are recorded as absolute indices.
constexpr int kLeaf = 4;
__global__ __launch_bounds__(kPanelThreads) void lu_leaf(double *A, std::uint32_t n, std::uint32_t k0, std::uint32_t j0,
                                                        std::uint32_t w, std::uint32_t pe, std::int32_t *piv, int *info) {
    __shared__ double best[kPanelThreads / 64];
    __shared__ std::uint32_t where[kPanelThreads / 64];
    __shared__ double2 u[kLeaf];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid / 64;
    double2 *A2 = reinterpret_cast<double2 *>(A);
    auto at = [&](std::uint32_t c, std::uint32_t r) -> double2 & { return A2[static_cast<std::size_t>(c) * n + r]; };
    const std::uint32_t je = j0 + w;
    for (std::uint32_t j = j0; j < je; ++j) {
        double bv = -1;
        std::uint32_t bi = j;
        for (std::uint32_t r = j + tid; r < n; r += kPanelThreads) {
            const double2 v = at(j, r);
            const double m = v.x * v.x + v.y * v.y;
            if (m > bv) {
                bv = m;
                bi = r;
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const double ov = __shfl_xor(bv, off, 64);
            const std::uint32_t oi = __shfl_xor(bi, off, 64);
            if (ov > bv || (ov == bv && oi < bi)) {
                bv = ov;
                bi = oi;
            }
        }
        if (lane == 0) {
            best[wave] = bv;
            where[wave] = bi;
        }
        __syncthreads(); // (1)
        double v = best[0];
        std::uint32_t p = where[0];
        for (int q = 1; q < kPanelThreads / 64; ++q)
            if (best[q] > v || (best[q] == v && where[q] < p)) {
                v = best[q];
                p = where[q];
            }
        if (tid < static_cast<int>(je - j))
            u[tid] = at(j + tid, p);
        if (tid == 0) {
            piv[j] = static_cast<std::int32_t>(p);
            if (!(v > 0))
                report_zero_pivot(info, static_cast<int>(j) + 1);
        }
        __syncthreads(); // (2): every thread has p and the pivot row's leaf entries
        const double2 d = u[0];
        const double dd = d.x * d.x + d.y * d.y;
        const double ir = dd > 0 ? d.x / dd : 0.0, ii = dd > 0 ? -d.y / dd : 0.0; // 1/a = conj(a)/|a|^2
        for (std::uint32_t r = j + 1 + tid; r < n; r += kPanelThreads) {
            const std::uint32_t src = r == p ? j : r; // row p receives the old row j
            const double2 a = at(j, src);
            const double lr = a.x * ir - a.y * ii, li = a.x * ii + a.y * ir;
            for (std::uint32_t c = j + 1; c < je; ++c) {
                const double2 b = at(c, src), uc = u[c - j];
                at(c, r) = double2{b.x - (lr * uc.x - li * uc.y), b.y - (lr * uc.y + li * uc.x)};
            }
            at(j, r) = double2{lr, li};
            if (r == p) // this thread read the old row j; the pivot row takes its place
                for (std::uint32_t c = j; c < je; ++c)
                    at(c, j) = u[c - j];
        }
        if (p != j) // the other panel columns (incl. this leaf's L columns before j): interchange rows j and p
            for (std::uint32_t c = k0 + tid; c < pe; c += kPanelThreads)
                if (c < j || c >= je) {
                    const double2 t = at(c, j);
                    at(c, j) = at(c, p);
                    at(c, p) = t;
                }
        __syncthreads(); // (3)
    }
}

// Apply the panel's row interchanges to the columns outside it.
__global__ void lu_swap(double *A, std::uint32_t n, std::uint32_t k0, std::uint32_t nb, const std::int32_t *piv) {
    const std::uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n || (c >= k0 && c < k0 + nb))
        return;
    double *col = A + 2 * static_cast<std::size_t>(c) * n;
    for (std::uint32_t j = k0; j < k0 + nb; ++j) {
        const std::uint32_t p = static_cast<std::uint32_t>(piv[j]);
        if (p != j) {
            const double t0 = col[2 * j], t1 = col[2 * j + 1];
            col[2 * j] = col[2 * p];
            col[2 * j + 1] = col[2 * p + 1];
            col[2 * p] = t0;
            col[2 * p + 1] = t1;
        }
    }
}

// U12 = L11^{-1} A12 (unit lower nb x nb L11 at [k0, k0 + nb)) for the columns
// [k0 + nb, c_end): 64 threads per 64 columns. The block's nb x 64 slice of A12 is
// staged through LDS with consecutive threads on consecutive rows of a column
// (coalesced), each thread solves one column from LDS, and the slice is written back
// the same way. Rows of the staged slice are padded against LDS bank conflicts.
__global__ __launch_bounds__(64) void lu_trsm(double *A, std::uint32_t n, std::uint32_t k0, std::uint32_t nb,
                                              std::uint32_t c_end) {
    __shared__ double L[kPanel][kPanel][2];
    __shared__ double2 X[64][kPanel + 1];
    for (std::uint32_t e = threadIdx.x; e < nb * nb; e += 64) {
        const std::uint32_t r = e % nb, c = e / nb;
        L[r][c][0] = A[2 * ((static_cast<std::size_t>(k0) + c) * n + k0 + r)];
        L[r][c][1] = A[2 * ((static_cast<std::size_t>(k0) + c) * n + k0 + r) + 1];
    }
    const std::uint32_t c_first = k0 + nb + blockIdx.x * 64;
    const std::uint32_t cols = min(64u, c_end - c_first);
    double2 *A2 = reinterpret_cast<double2 *>(A);
    for (std::uint32_t e = threadIdx.x; e < cols * nb; e += 64) {
        const std::uint32_t q = e / nb, r = e % nb;
        X[q][r] = A2[static_cast<std::size_t>(c_first + q) * n + k0 + r];
    }
    __syncthreads();
    const std::uint32_t t = threadIdx.x;
    if (t < cols) {
        double xr[kPanel], xi[kPanel];
        for (std::uint32_t i = 0; i < nb; ++i) {
            double vr = X[t][i].x, vi = X[t][i].y;
            for (std::uint32_t j = 0; j < i; ++j) {
                vr -= L[i][j][0] * xr[j] - L[i][j][1] * xi[j];
                vi -= L[i][j][0] * xi[j] + L[i][j][1] * xr[j];
            }
            xr[i] = vr;
            xi[i] = vi;
            X[t][i] = double2{vr, vi};
        }
    }
    __syncthreads();
    for (std::uint32_t e = threadIdx.x; e < cols * nb; e += 64) {
        const std::uint32_t q = e / nb, r = e % nb;
        A2[static_cast<std::size_t>(c_first + q) * n + k0 + r] = X[q][r];
    }
}


// ---- solves ----

// Every interchange applied to the right-hand sides (one workgroup each), n <= 16384: the
// permutation is composed in LDS, the net effect of 16 panels at a time found by 16
// wavefronts and applied in order, and the entries move once: 78 us at n = 4099, where the
// chain of single interchanges in memory below took 1.4 ms.
constexpr std::uint32_t kPermuteRows = kLuPermuteRows;
__global__ __launch_bounds__(1024) void permute_rows(double *B, std::uint32_t n, const std::int32_t *piv) {
    __shared__ std::uint16_t at[kPermuteRows];
    __shared__ std::uint16_t to[16][2 * kBlock], from[16][2 * kBlock];
    __shared__ std::uint32_t count[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double2 *b = reinterpret_cast<double2 *>(B) + static_cast<std::size_t>(blockIdx.x) * n;
    for (std::uint32_t i = tid; i < n; i += 1024)
        at[i] = static_cast<std::uint16_t>(i);
    for (std::uint32_t base = 0; base < n; base += 16 * kBlock) {
        const std::uint32_t j0 = base + wave * kBlock;
        u64 moved = 0;
        if (j0 < n) {
            const std::uint32_t nb = min(static_cast<std::uint32_t>(kBlock), n - j0);
            const std::uint32_t p = static_cast<std::uint32_t>(lane) < nb ? static_cast<std::uint32_t>(piv[j0 + lane])
                                                                          : j0 + lane;
            const Interchange x = net_interchange(p, j0, nb);
            moved = x.moved;
            const u64 owners = __ballot(x.owner);
            const int slot = __popcll(owners & ((1ull << lane) - 1));
            if (moved) {
                if (static_cast<std::uint32_t>(lane) < nb) {
                    to[wave][lane] = static_cast<std::uint16_t>(j0 + lane);
                    from[wave][lane] = static_cast<std::uint16_t>(x.inside);
                }
                if (x.owner) {
                    to[wave][nb + slot] = static_cast<std::uint16_t>(p);
                    from[wave][nb + slot] = static_cast<std::uint16_t>(x.outside);
                }
            }
            if (lane == 0)
                count[wave] = moved ? nb + static_cast<std::uint32_t>(__popcll(owners)) : 0;
        } else if (lane == 0) {
            count[wave] = 0;
        }
        __syncthreads();
        for (int w = 0; w < 16; ++w) { // in order; all entries of one panel read before any is written
            const std::uint32_t m = count[w];
            if (!m)
                continue;
            std::uint16_t x = 0;
            if (static_cast<std::uint32_t>(tid) < m)
                x = at[from[w][tid]];
            __syncthreads();
            if (static_cast<std::uint32_t>(tid) < m)
                at[to[w][tid]] = x;
            __syncthreads();
        }
        __syncthreads();
    }
    double2 value[kPermuteRows / 1024];
#pragma unroll
    for (std::uint32_t k = 0; k < kPermuteRows / 1024; ++k) {
        const std::uint32_t i = tid + 1024 * k;
        value[k] = i < n ? b[at[i]] : double2{0.0, 0.0};
    }
    drain_memory(); // every entry has been read
    __syncthreads();
#pragma unroll
    for (std::uint32_t k = 0; k < kPermuteRows / 1024; ++k) {
        const std::uint32_t i = tid + 1024 * k;
        if (i < n)
            b[i] = value[k];
    }
}

// Row interchanges of every panel applied to the right-hand sides.
__global__ void apply_pivots(double *B, std::uint32_t n, const std::int32_t *piv, std::uint32_t nrhs) {
    const std::uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nrhs)
        return;
    double *x = B + 2 * static_cast<std::size_t>(e) * n;
    for (std::uint32_t j = 0; j < n; ++j) {
        const std::uint32_t p = static_cast<std::uint32_t>(piv[j]);
        if (p != j) {
            const double t0 = x[2 * j], t1 = x[2 * j + 1];
            x[2 * j] = x[2 * p];
            x[2 * j + 1] = x[2 * p + 1];
            x[2 * p] = t0;
            x[2 * p + 1] = t1;
        }
    }
}

// One block step of a sweep: the 64 unknowns of block t (already solved; t < 0 or t >= blocks:
// none) are eliminated from one 64-row tile per workgroup, and the first workgroup, whose tile
// is the next block of the sweep, solves it. A wavefront then has a row per lane and
// takes the unknowns in order from a lane's registers (readlane), so the triangle costs no
// barriers; rows of the upper triangle are scaled by the inverse of their pivot first. Four
// right-hand sides at a time, one per wavefront. Bound by the latency of one launch per block:
// 15 us, against 38 us for a substitution with barriers and an elimination in two launches.
template <bool kUpper>
__global__ __launch_bounds__(256) void solve_step(const double *LU, std::uint32_t n, double *B, std::uint32_t nrhs,
                                                  std::int32_t t) {
    __shared__ double2 triangle[kBlock][kBlock + 1]; // [c][r], the first workgroup's
    __shared__ double2 x[4][kBlock], part[4][4][kBlock];
    const double2 *LU2 = reinterpret_cast<const double2 *>(LU);
    double2 *B2 = reinterpret_cast<double2 *>(B);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const std::uint32_t blocks = (n + kBlock - 1) / kBlock;
    const bool eliminate = kUpper ? t < static_cast<std::int32_t>(blocks) : t >= 0;
    const std::uint32_t tile = kUpper ? t - 1 - blockIdx.x : t + 1 + blockIdx.x;
    const std::uint32_t r0 = tile * kBlock, row = r0 + lane, rows = min(static_cast<std::uint32_t>(kBlock), n - r0);
    const bool in = static_cast<std::uint32_t>(lane) < rows, solve = blockIdx.x == 0;
    double2 l[16];
    if (eliminate) {
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const std::uint32_t col = static_cast<std::uint32_t>(t) * kBlock + 16 * wave + c;
            l[c] = in && col < n ? LU2[static_cast<std::size_t>(col) * n + row] : double2{0.0, 0.0};
        }
    }
    double2 scale = {1.0, 0.0};
    if (solve) {
        if (kUpper && in) {
            const double2 u = LU2[static_cast<std::size_t>(row) * n + row];
            const double d = u.x * u.x + u.y * u.y;
            scale = {u.x / d, -u.y / d};
        }
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const std::uint32_t q = 16 * wave + c;
            double2 a = {0.0, 0.0};
            if (in && q < rows && (kUpper ? static_cast<std::uint32_t>(lane) < q : static_cast<std::uint32_t>(lane) > q))
                a = LU2[static_cast<std::size_t>(r0 + q) * n + row];
            triangle[q][lane] = {a.x * scale.x - a.y * scale.y, a.x * scale.y + a.y * scale.x};
        }
    }
    for (std::uint32_t e0 = 0; e0 < nrhs; e0 += 4) {
        const std::uint32_t e = e0 + wave;
        double2 b = {0.0, 0.0};
        if (e < nrhs && in)
            b = B2[static_cast<std::size_t>(e) * n + row];
        if (eliminate) {
            const std::uint32_t known = static_cast<std::uint32_t>(t) * kBlock + lane;
            x[wave][lane] = e < nrhs && known < n ? B2[static_cast<std::size_t>(e) * n + known] : double2{0.0, 0.0};
            __syncthreads();
            const int count = min(4u, nrhs - e0);
            for (int f = 0; f < count; ++f) {
                double2 s = {0.0, 0.0};
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    const double2 y = x[f][16 * wave + c];
                    s.x += l[c].x * y.x - l[c].y * y.y;
                    s.y += l[c].x * y.y + l[c].y * y.x;
                }
                part[f][wave][lane] = s;
            }
            __syncthreads();
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                b.x -= part[wave][w][lane].x;
                b.y -= part[wave][w][lane].y;
            }
        } else {
            __syncthreads();
        }
        if (solve && e < nrhs) {
            if (kUpper)
                b = {b.x * scale.x - b.y * scale.y, b.x * scale.y + b.y * scale.x};
            auto take = [&](int j) {
                auto lane_value = [j](double v) {
                    const u64 w = __builtin_bit_cast(u64, v);
                    const std::uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(w), j),
                                        hi = __builtin_amdgcn_readlane(static_cast<int>(w >> 32), j);
                    return __builtin_bit_cast(double, static_cast<u64>(hi) << 32 | lo);
                };
                const double xr = lane_value(b.x), xi = lane_value(b.y);
                const double2 a = triangle[j][lane]; // zero on and beyond the diagonal
                b.x -= a.x * xr - a.y * xi;
                b.y -= a.x * xi + a.y * xr;
            };
            if (kUpper) {
#pragma unroll 8
                for (int j = kBlock - 1; j >= 0; --j)
                    take(j);
            } else {
#pragma unroll 8
                for (int j = 0; j < kBlock; ++j)
                    take(j);
            }
        }
        if (e < nrhs && in)
            B2[static_cast<std::size_t>(e) * n + row] = b;
        __syncthreads();
    }
}

} // namespace

namespace {

// Panel workgroups of this process that may wait for each other, per device: one per compute
// unit. (Two fit on an empty one, but a workgroup that was placed beside another kernel's may
// leave its LDS in two parts, neither large enough for a second.) Counted in whole rounds of
// the dies that take workgroups in turn, so that no die gets more than its compute units.
constexpr std::uint32_t kDies = 8;
constexpr int kMaxDevices = 64;
struct PanelBudget {
    std::mutex mutex;
    std::condition_variable freed;
    std::uint32_t capacity{}, used{};
};

PanelBudget &budget_of(int device) {
    static std::array<PanelBudget, kMaxDevices> budgets;
    if (device < 0 || device >= kMaxDevices)
        throw std::invalid_argument("device ordinal out of range for the LU factorization");
    PanelBudget &b = budgets[device];
    std::lock_guard lock(b.mutex);
    if (!b.capacity) {
        int units = 0, resident = 0;
        hip_check(hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device), "compute units");
        hip_check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&resident, lu_step, kStepThreads, 0), "LU occupancy");
        b.capacity = resident > 0 ? std::max(units, 1) : 1;
    }
    return b;
}

// The workgroups that a factorization of n rows may use for a panel, reserved until this object
// goes. Waits for others to finish theirs, but not for ever: after two seconds it takes what
// is left, if need be one, which waits for nobody.
class PanelGroups {
  public:
    PanelGroups(std::uint32_t n, std::uint32_t limit) {
        const std::uint32_t wanted = std::min((n + kPanelRows - 1) / kPanelRows, std::clamp(limit, 1u, kMaxPanelGroups));
        if (wanted <= 1)
            return;
        int device = 0;
        hip_check(hipGetDevice(&device), "current device");
        budget_ = &budget_of(device);
        std::unique_lock lock(budget_->mutex);
        const std::uint32_t whole = std::min((wanted + kDies - 1) / kDies * kDies, budget_->capacity);
        budget_->freed.wait_for(lock, std::chrono::seconds(2),
                                [&] { return budget_->used + whole <= budget_->capacity; });
        const std::uint32_t left = budget_->capacity - budget_->used;
        reserved_ = left >= whole ? whole : left / kDies * kDies;
        count_ = std::clamp(reserved_, 1u, wanted);
        budget_->used += reserved_;
    }
    ~PanelGroups() {
        if (!reserved_)
            return;
        {
            std::lock_guard lock(budget_->mutex);
            budget_->used -= reserved_;
        }
        budget_->freed.notify_all();
    }
    PanelGroups(const PanelGroups &) = delete;
    PanelGroups &operator=(const PanelGroups &) = delete;
    std::uint32_t count() const { return count_; }

  private:
    PanelBudget *budget_{};
    std::uint32_t reserved_{}, count_{1};
};

void step(double *A, std::uint32_t n, const PanelArgs &P, const UpdateArgs &U, hipStream_t stream) {
    const std::uint32_t rows = (U.r_end - U.r_begin + kBlock - 1) / kBlock,
                        columns = (U.c_end - U.c_begin + kBlock - 1) / kBlock;
    const std::uint32_t blocks = P.groups + rows * columns;
    if (blocks)
        hipLaunchKernelGGL(lu_step, dim3(blocks), dim3(kStepThreads), 0, stream, A, n, P, U);
}

// C -= L U over rows [r0, r1) x columns [c0, c1) with K = A's columns / rows [k0, k0 + nb).
void update(double *A, std::uint32_t n, std::uint32_t k0, std::uint32_t nb, std::uint32_t r0, std::uint32_t r1,
            std::uint32_t c0, std::uint32_t c1, hipStream_t stream) {
    if (r1 > r0 && c1 > c0)
        step(A, n, PanelArgs{}, UpdateArgs{k0, nb, r0, r1, c0, c1}, stream);
}

// The leaves of panel [k0, k0 + nb): pivoted 4-column leaves (row interchanges inside the
// panel), each leaf's U rows of the panel and the rank-4 update of the panel below it.
void factor_panel_leaves(double *A, std::uint32_t n, std::uint32_t k0, std::uint32_t nb, std::int32_t *piv, int *info,
                         hipStream_t stream) {
    const std::uint32_t pe = k0 + nb;
    for (std::uint32_t j0 = k0; j0 < pe; j0 += kLeaf) {
        const std::uint32_t w = std::min<std::uint32_t>(kLeaf, pe - j0);
        hipLaunchKernelGGL(lu_leaf, dim3(1), dim3(kPanelThreads), 0, stream, A, n, k0, j0, w, pe, piv, info);
        if (j0 + w >= pe)
            continue;
        hipLaunchKernelGGL(lu_trsm, dim3(1), dim3(64), 0, stream, A, n, j0, w, pe);
        update(A, n, j0, w, j0 + w, n, j0 + w, pe, stream);
    }
}

// The launches of a factorization whose panels may have `groups` workgroups.
void factor_launches(double *A, std::uint32_t n, std::int32_t *piv, int *info, double *work, std::uint32_t groups,
                     hipStream_t stream) {
    const std::uint32_t most = groups * kPanelRows;
    // While more rows are left than the panel's workgroups hold: pairs of 32-column panels
    // P1 = [k0, e1), P2 = [e1, e2), factored on one workgroup leaf by leaf, with one rank-64
    // trailing update. P1 is factored, its interchanges applied and its U rows solved over every
    // later column; P1's update reaches P2's columns before P2 is factored; after P2's
    // interchanges (applied to the still un-updated trailing rows and to P1's L rows alike)
    // P1's update reaches P2's U rows, P2's U rows are solved, and the rows below P2 take
    // both panels' updates at once.
    std::uint32_t k0 = 0;
    for (; n - k0 > most; k0 += 2 * kPanel) {
        const std::uint32_t e1 = k0 + kPanel, e2 = e1 + kPanel;
        factor_panel_leaves(A, n, k0, kPanel, piv, info, stream);
        hipLaunchKernelGGL(lu_swap, dim3((n + 63) / 64), dim3(64), 0, stream, A, n, k0, kPanel, piv);
        hipLaunchKernelGGL(lu_trsm, dim3((n - e1 + 63) / 64), dim3(64), 0, stream, A, n, k0, kPanel, n);
        update(A, n, k0, kPanel, e1, n, e1, e2, stream);
        factor_panel_leaves(A, n, e1, kPanel, piv, info, stream);
        hipLaunchKernelGGL(lu_swap, dim3((n + 63) / 64), dim3(64), 0, stream, A, n, e1, kPanel, piv);
        update(A, n, k0, kPanel, e1, e2, e2, n, stream);
        hipLaunchKernelGGL(lu_trsm, dim3((n - e2 + 63) / 64), dim3(64), 0, stream, A, n, e1, kPanel, n);
        update(A, n, k0, 2 * kPanel, e2, n, e2, n, stream);
    }
    // 64-column panels. Per panel: its interchanges and U rows in the other columns; its update of
    // the next panel's columns; then one launch that factors the next panel and updates the rest.
    auto *exchange = reinterpret_cast<u64 *>(work);
    auto *moves = reinterpret_cast<PanelMoves *>(work + kRing * kMaxPanelGroups * kSlotWords);
    auto panel = [&](std::uint32_t first) {
        PanelArgs P{};
        P.k0 = first;
        P.nb = std::min<std::uint32_t>(kBlock, n - first);
        P.groups = (n - first + kPanelRows - 1) / kPanelRows;
        P.piv = piv;
        P.info = info;
        P.exchange = exchange;
        P.moves = moves;
        return P;
    };
    if (n - k0 > static_cast<std::uint32_t>(kPanelRows)) {
        constexpr std::uint32_t words = kRing * kMaxPanelGroups * kSlotWords;
        hipLaunchKernelGGL(clear_exchange, dim3((words + 255) / 256), dim3(256), 0, stream, exchange, words);
    }
    step(A, n, panel(k0), UpdateArgs{}, stream);
    for (; k0 < n; k0 += kBlock) {
        const std::uint32_t nb = std::min<std::uint32_t>(kBlock, n - k0), e = k0 + nb;
        const std::uint32_t others = k0 / kBlock + (n - e + kBlock - 1) / kBlock;
        if (others)
            hipLaunchKernelGGL(lu_rows, dim3(others), dim3(256), 0, stream, A, n, k0, nb, moves, info);
        if (e == n)
            break;
        const std::uint32_t next = std::min<std::uint32_t>(kBlock, n - e);
        hipLaunchKernelGGL(lu_update_small, dim3((n - e + kSmall - 1) / kSmall, (next + kSmall - 1) / kSmall), dim3(256), 0,
                           stream, A, n, UpdateArgs{k0, nb, e, n, e, e + next});
        step(A, n, panel(e), UpdateArgs{k0, nb, e, n, e + next, n}, stream);
    }
}

} // namespace

void lu_factor(const std::function<void()> &fill, double *A, std::uint32_t n, std::int32_t *piv, int *info, double *work,
               hipStream_t stream, const char *singular, const LuLimits &limits) {
    int code = 0;
    auto attempt = [&](std::uint32_t most, int status) {
        if (fill)
            fill();
        const PanelGroups groups(n, most); // until the stream has been waited for
        hipLaunchKernelGGL(set_status, dim3(1), dim3(1), 0, stream, info, status);
        hip_check(hipGetLastError(), "LU status");
        factor_launches(A, n, piv, info, work, groups.count(), stream);
        hip_check(hipMemcpyAsync(&code, info, sizeof(int), hipMemcpyDeviceToHost, stream), "LU status download");
        hip_check(hipStreamSynchronize(stream), "LU sync");
    };
    attempt(limits.panel_groups, limits.status);
    if (code == kWaitFailed && fill && !limits.once)
        attempt(1, 0);
    if (code == kWaitFailed)
        throw std::runtime_error("LU factorization: the panel's workgroups did not all become resident");
    if (code)
        throw std::runtime_error(singular + std::to_string(code));
}

void lu_solve(const double *LU, std::uint32_t n, const std::int32_t *piv, double *B, std::uint32_t nrhs,
              hipStream_t stream, const LuLimits &limits) {
    if (n <= std::min(limits.permute_rows, kPermuteRows))
        hipLaunchKernelGGL(permute_rows, dim3(nrhs), dim3(1024), 0, stream, B, n, piv);
    else
        hipLaunchKernelGGL(apply_pivots, dim3((nrhs + 63) / 64), dim3(64), 0, stream, B, n, piv, nrhs);
    const auto blocks = static_cast<std::int32_t>((n + kBlock - 1) / kBlock);
    for (std::int32_t t = -1; t + 1 < blocks; ++t)
        hipLaunchKernelGGL(solve_step<false>, dim3(t < 0 ? 1 : blocks - 1 - t), dim3(256), 0, stream, LU, n, B, nrhs, t);
    for (std::int32_t t = blocks; t > 0; --t)
        hipLaunchKernelGGL(solve_step<true>, dim3(t == blocks ? 1 : t), dim3(256), 0, stream, LU, n, B, nrhs, t);
}

} // namespace hsbem::dev
