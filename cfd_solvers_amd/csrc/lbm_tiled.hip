// lbm_tiled.hip -- several D2Q9 time steps in one launch, on tiles held in LDS.
//
// A single in-place step reads and writes every population once, so a large 2-D lattice is bound by
// HBM and a small one by the launch.  Here a block loads a tile with a halo of K cells, takes K steps
// on it in LDS and writes the interior into a second lattice array (the halo cells' old state is
// read by several blocks, so the result cannot overwrite it).  The halo is recomputed: level s (1..K)
// updates the cells at least s away from the tile's edge.
//
// The tile is kept in the lattice's own esoteric slot map: level 1 loads from the global slots and
// stores into LDS slots, the levels between work in place on LDS (each slot is read and written by one
// cell, so one barrier a level is enough and nothing is double-buffered), level K stores to the global
// slots.  Every level rounds to the storage type and uses the step kernel's arithmetic, so K steps here
// are K single steps bit for bit, the slots left behind at walls included.
#include "lbm_tiled.hpp"
#include "lbm_cell.hpp"

#include <hip/hip_runtime.h>

#include <stdexcept>
#include <string>

namespace cfd_hip {

namespace {

constexpr int Q = 9;
constexpr int W = 64;  // slots of a tile row

// Populations of the cell at LDS slot `c` (Odd: parity of the step), and back.
template <class T, bool Odd, bool Bounded, int P>
__device__ __forceinline__ void load_tile(const T* t, int c, uint32_t desc, typename Storage<T>::Real (&f)[Q]) {
    using L = Lattice<Q>;
    using S = Storage<T>;
    f[0] = S::template decode<Q, 0>(t[c]);
    static_for<(Q - 1) / 2>([&](auto PP) {
        constexpr int i = 2 * decltype(PP)::value + 1;
        constexpr int up = -(L::cy[i] * W + L::cx[i]);
        if constexpr (Bounded) {
            const bool wup = ((desc >> (i - 1)) & 1U) != 0U, wdn = ((desc >> i) & 1U) != 0U;
            f[i] = S::template decode<Q, i>(t[c + up + (Odd != wup ? i + 1 : i) * P]);
            f[i + 1] = S::template decode<Q, i + 1>(t[c + (Odd != wdn ? i : i + 1) * P]);
        } else {
            f[i] = S::template decode<Q, i>(t[c + up + (Odd ? i + 1 : i) * P]);
            f[i + 1] = S::template decode<Q, i + 1>(t[c + (Odd ? i : i + 1) * P]);
        }
    });
}
template <class T, bool Odd, int P>
__device__ __forceinline__ void store_tile(T* t, int c, const typename Storage<T>::Real (&f)[Q]) {
    using L = Lattice<Q>;
    using S = Storage<T>;
    t[c] = S::template encode<Q, 0>(f[0]);
    static_for<(Q - 1) / 2>([&](auto PP) {
        constexpr int i = 2 * decltype(PP)::value + 1;
        constexpr int up = -(L::cy[i] * W + L::cx[i]);
        t[c + (Odd ? i : i + 1) * P] = S::template encode<Q, i>(f[i]);
        t[c + up + (Odd ? i + 1 : i) * P] = S::template encode<Q, i + 1>(f[i + 1]);
    });
}

// All K levels of one tile: W x H slots in LDS, the thread's column rx, rows ry0, ry0 + Rows, ...;
// `w` x `h` of them are used: the interior, which ends with the lattice, and its halo.
template <class T, bool Bounded, bool Forced, int K, int H, int Rows>
__device__ __forceinline__ void advance_tile(const void* src, void* dst, const Geometry& g,
                                             const Physics<typename Storage<T>::Real>& p, T* t, int rx, int ry0,
                                             uint32_t x, int y_first, int w, int h) {
    using Real = typename Storage<T>::Real;
    using S = Storage<T>;
    constexpr int P = W * H;
    static_for<K>([&](auto LL) {
        constexpr int s = decltype(LL)::value + 1;
        constexpr bool Odd = (s & 1) == 0;  // the tile starts at even parity
        if (rx >= s && rx < w - s)
            for (int ry = ry0 + s; ry < h - s; ry += Rows) {
                int yy = y_first + ry;  // -K .. ny + K - 1
                if (yy < 0) yy += static_cast<int>(g.ny);
                if (yy >= static_cast<int>(g.ny)) yy -= static_cast<int>(g.ny);
                const uint32_t y = static_cast<uint32_t>(yy);
                const uint32_t n = y * g.nx + x;
                uint32_t desc = 0U;
                if constexpr (Bounded) desc = p.links[n];
                const uint32_t type = (desc >> kTypeShift) & 3U;
                if (Bounded && type == kTypeWall) continue;
                const int c = ry * W + rx;
                Real f[Q];
                if constexpr (s == 1) {
                    PairSlots<Q> slots;
                    load_cell<Q, T, Odd, Bounded>(src, g, desc, neighbourhood(g, x, y, 0U), f, slots);
                } else {
                    load_tile<T, Odd, Bounded, P>(t, c, desc, f);
                }
                [[maybe_unused]] Real fin[Q];
                if constexpr (Bounded && s == K)
                    static_for<Q>([&](auto DD) { fin[decltype(DD)::value] = f[decltype(DD)::value]; });
                const Real rho = collide<Q, Forced, S>(p, static_cast<const Real*>(nullptr), g,
                                                       static_cast<uint8_t>(type), n, y, 0U, f);
                if constexpr (s < K) {
                    if constexpr (Bounded) moving_wall_terms<Q, S>(p, desc, n, rho, f);
                    store_tile<T, Odd, P>(t, c, f);
                } else {
                    const Neighbourhood nb = neighbourhood(g, x, y, 0U);
                    PairSlots<Q> slots;
                    slots.self = nb.cell(0, 0, 0) * static_cast<uint32_t>(sizeof(T));
                    slots.desc = desc;
                    static_for<(Q - 1) / 2>([&](auto PP) {
                        constexpr int i = 2 * decltype(PP)::value + 1;
                        using L = Lattice<Q>;
                        slots.up[i] = nb.cell(-L::cx[i], -L::cy[i], 0) * static_cast<uint32_t>(sizeof(T));
                        // A wall link's population was read from the slot of the other parity, which the
                        // in-place step leaves as it was.
                        if constexpr (Bounded) {
                            if (slots.is_wall_link(i - 1))
                                store_at<T>(plane<T>(dst, g, Odd ? i : i + 1), slots.up[i],
                                            S::template encode<Q, i>(fin[i]));
                            if (slots.is_wall_link(i))
                                store_at<T>(plane<T>(dst, g, Odd ? i + 1 : i), slots.self,
                                            S::template encode<Q, i + 1>(fin[i + 1]));
                        }
                    });
                    store_cell<Q, T, Odd, Bounded>(dst, g, p, n, x, y, 0U, rho, f, slots);
                }
            }
        if constexpr (s < K) __syncthreads();
    });
}

template <class T, bool Bounded, bool Forced, int K, int H, int Rows>
__global__ __launch_bounds__(W* Rows) void tiled_step(const void* __restrict__ src, void* __restrict__ dst,
                                                      const Geometry g,
                                                      const Physics<typename Storage<T>::Real> p, uint32_t tiles_x,
                                                      uint32_t rows) {
    __shared__ T tile[Q * W * H];
    const int rx = static_cast<int>(threadIdx.x) % W, ry0 = static_cast<int>(threadIdx.x) / W;
    const uint32_t bx = blockIdx.x % tiles_x, by = blockIdx.x / tiles_x;
    const int x0 = static_cast<int>(bx) * (W - 2 * K), y0 = static_cast<int>(by * rows);
    const int w = min(W, static_cast<int>(g.nx) - x0 + 2 * K), h = min(static_cast<int>(rows), static_cast<int>(g.ny) - y0) + 2 * K;
    int xx = x0 + rx - K;  // beyond w: not used
    if (xx < 0) xx += static_cast<int>(g.nx);
    if (xx >= static_cast<int>(g.nx)) xx -= static_cast<int>(g.nx);
    const uint32_t x = static_cast<uint32_t>(xx);
    if constexpr (Bounded) {
        // A tile whose cells are all plain fluid with plain-fluid neighbours takes the periodic path.
        int marked = 0;
        if (rx < w && (rx == 0 || rx == w - 1 || (x & 63U) == 0U))  // one lane of every segment touched
            for (int ry = ry0; ry < h; ry += Rows) {
                int yy = y0 + ry - K;
                if (yy < 0) yy += static_cast<int>(g.ny);
                if (yy >= static_cast<int>(g.ny)) yy -= static_cast<int>(g.ny);
                marked |= static_cast<int>(p.segments[static_cast<uint32_t>(yy) * p.seg_x + (x >> 6)] & kSpanBits);
            }
        if (__syncthreads_or(marked) != 0) {
            advance_tile<T, true, Forced, K, H, Rows>(src, dst, g, p, tile, rx, ry0, x, y0 - K, w, h);
            return;
        }
    }
    advance_tile<T, false, Forced, K, H, Rows>(src, dst, g, p, tile, rx, ry0, x, y0 - K, w, h);
}

constexpr uint32_t kHalo = 4;  // the largest K

// Two tiles, both 64 slots (one wavefront) wide.  34 rows (FP32: 77 KiB of LDS, two blocks a CU)
// recompute 18 % of the cells at K = 4 and are bound by the vector units: 4096^2 cavity FP32 91 us a step
// in calls of 40 against 196 single (periodic 83 against 204, FP16S 76 against 109), 1400^2 13.6 against
// 24.0.  When they were chosen, at 134 us, 26 rows measured 137-142, 42 rows 152, 8 rows of threads
// instead of 16 139.
//
// Below about 200 000 cells those tiles are too few to fill the chip, and the launch and the chain of
// levels count: up to 16 rows, 12 of them at a time, and as many interior rows as make the fewest
// wavefronts of the busiest CU (tile_rows).  256^2 FP32 periodic: 1.8 us a step against 4.2 single; 330^2:
// 2.0 against 3.9; 400^2: 2.1 against 3.9; 100 x 500: 1.7 against 4.1.  When they were chosen, at 2.0, 2.2,
// 2.6 and 1.9, tiles of 32 x 16 slots measured 2.1, 2.4, 2.9 and 2.1, the large tile 2.9 at 256^2 and 3.0
// at 400^2; it was ahead at 600^2 (3.6 against 4.6).
constexpr uint32_t kLargeTileCells = 200000U;
constexpr uint32_t kLargeRows = 34U - 2U * kHalo;  // interior rows of the large tile

// Interior rows (2 to `most`) of tiles with `strips` columns: blocks are dealt to 256 CUs, and a block
// issues K rows + K (K - 1) wavefronts over its levels (rows + 2 (K - s) at level s).
uint32_t tile_rows(uint32_t strips, uint32_t ny, uint32_t k, uint32_t most) {
    uint32_t best = most;
    uint64_t least = ~uint64_t{0};
    for (uint32_t rows = most; rows >= 2U; --rows) {
        const uint64_t blocks = static_cast<uint64_t>(strips) * ((ny + rows - 1U) / rows);
        const uint64_t waves = (blocks + 255U) / 256U * (k * rows + k * (k - 1U));
        if (waves < least) {
            least = waves;
            best = rows;
        }
    }
    return best;
}

template <class T, bool Bounded, bool Forced, int K> void launch(const LaunchState& st, const void* src, void* dst) {
    using Real = typename Storage<T>::Real;
    constexpr uint32_t kInner = 64U - 2U * K;
    const uint32_t tx = (st.geo.nx + kInner - 1U) / kInner;
    const auto go = [&](auto kernel, uint32_t rows, uint32_t threads) {
        hipLaunchKernelGGL(kernel, dim3(tx * ((st.geo.ny + rows - 1U) / rows)), dim3(threads), 0, st.stream, src, dst,
                           st.geo, *static_cast<const Physics<Real>*>(st.physics), tx, rows);
    };
    if (st.cells < kLargeTileCells)
        go(tiled_step<T, Bounded, Forced, K, 16, 12>, tile_rows(tx, st.geo.ny, K, 16U - 2U * K), 768U);
    else if constexpr (K == 4) go(tiled_step<T, Bounded, Forced, K, 34, 16>, kLargeRows, 1024U);
    else throw std::invalid_argument("tiled_steps: two steps in one launch only on small lattices");
    if (const hipError_t e = hipGetLastError(); e != hipSuccess)
        throw std::runtime_error(std::string("tiled_step launch: ") + hipGetErrorString(e));
}

template <class T> void steps(const LaunchState& st, int k, bool bounded, bool forced, const void* src, void* dst) {
    const auto with = [&](auto B, auto F) {
        constexpr bool b = decltype(B)::value, f = decltype(F)::value;
        if (k == 4) launch<T, b, f, 4>(st, src, dst);
        else if (k == 2) launch<T, b, f, 2>(st, src, dst);
        else throw std::invalid_argument("tiled_steps takes 2 or 4 steps");
    };
    if (bounded) forced ? with(std::true_type{}, std::true_type{}) : with(std::true_type{}, std::false_type{});
    else forced ? with(std::false_type{}, std::true_type{}) : with(std::false_type{}, std::false_type{});
}

}  // namespace

// The coordinates wrap once, so the lattice is at least as large as the halo; FP64 stays with the single
// step (its tile would be half as large).
//
// On small lattices both widths are ahead of the single step (64 000 cells of any shape: 4 steps 0.5-0.8 of
// its time, 2 steps 0.6-0.95; only FP16S rows of 8 cells next to walls take 1.07 with 2).  In the large
// tile 2 steps move nearly as much memory as 2 single ones and wait for it longer: 0.8-1.1 of the single
// step's time in FP32, up to 1.5 in FP16S (4096^2 periodic 1.19, 128 x 62500 cavity 1.52), so what 4 steps
// leave over runs singly there.
//
// 4 steps pay there by the wavefronts that a level issues for one of the single step (64-cell segments):
// strips x (ny + 3 tile rows) / (segments x ny), 1.2 to 1.4 for most lattices, 1.67 for 128-wide rows, 2.2
// for 57- to 64-wide ones.
//  * FP32 and FP32S, unforced, are bound by memory as single steps: 0.4-0.8 of the single step's time, 0.6-0.97
//    in 57- to 64-wide rows.  No limit.
//  * Forced and LES steps issue more: 0.5-1.0 up to 1.67, 1.0-1.3 in 57- to 64-wide rows.  Limit 2.
//  * FP16S moves half the bytes.  Periodic: 0.5-0.95 up to 1.67, 0.8-1.2 in 57- to 64-wide rows; limit 2.
//    Next to walls: 0.6-0.95 up to 1.4, 0.8-1.19 in 128-wide rows, 1.0-1.46 in 57- to 64-wide ones; limit
//    1.5, and 1.3 where one lattice fits the 256 MiB Infinity Cache but two do not, since only the single
//    step is served from it (8 M cells, cavity: 100000 x 80 at 1.31 1.11, 256-wide at 1.39 1.02, 2048- and
//    4096-wide at 1.29 0.86 and 0.82).
bool tiled_pays(int q, int storage, size_t nx, size_t ny, size_t bytes, int k, bool bounded, bool forced) {
    if (q != 9 || (storage != 0 && storage != 1 && storage != 3) || nx < 2 * kHalo || ny < 2 * kHalo) return false;
    if (nx * ny < kLargeTileCells) return k == 2 || k == 4;
    if (k != 4) return false;
    const uint64_t strips = (nx + 55U) / 56U, segments = (nx + 63U) / 64U;
    const uint64_t launched = strips * (ny + (kHalo - 1U) * ((ny + kLargeRows - 1U) / kLargeRows));
    const uint64_t single = segments * ny;
    if (storage == 1 && bounded) {
        const uint64_t cache = uint64_t{256} << 20;
        return 100U * launched < (bytes <= cache && 2U * bytes > cache ? 130U : 150U) * single;
    }
    return (!forced && storage != 1) || launched < 2U * single;
}

void tiled_steps(int storage, const LaunchState& st, int k, bool bounded, bool forced, const void* src, void* dst) {
    switch (storage) {
    case 0: return steps<float>(st, k, bounded, forced, src, dst);
    case 1: return steps<_Float16>(st, k, bounded, forced, src, dst);
    case 3: return steps<F32Dev>(st, k, bounded, forced, src, dst);
    default: throw std::invalid_argument("tiled_steps: storage must be FP32, FP16S or FP32S");
    }
}

}  // namespace cfd_hip
