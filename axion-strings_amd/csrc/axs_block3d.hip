// axs_block3d.hip -- several steps per pass on small 3D lattices (a side below
// 64, which the marching kernels do not take): one work-group per cube of
// sites, every site in flight.
//
// A work-group of 1024 work-items loads a 16^3 region, four consecutive planes
// (i) of one (j, k) column each, and advances it up to four steps of the 7-point
// stencil: the drifted field sits in LDS (two buffers, one barrier per step),
// the sites' velocity and force in registers.  A step makes the region's
// outermost sites invalid, so the inner 8^3 are written.
//
// Such lattices took one launch a step, of which the chain of 7 gathered sites
// and the launch itself are all: 48^3 FP64 8.1 us.  Here four steps take one
// launch of 16 us (4.1 us a step): half of each region's width is recomputed,
// which a lattice of a few hundred regions (216 at 48^3) has the idle CUs for.
//
// The sums run in the one-step kernels' order with the forms' expressions, so
// a pass is bit-identical to d one-step launches.
#include "axs_forms.hpp"
#include "axs_internal.hpp"
#include "axs_lattice.hpp"

#include <type_traits>

namespace axs {

constexpr int kCubeSide = 16;
constexpr int kCubeRows = 4;                        // planes per work-item
constexpr int kCubeItems = kCubeSide * kCubeSide * kCubeSide / kCubeRows;

constexpr int kCubeDepth = 4;                       // most steps of a pass
constexpr int kCubeOut = kCubeSide - 2 * kCubeDepth;

// d <= kCubeDepth steps of cube `t` of lattice m
template <class Tr>
__device__ __forceinline__ void block3d_tile(const BatchMember &m, const uint32_t t, const int d,
                                             const LevelScalars<typename Tr::Sc, kCubeDepth> &sc)
{
    using T = typename Tr::T;
    typedef T T2 __attribute__((ext_vector_type(2)));
    constexpr int H = kCubeDepth, TS = kCubeOut, R = kCubeRows;
    constexpr int SJ = kCubeSide, SI = kCubeSide * kCubeSide;    // strides of j and i
    // the rim sites' neighbour reads end in unwritten padding before, between
    // and after the buffers (their values reach no written site)
    constexpr int PAD = SI + SJ + 1, BUF = kCubeSide * SI + PAD;
    __shared__ T2 X[2 * BUF + PAD];

    const int N = m.N;
    const uint32_t nt = (uint32_t)m.nTj;
    const int tk = (int)(t % nt), tj = (int)(t / nt % nt), ti = (int)(t / nt / nt);
    const int ck = (int)(threadIdx.x % SJ), cj = (int)(threadIdx.x / SJ % kCubeSide);
    const int ci = (int)(threadIdx.x / SI) * R;
    const int i0 = ti * TS, j0 = tj * TS, k0 = tk * TS;
    auto wrap = [N](int x) {                 // any side, also below the region's
        x %= N;
        return x < 0 ? x + N : x;
    };
    const uint32_t un = (uint32_t)N;
    const uint32_t col = (uint32_t)wrap(j0 - H + cj) * un + (uint32_t)wrap(k0 - H + ck);
    const bool inner = cj >= H && cj < H + TS && j0 + cj - H < N && ck >= H && ck < H + TS &&
                       k0 + ck - H < N;
    uint32_t q[R];
    typename Tr::Raw raw[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        q[r] = (uint32_t)wrap(i0 - H + ci + r) * un * un + col;
        Tr::fetch(form_in<Tr>(m.in), q[r], raw[r]);
    }
    const typename Tr::Vc vc = Tr::vconst(sc.s[0]);
    T x[R], y[R];
    typename Tr::Own own[R];
#pragma unroll
    for (int r = 0; r < R; ++r) Tr::drift0(raw[r], sc.s[0], x[r], y[r], own[r]);
    const int o = PAD + ci * SI + cj * SJ + ck;
    for (int l = 0; l < d; ++l) {
        const typename Tr::Sc &s = sc.s[l];
        const typename Tr::Sc &sn = sc.s[l + 1 < d ? l + 1 : l];
        // buffer l & 1 was last read two steps ago: every wave has passed a
        // barrier since
        T2 *B = X + (l & 1) * BUF;
#pragma unroll
        for (int r = 0; r < R; ++r) B[o + r * SI] = T2{x[r], y[r]};
        __syncthreads();
        T nx[R], ny[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            // a plane of the column, from the work-item's own where it holds it
            auto plane = [&](int rr) -> T2 {
                return (rr >= 0 && rr < R) ? T2{x[rr < 0 ? 0 : (rr < R ? rr : 0)],
                                                y[rr < 0 ? 0 : (rr < R ? rr : 0)]}
                                           : B[o + rr * SI];
            };
            const T2 *b = B + o + r * SI;
            // the 7-point stencil's coefficient is 1: its products are exact
            // and left out
            T a = Tr::centre(s, x[r]), c = Tr::centre(s, y[r]);
            auto add = [&](T2 v) {
                a = a + v.x;
                c = c + v.y;
            };
            add(plane(r + 1));
            add(plane(r - 1));
            add(b[SJ]);
            add(b[-SJ]);
            add(b[1]);
            add(b[-1]);
            typename Tr::Own on;
            Tr::level(x[r], y[r], a, c, own[r], s, sn, vc, on, nx[r], ny[r]);
            own[r] = on;
        }
        if (l + 1 < d) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                x[r] = nx[r];
                y[r] = ny[r];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int e = ci + r;
        if (inner && e >= H && e < H + TS && i0 + e - H < N)
            Tr::store(form_out<Tr>(m.out), q[r], x[r], y[r], own[r]);
    }
}

// one cube per work-group; a single lattice by value (no member table to read)
template <class Tr>
__global__ void __launch_bounds__(kCubeItems)
block3d_kernel(BatchMember one, int d, LevelScalars<typename Tr::Sc, kCubeDepth> sc)
{
    block3d_tile<Tr>(one, blockIdx.x, d, sc);
}

template <class Tr>
__global__ void __launch_bounds__(kCubeItems)
block3d_batch_kernel(const BatchMember *__restrict__ mem, int n_members, int d,
                     LevelScalars<typename Tr::Sc, kCubeDepth> sc)
{
    int lo = 0, hi = n_members - 1;            // last member starting at or before the cube
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (mem[mid].item_begin <= blockIdx.x)
            lo = mid;
        else
            hi = mid - 1;
    }
    const BatchMember &m = mem[lo];
    block3d_tile<Tr>(m, blockIdx.x - m.item_begin, d, sc);
}

// Runs where the marching kernels do not (a member with a side below 64), with
// the 7-point stencil, up to the launch limit (2^22 cubes).  In FP64 one group
// is resident per CU, so a pass takes as long as its rounds of one cube per CU,
// 4.1 us a step each, against about 6 us and 22 ps a site for the one-step
// kernel: the cubes run while that is less, and for four rounds at most (as far
// as was measured).  In us a step, cubes / one-step kernel: 48^3 4.2 / 8.2, two
// of 48^3 8.2 / 8.8, four (864 cubes) 16.1 / 15.6, 62^3 7.0 / 9.9, two 14.2 / 15.6,
// 37 of 24^3 16.5 / 17.5, but of 20^3, whose cubes are half empty, 14.4 / 12.0.
// In FP32 the one-step kernel is nowhere far ahead: 16^3 1.7 / 2.6, 62^3 3.0 /
// 6.0; forty of 32^3 11.3 / 13.4, 120 35.5 / 33.0, 480 121 / 138; of 62^3
// sixteen 38.1 / 35.1, 64 127 / 141; of 48^3 64 62.7 / 70.5; and a small member
// beside large ones 32 and 192 61 / 58, 32 and 200 73 / 82, 24 and 400 474 / 671.
// Wider stencils gain at most 1.2x (radius 2, 62^3) and lose up to 2x: not built.
int block3d_depth(const Context *c)
{
    if (c->nd != 3 || c->p.laplacian != AXS_LAPLACIAN_STENCIL || c->tune.configured ||
        stencil_radius_of(c) != 1)
        return 0;
    bool small = false;
    uint64_t cubes = 0, sites = 0;
    for (const Member &m : c->members) {
        small = small || !march2_supported(c, m.N);
        const uint64_t t = (uint64_t)((m.N + kCubeOut - 1) / kCubeOut);
        cubes += t * t * t;
        sites += (uint64_t)m.L;
    }
    if (!small || cubes * kCubeItems > kMaxGridItems) return 0;
    if (c->prec == AXS_FP64) {
        const uint64_t cus = (uint64_t)(c->num_cu > 0 ? c->num_cu : 1);
        const uint64_t rounds = (cubes + cus - 1) / cus;
        if (rounds > 4 || 4.1 * (double)rounds > 6.0 + 22e-6 * (double)sites) return 0;
    }
    return kCubeDepth;
}

int prepare_block3d(Context *c)
{
    return (c->blk.key == 3) ? AXS_OK : block_tables(c, kCubeOut, kCubeOut, 3);
}

template <class Tr>
static void launch_cubes(Context *c, int src, const StepScalars *s, int d)
{
    LevelScalars<typename Tr::Sc, kCubeDepth> sc{};
    for (int l = 0; l < d; ++l) {
        if constexpr (std::is_same<typename Tr::Sc, StepScalarsF>::value)
            sc.s[l] = to_float(s[l]);
        else
            sc.s[l] = s[l];
    }
    if (c->members.size() > 1)
        hipLaunchKernelGGL((block3d_batch_kernel<Tr>), dim3(c->blk.items), dim3(kCubeItems), 0,
                           c->stream, c->blk.tab[src], (int)c->members.size(), d, sc);
    else
        hipLaunchKernelGGL((block3d_kernel<Tr>), dim3(c->blk.items), dim3(kCubeItems), 0,
                           c->stream, c->blk_one[src], d, sc);
}

int launch_block3d(Context *c, const StepScalars *s, int d)
{
    const int src = c->cur;
    if (c->prec == AXS_FP32)
        launch_cubes<F32Form>(c, src, s, d);
    else if (c->p.eom == AXS_EOM_HAMILTONIAN)
        launch_cubes<F64FormT<true>>(c, src, s, d);
    else
        launch_cubes<F64FormT<false>>(c, src, s, d);
    AXS_HIP_TRY(hipGetLastError());
    c->cur = src ^ 1;
    return AXS_OK;
}

}  // namespace axs
