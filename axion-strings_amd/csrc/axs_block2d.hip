// axs_block2d.hip -- several steps per pass on small 2D lattices: one
// work-group per square block of sites, every site of the block in flight.
//
// The strip kernels (axs_march2d.hpp) march a wave along j, so a pass takes
// as long as one wave's chain of rows however small the lattice is.  Here a
// work-group of 1024 work-items loads a 32 x 32 region, one site each, and
// advances it d steps: the drifted field sits in LDS (two buffers, one
// barrier per step), the site's own velocity and force in registers.  A step
// makes the outermost RAD columns and rows of the region invalid, so the
// inner (32 - 2 H)^2 sites, H = D RAD, are written.  Once the blocks no
// longer fit the chip at once, a work-item holds two rows (32 x 64 regions).
//
// What bounds it: on the smallest lattices the launch, load and store around
// the steps (2D 256^2 FP64: 8.7 us for a pass of six, where the strips took
// 43); on larger ones the FP64 issue of the 16 waves, of which the inner
// block's share is (20/32)^2 at one row per work-item and 20/32 52/64 at two.
//
// The sums run in the one-step kernels' order with the forms' expressions,
// so a pass is bit-identical to d one-step launches.
#include "axs_forms.hpp"
#include "axs_internal.hpp"
#include "axs_lattice.hpp"

#include <type_traits>

namespace axs {

constexpr int kBlkSide = 32;                        // region side (sites)
constexpr int kBlkItems = kBlkSide * kBlkSide;      // work-items of a group

// most steps of a pass by stencil radius: a halo of six or eight sites
constexpr int blk_depth(int RAD) { return RAD == 1 ? 6 : 8 / RAD; }
constexpr int blk_cols(int RAD) { return kBlkSide - 2 * blk_depth(RAD) * RAD; }
constexpr int blk_rows(int RAD, int R) { return kBlkSide * R - 2 * blk_depth(RAD) * RAD; }

// d <= blk_depth(RAD) steps of block `t` of lattice m; R consecutive rows per
// work-item, a region of 32 columns and 32 R rows
template <class Tr, int RAD, int R>
__device__ __forceinline__ void block2d_tile(const BatchMember &m, const uint32_t t, const int d,
                                             const LevelScalars<typename Tr::Sc, kMaxDepth> &sc)
{
    using T = typename Tr::T;
    typedef T T2 __attribute__((ext_vector_type(2)));
    constexpr int H = blk_depth(RAD) * RAD, TI = blk_cols(RAD), TJ = blk_rows(RAD, R);
    // the rim sites' neighbour reads stay inside the array (their values
    // reach no written site)
    constexpr int PAD = RAD * kBlkSide + RAD;
    __shared__ T2 X[2][kBlkItems * R + 2 * PAD];

    const int N = m.N;
    const int ti = (int)(t % (uint32_t)m.nTk), tj = (int)(t / (uint32_t)m.nTk);
    const int ci = (int)(threadIdx.x % kBlkSide), cj = (int)(threadIdx.x / kBlkSide) * R;
    const int i0 = ti * TI, j0 = tj * TJ;
    auto wrap = [N](int x) {                 // any side, also below the region's
        x %= N;
        return x < 0 ? x + N : x;
    };
    const uint32_t qi = (uint32_t)wrap(i0 - H + ci);
    const bool icol = ci >= H && ci < H + TI && i0 + ci - H < N;
    uint32_t q[R];
    typename Tr::Raw raw[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        q[r] = (uint32_t)wrap(j0 - H + cj + r) * (uint32_t)N + qi;
        Tr::fetch(form_in<Tr>(m.in), q[r], raw[r]);
    }
    const typename Tr::Vc vc = Tr::vconst(sc.s[0]);
    T x[R], y[R];
    typename Tr::Own own[R];
#pragma unroll
    for (int r = 0; r < R; ++r) Tr::drift0(raw[r], sc.s[0], x[r], y[r], own[r]);
    const int o = PAD + cj * kBlkSide + ci;
    for (int l = 0; l < d; ++l) {
        const typename Tr::Sc &s = sc.s[l];
        const typename Tr::Sc &sn = sc.s[l + 1 < d ? l + 1 : l];
        // buffer l & 1 was last read two steps ago: every wave has passed a
        // barrier since
        T2 *B = X[l & 1];
#pragma unroll
        for (int r = 0; r < R; ++r) B[o + r * kBlkSide] = T2{x[r], y[r]};
        __syncthreads();
        T nx[R], ny[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            // a row of the column, from the work-item's own rows where it holds it
            auto row = [&](int rr) -> T2 {
                return (rr >= 0 && rr < R) ? T2{x[rr < 0 ? 0 : (rr < R ? rr : 0)],
                                                y[rr < 0 ? 0 : (rr < R ? rr : 0)]}
                                           : B[o + rr * kBlkSide];
            };
            T a = Tr::centre(s, x[r]), c = Tr::centre(s, y[r]);
#pragma unroll
            for (int e = 1; e <= RAD; ++e) {
                // the 5-point stencil's coefficient is 1: its products are
                // exact and left out
                const T cm = (T)s.c[e];
                auto add = [&](T2 v) {
                    a = (RAD == 1) ? a + v.x : Tr::acc(a, cm, v.x);
                    c = (RAD == 1) ? c + v.y : Tr::acc(c, cm, v.y);
                };
                const T2 ip = B[o + r * kBlkSide + e], im = B[o + r * kBlkSide - e];
                const T2 jp = row(r + e), jm = row(r - e);
                if constexpr (std::is_same<T, float>::value) {
                    add(jp);                 // the FP32 form's order: j, then i
                    add(jm);
                    add(ip);
                    add(im);
                } else {
                    add(ip);                 // FP64: the reference's COO order
                    add(im);
                    add(jp);
                    add(jm);
                }
            }
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
        const int e = cj + r;
        if (icol && e >= H && e < H + TJ && j0 + e - H < N)
            Tr::store(form_out<Tr>(m.out), q[r], x[r], y[r], own[r]);
    }
}

// one block per work-group.  A single lattice comes by value: the member
// table would cost a chain of loads before the first site is fetched
template <class Tr, int RAD, int R>
__global__ void __launch_bounds__(kBlkItems)
block2d_kernel(BatchMember one, int d, LevelScalars<typename Tr::Sc, kMaxDepth> sc)
{
    block2d_tile<Tr, RAD, R>(one, blockIdx.x, d, sc);
}

template <class Tr, int RAD, int R>
__global__ void __launch_bounds__(kBlkItems)
block2d_batch_kernel(const BatchMember *__restrict__ mem, int n_members, int d,
                     LevelScalars<typename Tr::Sc, kMaxDepth> sc)
{
    int lo = 0, hi = n_members - 1;            // last member starting at or before the block
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (mem[mid].item_begin <= blockIdx.x)
            lo = mid;
        else
            hi = mid - 1;
    }
    const BatchMember &m = mem[lo];
    block2d_tile<Tr, RAD, R>(m, blockIdx.x - m.item_begin, d, sc);
}

static uint64_t block2d_tiles(const Context *c, int R)
{
    const int RAD = stencil_radius_of(c);
    uint64_t n = 0;
    for (const Member &m : c->members)
        n += (uint64_t)((m.N + blk_cols(RAD) - 1) / blk_cols(RAD)) *
             (uint64_t)((m.N + blk_rows(RAD, R) - 1) / blk_rows(RAD, R));
    return n;
}

// Rows per work-item: one while the blocks fit the chip at once (two groups of
// 1024 work-items are resident per CU), else two, which halve the region's
// height overhead: FP64 1000^2 6.8 -> 5.9 us a step, fourth order 13.6 -> 10.1;
// FP32 3.7 -> 2.7.  FP64 radius 3 and 4 keep one (two rows of their sums leave
// one group per CU: 17.3 against 19.1 us at 1000^2, radius 3).
constexpr bool two_rows_built(bool f64, int RAD) { return !f64 || RAD <= 2; }
static int block2d_rows(const Context *c)
{
    if (!two_rows_built(c->prec == AXS_FP64, stencil_radius_of(c))) return 1;
    return block2d_tiles(c, 1) <= 2 * (uint64_t)c->num_cu ? 1 : 2;
}

// Where the blocks run: everywhere the strips cannot (a side below 64, where
// the alternative is one launch a step), and up to the number of sites where
// the strips catch up.  Measured in us a step, blocks against the best strips
// chunk: FP64 256^2 1.5 / 3.5, 1000^2 5.9 / 6.6, 2048^2 18.3 / 21.8 (4096^2:
// strips); fourth order 256^2 1.9 / 5.9, 1000^2 10.1 / 13.8, 2048^2 33.6 / 47.4
// and the strips never catch up (8.0 against 10.0 ps a site at 4096^2, whose
// two-step passes the register rings limit); radius 3 1000^2 17.3 / 18.0;
// radius 4 720^2 12.9 / 15.0, 1000^2 22.3 / 22.1; FP32 1440^2 4.28 / 4.40,
// 2048^2 7.6 / 6.9 (radius 2-4 the same line within 2%).
int block2d_depth(const Context *c)
{
    if (c->nd != 2 || c->p.laplacian != AXS_LAPLACIAN_STENCIL || c->tune.configured) return 0;
    const int RAD = stencil_radius_of(c);
    bool strips = true;
    int64_t sites = 0;
    for (const Member &m : c->members) {
        strips = strips && march2d_supported(c, m.N);
        sites += m.L;
    }
    if (strips) {
        int64_t most;
        if (c->prec == AXS_FP32)
            most = (int64_t)1 << 21;
        else
            most = (RAD == 1) ? (int64_t)1 << 22 : (RAD == 2) ? INT64_MAX : (int64_t)1 << 20;
        if (sites > most) return 0;
    }
    // the grid: one group per block
    if (block2d_tiles(c, block2d_rows(c)) * kBlkItems > kMaxGridItems) return 0;
    return blk_depth(RAD);
}

// member tables of the block kernels, for blocks of TI columns and TJ rows (2D)
// or TI^3 sites (3D)
int block_tables(Context *c, int TI, int TJ, int key)
{
    Context::MultiTables &mt = c->blk;
    std::vector<BatchMember> tab[2];
    uint32_t items = 0;
    for (const Member &m : c->members) {
        BatchMember b{};
        b.N = m.N;
        b.L = (uint32_t)m.L;
        b.item_begin = items;
        b.nTj = (m.N + TJ - 1) / TJ;
        b.nTk = (m.N + TI - 1) / TI;
        items += (uint32_t)b.nTj * (uint32_t)b.nTk * (c->nd == 3 ? (uint32_t)b.nTj : 1u);
        for (int h = 0; h < 2; ++h) {
            for (int a = 0; a < 3; ++a) {
                b.in[a] = m.state[h][a];
                b.out[a] = m.state[h ^ 1][a];
            }
            tab[h].push_back(b);
        }
    }
    for (int h = 0; h < 2; ++h) {
        c->blk_one[h] = tab[h][0];
        if (c->members.size() < 2) continue;
        if (!mt.tab[h])
            AXS_HIP_TRY(hipMalloc(&mt.tab[h], c->members.size() * sizeof(BatchMember)));
        AXS_HIP_TRY(hipMemcpyAsync(mt.tab[h], tab[h].data(),
                                   tab[h].size() * sizeof(BatchMember), hipMemcpyHostToDevice,
                                   c->stream));
    }
    if (c->members.size() > 1) AXS_HIP_TRY(hipStreamSynchronize(c->stream));
    mt.items = items;
    mt.key = key;
    return AXS_OK;
}

int prepare_block2d(Context *c)
{
    const int RAD = stencil_radius_of(c), R = block2d_rows(c);
    if (c->blk.key == R) return AXS_OK;
    return block_tables(c, blk_cols(RAD), blk_rows(RAD, R), R);
}

int block_depth(const Context *c)
{
    return (c->nd == 2) ? block2d_depth(c) : block3d_depth(c);
}

int prepare_blocks(Context *c)
{
    return (c->nd == 2) ? prepare_block2d(c) : prepare_block3d(c);
}

int launch_blocks(Context *c, const StepScalars *s, int d)
{
    return (c->nd == 2) ? launch_block2d(c, s, d) : launch_block3d(c, s, d);
}

template <class Tr, int RAD, int R>
static void launch_rows(Context *c, int src, const LevelScalars<typename Tr::Sc, kMaxDepth> &sc,
                        int d)
{
    if (c->members.size() > 1)
        hipLaunchKernelGGL((block2d_batch_kernel<Tr, RAD, R>), dim3(c->blk.items),
                           dim3(kBlkItems), 0, c->stream, c->blk.tab[src],
                           (int)c->members.size(), d, sc);
    else
        hipLaunchKernelGGL((block2d_kernel<Tr, RAD, R>), dim3(c->blk.items), dim3(kBlkItems), 0,
                           c->stream, c->blk_one[src], d, sc);
}

template <class Tr, int RAD>
static void launch_rad(Context *c, int src, const StepScalars *s, int d)
{
    LevelScalars<typename Tr::Sc, kMaxDepth> sc{};
    for (int l = 0; l < d; ++l) {
        if constexpr (std::is_same<typename Tr::Sc, StepScalarsF>::value)
            sc.s[l] = to_float(s[l]);
        else
            sc.s[l] = s[l];
    }
    if constexpr (two_rows_built(!std::is_same<Tr, F32Form>::value, RAD))
        if (c->blk.key == 2) return launch_rows<Tr, RAD, 2>(c, src, sc, d);
    launch_rows<Tr, RAD, 1>(c, src, sc, d);
}

template <class Tr>
static void launch_form(Context *c, int src, const StepScalars *s, int d)
{
    switch (stencil_radius_of(c)) {
    case 1: return launch_rad<Tr, 1>(c, src, s, d);
    case 2: return launch_rad<Tr, 2>(c, src, s, d);
    case 3: return launch_rad<Tr, 3>(c, src, s, d);
    default: return launch_rad<Tr, 4>(c, src, s, d);
    }
}

int launch_block2d(Context *c, const StepScalars *s, int d)
{
    const int src = c->cur;
    if (c->prec == AXS_FP32)
        launch_form<F32Form>(c, src, s, d);
    else if (c->p.eom == AXS_EOM_HAMILTONIAN)
        launch_form<F64FormT<true>>(c, src, s, d);
    else
        launch_form<F64FormT<false>>(c, src, s, d);
    AXS_HIP_TRY(hipGetLastError());
    c->cur = src ^ 1;
    return AXS_OK;
}

}  // namespace axs
