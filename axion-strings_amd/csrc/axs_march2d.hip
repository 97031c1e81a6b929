// axs_march2d.hip -- the 2D multi-step kernels (axs_march2d.hpp) for the
// 5-point stencil in the FP32 form and the bit-exact FP64 form
// (field-rescaled or Hamiltonian), and the 2D work lists.  Radii 2-4
// (stencil_setting 1-3) are instantiated in axs_march2d_hi.hip.
#include "axs_march2d.hpp"

namespace axs {

bool march2d_supported(const Context *c, int N)
{
    return c->nd == 2 && c->p.laplacian == AXS_LAPLACIAN_STENCIL && N >= kW2;
}

// radius 1: 2, 3, 4, 6 or 8 steps per pass; radii 2-4: 1-4 steps (FP32),
// 1-2 steps (FP64: the register rings grow with the radius)
bool march2d_depth_built(int D, int RAD, int prec)
{
    if (RAD == 1) return D == 2 || D == 3 || D == 4 || D == 6 || D == 8;
    if (RAD > 4) return false;
    return D >= 1 && D <= ((prec == AXS_FP64) ? 2 : 4);
}

// Rows per chunk, unless configured, by a cost model.  A wave marches chunk +
// 2H rows (H = halo); w = waves per SIMD share its issue, and a wave alone
// leaves a SIMD idle for the row's dependent chain and its loads.  A pass
// takes about (w + b) (chunk + 2H), b = 3 in FP32 and 1 in FP64 (whose rows
// fill the issue): fitted to chunks 8..128 at sides 720..2048 and 4096, where
// it is within 10% of the best chunk measured.  It keeps 128 for the
// 512-lattice ensemble and 32 (FP32) / 64 (FP64) at 4096^2; at 1000^2 it
// takes 10-row chunks (FP64 depth 6: 46 -> 40 us a pass; FP64 second order,
// depth 2: 35 -> 28 us; FP32 22 -> 16 us), where 32 rows left half the SIMDs
// without a wave.
static int pick_cap(const Context *c, int TI, int H)
{
    const double simds = 4.0 * (c->num_cu > 0 ? c->num_cu : 1);
    const double b = (c->prec == AXS_FP32) ? 3.0 : 1.0;
    int best = 8;
    double best_cost = 1e300;
    for (int cap = 128; cap >= 8; cap >>= 1) {
        double waves = 0.0;
        for (const Member &m : c->members)
            waves += (double)((m.N + TI - 1) / TI) * (double)((m.N + cap - 1) / cap);
        const double cost = (waves / simds + b) * (double)(cap + 2 * H);
        if (cost < best_cost) {
            best_cost = cost;
            best = cap;
        }
    }
    return best;
}

int prepare_march2d_items(Context *c, int D)
{
    if (D < 1) return AXS_OK;
    Context::MultiTables &mt = c->mtab[D];
    const int RAD = stencil_radius_of(c);
    const int key = ((D * 10 + RAD) * 100 + 2) * 10000 + c->tune.ci32;
    if (key == mt.key && mt.tab[0]) return AXS_OK;
    const int TI = kW2 - 2 * D * RAD;
    const int cap = pick_cap(c, TI, D * RAD);
    std::vector<BatchMember> tab[2];
    uint32_t items = 0;
    for (const Member &m : c->members) {
        BatchMember b{};
        b.N = m.N;
        b.L = (uint32_t)m.L;
        b.item_begin = items;
        b.nTj = (m.N + TI - 1) / TI;       // strips
        b.nTk = 1;
        const int cfg = c->tune.ci32;      // rows per chunk
        b.CI = (cfg > 0 && m.N % cfg == 0) ? cfg : equal_chunk(m.N, cap);   // last one shorter
        items += (uint32_t)b.nTj * (uint32_t)((m.N + b.CI - 1) / b.CI);
        for (int h = 0; h < 2; ++h) {
            for (int a = 0; a < 3; ++a) {
                b.in[a] = m.state[h][a];
                b.out[a] = m.state[h ^ 1][a];
            }
            tab[h].push_back(b);
        }
    }
    for (int h = 0; h < 2; ++h) {
        if (!mt.tab[h])
            AXS_HIP_TRY(hipMalloc(&mt.tab[h], c->members.size() * sizeof(BatchMember)));
        AXS_HIP_TRY(hipMemcpyAsync(mt.tab[h], tab[h].data(),
                                   tab[h].size() * sizeof(BatchMember), hipMemcpyHostToDevice,
                                   c->stream));
    }
    AXS_HIP_TRY(hipStreamSynchronize(c->stream));
    mt.items = items;
    mt.key = key;
    return AXS_OK;
}

template <class Tr>
static int launch_form2d(Context *c, int src, const StepScalars *s, int depth, bool pf)
{
    switch (depth) {
    case 2: return launch_march2d_pass<Tr, 2, 1>(c, src, s, pf);
    case 3: return launch_march2d_pass<Tr, 3, 1>(c, src, s, pf);
    case 4: return launch_march2d_pass<Tr, 4, 1>(c, src, s, pf);
    case 6: return launch_march2d_pass<Tr, 6, 1>(c, src, s, pf);
    case 8: return launch_march2d_pass<Tr, 8, 1>(c, src, s, pf);
    default:
        set_error("2D depth %d is not built", depth);
        return AXS_ERR_UNSUPPORTED;
    }
}

int launch_march2d(Context *c, int src, const StepScalars *s, int depth)
{
    if (depth < 1 || depth > kMaxDepth || !c->mtab[depth].tab[src]) {
        set_error("2D multi-step work list missing");
        return AXS_ERR_STATE;
    }
    const bool pf = (c->tune.flags & kTunePrefetch) != 0;
    if (stencil_radius_of(c) > 1) return launch_march2d_high_order(c, src, s, depth, pf);
    if (c->prec == AXS_FP32) return launch_form2d<F32Form>(c, src, s, depth, pf);
    if (c->p.eom == AXS_EOM_HAMILTONIAN) return launch_form2d<F64FormT<true>>(c, src, s, depth, pf);
    return launch_form2d<F64FormT<false>>(c, src, s, depth, pf);
}

}  // namespace axs
