// Lookup of the compiled Stockham leaf kernels (generated instance tables).
#include <cstdlib>
#include <map>

#include "plan.h"

namespace sip {

#define SIP_STOCKHAM_PART(k)                                \
    extern const StockhamInstance g_stockham_part_##k[];    \
    extern const int g_stockham_part_##k##_count;
#include "stockham_parts.inc"
#undef SIP_STOCKHAM_PART

static const std::map<int64_t, const StockhamInstance *> &instances()
{
    static const std::map<int64_t, const StockhamInstance *> m = [] {
        std::map<int64_t, const StockhamInstance *> r;
#define SIP_STOCKHAM_PART(k)                                        \
    for (int i = 0; i < g_stockham_part_##k##_count; i++)           \
        r[g_stockham_part_##k[i].L] = &g_stockham_part_##k[i];
#include "stockham_parts.inc"
#undef SIP_STOCKHAM_PART
        return r;
    }();
    return m;
}

const StockhamInstance *find_instance(int64_t L)
{
    const auto &m = instances();
    auto it = m.find(L);
    return it == m.end() ? nullptr : it->second;
}

int64_t instance_count() { return (int64_t)instances().size(); }

extern const Stockham2dInstance g_stockham2d[9];
extern const Stockham2dInstance g_stockham2d_planes[1];

const Stockham2dInstance *find_2d_instance(int64_t X, int64_t Y)
{
    // tuning switch: the two-plane tile of 128 x 128 slices
    if (X == 128 && Y == 128) {
        const char *e = std::getenv("SIP_FFT_TILE2D_SPLIT");
        if (e && std::atoi(e) == 0) return &g_stockham2d_planes[0];
    }
    for (const Stockham2dInstance &t : g_stockham2d)
        if (t.X == X && t.Y == Y) return &t;
    return nullptr;
}

extern const BluesteinInstance g_bluestein[];
extern const int g_bluestein_count;

const BluesteinInstance *find_bluestein_instance(int64_t min_m)
{
    for (int i = 0; i < g_bluestein_count; i++)  // ascending M
        if (g_bluestein[i].M >= min_m) return &g_bluestein[i];
    return nullptr;
}

#define SIP_ROLE_PART(name)                   \
    extern const RoleInstance g_##name[];     \
    extern const int g_##name##_count;
#include "role_parts.inc"
#undef SIP_ROLE_PART

const RoleInstance *find_role(Role role, int64_t L)
{
    static const auto m = [] {
        std::map<std::pair<int, int64_t>, const RoleInstance *> r;
#define SIP_ROLE_PART(name) \
    for (int i = 0; i < g_##name##_count; i++) r[{g_##name[i].role, g_##name[i].inst.L}] = &g_##name[i];
#include "role_parts.inc"
#undef SIP_ROLE_PART
        return r;
    }();
    auto it = m.find({role, L});
    return it == m.end() ? nullptr : it->second;
}

const char *kernel_set()
{
    return
#include "kernel_set.inc"
        ;
}

std::pair<int, int> split_rates(int64_t L)
{
    static const std::map<int64_t, std::pair<int, int>> m = {
#include "split_rates.inc"
    };
    auto it = m.find(L);
    return it == m.end() ? std::pair<int, int>{0, 0} : it->second;
}

#define SIP_ISTFT_PART(k)                            \
    extern const IstftInstance g_istft_part_##k[];   \
    extern const int g_istft_part_##k##_count;
#include "istft_parts.inc"
#undef SIP_ISTFT_PART

const IstftInstance *find_istft_instance(int64_t n)
{
#define SIP_ISTFT_PART(k)                                 \
    for (int i = 0; i < g_istft_part_##k##_count; i++)    \
        if (g_istft_part_##k[i].L == n) return &g_istft_part_##k[i];
#include "istft_parts.inc"
#undef SIP_ISTFT_PART
    return nullptr;
}

}  // namespace sip
