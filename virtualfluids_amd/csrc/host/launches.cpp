// Sequences of launches: the entry points of a time step enqueued from a native loop.
#include "../vf_common.h"

#include <algorithm>
#include <cstdint>
#include <new>
#include <utility>
#include <vector>

extern "C" int vf_run_launches(const vf_launch* list, uint32_t n, uint32_t repeats, void* stream)
{
    using namespace vfa;
    if (n && !list) {
        set_last_error("run_launches: null list");
        return VF_ERR_INVALID_ARGUMENT;
    }
    for (uint32_t i = 0; i < n; ++i) {
        const vf_launch& l = list[i];
        const bool scaling = l.kind == VF_LAUNCH_COARSE_TO_FINE || l.kind == VF_LAUNCH_FINE_TO_COARSE;
        if (l.kind < VF_LAUNCH_BOX || l.kind > VF_LAUNCH_FINE_TO_COARSE || !l.level ||
            (l.kind == VF_LAUNCH_BC && !l.bc && !l.pair) || (scaling && !l.fine)) {
            set_last_error("run_launches: an entry of unknown kind, without a level, a launcher or a fine level");
            return VF_ERR_INVALID_ARGUMENT;
        }
    }
    for (uint32_t r = 0; r < repeats; ++r) {
        for (uint32_t i = 0; i < n; ++i) {
            const vf_launch& l = list[i];
            int rc = VF_OK;
            switch (l.kind) {
            case VF_LAUNCH_BOX: rc = vf_k17_run_box(l.level, l.collisionTemplate, stream); break;
            case VF_LAUNCH_BOX_BOUNCE_BACK:
                rc = vf_k17_run_box_bounce_back(l.level, l.collisionTemplate, l.bounceBack, stream);
                break;
            case VF_LAUNCH_INDICES:
                rc = vf_k17_run_on_indices(l.level, l.level->fluidNodeIndices, l.level->numberOfFluidNodes,
                                           l.collisionTemplate, stream);
                break;
            case VF_LAUNCH_BC: rc = l.pair ? l.pair(l.level, l.list, l.list2, stream) : l.bc(l.level, l.list, stream); break;
            case VF_LAUNCH_SWAP: l.level->isEvenTimestep = l.level->isEvenTimestep ? 0 : 1; break;
            case VF_LAUNCH_COARSE_TO_FINE:
                rc = vf_ScaleCoarseToFineCompressible(l.level, l.fine, l.cells, l.offsets, stream);
                break;
            default: rc = vf_ScaleFineToCoarseCompressible(l.level, l.fine, l.cells, l.offsets, stream); break;
            }
            if (rc != VF_OK) return rc;
        }
    }
    return VF_OK;
}

namespace {

struct HostList {
    uint32_t n;
    const int32_t* k;
    const double* q;
    const double* at(int d, uint32_t i) const { return q + (uint64_t)d * n + i; }
    // as the kernels see it, which read the distances in FP32 (1 + 1e-9 is a link there)
    static bool link(const double* v) { const float q = (float)*v; return q >= 0.0f && q <= 1.0f; }
};

// The shorter list's nodes (a) in a table over their extent; only nodes of the other within a node
// of that extent (an inflow face: the walls' rim) look their neighbourhood up.
bool lists_independent(const int32_t (&size)[3], HostList a, HostList b)
{
    if (a.n > b.n) std::swap(a, b);
    // the coordinates of node k; c holds those of node `last` (lists run along x for the most part)
    int32_t last = -2;
    const auto coordinates = [nx = size[0], ny = size[1], &last](int32_t k, int32_t (&c)[3]) {
        if (k == last + 1 && c[0] + 1 < nx) {
            ++c[0];
        } else {
            const int32_t t = k / nx;
            c[2] = t / ny;
            c[0] = k - t * nx;
            c[1] = t - c[2] * ny;
        }
        last = k;
    };
    int32_t c[3] = {}, lo[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, hi[3] = {-1, -1, -1};
    for (uint32_t i = 0; i < a.n; ++i) {
        coordinates(a.k[i], c);
        for (int x = 0; x < 3; ++x) {
            lo[x] = std::min(lo[x], c[x]);
            hi[x] = std::max(hi[x], c[x]);
        }
    }
    const int64_t ex = hi[0] - lo[0] + 1, ey = hi[1] - lo[1] + 1, ez = hi[2] - lo[2] + 1;
    std::vector<uint32_t> table((size_t)(ex * ey * ez), 0); // index + 1 in a
    const auto place = [&](const int32_t (&v)[3]) {
        return (size_t)(v[0] - lo[0] + ex * (v[1] - lo[1] + ey * (v[2] - lo[2])));
    };
    for (uint32_t i = 0; i < a.n; ++i) {
        coordinates(a.k[i], c);
        table[place(c)] = i + 1;
    }
    // lowest and highest coordinate beside the extent; a box that wraps around has others as well
    const auto beside = [&](int x, int32_t v) {
        return (v >= lo[x] - 1 && v <= hi[x] + 1) || (lo[x] == 0 && v == size[x] - 1) || (hi[x] == size[x] - 1 && v == 0);
    };
    // the distances to look at lie a cache line apart each: fetched ahead, tested afterwards
    std::vector<const double*> alone;                          // no link may be here
    std::vector<std::pair<const double*, const double*>> both; // not both may be links
    const auto fetch = [](const double* v) {
        __builtin_prefetch(v);
        return v;
    };
    for (uint32_t i = 0; i < b.n; ++i) {
        coordinates(b.k[i], c);
        if (!beside(0, c[0]) || !beside(1, c[1]) || !beside(2, c[2])) continue;
        for (int d = 0; d < 27; ++d) {
            int32_t v[3] = {c[0] + vfa::cx(d), c[1] + vfa::cy(d), c[2] + vfa::cz(d)};
            bool in = true;
            for (int x = 0; x < 3; ++x) {
                v[x] = v[x] < 0 ? size[x] - 1 : v[x] >= size[x] ? 0 : v[x];
                in = in && v[x] >= lo[x] && v[x] <= hi[x];
            }
            const uint32_t j = in ? table[place(v)] : 0;
            if (j == 0) continue;
            if (d == 0) {
                for (int e = 1; e < 27; ++e) both.emplace_back(fetch(a.at(e, j - 1)), fetch(b.at(e, i)));
            } else {
                alone.push_back(fetch(b.at(d, i)));
                alone.push_back(fetch(a.at(vfa::inv(d), j - 1)));
            }
        }
    }
    return std::none_of(alone.begin(), alone.end(), HostList::link) &&
           std::none_of(both.begin(), both.end(),
                        [](const auto& p) { return HostList::link(p.first) && HostList::link(p.second); });
}

} // namespace

extern "C" int vf_bc_lists_independent(int32_t nx, int32_t ny, int32_t nz, uint32_t na, const int32_t* ka,
                                       const double* qa, uint32_t nb, const int32_t* kb, const double* qb,
                                       int32_t* independent)
{
    using namespace vfa;
    const int64_t nodes = nx > 0 && ny > 0 && nz > 0 ? (int64_t)nx * ny * nz : 0;
    const auto inside = [&](uint32_t n, const int32_t* k) {
        return std::all_of(k, k + n, [&](int32_t v) { return v >= 0 && v < nodes; });
    };
    if (nodes == 0 || nodes > INT32_MAX || !independent || (na && (!ka || !qa)) || (nb && (!kb || !qb)) || !inside(na, ka) ||
        !inside(nb, kb)) {
        set_last_error("bc_lists_independent: missing arrays or a node outside the box");
        return VF_ERR_INVALID_ARGUMENT;
    }
    *independent = 1;
    if (na == 0 || nb == 0) return VF_OK;
    try {
        *independent = lists_independent({nx, ny, nz}, {na, ka, qa}, {nb, kb, qb}) ? 1 : 0;
        return VF_OK;
    } catch (const std::bad_alloc&) {
        set_last_error("bc_lists_independent: out of memory");
        return VF_ERR_INVALID_ARGUMENT;
    }
}
