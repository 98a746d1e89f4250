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

// bit d of links: a link along d, as the kernels see it, which read the distances in FP32 (1 + 1e-9 is a
// link there)
struct DistanceList {
    uint32_t n;
    const int32_t* k;
    const double* q;
    uint32_t links(uint32_t i) const
    {
        uint32_t m = 0;
        for (int d = 1; d < 27; ++d) {
            const float v = (float)q[(uint64_t)d * n + i];
            m |= (v >= 0.0f && v <= 1.0f ? 1u : 0u) << d;
        }
        return m;
    }
};
struct LinkList {
    uint32_t n;
    const int32_t* k;
    const uint32_t* q;
    uint32_t links(uint32_t i) const { return q[i] & ~1u; }
};

// The shorter list's nodes (a) in a hash table, and the x, y and z planes that hold any of them; only
// nodes of the other list beside such planes (an inflow face: the walls' rim) look their
// neighbourhood up. Memory and time follow the lists, not the box: two opposite faces of 384^3 and its
// walls (874 000 nodes) 231 -> 14 ms and no 230 MB table.
template <class List> bool lists_independent(const int32_t (&size)[3], List a, List b)
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
    int bits = 4;
    while ((1ull << bits) < 2ull * a.n) ++bits;
    const uint32_t mask = (uint32_t)((1ull << bits) - 1);
    const auto hash = [bits](int32_t k) { return (uint32_t)(((uint64_t)(uint32_t)k * 0x9e3779b97f4a7c15ull) >> (64 - bits)); };
    std::vector<uint32_t> table((size_t)mask + 1, 0); // index + 1 in a
    std::vector<uint8_t> held[3], beside[3];          // planes that hold nodes of a; those and the ones beside
    for (int x = 0; x < 3; ++x) held[x].assign(size[x], 0);
    int32_t c[3] = {};
    for (uint32_t i = 0; i < a.n; ++i) {
        coordinates(a.k[i], c);
        for (int x = 0; x < 3; ++x) held[x][c[x]] = 1;
        uint32_t h = hash(a.k[i]);
        while (table[h]) h = (h + 1) & mask;
        table[h] = i + 1;
    }
    const auto wrapped = [&size](int x, int32_t v) { return v < 0 ? size[x] - 1 : v >= size[x] ? 0 : v; };
    for (int x = 0; x < 3; ++x) {
        beside[x] = held[x];
        for (int32_t v = 0; v < size[x]; ++v)
            if (held[x][wrapped(x, v - 1)] || held[x][wrapped(x, v + 1)]) beside[x][v] = 1;
    }
    for (uint32_t i = 0; i < b.n; ++i) {
        coordinates(b.k[i], c);
        if (!beside[0][c[0]] || !beside[1][c[1]] || !beside[2][c[2]]) continue;
        const uint32_t links = b.links(i);
        for (int d = 0; d < 27; ++d) {
            const int32_t v[3] = {wrapped(0, c[0] + vfa::cx(d)), wrapped(1, c[1] + vfa::cy(d)), wrapped(2, c[2] + vfa::cz(d))};
            if (!held[0][v[0]] || !held[1][v[1]] || !held[2][v[2]]) continue;
            const int32_t k = v[0] + size[0] * (v[1] + size[1] * v[2]);
            for (uint32_t h = hash(k); table[h]; h = (h + 1) & mask) {
                const uint32_t j = table[h] - 1;
                if (a.k[j] != k) continue;
                // a link in common, or one of either that leads to the other's node
                if (d == 0 ? (links & a.links(j)) != 0 : (links >> d & 1u) || (a.links(j) >> vfa::inv(d) & 1u)) return false;
            }
        }
    }
    return true;
}

template <class List>
int independent_in_box(int32_t nx, int32_t ny, int32_t nz, const List& a, const List& b, int32_t* independent)
{
    using namespace vfa;
    const int64_t nodes = nx > 0 && ny > 0 && nz > 0 ? (int64_t)nx * ny * nz : 0;
    const auto valid = [&](const List& l) {
        return l.n == 0 || (l.k && l.q && std::all_of(l.k, l.k + l.n, [&](int32_t v) { return v >= 0 && v < nodes; }));
    };
    if (nodes == 0 || nodes > INT32_MAX || !independent || !valid(a) || !valid(b)) {
        set_last_error("bc lists independent: missing arrays or a node outside the box");
        return VF_ERR_INVALID_ARGUMENT;
    }
    *independent = 1;
    if (a.n == 0 || b.n == 0) return VF_OK;
    try {
        *independent = lists_independent({nx, ny, nz}, a, b) ? 1 : 0;
    } catch (const std::bad_alloc&) {
        *independent = 0; // not found out: the lists keep their launches
    }
    return VF_OK;
}

} // namespace

extern "C" int vf_bc_lists_independent(int32_t nx, int32_t ny, int32_t nz, uint32_t na, const int32_t* ka,
                                       const double* qa, uint32_t nb, const int32_t* kb, const double* qb,
                                       int32_t* independent)
{
    return independent_in_box(nx, ny, nz, DistanceList{na, ka, qa}, DistanceList{nb, kb, qb}, independent);
}

extern "C" int vf_bc_links_independent(int32_t nx, int32_t ny, int32_t nz, uint32_t na, const int32_t* ka,
                                       const uint32_t* linksA, uint32_t nb, const int32_t* kb, const uint32_t* linksB,
                                       int32_t* independent)
{
    return independent_in_box(nx, ny, nz, LinkList{na, ka, linksA}, LinkList{nb, kb, linksB}, independent);
}
