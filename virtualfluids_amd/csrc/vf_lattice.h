// Device helpers shared by the boundary, initialisation and output kernels:
// cell-node lookup (neighbour arrays or dense periodic box) and esoteric-twist
// reads/writes with a runtime parity flag.
#pragma once

#include "vf_common.h"

namespace vfa {

#define VF_PLANE_HD __host__ __device__ __forceinline__

struct Addr {
    uint64_t N;
    const uint32_t* nbx; // +x/+y/+z neighbour arrays (sparse grids)
    const uint32_t* nby;
    const uint32_t* nbz;
    int nx, ny, nz; // dense periodic box when nbx == nullptr
};

inline Addr make_addr(const vf_lbm_parameter& p)
{
    return Addr{p.numberOfNodes, p.neighborX, p.neighborY, p.neighborZ, p.nx, p.ny, p.nz};
}

// The 8 nodes of the cell at k: bit0 = +x, bit1 = +y, bit2 = +z
// (ListIndices, src/gpu/core/Utilities/KernelUtilities.h:221-245).
__device__ __forceinline__ void cell_nodes(const Addr& a, uint32_t k, uint32_t (&n)[8])
{
    if (a.nbx) {
        n[0] = k;
        n[1] = a.nbx[k];
        n[2] = a.nby[k];
        n[4] = a.nbz[k];
        n[3] = a.nby[n[1]];
        n[5] = a.nbz[n[1]];
        n[6] = a.nbz[n[2]];
        n[7] = a.nbz[n[3]];
    } else {
        const uint32_t nx = (uint32_t)a.nx, ny = (uint32_t)a.ny, nz = (uint32_t)a.nz;
        const uint32_t x = k % nx, t = k / nx, y = t % ny, z = t / ny;
        const uint32_t xp = x + 1 == nx ? 0 : x + 1, yp = y + 1 == ny ? 0 : y + 1, zp = z + 1 == nz ? 0 : z + 1;
        const uint32_t r00 = nx * (y + ny * z), r10 = nx * (yp + ny * z), r01 = nx * (y + ny * zp),
                       r11 = nx * (yp + ny * zp);
        n[0] = r00 + x; n[1] = r00 + xp; n[2] = r10 + x; n[3] = r10 + xp;
        n[4] = r01 + x; n[5] = r01 + xp; n[6] = r11 + x; n[7] = r11 + xp;
    }
}

// Plane-flat numbering of the one-node-per-thread box kernels: a launch of (plane_blocks, nz)
// workgroups of kPlaneBlock threads gives thread t of plane z the node t of the plane's nx * ny
// nodes, so every lane has a node whatever nx is. y = t / nx comes from a double reciprocal:
// v = (t + 1/2) / nx lies at least 1/(2 nx) from an integer, and the two roundings (of 1/nx and
// of the product) err by at most v 2^-52 < 1/(2 nx) for every t < 2^51, so the truncation is
// exact.
constexpr int kPlaneBlock = 256;
struct PlaneDiv {
    uint32_t nx;
    uint32_t planeNodes; // nx * ny
    double invNx;        // 1 / nx
};
inline PlaneDiv make_plane_div(int nx, int ny)
{
    return PlaneDiv{(uint32_t)nx, (uint32_t)nx * (uint32_t)ny, 1.0 / (double)nx};
}
inline unsigned plane_blocks(int nx, int ny)
{
    return (unsigned)(((uint64_t)nx * (uint64_t)ny + kPlaneBlock - 1) / kPlaneBlock);
}
VF_PLANE_HD uint32_t plane_row(uint32_t t, const PlaneDiv& p) { return (uint32_t)(((double)t + 0.5) * p.invNx); }
// (x, y) of this thread's node in its plane (blockIdx.y); false for threads beyond the plane
__device__ __forceinline__ bool plane_xy(const PlaneDiv& p, int& x, int& y)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= p.planeNodes) return false;
    const uint32_t r = plane_row(t, p);
    y = (int)r;
    x = (int)(t - r * p.nx);
    return true;
}

// Flat numbering of a box's nodes, k = x + nx (y + ny z), for kernels that walk the whole box whatever its
// planes are. k / d of k < 2^30 (numberOfNodes is checked) by a multiplication: with 2^(s-1) < d <= 2^s and
// m = floor(2^(30+s) / d) + 1, m d exceeds 2^(30+s) by at most d <= 2^s, so k m / 2^(30+s) exceeds k / d by
// less than 1 / d and has the same integer part.
struct Divider {
    uint32_t d, m;
    int s;
};
inline Divider make_divider(uint32_t d)
{
    int s = 0;
    while ((1u << s) < d) ++s;
    return Divider{d, (uint32_t)((1ull << (30 + s)) / d + 1), s};
}
VF_PLANE_HD uint32_t divide(uint32_t k, const Divider& v) { return (uint32_t)(((uint64_t)(k << 2) * v.m) >> 32) >> v.s; }
struct BoxDiv {
    Divider plane, row; // by nx ny and by nx
};
inline BoxDiv make_box_div(int nx, int ny)
{
    return BoxDiv{make_divider((uint32_t)nx * (uint32_t)ny), make_divider((uint32_t)nx)};
}

// A reduction over a lattice ends in one FP64 atomic per workgroup and sum on the same few words,
// about 10 ns a workgroup one after the other (64^3 moment sums: 18.4 us with 1024 workgroups, 10.6
// with 256). So the sums take one workgroup of 16 waves per CU, as few as keep HBM busy, and up to 48 k
// nodes workgroups of four waves, which start and end sooner (moment sums of 20^3 nodes 7.0 -> 5.8 us).
// A box is walked in pieces of a workgroup's size: of its planes (SUM_PLANES: the plane is the same for all
// lanes, and so are the offsets to its neighbours: kinetic energy of 448 x 69 x 231 33.8 us, 38.1 flat) where
// these fill their last pieces to 9/10 in the mean, else of the flat numbering (2 x 2 x 9000: 5.6, 20.7 by planes).
constexpr int kReduceThreads = 1024;
constexpr unsigned kReduceGroups = 256;
enum SumForm { SUM_INDEXED, SUM_FLAT, SUM_PLANES };
struct SumLaunch {
    SumForm form;
    uint32_t groups, threads; // the launch, also as kernel arguments (reading blockDim costs a load before all else)
    BoxDiv box;
};
inline SumLaunch sum_launch(const vf_lbm_parameter& p)
{
    const uint64_t n = p.numberOfNodes;
    const unsigned threads = n <= 48 * 1024 ? 256 : kReduceThreads;
    SumForm form = SUM_INDEXED;
    uint64_t pieces = (n + threads - 1) / threads;
    if (!p.neighborX) {
        const uint64_t planes = ((uint64_t)p.nx * p.ny + threads - 1) / threads * p.nz;
        form = planes * threads * 9 <= n * 10 ? SUM_PLANES : SUM_FLAT;
        if (form == SUM_PLANES) pieces = planes;
    }
    return {form, (uint32_t)(pieces < kReduceGroups ? pieces : kReduceGroups), threads,
            form == SUM_INDEXED ? BoxDiv{} : make_box_div(p.nx, p.ny)};
}
// f(k, z, t) for this thread's nodes k = t + nx ny z of a box (z, t: 0 and k on neighbour arrays)
template <SumForm FORM, class F> __device__ __forceinline__ void sum_nodes(const Addr& a, const SumLaunch& l, F f)
{
    const BoxDiv& b = l.box;
    if constexpr (FORM == SUM_PLANES) {
        const uint32_t P = b.plane.d, nz = (uint32_t)a.nz, per = (P + l.threads - 1) / l.threads;
        // piece i of plane z, and the step to this workgroup's next one
        uint32_t z = blockIdx.x / per, i = blockIdx.x - z * per;
        const uint32_t dz = l.groups / per, di = l.groups - dz * per;
        while (z < nz) {
            const uint32_t t = i * l.threads + threadIdx.x;
            if (t < P) f(P * z + t, z, t);
            z += dz;
            i += di;
            if (i >= per) {
                i -= per;
                ++z;
            }
        }
    } else {
        for (uint64_t kk = (uint64_t)blockIdx.x * l.threads + threadIdx.x; kk < a.N; kk += (uint64_t)l.groups * l.threads) {
            const uint32_t k = (uint32_t)kk, z = FORM == SUM_FLAT ? divide(k, b.plane) : 0;
            f(k, z, k - b.plane.d * z);
        }
    }
}

template <class S> __device__ __forceinline__ S* slot_ptr(S* f, uint64_t N, int d, bool even)
{
    return f + (uint64_t)(even ? d : inv(d)) * N;
}

// pre-collision value of direction d (the value a collision at this cell would read)
template <class S> __device__ __forceinline__ float read_pre(const S* f, const Addr& a, const uint32_t (&n)[8], int d, bool even)
{
    return Codec<S>::load(slot_ptr(const_cast<S*>(f), a.N, d, even) + n[node_sel(d)]);
}
template <class S> __device__ __forceinline__ void write_pre(S* f, const Addr& a, const uint32_t (&n)[8], int d, bool even, float v)
{
    Codec<S>::store(slot_ptr(f, a.N, d, even) + n[node_sel(d)], v);
}
// post-collision value of direction d (stored in the slot of inv(d) at inv(d)'s node)
template <class S> __device__ __forceinline__ float read_post(const S* f, const Addr& a, const uint32_t (&n)[8], int d, bool even)
{
    return read_pre(f, a, n, inv(d), even);
}

__device__ __forceinline__ float c_dot(int d, float ux, float uy, float uz)
{
    float s = 0.0f;
    if (cx(d)) s += float(cx(d)) * ux;
    if (cy(d)) s += float(cy(d)) * uy;
    if (cz(d)) s += float(cz(d)) * uz;
    return s;
}

// VelocityBounceBack: the incoming population inv(d) from the post-collision value of the wall
// link d, f_inv(d) = f_d - 6 w_d c_d.U (getBounceBackDistributionForVeloBC,
// src/gpu/core/Utilities/KernelUtilities.h:186-190); NoSlipBounceBack returns f_d itself
__device__ __forceinline__ float velocity_bounce_back(float post_d, int d, float Ux, float Uy, float Uz)
{
    return post_d - 6.0f * weight(d) * c_dot(d, Ux, Uy, Uz);
}

// Full shifted equilibrium w_d (drho + (1+drho)(3 c.u + 9/2 (c.u)^2 - 3/2 u^2))
// (InitNavierStokesCompressible_Device.cu:173-201).
__device__ __forceinline__ float feq_shifted(int d, float drho, float ux, float uy, float uz, float cu_sq)
{
    if (d == 0) return (8.0f / 27.0f) * (drho - cu_sq * (1.0f + drho));
    const float cu = c_dot(d, ux, uy, uz);
    return weight(d) * (drho + (1.0f + drho) * (3.0f * cu + 4.5f * cu * cu - cu_sq));
}

} // namespace vfa
