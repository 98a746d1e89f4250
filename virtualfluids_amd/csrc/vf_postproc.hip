// Post-processing reductions in FP64: drag and lift by momentum exchange on a BC node list,
// and the kinetic-energy analyzer. These are the objectives of the flow cases (drag on a body,
// decay of the kinetic energy), evaluated on the device without copying fields to the host.
//
//  * vf_DragLiftPostD27 / vf_DragLiftPreD27: the two per-node halves of the reference
//    (src/gpu/core/PostProcessor/DragLift.cu:50-556), one double per node and axis.
//  * vf_DragLiftSum: their sum over the nodes, pre - post (DragLift.cpp:67-72), from the state
//    after the step alone. Both halves sit in cells no kernel touches between the two reference
//    calls: the population e a node sends towards the wall lands in the cell of the solid node
//    across the link, which nothing reads or writes, and the BC writes the returning population
//    inv(e) into the node's own next-step cell. With the parity after the swap both are the
//    slots e and inv(e) at the node that stores inv(e). One workgroup, fixed summation order:
//    the result does not change from run to run.
//  * vf_KineticEnergy: kineticEnergyKernel's node selection (the node, its six face neighbours
//    and its (-1,-1,-1) neighbour are fluid) and energy
//    (src/gpu/core/PostProcessor/KineticEnergyAnalyzer.cu:99-153), summed in double.
#include "vf_lattice.h"

namespace vfa {

namespace {

// One workgroup sums a list (a fixed order without a workspace): its 16 waves are all the
// loads in flight there are
constexpr int kSumThreads = 1024;

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

__device__ __forceinline__ bool link_active(float q) { return q >= 0.0f && q <= 1.0f; }

template <class S, bool POST>
__global__ __launch_bounds__(256) void drag_lift_kernel(const S* __restrict__ f, Addr a, const int32_t* __restrict__ k,
                                                        const float* __restrict__ q, uint32_t nbc, int even_flag,
                                                        double* dx, double* dy, double* dz)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nbc) return;
    const bool even = even_flag != 0;
    uint32_t n[8];
    cell_nodes(a, (uint32_t)k[i], n);
    double sx = 0.0, sy = 0.0, sz = 0.0;
#pragma unroll
    for (int e = 1; e < 27; ++e) {
        if (!link_active(q[(uint64_t)e * nbc + i])) continue;
        // post half: the population e leaving towards the wall; pre half: inv(e) coming back
        const int d = POST ? e : inv(e);
        const double v = POST ? (double)read_post(f, a, n, d, even) : (double)read_pre(f, a, n, d, even);
        sx += cx(d) * v;
        sy += cy(d) * v;
        sz += cz(d) * v;
    }
    dx[i] = -sx;
    dy[i] = -sy;
    dz[i] = -sz;
}

// force[0..2] = sum over links c_e (f_e leaving + f_inv(e) returning), state after the swap
template <class S>
__global__ __launch_bounds__(kSumThreads) void drag_sum_kernel(const S* __restrict__ f, Addr a,
                                                               const int32_t* __restrict__ k,
                                                               const float* __restrict__ q, uint32_t nbc,
                                                               int even_flag, double* force)
{
    __shared__ double part[kSumThreads / 64][3];
    const bool even = even_flag != 0;
    double acc[3] = {0.0, 0.0, 0.0};
    for (uint32_t i = threadIdx.x; i < nbc; i += kSumThreads) {
        uint32_t n[8];
        cell_nodes(a, (uint32_t)k[i], n);
        // every distance, then every active link's two populations, each before the first is used:
        // a chain of 26 distance -> population latencies per node otherwise (sphere channel, 3 000
        // nodes: 82 us with 256 threads and the chain, 25 us so)
        uint32_t active = 0;
#pragma unroll
        for (int e = 1; e < 27; ++e) active |= (link_active(q[(uint64_t)e * nbc + i]) ? 1u : 0u) << e;
        float out[27], back[27];
#pragma unroll
        for (int e = 1; e < 27; ++e) {
            const uint32_t m = n[node_sel(inv(e))];
            out[e] = back[e] = 0.0f;
            if (active >> e & 1u) {
                out[e] = Codec<S>::load(slot_ptr(const_cast<S*>(f), a.N, e, even) + m);
                back[e] = Codec<S>::load(slot_ptr(const_cast<S*>(f), a.N, inv(e), even) + m);
            }
        }
#pragma unroll
        for (int e = 1; e < 27; ++e) {
            const double s = (double)out[e] + (double)back[e];
            acc[0] += cx(e) * s;
            acc[1] += cy(e) * s;
            acc[2] += cz(e) * s;
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const double s = wave_sum(acc[j]);
        if (lane == 0) part[wave][j] = s;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        double s = 0.0;
        for (int w = 0; w < kSumThreads / 64; ++w) s += part[w][threadIdx.x];
        force[threadIdx.x] = s;
    }
}

__global__ void zero2_kernel(double* out)
{
    if (threadIdx.x < 2) out[threadIdx.x] = 0.0;
}

// the node k, its six face neighbours and its (-1,-1,-1) neighbour are fluid
// (kineticEnergyFunction checks the diagonal node it reaches the -x/-y/-z neighbours through)
__device__ __forceinline__ bool interior_fluid(const Addr& a, const uint32_t* nbinv, const uint32_t* geo, uint32_t k)
{
    auto fl = [&](uint32_t j) { return geo[j] == VF_GEO_FLUID; };
    if (!fl(k)) return false;
    const uint32_t m = nbinv[k];
    return fl(a.nbx[k]) && fl(a.nby[k]) && fl(a.nbz[k]) && fl(m) && fl(a.nbz[a.nby[m]]) && fl(a.nbz[a.nbx[m]]) &&
           fl(a.nby[a.nbx[m]]);
}

__device__ __forceinline__ double node_energy(float vx, float vy, float vz, float rho)
{
    const double ux = vx, uy = vy, uz = vz;
    return 0.5 * (ux * ux + uy * uy + uz * uz) * ((double)rho + 1.0);
}

// FORM: sum_launch. The seven neighbours of a box's node are offsets; their types and the node's fields
// are loaded together (one by one behind the previous test they are eight memory latencies a node).
// Bound by HBM: 20 bytes a node. 256^3: 155 us with the chain, a division per coordinate and 2048
// workgroups, 72 us so.
template <SumForm FORM>
__global__ __launch_bounds__(kReduceThreads) void kinetic_energy_kernel(Addr a, const uint32_t* nbinv, const uint32_t* geo,
                                                             const float* vx, const float* vy, const float* vz,
                                                             const float* rho, SumLaunch l, double* out)
{
    __shared__ double part[kReduceThreads / 64][2];
    double e = 0.0, c = 0.0;
    const uint32_t nx = l.box.row.d, ny = (uint32_t)a.ny, nz = (uint32_t)a.nz, P = l.box.plane.d;
    sum_nodes<FORM>(a, l, [&](uint32_t k, uint32_t z, uint32_t t) {
        if constexpr (FORM == SUM_INDEXED) {
            if (!interior_fluid(a, nbinv, geo, k)) return;
            e += node_energy(vx[k], vy[k], vz[k], rho[k]);
            c += 1.0;
        } else {
            const uint32_t y = divide(t, l.box.row), x = t - y * nx;
            const uint32_t xp = x + 1 == nx ? t + 1 - nx : t + 1, xm = x == 0 ? t + nx - 1 : t - 1;
            const uint32_t yp = y + 1 == ny ? x : t + nx, ym = y == 0 ? t + (P - nx) : t - nx;
            const uint32_t xym = y == 0 ? xm + (P - nx) : xm - nx;
            const uint32_t zo = P * z, zp = P * (z + 1 == nz ? 0 : z + 1), zm = P * (z == 0 ? nz - 1 : z - 1);
            const uint32_t g[8] = {geo[k],       geo[zo + xp], geo[zo + xm], geo[zo + yp],
                                   geo[zo + ym], geo[zp + t],  geo[zm + t],  geo[zm + xym]};
            float ux = vx[k], uy = vy[k], uz = vz[k], r = rho[k];
            // needed here: the compiler would move these loads behind the test of the types (256^3 72 -> 95 us)
            asm volatile("" : "+v"(ux), "+v"(uy), "+v"(uz), "+v"(r));
            bool in = true;
#pragma unroll
            for (int j = 0; j < 8; ++j) in &= g[j] == VF_GEO_FLUID;
            if (in) {
                e += node_energy(ux, uy, uz, r);
                c += 1.0;
            }
        }
    });
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    e = wave_sum(e);
    c = wave_sum(c);
    if (lane == 0) {
        part[wave][0] = e;
        part[wave][1] = c;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double s = 0.0;
        for (unsigned w = 0; w < l.threads / 64; ++w) s += part[w][threadIdx.x];
        atomicAdd(out + threadIdx.x, s);
    }
}

template <template <class> class K, class... A> int by_storage(int storage, A&&... args)
{
    switch (storage) {
    case VF_STORAGE_FP32: K<float>::run(args...); return VF_OK;
    case VF_STORAGE_FP16: K<__half>::run(args...); return VF_OK;
    case VF_STORAGE_BF16: K<__hip_bfloat16>::run(args...); return VF_OK;
    default: set_last_error("unknown storage type"); return VF_ERR_INVALID_ARGUMENT;
    }
}

template <bool POST> struct DragL {
    template <class S> struct L {
        static void run(const vf_lbm_parameter& p, const vf_q_boundary_conditions& b, double* dx, double* dy,
                        double* dz, hipStream_t s)
        {
            const dim3 grid((b.numberOfBCnodes + 255) / 256);
            hipLaunchKernelGGL((drag_lift_kernel<S, POST>), grid, dim3(256), 0, s, (const S*)p.distributions,
                               make_addr(p), b.k, b.q27, b.numberOfBCnodes, p.isEvenTimestep, dx, dy, dz);
        }
    };
};

template <class S> struct DragSumL {
    static void run(const vf_lbm_parameter& p, const vf_q_boundary_conditions& b, double* force, hipStream_t s)
    {
        hipLaunchKernelGGL(drag_sum_kernel<S>, dim3(1), dim3(kSumThreads), 0, s, (const S*)p.distributions,
                           make_addr(p), b.k, b.q27, b.numberOfBCnodes, p.isEvenTimestep, force);
    }
};

int check_drag(const vf_lbm_parameter* p, const vf_q_boundary_conditions* bc)
{
    if (!p || !bc || !p->distributions) {
        set_last_error("drag/lift: null parameter, boundary condition or distributions");
        return VF_ERR_INVALID_ARGUMENT;
    }
    if (p->numberOfNodes == 0 || p->numberOfNodes >= (1ull << 30)) {
        set_last_error("drag/lift: numberOfNodes must lie in [1, 2^30)");
        return VF_ERR_INVALID_ARGUMENT;
    }
    if (!p->neighborX && (uint64_t)p->nx * p->ny * p->nz != p->numberOfNodes) {
        set_last_error("drag/lift: needs neighbour arrays or a dense box");
        return VF_ERR_INVALID_ARGUMENT;
    }
    if (bc->numberOfBCnodes > 0 && (!bc->k || !bc->q27)) {
        set_last_error("drag/lift: BC nodes without k or q27");
        return VF_ERR_INVALID_ARGUMENT;
    }
    return VF_OK;
}

template <bool POST>
int drag_half(const vf_lbm_parameter* p, const vf_q_boundary_conditions* bc, double* dx, double* dy, double* dz,
              void* stream, const char* name)
{
    int rc = check_drag(p, bc);
    if (rc) return rc;
    if (bc->numberOfBCnodes == 0) return VF_OK;
    if (!dx || !dy || !dz) {
        set_last_error("drag/lift: null output array");
        return VF_ERR_INVALID_ARGUMENT;
    }
    rc = by_storage<DragL<POST>::template L>(p->storage, *p, *bc, dx, dy, dz, (hipStream_t)stream);
    return rc ? rc : check_launch(name);
}

} // namespace
} // namespace vfa

using namespace vfa;

extern "C" int vf_DragLiftPostD27(const vf_lbm_parameter* p, const vf_q_boundary_conditions* bc, double* dragX,
                                  double* dragY, double* dragZ, void* stream)
{
    return drag_half<true>(p, bc, dragX, dragY, dragZ, stream, "DragLiftPost27 execution failed");
}

extern "C" int vf_DragLiftPreD27(const vf_lbm_parameter* p, const vf_q_boundary_conditions* bc, double* dragX,
                                 double* dragY, double* dragZ, void* stream)
{
    return drag_half<false>(p, bc, dragX, dragY, dragZ, stream, "DragLiftPre27 execution failed");
}

extern "C" int vf_DragLiftSum(const vf_lbm_parameter* p, const vf_q_boundary_conditions* bc, double* force3,
                              void* stream)
{
    int rc = check_drag(p, bc);
    if (rc) return rc;
    if (!force3) {
        set_last_error("drag/lift: null output");
        return VF_ERR_INVALID_ARGUMENT;
    }
    rc = by_storage<DragSumL>(p->storage, *p, *bc, force3, (hipStream_t)stream);
    return rc ? rc : check_launch("DragLiftSum");
}

extern "C" int vf_KineticEnergy(const vf_lbm_parameter* p, const uint32_t* neighborInverse, double* out2, void* stream)
{
    if (!p || !out2 || !p->typeOfGridNode || !p->rho || !p->velocityX || !p->velocityY || !p->velocityZ) {
        set_last_error("kinetic energy: needs typeOfGridNode, rho, velocityX/Y/Z and an output");
        return VF_ERR_INVALID_ARGUMENT;
    }
    if (p->numberOfNodes == 0 || p->numberOfNodes >= (1ull << 30)) {
        set_last_error("kinetic energy: numberOfNodes must lie in [1, 2^30)");
        return VF_ERR_INVALID_ARGUMENT;
    }
    if (p->neighborX && !neighborInverse) {
        set_last_error("kinetic energy on neighbour arrays needs neighborInverse");
        return VF_ERR_INVALID_ARGUMENT;
    }
    if (!p->neighborX && (uint64_t)p->nx * p->ny * p->nz != p->numberOfNodes) {
        set_last_error("kinetic energy: needs neighbour arrays or a dense box");
        return VF_ERR_INVALID_ARGUMENT;
    }
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(zero2_kernel, dim3(1), dim3(64), 0, s, out2);
    const SumLaunch l = sum_launch(*p);
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(l.groups), dim3(l.threads), 0, s, make_addr(*p), neighborInverse,
                           p->typeOfGridNode, p->velocityX, p->velocityY, p->velocityZ, p->rho, l, out2);
    };
    if (l.form == SUM_INDEXED) launch(kinetic_energy_kernel<SUM_INDEXED>);
    else if (l.form == SUM_PLANES) launch(kinetic_energy_kernel<SUM_PLANES>);
    else launch(kinetic_energy_kernel<SUM_FLAT>);
    return check_launch("kineticEnergyKernel execution failed");
}
