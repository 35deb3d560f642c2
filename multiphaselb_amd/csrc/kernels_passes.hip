// Fused passes of the per-routine arithmetic (FP64, and FP32 without the fused kernels).
//
// Between the first collision and the last macroscopic update of a run of steps the only
// state that has to reach memory is the post-collision populations, so a step is two
// passes (three with heat transfer) instead of one launch per reference routine:
//   density   pull-stream f (and g): rho and psi, or rho and the sum of g;
//   heat      (thermal) heat source from the rho, T and U stencils, new T, psi;
//   collide   pull again, psi stencil -> force -> velocity, then the collisions of the next
//             step, written to the other buffer.  The last step of a run writes the
//             post-stream populations and all macroscopic fields instead, so that between
//             runs the state is the one the per-routine kernels keep.
// Every node uses the expressions of node.h in the reference's order (this file is built
// with -ffp-contract=off): results equal the per-routine kernels' bit for bit.
//
// Bound: HBM.  Per node and step the per-routine kernels move about 1000 B (D3Q15, FP64,
// isothermal: f is read four times and written twice, with the neighbour table each time)
// and 2100 B with heat transfer; the passes move 2 x 120 + 120 + 24 = 384 B and about
// 880 B.  Neighbours are computed from coordinates, not read (boxidx.h); 256 consecutive
// nodes per block keep every population plane's rows contiguous.
#include <hip/hip_runtime.h>

#include "boxidx.h"
#include "node.h"
#include "passes.h"

namespace mplb {

namespace {

constexpr int kBlock = 256;

template <typename T>
__device__ inline void put(T* p, int64_t i, T v) {
    __builtin_nontemporal_store(v, p + i);
}

// Post-stream, post-boundary populations of one field: boundary nodes were prepared in
// the output buffer
template <class L, typename T>
__device__ inline void pull(const PassArgs<T>& a, const NodePos& p, const T* in, const T* out, const uint8_t* order,
                            T* v) {
    if (p.table && order && order[p.id] != 255) {
#pragma unroll
        for (int q = 0; q < L::Q; q++) v[q] = out[q * a.N + p.id];
    } else if constexpr (L::D == 2) {
        // one branch for the node (D2Q9 FP64 700^2 47.4 -> 43.2 us per step); in 3D the ids of
        // all populations at once cost registers (75 x 90 x 120 with heat transfer 176 -> 181)
        unsigned up[L::Q];
        upstreams<L>(a, p, up);
#pragma unroll
        for (int q = 0; q < L::Q; q++) v[q] = in[q * a.N + up[q]];
    } else {
#pragma unroll
        for (int q = 0; q < L::Q; q++) v[q] = in[q * a.N + upstream<L>(a, p, q)];
    }
}

template <class L, typename T>
__global__ void __launch_bounds__(kBlock) k_pass_boundary(PassArgs<T> a, int fld, int order, BdList b) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= b.n) return;
    const int64_t id = b.nodes[i], N = a.N;
    const T* in = fld == 0 ? a.fin : a.gin;
    T* out = fld == 0 ? a.fout : a.gout;
    const uint8_t* ord = a.order[fld];
    T v[L::Q];
    int up[L::Q];
#pragma unroll
    for (int q = 0; q < L::Q; q++) up[q] = a.nb[q * N + id];
#pragma unroll
    for (int q = 0; q < L::Q; q++) v[q] = in[q * N + (up[q] == -1 ? id : (int64_t)up[q])];
    if (b.type == BD_BBACK) {
        bool miss[L::Q];
#pragma unroll
        for (int q = 0; q < L::Q; q++) miss[q] = up[q] == -1;
        node_bounce_back<L, T>(v, miss);
    } else {
        // fixedT.c:45-122 and fixedRandomT.c:48-112 (see bc_fixed_temp): the neighbour's
        // post-stream population is pulled directly unless an earlier list corrected it
        const bool random = b.type == BD_FRDT;
        T minT = 0, maxT = 0;
        int draw = 0;
        if (random) {
            minT = T(b.value[0]) * (T(100.0) - T(b.pert)) / T(100.0);
            maxT = T(b.value[0]) * (T(100.0) + T(b.pert)) / T(100.0);
            draw = b.rnd_off[i];
        }
#pragma unroll
        for (int q = 0; q < L::Q; q++) {
            if (up[q] != -1) continue;
            const int nbid = up[L::t.rev[q]];
            if (nbid == -1) continue;
            const int s2 = a.nb[q * N + nbid];
            const T gnb = ord[nbid] < order ? out[q * N + nbid] : in[q * N + (s2 == -1 ? nbid : s2)];
            const T Unb[3] = {a.U[nbid], a.U[N + nbid], a.U[2 * N + nbid]};
            const T eq_nb = node_geq<L, T>(a.gp, q, a.temp[nbid], Unb);
            T Tw = T(b.value[0]);
            if (random && b.draw) {
                const T r = T(b.rnd[draw++]);
                Tw = minT + (maxT - minT) * r;
            }
            v[q] = node_geq<L, T>(a.gp, q, Tw, Unb) + (gnb - eq_nb);
        }
    }
#pragma unroll
    for (int q = 0; q < L::Q; q++) out[q * N + id] = v[q];
}

template <class L, typename T, bool THERMAL>
__global__ void __launch_bounds__(kBlock) k_pass_density(PassArgs<T> a) {
    const NodePos p = node_pos<L>(a);
    if (!p.valid) return;
    T v[L::Q];
    pull<L, T>(a, p, a.fin, a.fout, a.order[0], v);
    if (THERMAL) {
        T w[L::Q];
        pull<L, T>(a, p, a.gin, a.gout, a.order[1], w);
        a.rho[p.id] = node_sum<L, T>(v);
        a.sumg[p.id] = node_sum<L, T>(w);
    } else {
        const T rho = node_sum<L, T>(v);
        a.rho[p.id] = rho;
        a.psi[p.id] = potential<T>(a.eos, rho, a.temp[p.id]);
    }
}

template <class L, typename T>
__global__ void __launch_bounds__(kBlock) k_pass_heat(PassArgs<T> a) {
    const NodePos p = node_pos<L>(a);
    if (!p.valid) return;
    const int64_t id = p.id;
    const T rho = a.rho[id], temp = a.temp[id];
    T dot = 0, divU = 0;
    T gT[3] = {0, 0, 0}, gR[3] = {0, 0, 0};
#pragma unroll
    for (int ax = 0; ax < L::D; ax++) {
        // fd_plus's upstream node is x + e, fd_minus's is x - e
        const int64_t na = downstream<L>(a, p, L::t.rev[L::fd_plus[ax]]);
        const int64_t nb = downstream<L>(a, p, L::t.rev[L::fd_minus[ax]]);
        const bool ha = na != -1, hb = nb != -1;
        const int64_t ia = ha ? na : id, ib = hb ? nb : id;
        const T* Uax = a.U + ax * a.N;
        gT[ax] = node_fd<T>(a.temp[ia], ha, a.temp[ib], hb, temp, false);
        gR[ax] = node_fd<T>(a.rho[ia], ha, a.rho[ib], hb, rho, true);
        divU += node_fd<T>(Uax[ia], ha, Uax[ib], hb, Uax[id], false);
    }
#pragma unroll
    for (int k = 0; k < 3; k++) dot += gT[k] * gR[k];
    const T s = node_heat<L, T>(a.eos, a.gp, rho, temp, dot, divU);
    T ss = s, t = a.sumg[id];
    if (a.gp.model == M_MYMRT) {
        t = t + T(0.5) * ss;
    } else {
        const T oldss = a.first_call ? T(0) : a.ss[id];
        ss = s + T(0.5) * (s - oldss);
    }
    a.ss[id] = ss;
    a.sumg[id] = t;
    a.psi[id] = potential<T>(a.eos, rho, t);
}

template <class L, typename T, bool THERMAL, bool LAST>
__global__ void __launch_bounds__(kBlock) k_pass_collide(PassArgs<T> a) {
    const NodePos p = node_pos<L>(a);
    if (!p.valid) return;
    const int64_t id = p.id, N = a.N;
    T v[L::Q], psin[L::Q];
    pull<L, T>(a, p, a.fin, a.fout, a.order[0], v);
    const T psi = a.psi[id], rho = a.rho[id];
    bool full = true;
    int dn[L::Q];
    if constexpr (L::D == 2) downstreams<L>(a, p, dn);
#pragma unroll
    for (int q = 1; q < L::Q; q++) {
        const int64_t n = L::D == 2 ? (int64_t)dn[q] : downstream<L>(a, p, q);
        full = full && n != -1;
        psin[q] = a.psi[n == -1 ? id : n];
    }
    const bool interior = !p.table || a.onbnd[id] == 0;
    T Fi[3], Ft[3], U[3];
    node_force<L, T>(a.eos, psin, psi, interior, Fi);
    node_total_force<T>(a.eos, Fi, rho, a.rho0, interior, Ft);
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const T F = L::D == 2 ? Ft[j] : Fi[j] + (rho - a.rho0) * T(a.eos.g[j]);
        U[j] = node_velocity<L, T>(v, rho, F, j);
    }
    if (!LAST) {
        T C[L::Q];
        if (a.fp.surf) {
#pragma unroll
            for (int k = 0; k < L::Q; k++) C[k] = T(0);
            if (full) node_surface_tension<L, T>(a.eos, a.fp, psin, psi, C);
        }
        if constexpr (L::D == 2) node_collide_limrt<L, T>(a.fp, v, rho, U, Ft, Fi[0], Fi[1], psi, C);
        else node_collide_xumrt<L, T>(a.eos, a.fp, v, rho, U, Fi, psi, a.rho0, C);
    }
#pragma unroll
    for (int q = 0; q < L::Q; q++) put<T>(a.fout, q * N + id, v[q]);
    if (THERMAL) {
        const T t = a.sumg[id];
        pull<L, T>(a, p, a.gin, a.gout, a.order[1], v);
        if (!LAST) {
            if (L::D == 3 || a.gp.model == M_MYMRT) node_collide_my<L, T>(a.gp, v, t, U, a.ss[id]);
            else node_collide_litemp<L, T>(a.gp, v, t, U, a.ss[id]);
        }
#pragma unroll
        for (int q = 0; q < L::Q; q++) put<T>(a.gout, q * N + id, v[q]);
        a.temp[id] = t;
    }
    if (THERMAL || LAST) {
#pragma unroll
        for (int j = 0; j < 3; j++) a.U[j * N + id] = U[j];
    }
    if (LAST) {
#pragma unroll
        for (int j = 0; j < 3; j++) {
            a.Fi[j * N + id] = Fi[j];
            a.Ft[j * N + id] = Ft[j];
        }
    }
}

// ---------------------------------------------------------------------------
// The isothermal step of a fully periodic D3Q15 box in one pass: a workgroup owns a 32 x 8
// column of sites over a chunk of z planes and walks up the chunk; plane z + 1 is pulled for
// the column and the one-site ring around it and turned into psi in an LDS ring of four
// planes, then plane z collides from the populations pulled one plane earlier and the psi
// stencil in LDS.  psi and rho do not go to memory (the last step of a run writes them) and
// the populations are read once: 240 B per node and step in FP64 instead of 384.
//
// Bound: half the time is FP64 arithmetic in the reference's order (no contraction), at two
// waves per SIMD (the two planes' populations and the collision take 200 registers; three
// waves spill: 160^3 0.367 ms).  FP64 160^3 0.310 -> 0.266 ms per step, 128^3 0.177 -> 0.137,
// 256 x 128^2 0.333 -> 0.265.  Columns of 64 x 4 (a ring of 140 sites instead of 84) run 160^3
// at 0.292 ms and 128^3 at 0.134, 16 x 16 (rows of 128 bytes) at 0.283 and 0.143.
constexpr int MX = 32, MY = kBlock / MX, MHX = MX + 2, MHY = MY + 2, MSLOT = MHX * MHY, MRING = 2 * MHX + 2 * MY;
static_assert(MRING <= kBlock, "one thread per ring site");

__device__ inline int wrapd(int u, int n) { return u < 0 ? u + (n - 1) : (u > n - 1 ? u - (n - 1) : u); }

template <typename T, bool LAST>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2)))
k_pass_march(PassArgs<T> a, int mtx, int mtiles, int mitems, int mper, int mzc) {
    using L = D3Q15;
    __shared__ T ring[4][MSLOT];
    const unsigned wi = (blockIdx.x & 7u) * (unsigned)mper + (blockIdx.x >> 3);
    if (wi >= (unsigned)mitems) return;
    const int chunk = (int)(wi / (unsigned)mtiles), tile = (int)(wi - (unsigned)chunk * (unsigned)mtiles);
    const int x0 = (tile % mtx) * MX, y0 = (tile / mtx) * MY;
    const int z0 = chunk * mzc, z1 = min(z0 + mzc, a.nz);
    const int t = threadIdx.x, tx = t % MX, ty = t / MX;
    const int x = x0 + tx, y = y0 + ty;
    const bool owner = x < a.nx && y < a.ny;
    const bool edge = x <= a.nx && y <= a.ny;          // raw n wraps onto site 1
    const int ex = wrapd(x, a.nx), ey = wrapd(y, a.ny);
    int rhx = 0, rhy = 0;
    if (t < MHX) {
        rhx = t;
    } else if (t < 2 * MHX) {
        rhx = t - MHX;
        rhy = MHY - 1;
    } else if (t < 2 * MHX + MY) {
        rhy = 1 + (t - 2 * MHX);
    } else {
        rhx = MHX - 1;
        rhy = 1 + (t - 2 * MHX - MY);
    }
    const bool ring_site = t < MRING && x0 + rhx - 1 <= a.nx && y0 + rhy - 1 <= a.ny;
    const int rx = wrapd(x0 + rhx - 1, a.nx), ry = wrapd(y0 + rhy - 1, a.ny);
    T fc[L::Q], fn[L::Q];
    // populations of site (px, py) of plane zw, their sum, and psi into the ring
    auto site = [&](int px, int py, int zw, T* v, T* slot) __attribute__((always_inline)) {
        const unsigned nx = (unsigned)a.nx, nxy = (unsigned)a.nxy;
        const unsigned X[3] = {(unsigned)wrapd(px - 1, a.nx), (unsigned)px, (unsigned)wrapd(px + 1, a.nx)};
        const unsigned Y[3] = {(unsigned)wrapd(py - 1, a.ny) * nx, (unsigned)py * nx, (unsigned)wrapd(py + 1, a.ny) * nx};
        const unsigned Z[3] = {(unsigned)wrapd(zw - 1, a.nz) * nxy, (unsigned)zw * nxy, (unsigned)wrapd(zw + 1, a.nz) * nxy};
#pragma unroll
        for (int q = 0; q < L::Q; q++)
            v[q] = a.fin[q * a.N + (X[1 - L::t.c[q][0]] + Y[1 - L::t.c[q][1]] + Z[1 - L::t.c[q][2]])];
        *slot = potential<T>(a.eos, node_sum<L, T>(v), a.temp[X[1] + Y[1] + Z[1]]);
    };
    auto plane = [&](int zr) __attribute__((always_inline)) {
        const int zw = wrapd(zr, a.nz);
        T* sl = ring[(zr - z0 + 1) & 3];
        __builtin_amdgcn_s_setprio(2);
        if (edge) site(ex, ey, zw, fn, &sl[(ty + 1) * MHX + tx + 1]);
        if (ring_site) {
            T tmp[L::Q];
            site(rx, ry, zw, tmp, &sl[rhy * MHX + rhx]);
        }
        __builtin_amdgcn_s_setprio(0);
    };
    plane(z0 - 1);
    plane(z0);
#pragma unroll
    for (int q = 0; q < L::Q; q++) fc[q] = fn[q];
    for (int z = z0; z < z1; z++) {
        plane(z + 1);
        __syncthreads();
        if (owner) {
            const T rho = node_sum<L, T>(fc);
            T psin[L::Q];
#pragma unroll
            for (int q = 0; q < L::Q; q++)
                psin[q] = ring[(z + L::t.c[q][2] - z0 + 1) & 3][(ty + 1 + L::t.c[q][1]) * MHX + tx + 1 + L::t.c[q][0]];
            T Fi[3], Ft[3], U[3];
            node_force<L, T>(a.eos, psin, psin[0], true, Fi);
            node_total_force<T>(a.eos, Fi, rho, a.rho0, true, Ft);
#pragma unroll
            for (int j = 0; j < 3; j++)
                U[j] = node_velocity<L, T>(fc, rho, Fi[j] + (rho - a.rho0) * T(a.eos.g[j]), j);
            const int64_t id = (int64_t)x + (int64_t)y * a.nx + (int64_t)z * a.nxy, N = a.N;
            if (!LAST) {
                T C[L::Q];
                if (a.fp.surf) node_surface_tension<L, T>(a.eos, a.fp, psin, psin[0], C);
                node_collide_xumrt<L, T>(a.eos, a.fp, fc, rho, U, Fi, psin[0], a.rho0, C);
            }
#pragma unroll
            for (int q = 0; q < L::Q; q++) put<T>(a.fout, q * N + id, fc[q]);
            if (LAST) {
                a.rho[id] = rho;
                a.psi[id] = psin[0];
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    a.U[j * N + id] = U[j];
                    a.Fi[j * N + id] = Fi[j];
                    a.Ft[j * N + id] = Ft[j];
                }
            }
        }
#pragma unroll
        for (int q = 0; q < L::Q; q++) fc[q] = fn[q];
    }
}

template <typename Fn>
void for_lattice(int model, Fn fn) {
    if (model == 0) fn(D2Q9{});
    else fn(D3Q15{});
}

template <typename T>
dim3 grid_of(const PassArgs<T>& a) {
    return dim3((unsigned)((a.N + kBlock - 1) / kBlock));
}

}  // namespace

template <typename T>
void PassOps<T>::boundary(int model, hipStream_t s, const PassArgs<T>& a, int fld, int order, const BdList& b) {
    if (b.n <= 0) return;
    const dim3 grid((unsigned)((b.n + kBlock - 1) / kBlock));
    for_lattice(model, [&](auto l) { k_pass_boundary<decltype(l), T><<<grid, kBlock, 0, s>>>(a, fld, order, b); });
}

template <typename T>
void PassOps<T>::density(int model, hipStream_t s, const PassArgs<T>& a, bool thermal) {
    for_lattice(model, [&](auto l) {
        if (thermal) k_pass_density<decltype(l), T, true><<<grid_of(a), kBlock, 0, s>>>(a);
        else k_pass_density<decltype(l), T, false><<<grid_of(a), kBlock, 0, s>>>(a);
    });
}

template <typename T>
void PassOps<T>::heat(int model, hipStream_t s, const PassArgs<T>& a) {
    for_lattice(model, [&](auto l) { k_pass_heat<decltype(l), T><<<grid_of(a), kBlock, 0, s>>>(a); });
}

template <typename T>
void PassOps<T>::collide(int model, hipStream_t s, const PassArgs<T>& a, bool thermal, bool last) {
    for_lattice(model, [&](auto l) {
        using L = decltype(l);
        if (thermal && last) k_pass_collide<L, T, true, true><<<grid_of(a), kBlock, 0, s>>>(a);
        else if (thermal) k_pass_collide<L, T, true, false><<<grid_of(a), kBlock, 0, s>>>(a);
        else if (last) k_pass_collide<L, T, false, true><<<grid_of(a), kBlock, 0, s>>>(a);
        else k_pass_collide<L, T, false, false><<<grid_of(a), kBlock, 0, s>>>(a);
    });
}

// Which boxes march: rows of whole columns in more than 2^19 nodes.  Elsewhere idle lanes and
// stores that share sectors cost more than the passes' second read (FP64 101^3 0.098 against
// 0.084 ms, 201 x 150 x 180 0.523 against 0.414, 144 x 100 x 90, 112^3 and 200^3 equal), and
// small boxes are short chains of launches either way (64^3 0.0237 against 0.0223; 128 x 64 x 64,
// 2^19 nodes, 0.0406 against 0.0451 in FP64 and 0.0268 against 0.0260 in FP32; 96^3 0.0616
// against 0.0664, FP32 0.0381 against 0.0417).
//
// z chunks of the march: the work items run in rounds of the workgroups that are resident at
// once, so the count that minimises rounds x (planes per chunk + 2 halo planes)
template <typename T>
int PassOps<T>::march_plan(int device, int nx, int ny, int nz, PassMarch* p) {
    if (nx % MX || (int64_t)nx * ny * nz <= (1 << 19) || ny < 3 || nz < 3) return 0;
    int bpc = 0, cus = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&bpc, k_pass_march<T, false>, kBlock, 0);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
    if (e != hipSuccess) return (int)e;
    p->mtx = (nx + MX - 1) / MX;
    p->tiles = p->mtx * ((ny + MY - 1) / MY);
    const long long resident = bpc > 0 && cus > 0 ? (long long)bpc * cus : 1;
    int chunks = 1;
    long long best = -1;
    for (int n = 1; n <= nz; n++) {
        const long long cost = ((long long)p->tiles * n + resident - 1) / resident * ((nz + n - 1) / n + 2);
        if (best < 0 || cost < best) {
            best = cost;
            chunks = n;
        }
    }
    p->zc = (nz + chunks - 1) / chunks;
    p->items = p->tiles * ((nz + p->zc - 1) / p->zc);
    p->per = (p->items + 7) / 8;
    return 0;
}

template <typename T>
void PassOps<T>::march(hipStream_t s, const PassArgs<T>& a, const PassMarch& p, bool last) {
    const dim3 grid(8u * (unsigned)p.per);
    if (last) k_pass_march<T, true><<<grid, kBlock, 0, s>>>(a, p.mtx, p.tiles, p.items, p.per, p.zc);
    else k_pass_march<T, false><<<grid, kBlock, 0, s>>>(a, p.mtx, p.tiles, p.items, p.per, p.zc);
}

template struct PassOps<double>;
template struct PassOps<float>;

}  // namespace mplb
