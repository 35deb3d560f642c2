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
#pragma unroll
    for (int q = 1; q < L::Q; q++) {
        const int64_t n = downstream<L>(a, p, q);
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

template struct PassOps<double>;
template struct PassOps<float>;

}  // namespace mplb
