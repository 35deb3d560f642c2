// Several time steps per launch for lattices too small to fill the chip.
//
// A step of a lattice of a few thousand nodes is a handful of launches of a few
// microseconds each, whatever the nodes cost.  Here a workgroup owns a block of nodes and
// loads with them every node whose state can reach them within S steps (its halo: two
// neighbours per step, pull and psi stencil; three with heat transfer), one thread per
// node, populations in LDS, and advances the whole set S steps, the valid set shrinking
// by the halo of a step each time.  What neighbouring workgroups compute twice they
// compute alike, so there is nothing to exchange before the next launch.  The state before
// and after is the per-routine kernels' (node.h arithmetic in the reference's order,
// compiled with -ffp-contract=off): results equal theirs bit for bit.
//
// Neighbours come from a per-tile table built on the host from the lattice's own
// neighbour table, so walls, duplicate end nodes and corner links are followed exactly.
// Bound: latency (launch, barriers, and the dependent FP64 arithmetic of one node per
// lane at one to three wavefronts per SIMD), not bandwidth.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "node.h"
#include "tiles.h"

namespace mplb {

namespace {

// LDS values per node: f (and g) populations and psi; with heat transfer also rho, T, U
template <class L, bool THERMAL>
constexpr int kSlots = THERMAL ? 2 * L::Q + 3 + L::D : L::Q + 1;

constexpr int kLdsBytes = 160 * 1024;

// workgroup sizes that fit LDS and keep a node's step in registers (at 768 threads the
// thermal kernels spill, D3Q15 FP64 with heat transfer already at 512)
template <class L, typename T, bool THERMAL, int NT>
constexpr bool kFits = kSlots<L, THERMAL> * NT * (int)sizeof(T) <= kLdsBytes &&
                       NT <= (!THERMAL ? 768 : (L::Q == 15 && sizeof(T) == 8 ? 256 : 512));

// node i's g after bounceBack (done by the caller) or fixedT / fixedRandomT
template <class L, typename T, int NT>
__device__ inline void tile_fixed_temp(const TileArgs<T>& a, const TileList& b, int draw, const int* nb,
                                       const int* inner, int step, const T (*gs)[NT], const T* sT, const T (*sU)[NT],
                                       T* v) {
    const bool random = b.type == BD_FRDT;
    T minT = 0, maxT = 0;
    if (random) {
        minT = T(b.value) * (T(100.0) - T(b.pert)) / T(100.0);
        maxT = T(b.value) * (T(100.0) + T(b.pert)) / T(100.0);
    }
#pragma unroll
    for (int q = 0; q < L::Q; q++) {
        if (nb[q] != -1) continue;
        const int n = nb[L::t.rev[q]];
        if (n == -1) continue;
        const T gnb = gs[q][inner[q]];
        const T Unb[3] = {sU[0][n], sU[1][n], L::D == 3 ? sU[L::D - 1][n] : T(0)};
        const T eq_nb = node_geq<L, T>(a.gp, q, sT[n], Unb);
        T Tw = T(b.value);
        if (random && step < b.left) {
            const T r = T(a.rnd[draw++]);
            Tw = minT + (maxT - minT) * r;
        }
        v[q] = node_geq<L, T>(a.gp, q, Tw, Unb) + (gnb - eq_nb);
    }
}

template <class L, typename T, bool THERMAL, int NT>
__global__ void __launch_bounds__(NT) k_tile(TileArgs<T> a) {
    __shared__ T fs[L::Q][NT];
    __shared__ T gs[THERMAL ? L::Q : 1][THERMAL ? NT : 1];
    __shared__ T s_psi[NT], s_rho[THERMAL ? NT : 1], s_T[THERMAL ? NT : 1], s_U[L::D][THERMAL ? NT : 1];
    constexpr int H = THERMAL ? 3 : 2;
    const int i = threadIdx.x;
    const int64_t e = (int64_t)blockIdx.x * a.t.stride + i, N = a.N;
    const bool surf = a.fp.surf != 0;
    // depth up to which the collision is needed; with surface tension the first one reads
    // its neighbours' psi, so one more level is loaded
    int R = H * a.steps + (surf ? 1 : 0);
    T v[L::Q], w[THERMAL ? L::Q : 1];
    T U[3] = {0, 0, 0}, Fi[3] = {0, 0, 0}, Ft[3] = {0, 0, 0};
    T rho = 0, temp = 0, ss = 0, psi = 0;
    int nb[L::Q], inner[THERMAL ? L::Q : 1], draw = 0;
    int64_t id = 0;
    const int meta = i < a.t.stride ? a.t.meta[e] : 255 << 24;
    const int depth = meta >> 24 & 0xFF;
    auto collide = [&](const T* psin, bool full) __attribute__((always_inline)) {
        T C[L::Q];
        if (surf) {
#pragma unroll
            for (int k = 0; k < L::Q; k++) C[k] = T(0);
            if (full) node_surface_tension<L, T>(a.eos, a.fp, psin, psi, C);
        }
        if constexpr (L::D == 2) node_collide_limrt<L, T>(a.fp, v, rho, U, Ft, Fi[0], Fi[1], psi, C);
        else node_collide_xumrt<L, T>(a.eos, a.fp, v, rho, U, Fi, psi, a.rho0, C);
#pragma unroll
        for (int q = 0; q < L::Q; q++) fs[q][i] = v[q];
        if constexpr (THERMAL) {
            if (L::D == 3 || a.gp.model == M_MYMRT) node_collide_my<L, T>(a.gp, w, temp, U, ss);
            else node_collide_litemp<L, T>(a.gp, w, temp, U, ss);
#pragma unroll
            for (int q = 0; q < L::Q; q++) gs[q][i] = w[q];
            s_T[i] = temp;
#pragma unroll
            for (int d = 0; d < L::D; d++) s_U[d][i] = U[d];
        }
    };
    // psi at the downstream nodes (own psi where the link is missing)
    auto stencil = [&](T* psin) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 1; q < L::Q; q++) {
            const int n = nb[L::t.rev[q]];
            psin[q] = n == -1 ? psi : s_psi[n];
        }
    };
    // the first collision, from the state in memory
    if (depth <= R) {
        id = a.t.gid[e];
#pragma unroll
        for (int q = 0; q < L::Q; q++) nb[q] = a.t.nb[q * a.t.total + e];
        if constexpr (THERMAL) {
            if (a.t.inner && (meta >> 8 & 0xFF) != 0xFF) {
#pragma unroll
                for (int q = 0; q < L::Q; q++) inner[q] = a.t.inner[q * a.t.total + e];
                if (a.t.draw) draw = a.t.draw[e];
            }
        }
#pragma unroll
        for (int q = 0; q < L::Q; q++) {
            v[q] = a.in.f[q * N + id];
            if constexpr (THERMAL) w[q] = a.in.g[q * N + id];
        }
        rho = a.in.rho[id];
        temp = a.in.temp[id];
        psi = a.in.psi[id];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            U[j] = a.in.U[j * N + id];
            Fi[j] = a.in.Fi[j * N + id];
            Ft[j] = a.in.Ft[j * N + id];
        }
        if constexpr (THERMAL) ss = a.in.ss[id];
        s_psi[i] = psi;
    }
    const bool interior = (meta >> 16 & 1) != 0, full = (meta >> 17 & 1) != 0;
    if (surf) __syncthreads();
    if (depth <= R) {
        T psin[L::Q];
        if (surf && depth < R) stencil(psin);
        collide(psin, full && depth < R);
    }
    __syncthreads();
    if (surf) R--;
    for (int s = 0; s < a.steps; s++) {
        if (depth <= R - 1) {
#pragma unroll
            for (int q = 0; q < L::Q; q++) v[q] = fs[q][nb[q] == -1 ? i : nb[q]];
            const int bf = meta & 0xFF;
            if (bf != 0xFF) {
                bool miss[L::Q];
#pragma unroll
                for (int q = 0; q < L::Q; q++) miss[q] = nb[q] == -1;
                node_bounce_back<L, T>(v, miss);
            }
            rho = node_sum<L, T>(v);
            if constexpr (THERMAL) {
                s_rho[i] = rho;
#pragma unroll
                for (int q = 0; q < L::Q; q++) w[q] = gs[q][nb[q] == -1 ? i : nb[q]];
                const int bg = meta >> 8 & 0xFF;
                if (bg != 0xFF) {
                    if (a.lists[1][bg].type == BD_BBACK) {
                        bool miss[L::Q];
#pragma unroll
                        for (int q = 0; q < L::Q; q++) miss[q] = nb[q] == -1;
                        node_bounce_back<L, T>(w, miss);
                    } else {
                        tile_fixed_temp<L, T, NT>(a, a.lists[1][bg], draw, nb, inner, s, gs, s_T, s_U, w);
                    }
                }
            } else {
                psi = potential<T>(a.eos, rho, temp);
                s_psi[i] = psi;
            }
        }
        __syncthreads();
        if constexpr (THERMAL) {
            if (depth <= R - 2) {
                T dot = 0, divU = 0;
                T gT[3] = {0, 0, 0}, gR[3] = {0, 0, 0};
#pragma unroll
                for (int ax = 0; ax < L::D; ax++) {
                    const int na = nb[L::fd_plus[ax]], nm = nb[L::fd_minus[ax]];
                    const bool ha = na != -1, hb = nm != -1;
                    const int ia = ha ? na : i, ib = hb ? nm : i;
                    gT[ax] = node_fd<T>(s_T[ia], ha, s_T[ib], hb, temp, false);
                    gR[ax] = node_fd<T>(s_rho[ia], ha, s_rho[ib], hb, rho, true);
                    divU += node_fd<T>(s_U[ax][ia], ha, s_U[ax][ib], hb, U[ax], false);
                }
#pragma unroll
                for (int k = 0; k < 3; k++) dot += gT[k] * gR[k];
                const T src = node_heat<L, T>(a.eos, a.gp, rho, temp, dot, divU);
                T t = node_sum<L, T>(w);
                if (a.gp.model == M_MYMRT) {
                    ss = src;
                    t = t + T(0.5) * ss;
                } else {
                    const T old = s == a.first_level ? T(0) : ss;
                    ss = src + T(0.5) * (src - old);
                }
                temp = t;
                psi = potential<T>(a.eos, rho, t);
                s_psi[i] = psi;
            }
            __syncthreads();
        }
        R -= H;
        if (depth <= R) {
            T psin[L::Q];
            stencil(psin);
            node_force<L, T>(a.eos, psin, psi, interior, Fi);
            node_total_force<T>(a.eos, Fi, rho, a.rho0, interior, Ft);
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const T F = L::D == 2 ? Ft[j] : Fi[j] + (rho - a.rho0) * T(a.eos.g[j]);
                U[j] = node_velocity<L, T>(v, rho, F, j);
            }
            if (s + 1 < a.steps) collide(psin, full);
        }
        __syncthreads();
    }
    if (depth == 0) {
#pragma unroll
        for (int q = 0; q < L::Q; q++) {
            a.out.f[q * N + id] = v[q];
            if constexpr (THERMAL) a.out.g[q * N + id] = w[q];
        }
        a.out.rho[id] = rho;
        a.out.psi[id] = psi;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            a.out.U[j * N + id] = U[j];
            a.out.Fi[j * N + id] = Fi[j];
            a.out.Ft[j * N + id] = Ft[j];
        }
        if constexpr (THERMAL) {
            a.out.temp[id] = temp;
            a.out.ss[id] = ss;
        }
    }
}

template <class L, typename T, bool THERMAL, int NT>
bool launch(hipStream_t s, const TileArgs<T>& a, int nodes) {
    if constexpr (kFits<L, T, THERMAL, NT>) {
        if (nodes > NT) return false;
        k_tile<L, T, THERMAL, NT><<<(unsigned)a.t.tiles, NT, 0, s>>>(a);
        return true;
    }
    return false;
}

template <class L, typename T, bool THERMAL>
constexpr int max_of() {
    if (kFits<L, T, THERMAL, 768>) return 768;
    return kFits<L, T, THERMAL, 512> ? 512 : 256;
}

}  // namespace

template <typename T>
int TileOps<T>::max_nodes(int model, bool thermal) {
    if (model == 0) return thermal ? max_of<D2Q9, T, true>() : max_of<D2Q9, T, false>();
    return thermal ? max_of<D3Q15, T, true>() : max_of<D3Q15, T, false>();
}

template <typename T>
void TileOps<T>::run(int model, hipStream_t s, const TileArgs<T>& a, bool thermal, int nodes) {
    auto go = [&](auto l, auto th) {
        using L = decltype(l);
        constexpr bool TH = decltype(th)::value;
        (void)(launch<L, T, TH, 256>(s, a, nodes) || launch<L, T, TH, 512>(s, a, nodes) ||
               launch<L, T, TH, 768>(s, a, nodes));
    };
    if (model == 0 && thermal) go(D2Q9{}, std::true_type{});
    else if (model == 0) go(D2Q9{}, std::false_type{});
    else if (thermal) go(D3Q15{}, std::true_type{});
    else go(D3Q15{}, std::false_type{});
}

template struct TileOps<double>;
template struct TileOps<float>;

}  // namespace mplb
