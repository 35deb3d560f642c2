// Neighbours of a node of a structured box: computed from wrapped coordinates, or read from
// the neighbour table: on the faces that cover the nodes with odd links or a boundary
// condition (odd_faces, mesh.h), or everywhere where such nodes lie inside (plain_inside).
#pragma once

#include <hip/hip_runtime.h>

#include "lattice.h"

namespace mplb {

// bits of face_table: the faces x0 x1 y0 y1 z0 z1, and this one for all nodes
constexpr int kAllTable = 64;

struct NodePos {
    int i, j, k;
    int64_t id;
    bool table;         // links and boundary conditions come from the tables
    bool valid;
    unsigned X[3], Y[3], Z[3];   // wrapped coordinates u-1, u, u+1 premultiplied by the strides
};

// Block b covers the 256 consecutive node ids [256 b, 256 b + 256).  A: kernel arguments
// with nx, ny, nz, nxy, N, face_table and nb.
template <class L, class A>
__device__ inline NodePos node_pos(const A& a) {
    NodePos p;
    const unsigned id = blockIdx.x * 256u + threadIdx.x;     // N < 2^31
    const unsigned nxy = (unsigned)a.nxy, nx = (unsigned)a.nx;
    p.id = id;
    p.valid = p.id < a.N;
    const unsigned k = id / nxy, r = id - k * nxy, j = r / nx;
    p.k = (int)k;
    p.j = (int)j;
    p.i = (int)(r - j * nx);
    const bool x0 = p.i == 0, x1 = p.i == a.nx - 1, y0 = p.j == 0, y1 = p.j == a.ny - 1;
    const bool z0 = L::D == 3 && p.k == 0, z1 = L::D == 3 && p.k == a.nz - 1;
    const int m = a.face_table;
    p.table = (m & kAllTable) || (x0 && (m & 1)) || (x1 && (m & 2)) || (y0 && (m & 4)) || (y1 && (m & 8)) || (z0 && (m & 16)) ||
              (z1 && (m & 32));
    // periodic wrap with duplicate end nodes: u - 1 at 0 is n - 2, u + 1 at n - 1 is 1
    p.X[0] = x0 ? nx - 2 : p.i - 1;
    p.X[1] = p.i;
    p.X[2] = x1 ? 1 : p.i + 1;
    p.Y[0] = (y0 ? a.ny - 2 : p.j - 1) * nx;
    p.Y[1] = j * nx;
    p.Y[2] = (y1 ? 1 : p.j + 1) * nx;
    if (L::D == 3) {
        p.Z[0] = (z0 ? a.nz - 2 : p.k - 1) * nxy;
        p.Z[1] = k * nxy;
        p.Z[2] = (z1 ? 1 : p.k + 1) * nxy;
    } else {
        p.Z[0] = p.Z[1] = p.Z[2] = 0;
    }
    return p;
}

// upstream node x - c_q (lbstream.c:16-62: a missing link keeps the node's own value)
template <class L, class A>
__device__ inline unsigned upstream(const A& a, const NodePos& p, int q) {
    if (p.table) {
        const int s = a.nb[q * a.N + p.id];
        return s == -1 ? (unsigned)p.id : (unsigned)s;
    }
    return p.X[1 - L::t.c[q][0]] + p.Y[1 - L::t.c[q][1]] + p.Z[1 - L::t.c[q][2]];
}

// downstream node x + c_q (the interaction-force and stencil neighbour), -1 if missing
template <class L, class A>
__device__ inline int64_t downstream(const A& a, const NodePos& p, int q) {
    if (p.table) return a.nb[L::t.rev[q] * a.N + p.id];
    return (int64_t)(p.X[1 + L::t.c[q][0]] + p.Y[1 + L::t.c[q][1]] + p.Z[1 + L::t.c[q][2]]);
}

// All upstream / downstream nodes in one branch: a branch for each neighbour keeps a node's
// loads from going out together.
template <class L, class A>
__device__ inline void upstreams(const A& a, const NodePos& p, unsigned* up) {
    if (p.table) {
#pragma unroll
        for (int q = 0; q < L::Q; q++) {
            const int s = a.nb[q * a.N + p.id];
            up[q] = s == -1 ? (unsigned)p.id : (unsigned)s;
        }
    } else {
#pragma unroll
        for (int q = 0; q < L::Q; q++) up[q] = p.X[1 - L::t.c[q][0]] + p.Y[1 - L::t.c[q][1]] + p.Z[1 - L::t.c[q][2]];
    }
}

template <class L, class A>
__device__ inline void downstreams(const A& a, const NodePos& p, int* dn) {
    if (p.table) {
#pragma unroll
        for (int q = 0; q < L::Q; q++) dn[q] = a.nb[L::t.rev[q] * a.N + p.id];
    } else {
#pragma unroll
        for (int q = 0; q < L::Q; q++)
            dn[q] = (int)(p.X[1 + L::t.c[q][0]] + p.Y[1 + L::t.c[q][1]] + p.Z[1 + L::t.c[q][2]]);
    }
}

}  // namespace mplb
