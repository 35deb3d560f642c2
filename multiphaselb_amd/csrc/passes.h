// Launch interface of the fused passes of the per-routine arithmetic (kernels_passes.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"

namespace mplb {

// Device view of one step: populations are read from fin / gin (post-collision, pulled)
// and written to fout / gout.
template <typename T>
struct PassArgs {
    int nx, ny, nz;
    int64_t N, nxy;
    int face_table;              // faces read through the neighbour table (boxidx.h)
    const int* nb;               // [Q][N]
    const uint8_t* onbnd;
    const uint8_t* order[2];     // per field: the node's boundary list (255: none); null without lists
    EosParams eos;
    ModelParams fp, gp;
    T rho0;
    const T* fin;
    T* fout;
    const T* gin;
    T* gout;
    T* rho;
    T* temp;
    T* U;                        // [3][N]
    T* Fi;
    T* Ft;
    T* ss;
    T* psi;
    T* sumg;                     // sum of g, then the new temperature
    int first_call;              // liTempMRT heat source S_old = 0
};

// Work split of the single-pass march over a fully periodic D3Q15 box (items 0: not used)
struct PassMarch {
    int mtx = 0, tiles = 0, items = 0, per = 0, zc = 0;
};

template <typename T>
struct PassOps {
    // boundary condition of one list of field fld (0 f, 1 g): the nodes' pulled and
    // corrected populations go to fout / gout, where the passes pick them up
    static void boundary(int model, hipStream_t s, const PassArgs<T>& a, int fld, int order, const BdList& b);
    // rho, and psi (isothermal) or the sum of g (thermal)
    static void density(int model, hipStream_t s, const PassArgs<T>& a, bool thermal);
    // heat source, new temperature (in sumg) and psi
    static void heat(int model, hipStream_t s, const PassArgs<T>& a);
    // force, velocity and the collisions of the next step; last: no collision, the
    // post-stream populations and every macroscopic field instead
    static void collide(int model, hipStream_t s, const PassArgs<T>& a, bool thermal, bool last);
    // density and collide passes of an isothermal step in one (the plan stays empty where the
    // two passes are the better choice)
    static int march_plan(int device, int nx, int ny, int nz, PassMarch* p);
    static void march(hipStream_t s, const PassArgs<T>& a, const PassMarch& p, bool last);
};

}  // namespace mplb
