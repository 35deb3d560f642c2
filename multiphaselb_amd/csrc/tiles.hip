// Tile plans of small lattices: which nodes a workgroup of k_tile owns, how many steps it
// takes per launch, and the local node lists it works on.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "case.h"
#include "tiles.h"

namespace mplb {

namespace {

struct Plan {
    int b[3] = {0, 0, 0};        // owned block (structured boxes); b[0] consecutive nodes otherwise
    int steps = 0;
    double us = 0;               // estimated time of a step
};

#define TCHK(c, call)                                                           \
    do {                                                                        \
        hipError_t _e = (call);                                                 \
        if (_e != hipSuccess) {                                                 \
            (c)->err = std::string(#call) + ": " + hipGetErrorString(_e);       \
            return MPLB_E_HIP;                                                  \
        }                                                                       \
    } while (0)

int tile_reverse(const Mesh& m, int k) { return m.lbmodel == 0 ? D2Q9::t.rev[k] : D3Q15::t.rev[k]; }

// Time of one step with a plan, in microseconds: a launch with the load of its state, then
// per step a latency (barriers, LDS, the dependent arithmetic of one node) and the
// arithmetic of every 256 nodes, a wavefront on each SIMD; more tiles than CUs take turns.
// The constants fit D2Q9 FP64 runs on MI355X: 128^2 in 8 x 8 blocks 8.1, 10.7, 14.0 and 18.2
// us per launch of 1 to 4 steps (11.3 us per step in passes); 128^2 with heat transfer 11.8
// and 17.7 us for 1 and 2 steps (18.7); 3 x 301 with heat transfer 4.2 us per further step.
// Chosen by it, us per step in tiles against passes: D2Q9 64^2 3.6 / 10.7, 128^2 4.5 / 11.0,
// 256^2 7.9 / 12.3; with heat transfer 64^2 7.0 / 17.6, 128^2 8.8 / 18.4, 3 x 301 column 4.7 / 28.4
// (its walls are launches of their own in passes), 3 x 3 x 301 D3Q15 column 9.9 / 40.7.  From
// about 300^2 on the halo costs more than the launches it saves.
double plan_us(const Plan& p, const int n[3], bool thermal, bool d3, bool fp64, int cap, int extra, int cus) {
    const int H = thermal ? 3 : 2;
    const double scale = (d3 ? 1.7 : 1.0) * (fp64 ? 1.0 : 0.6);
    const double wait = (thermal ? 2.2 : 1.0) * scale, work = (thermal ? 2.0 : 1.05) * scale;
    double sum = 0, load = 0;
    int64_t tiles = 1;
    for (int d = 0; d < 3; d++) tiles *= (n[d] + p.b[d] - 1) / p.b[d];
    for (int s = p.steps; s > 0; s--) {
        int64_t local = 1;
        for (int d = 0; d < 3; d++) local *= std::min(n[d], p.b[d] + 2 * (H * s + extra) + 1);
        if (local > cap) return 1e30;
        if (s == p.steps) load = (double)local / (thermal ? 90 : 150);
        sum += wait + work * (double)((local + 255) / 256);
    }
    const double rounds = (double)((tiles + cus - 1) / cus);
    return (5.0 + (rounds > 1 ? 1.25 * rounds : 1.0) * (sum + load)) / p.steps;
}

// Time of one step in fused passes: its launches, and the bytes it moves
double passes_us(const mplb_case* c, bool thermal, bool fp64) {
    double us = 5.5 * (thermal ? 3 : 2);
    for (int f = 0; f < (thermal ? 2 : 1); f++)
        if (c->order[f])
            for (size_t b = 0; b < c->bd.size(); b++) us += c->fc[f].bctype[b] != BD_PERIODIC ? 2.5 : 0.0;
    const double per = (thermal ? 6.0 * c->mesh.Q + 20 : 3.0 * c->mesh.Q + 4) * (fp64 ? 8 : 4);
    return us + (double)c->mesh.N * per / 5e6;
}

Plan choose(mplb_case* c, int cap, bool thermal, bool fp64, int extra) {
    const Mesh& m = c->mesh;
    const bool d3 = m.d == 3;
    int cus = 256;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->opts.device);
    Plan best;
    best.us = 0.85 * passes_us(c, thermal, fp64);
    const int n[3] = {m.structured ? m.nx : (int)m.N, m.structured ? m.ny : 1, m.structured ? m.nz : 1};
    if (!m.structured) return best;      // no neighbourhood to size a block by
    static const int sizes[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 14, 16, 20, 24, 32, 48, 64, 128};
    for (int bx : sizes)
        for (int by : sizes)
            for (int bz : sizes) {
                if (!d3 && bz > 1) break;
                Plan p;
                const int want[3] = {bx, by, bz};
                bool ok = true;
                for (int d = 0; d < 3; d++) {
                    p.b[d] = std::min(want[d], n[d]);
                    ok = ok && (want[d] < 2 * n[d]);
                }
                if (!ok || (int64_t)p.b[0] * p.b[1] * p.b[2] > cap) continue;
                for (p.steps = 1; p.steps <= 12; p.steps++) {
                    p.us = plan_us(p, n, thermal, d3, fp64, cap, extra, cus);
                    if (p.us >= 1e29) break;
                    if (p.us < best.us) best = p;
                }
            }
    return best;
}

}  // namespace

// What a tiled case keeps on the device
struct Tiles {
    TileTable t{};
    int nodes = 0;               // largest tile
    int steps = 0;               // per launch
    std::vector<void*> owned;
};

void tiles_destroy(mplb_case* c) {
    if (!c->tiles) return;
    for (void* p : c->tiles->owned) (void)hipFree(p);
    delete c->tiles;
    c->tiles = nullptr;
    for (void*& p : c->alt) {
        if (p) (void)hipFree(p);
        p = nullptr;
    }
}

int tiles_create(mplb_case* c) {
    const Mesh& m = c->mesh;
    const bool thermal = c->fc[1].present && c->update[1], fp64 = c->scalar_bytes == 8;
    if (!c->passes || m.N > 1 << 20 || m.bd.size() > (size_t)kTileLists) return 0;
    const int cap = fp64 ? TileOps<double>::max_nodes(m.lbmodel, thermal) : TileOps<float>::max_nodes(m.lbmodel, thermal);
    const int H = thermal ? 3 : 2, extra = c->fc[0].mp.surf ? 1 : 0, Q = m.Q;
    Plan p = choose(c, cap, thermal, fp64, extra);
    // MPLB_TILES=bx,by,bz,steps sets the plan (steps 0: fused passes), for tests and timing sweeps
    if (const char* env = std::getenv("MPLB_TILES")) {
        if (std::sscanf(env, "%d,%d,%d,%d", &p.b[0], &p.b[1], &p.b[2], &p.steps) != 4) p.steps = 0;
        for (int d = 0; d < 3; d++) p.b[d] = std::max(1, p.b[d]);
    }
    if (p.steps <= 0) return 0;
    const int D = H * p.steps + extra;
    // the g lists of fixedT nodes, whose condition reads the population that their inner
    // neighbour pulled: it must not come from a list applied before
    std::vector<int> list[2];
    for (int f = 0; f < 2; f++) {
        list[f].assign(m.N, 255);
        if (!c->order[f]) continue;
        for (size_t b = 0; b < m.bd.size(); b++) {
            const int t = c->fc[f].bctype[b];
            if (t == BD_BBACK || t == BD_FT || t == BD_FRDT)
                for (int32_t id : m.bd[b]) list[f][id] = (int)b;
        }
    }
    auto fixed_t = [&](int64_t id) { return list[1][id] != 255 && c->fc[1].bctype[list[1][id]] != BD_BBACK; };
    std::vector<int> draws;
    if (thermal && c->rnd) {
        draws.assign(m.N, 0);
        for (size_t b = 0; b < m.bd.size(); b++) {
            if (c->fc[1].bctype[b] != BD_FRDT) continue;
            int n = 0;
            for (int32_t id : m.bd[b]) {
                draws[id] = n;
                for (int k = 0; k < Q; k++)
                    n += m.nb[(int64_t)id * Q + k] == -1 && m.nb[(int64_t)id * Q + tile_reverse(m, k)] != -1;
            }
        }
    }
    // owners, then each tile's halo level by level
    std::vector<std::vector<int>> own;
    {
        const int nx = m.structured ? m.nx : (int)m.N, ny = m.structured ? m.ny : 1, nz = m.structured ? m.nz : 1;
        for (int k0 = 0; k0 < nz; k0 += p.b[2])
            for (int j0 = 0; j0 < ny; j0 += p.b[1])
                for (int i0 = 0; i0 < nx; i0 += p.b[0]) {
                    own.emplace_back();
                    for (int k = k0; k < std::min(nz, k0 + p.b[2]); k++)
                        for (int j = j0; j < std::min(ny, j0 + p.b[1]); j++)
                            for (int i = i0; i < std::min(nx, i0 + p.b[0]); i++)
                                own.back().push_back((int)(i + (int64_t)j * nx + (int64_t)k * nx * ny));
                }
    }
    std::vector<int> mark(m.N, -1), slot(m.N, 0);
    std::vector<std::vector<int>> local(own.size()), level(own.size());   // nodes, and their depths
    size_t largest = 0;
    for (size_t t = 0; t < own.size(); t++) {
        std::vector<int>&nodes = local[t], &depth = level[t];
        int at = 0;
        auto add = [&](int64_t id) {
            if (id < 0 || mark[id] == (int)t) return;
            mark[id] = (int)t;
            slot[id] = (int)nodes.size();
            nodes.push_back((int)id);
            depth.push_back(at);
        };
        for (int id : own[t]) add(id);
        size_t from = 0;
        for (int d = 0; d < D; d++) {
            const size_t to = nodes.size();
            at = d + 1;
            for (size_t i = from; i < to; i++) {
                const int64_t id = nodes[i];
                for (int k = 0; k < Q; k++) add(m.nb[id * Q + k]);
                if (!fixed_t(id)) continue;
                for (int k = 0; k < Q; k++) {
                    const int64_t in = m.nb[id * Q + tile_reverse(m, k)];
                    if (m.nb[id * Q + k] != -1 || in == -1) continue;
                    if (list[1][in] < list[1][id]) return 0;
                    add(m.nb[in * Q + k]);
                }
            }
            from = to;
        }
        largest = std::max(largest, nodes.size());
        if (largest > (size_t)cap) return 0;
    }
    const size_t total = own.size() * largest;
    if (total > size_t(1) << 23 || D > 250) return 0;
    const bool any_fixed = thermal && c->order[1];
    std::vector<int16_t> nb(total * Q, -1), inner(any_fixed ? total * Q : 0, 0);
    std::vector<int> gid(total, 0), meta(total, 255 << 24), draw(draws.empty() ? 0 : total);
    for (size_t t = 0; t < own.size(); t++) {
        const std::vector<int>& nodes = local[t];
        const int stamp = (int)(own.size() + t);
        for (size_t i = 0; i < nodes.size(); i++) {
            mark[nodes[i]] = stamp;
            slot[nodes[i]] = (int)i;
        }
        // neighbours outside the tile belong to its rim and are never followed
        auto at = [&](int32_t n) { return (int16_t)(n != -1 && mark[n] == stamp ? slot[n] : -1); };
        for (size_t i = 0; i < nodes.size(); i++) {
            const int64_t id = nodes[i];
            const size_t e = t * largest + i;
            gid[e] = (int)id;
            bool full = true;
            for (int k = 0; k < Q; k++) {
                const int32_t n = m.nb[id * Q + k];
                full = full && n != -1;
                nb[k * total + e] = at(n);
                const int32_t in = m.nb[id * Q + tile_reverse(m, k)];
                if (any_fixed && fixed_t(id) && n == -1 && in != -1) {
                    // post-stream population k of the inner neighbour: its upstream node's, or its
                    // own where that link is missing
                    const int32_t up = m.nb[(int64_t)in * Q + k];
                    inner[k * total + e] = std::max<int16_t>(0, at(up == -1 ? in : up));
                }
            }
            meta[e] = list[0][id] | list[1][id] << 8 | (m.onbnd[id] == 0 ? 1 << 16 : 0) | (full ? 1 << 17 : 0) |
                      level[t][i] << 24;
            if (!draws.empty()) draw[e] = draws[id];
        }
    }
    Tiles* s = new Tiles();
    c->tiles = s;
    auto put = [&](const void* src, size_t bytes, const void** dst) -> int {
        void* q = nullptr;
        TCHK(c, hipMalloc(&q, bytes ? bytes : 1));
        s->owned.push_back(q);
        TCHK(c, hipMemcpy(q, src, bytes, hipMemcpyHostToDevice));
        *dst = q;
        return 0;
    };
    int rc = put(gid.data(), sizeof(int) * total, (const void**)&s->t.gid);
    if (!rc) rc = put(nb.data(), sizeof(int16_t) * nb.size(), (const void**)&s->t.nb);
    if (!rc && any_fixed) rc = put(inner.data(), sizeof(int16_t) * inner.size(), (const void**)&s->t.inner);
    if (!rc) rc = put(meta.data(), sizeof(int) * total, (const void**)&s->t.meta);
    if (!rc && !draw.empty()) rc = put(draw.data(), sizeof(int) * total, (const void**)&s->t.draw);
    if (rc) return rc;
    s->t.tiles = (int)own.size();
    s->t.stride = (int)largest;
    s->t.total = (int64_t)total;
    s->nodes = (int)largest;
    s->steps = p.steps;
    // second copies of the macroscopic fields: a launch reads one set and writes the other
    const int comps[7] = {1, 1, 3, 3, 3, 1, 1};
    for (int i = 0; i < 7; i++) TCHK(c, hipMalloc(&c->alt[i], c->scalar_bytes * comps[i] * m.N));
    return 0;
}

template <typename T>
void tiles_run(mplb_case* c, int m, int level0) {
    const Tiles* s = c->tiles;
    const bool thermal = c->fc[1].present && c->update[1];
    TileArgs<T> a{};
    a.t = s->t;
    a.N = c->mesh.N;
    a.eos = c->eos;
    a.fp = c->fc[0].mp;
    a.gp = c->fc[1].mp;
    a.rho0 = T(c->rho0);
    a.rnd = c->rnd;
    void** cur[7] = {&c->rho, &c->temp, &c->U, &c->Fi, &c->Ft, &c->ss, &c->psi};
    auto view = [&](void* f, void* g, bool other) {
        TileState<T> v;
        v.f = (T*)f;
        v.g = (T*)g;
        T** to[7] = {&v.rho, &v.temp, &v.U, &v.Fi, &v.Ft, &v.ss, &v.psi};
        for (int i = 0; i < 7; i++) *to[i] = (T*)(other ? c->alt[i] : *cur[i]);
        return v;
    };
    for (int done = 0; done < m;) {
        a.steps = std::min(s->steps, m - done);
        a.first_level = -1 - (level0 + done) >= 0 ? -1 - (level0 + done) : -1;
        for (int f = 0; f < (thermal ? 2 : 1); f++)
            for (size_t b = 0; b < c->bd.size(); b++) {
                FieldCfg& fc = c->fc[f];
                TileList& l = a.lists[f][b];
                l.type = fc.bctype[b];
                l.value = fc.bcval[b][0];
                l.pert = fc.pert[b];
                l.left = fc.psteps[b] - fc.localT[b];
                if (l.type == BD_FRDT) fc.localT[b] += a.steps;
            }
        a.in = view(c->f[0], c->f[1], false);
        a.out = view(c->f_alt[0], c->f_alt[1], true);
        TileOps<T>::run(c->mesh.lbmodel, c->stream, a, thermal, s->nodes);
        for (int f = 0; f < (thermal ? 2 : 1); f++) std::swap(c->f[f], c->f_alt[f]);
        for (int i = 0; i < 7; i++)
            if (thermal || (i != 1 && i != 5)) std::swap(*cur[i], c->alt[i]);
        done += a.steps;
    }
}

template void tiles_run<double>(mplb_case*, int, int);
template void tiles_run<float>(mplb_case*, int, int);

}  // namespace mplb
