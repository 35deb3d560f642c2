// Tile plans of small lattices: which nodes a workgroup of k_tile owns, how many steps it
// takes per launch, and the local node lists it works on.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <exception>
#include <memory>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "case.h"
#include "tiles.h"

namespace mplb {

namespace {

// rho, T, U, Fi, Ft, ss, psi (mplb_case::alt): those that change with heat transfer only
constexpr bool kHeatField[7] = {false, true, false, false, false, true, false};

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
double plan_us(const TilePlan& p, const int n[3], bool thermal, bool d3, bool fp64, int cap, int extra, int cus) {
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

}  // namespace

TilePlan tile_choose(const mplb_case* c, const std::vector<int>& sizes, double limit_us,
                     const std::function<double(const TilePlan&)>& us) {
    const Mesh& m = c->mesh;
    TilePlan best;
    best.us = limit_us;
    if (!m.structured) return best;      // no neighbourhood to size a block by
    const int n[3] = {m.nx, m.ny, m.nz};
    for (int bx : sizes)
        for (int by : sizes)
            for (int bz : sizes) {
                if (m.d == 2 && bz > 1) break;
                TilePlan p;
                const int want[3] = {bx, by, bz};
                bool ok = true;
                for (int d = 0; d < 3; d++) {
                    p.b[d] = std::min(want[d], n[d]);
                    ok = ok && (want[d] < 2 * n[d]);
                }
                if (!ok) continue;
                for (p.steps = 1; p.steps <= 12; p.steps++) {
                    p.us = us(p);
                    if (p.us >= 1e29) break;
                    if (p.us < best.us) best = p;
                }
            }
    return best;
}

void tile_override(TilePlan* p) {
    if (const char* env = std::getenv("MPLB_TILES")) {
        if (std::sscanf(env, "%d,%d,%d,%d", &p->b[0], &p->b[1], &p->b[2], &p->steps) != 4) p->steps = 0;
        for (int d = 0; d < 3; d++) p->b[d] = std::max(1, p->b[d]);
    }
}

void tiles_destroy(mplb_case* c) {
    if (!c->tiles) return;
    for (void* p : c->tiles->owned)
        if (p) (void)hipFree(p);
    delete c->tiles;
    c->tiles = nullptr;
    for (void*& p : c->alt) {
        if (p) (void)hipFree(p);
        p = nullptr;
    }
}

namespace {

// fn(t, mark, slot) for every tile, on a few threads; mark (-1 at first) and slot are a
// thread's own entries per node.  False: memory ran out.
template <typename Fn>
bool over_tiles(size_t tiles, int64_t N, const Fn& fn) {
    std::atomic<size_t> next{0};
    std::atomic<bool> ok{true};
    auto work = [&] {
        try {
            std::vector<int> mark, slot;
            for (size_t t; (t = next++) < tiles && ok;) {
                if (mark.empty()) {
                    mark.assign(N, -1);
                    slot.assign(N, 0);
                }
                fn(t, mark, slot);
            }
        } catch (const std::bad_alloc&) {
            ok = false;
        }
    };
    std::vector<std::thread> pool;
    for (size_t i = 1; i < std::min<size_t>(8, tiles / 8); i++) {
        try {
            pool.emplace_back(work);
        } catch (const std::exception&) {
            break;                       // fewer threads do the same
        }
    }
    work();
    for (std::thread& t : pool) t.join();
    return ok;
}

}  // namespace

void tiles_create(mplb_case* c) {
    const Mesh& m = c->mesh;
    const bool thermal = c->fc[1].present && c->update[1], fp64 = c->scalar_bytes == 8;
    if (!c->passes || m.N > 1 << 20 || m.bd.size() > (size_t)kTileLists) return;
    const int cap = fp64 ? TileOps<double>::max_nodes(m.lbmodel, thermal) : TileOps<float>::max_nodes(m.lbmodel, thermal);
    const int H = thermal ? 3 : 2, extra = c->fc[0].mp.surf ? 1 : 0;
    const int n[3] = {m.nx, m.ny, m.nz};
    const std::vector<int> sizes = {1, 2, 3, 4, 5, 6, 8, 10, 12, 14, 16, 20, 24, 32, 48, 64, 128};
    int cus = 256;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->opts.device);
    TilePlan p = tile_choose(c, sizes, 0.85 * passes_us(c, thermal, fp64), [&](const TilePlan& q) {
        return plan_us(q, n, thermal, m.d == 3, fp64, cap, extra, cus);
    });
    tile_override(&p);
    if (p.steps <= 0) return;
    const bool lists[2] = {c->order[0] != nullptr, c->order[1] != nullptr};
    if (!tile_tables(c, p, H * p.steps + extra, cap, lists)) return;
    // second copies of the macroscopic fields: a launch reads one set and writes the other
    // (T and the heat source change with heat transfer only)
    const int comps[7] = {1, 1, 3, 3, 3, 1, 1};
    for (int i = 0; i < 7; i++)
        if ((thermal || !kHeatField[i]) && !device_alloc(&c->alt[i], c->scalar_bytes * comps[i] * m.N)) return tiles_destroy(c);
}

namespace {

bool build_tables(mplb_case* c, const TilePlan& p, int D, int cap, const bool lists[2]);

}  // namespace

bool tile_tables(mplb_case* c, const TilePlan& p, int depth, int cap, const bool lists[2]) {
    try {
        if (build_tables(c, p, depth, cap, lists)) return true;
    } catch (const std::bad_alloc&) {
        // host memory ran out: without tiles as well
    }
    tiles_destroy(c);
    return false;
}

namespace {

bool build_tables(mplb_case* c, const TilePlan& p, int D, int cap, const bool lists[2]) {
    const Mesh& m = c->mesh;
    const int Q = m.Q;
    const bool thermal = c->fc[1].present && c->update[1];
    // the g lists of fixedT nodes, whose condition reads the population that their inner
    // neighbour pulled: it must not come from a list applied before
    std::vector<int> list[2];
    for (int f = 0; f < 2; f++) {
        list[f].assign(m.N, 255);
        if (!lists[f]) continue;
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
    // tile t's nodes from local[t * cap], level d ending at ends[t * (D + 1) + d]
    if (own.size() * (size_t)cap > size_t(1) << 26 || D > 250) return false;
    const std::unique_ptr<int[]> local(new int[own.size() * cap]), ends(new int[own.size() * (D + 1)]);
    std::atomic<bool> fits{true};
    const bool listed = over_tiles(own.size(), m.N, [&](size_t t, std::vector<int>& mark, std::vector<int>&) {
        int *nodes = &local[t * cap], *end = &ends[t * (D + 1)], n = 0;
        auto add = [&](int64_t id) {
            if (id < 0 || mark[id] == (int)t) return;
            mark[id] = (int)t;
            if (n < cap) nodes[n] = (int)id;
            n++;
        };
        for (int id : own[t]) add(id);
        int from = 0;
        for (int d = 0; d <= D && fits; d++) {
            if (n > cap) fits = false;
            if (!fits) break;
            // (in memory order, so that a wavefront's loads share sectors)
            std::sort(nodes + from, nodes + n);
            const int to = end[d] = n;
            for (int i = from; i < to && d < D; i++) {
                const int64_t id = nodes[i];
                for (int k = 0; k < Q; k++) add(m.nb[id * Q + k]);
                if (!fixed_t(id)) continue;
                for (int k = 0; k < Q; k++) {
                    const int64_t in = m.nb[id * Q + tile_reverse(m, k)];
                    if (m.nb[id * Q + k] != -1 || in == -1) continue;
                    if (list[1][in] < list[1][id]) fits = false;
                    add(m.nb[in * Q + k]);
                }
            }
            from = to;
        }
    });
    if (!listed || !fits) return false;
    size_t largest = 0;
    for (size_t t = 0; t < own.size(); t++) largest = std::max(largest, (size_t)ends[t * (D + 1) + D]);
    const size_t total = own.size() * largest;
    if (total > size_t(1) << 23) return false;
    const bool any_fixed = thermal && lists[1];
    std::vector<int16_t> nb(total * Q, -1), inner(any_fixed ? total * Q : 0, 0);
    std::vector<int> gid(total, 0), meta(total, 255 << 24), draw(draws.empty() ? 0 : total);
    const bool filled = over_tiles(own.size(), m.N, [&](size_t t, std::vector<int>& mark, std::vector<int>& slot) {
        const int *nodes = &local[t * cap], *end = &ends[t * (D + 1)];
        const int count = end[D];
        for (int i = 0; i < count; i++) {
            mark[nodes[i]] = (int)t;
            slot[nodes[i]] = i;
        }
        // neighbours outside the tile belong to its rim and are never followed
        auto at = [&](int32_t n) { return (int16_t)(n != -1 && mark[n] == (int)t ? slot[n] : -1); };
        for (int i = 0, depth = 0; i < count; i++) {
            while (i >= end[depth]) depth++;
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
                      depth << 24;
            if (!draws.empty()) draw[e] = draws[id];
        }
    });
    if (!filled) return false;
    Tiles* s = new Tiles();
    c->tiles = s;
    auto put = [&](const void* src, size_t bytes, const void** dst) {
        void* q = nullptr;
        s->owned.push_back(nullptr);
        if (!device_alloc(&q, bytes)) return false;
        s->owned.back() = q;
        *dst = q;
        return hipMemcpy(q, src, bytes, hipMemcpyHostToDevice) == hipSuccess;
    };
    if (!put(gid.data(), sizeof(int) * total, (const void**)&s->t.gid) ||
        !put(nb.data(), sizeof(int16_t) * nb.size(), (const void**)&s->t.nb) ||
        (any_fixed && !put(inner.data(), sizeof(int16_t) * inner.size(), (const void**)&s->t.inner)) ||
        !put(meta.data(), sizeof(int) * total, (const void**)&s->t.meta) ||
        (!draw.empty() && !put(draw.data(), sizeof(int) * total, (const void**)&s->t.draw)))
        return false;
    s->t.tiles = (int)own.size();
    s->t.stride = (int)largest;
    s->t.total = (int64_t)total;
    s->nodes = (int)largest;
    s->steps = p.steps;
    return true;
}

}  // namespace

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
            if (thermal || !kHeatField[i]) std::swap(*cur[i], c->alt[i]);
        done += a.steps;
    }
}

template void tiles_run<double>(mplb_case*, int, int);
template void tiles_run<float>(mplb_case*, int, int);

}  // namespace mplb
