// Runs SyncPlan's launches on the CPU against the ops applied one after the other.
//   sync_plan_check G BLOCKS [one_op]
// BLOCKS: m0xm1xm2:WALLS,...  (WALLS: the faces 0..5 that are solid, the others are
// far field).  Prints the number of launches and of values written; fails when a
// value differs, when another set of values is written, or when a lane reads or
// writes what another lane of the launch writes.  one_op: all walls in one op.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <memory>
#include <random>
#include <set>
#include <string>

#include "mercury_sync_plan.h"

using namespace merc;
namespace {

struct Blk {
    int m[3], off;
    bool wall[6];
};
int g = 2;
int at(const Blk &b, int i, int j, int k) { return b.off + ((i + g) * (b.m[1] + 2 * g) + j + g) * (b.m[2] + 2 * g) + k + g; }

constexpr int NC = 5, SLOT = 0;
using State = std::vector<double>;  // values, component major
double rho_floor = 0.6, p_floor = 0.05, gm1 = 5.0 / 3.0 - 1.0;
void reflect(double v[5]) {
    const double rho = std::max(v[0], rho_floor);
    double eint = v[4] - 0.5 * (v[1] * v[1] + v[2] * v[2] + v[3] * v[3]) / rho;
    if (eint < 0.0) eint = 0.0;
    v[0] = rho;
    v[1] = v[2] = v[3] = rho * 0.0;
    v[4] = std::max(gm1 * eint, p_floor) / gm1;
}

int fail(const char *what, long long n) {
    std::printf("%s %lld\n", what, n);
    return 1;
}

}  // namespace

int main(int argc, char **argv) {
    if (argc < 3) return 2;
    g = std::atoi(argv[1]);
    std::vector<Blk> blk;
    int V = 0;
    for (const char *s = argv[2]; *s;) {
        Blk b{};
        int n = 0;
        if (std::sscanf(s, "%dx%dx%d:%n", b.m, b.m + 1, b.m + 2, &n) != 3 || !n) return 2;
        for (s += n; *s >= '0' && *s <= '5'; ++s) b.wall[*s - '0'] = true;
        if (*s == ',') ++s;
        b.off = V;
        V += (b.m[0] + 2 * g) * (b.m[1] + 2 * g) * (b.m[2] + 2 * g);
        blk.push_back(b);
    }
    const bool one_op = argc > 3 && std::string(argv[3]) == "one_op";

    // far-field ghosts, walls face by face, then the corner ghosts from the nearest cell
    std::vector<std::unique_ptr<SyncOp>> ops;
    auto add = [&](OpType t) {
        ops.emplace_back(new SyncOp());
        ops.back()->type = t;
        for (int c = 0; c < NC; ++c) ops.back()->slots.push_back(SLOT + c);
        return ops.back().get();
    };
    SyncOp *far = add(OP_FILL);
    far->fillv = {1.0, 0.5, 0.25, 0.125, 3.0};
    std::vector<SyncOp *> wall;
    for (int f = 0; f < 6; ++f) wall.push_back(f == 0 || !one_op ? add(OP_WALLF) : wall[0]);
    SyncOp *corner = add(OP_COPY);
    for (const Blk &b : blk)
        for (int f = 0; f < 6; ++f) {
            const int a = f / 2, s = f & 1 ? 1 : -1;
            int n[3] = {b.m[0], b.m[1], b.m[2]};
            n[a] = 1;
            for (int i = 0; i < n[0]; ++i)
                for (int j = 0; j < n[1]; ++j)
                    for (int k = 0; k < n[2]; ++k) {
                        auto cell = [&](int l) {
                            int c[3] = {i, j, k};
                            c[a] = (f & 1 ? b.m[a] - 1 : 0) + l * s;
                            return at(b, c[0], c[1], c[2]);
                        };
                        if (b.wall[f]) wall[f]->hidx.insert(wall[f]->hidx.end(), {cell(0), cell(-1)});
                        for (int l = 1; l <= g; ++l) (b.wall[f] ? wall[f] : far)->hidx.push_back(cell(l));
                    }
        }
    for (const Blk &b : blk)
        for (int i = -g; i < b.m[0] + g; ++i)
            for (int j = -g; j < b.m[1] + g; ++j)
                for (int k = -g; k < b.m[2] + g; ++k) {
                    const int c[3] = {i, j, k};
                    int in[3], out = 0;
                    for (int a = 0; a < 3; ++a) out += (in[a] = std::min(std::max(c[a], 0), b.m[a] - 1)) != c[a];
                    if (out > 1) corner->hidx.insert(corner->hidx.end(), {at(b, i, j, k), at(b, in[0], in[1], in[2])});
                }

    std::mt19937 rng(7);
    std::uniform_real_distribution<double> u(0.1, 2.0);
    State start((size_t)V * NC);
    for (double &x : start) x = u(rng);
    auto load = [V](const State &s, int q, double v[5]) {
        for (int c = 0; c < NC; ++c) v[c] = s[(size_t)c * V + q];
    };
    auto store = [V](State &s, int q, const double v[5]) {
        for (int c = 0; c < NC; ++c) s[(size_t)c * V + q] = v[c];
    };

    State want = start;
    std::set<int> written;
    double v[5];
    auto put = [&](int q) {
        store(want, q, v);
        written.insert(q);
    };
    for (const auto &o : ops) {
        const std::vector<int> &x = o->hidx;
        if (o->type == OP_FILL)
            for (int q : x) {
                std::copy(o->fillv.begin(), o->fillv.end(), v);
                put(q);
            }
        else if (o->type == OP_COPY)
            for (size_t t = 0; t < x.size(); t += 2) {
                load(want, x[t + 1], v);
                put(x[t]);
            }
        else
            for (size_t t = 0; t < x.size(); t += 2 + g) {
                load(want, x[t + 1], v);
                reflect(v);
                put(x[t]);
                reflect(v);
                for (int l = 0; l < g; ++l) put(x[t + 2 + l]);
            }
    }

    std::vector<const SyncOp *> list;
    for (const auto &o : ops)
        if (!o->hidx.empty()) list.push_back(o.get());
    SyncPlan plan(V);
    try {
        plan.add(list, SLOT, NC, g);
    } catch (const std::logic_error &e) {
        std::printf("refused: %s\n", e.what());
        return 3;
    }

    State got = start;
    std::set<int> done;
    for (const SyncPlan::Host &H : plan.out) {
        const State before = got;
        std::map<int, long long> writer;  // value -> lane
        std::vector<std::pair<int, long long>> reads;
        long long clash = 0, lane = 0;
        auto write = [&](int q, long long ln) {
            store(got, q, v);
            clash += !writer.insert({q, ln}).second;
            done.insert(q);
        };
        for (const SyncWave &w : H.waves)
            for (int l = 0; l < 64; ++l, ++lane) {
                const int *e = &H.ent[2 * ((size_t)w.first + l)];
                if (e[0] < 0) continue;
                if (w.kind == SYNC_CONST) {
                    std::copy(H.val.begin() + e[1], H.val.begin() + e[1] + NC, v);
                    write(e[0], lane);
                    continue;
                }
                if (w.kind == SYNC_CHAIN || w.kind == SYNC_CHAIN_CONST) {
                    load(before, e[0], v);
                    reads.push_back({e[0], lane});
                    for (int n = 1; n <= w.np; ++n)
                        for (int h = 0; h < 2; ++h)
                            if (e[128 * n + h] >= 0) write(e[128 * n + h], lane);
                    if (w.kind == SYNC_CHAIN_CONST) std::copy(H.val.begin() + e[1], H.val.begin() + e[1] + NC, v);
                }
                if (w.kind != SYNC_CHAIN_CONST) {
                    load(before, e[1], v);
                    reads.push_back({e[1], lane});
                }
                for (int n = w.kind == SYNC_WALL2 ? 2 : w.kind == SYNC_WALL1 ? 1 : 0; n > 0; --n) reflect(v);
                write(e[0], lane);
            }
        for (const auto &r : reads) {
            const auto it = writer.find(r.first);
            clash += it != writer.end() && it->second != r.second;
        }
        if (clash) return fail("lanes that meet:", clash);
    }
    if (done != written) return fail("values written:", (long long)done.size() - (long long)written.size());
    long long bad = 0;
    for (size_t n = 0; n < want.size(); ++n) bad += !(want[n] == got[n]);
    if (bad) return fail("values that differ:", bad);
    std::printf("launches %zu values %zu\n", plan.out.size(), written.size());
    return 0;
}
