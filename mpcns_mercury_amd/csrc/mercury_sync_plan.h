// The sync programs of a field (halo, physical boundaries, owner -> alias) as
// index lists, and their planning into launches.  Host code only.
#pragma once
#include <algorithm>
#include <climits>
#include <cstring>
#include <functional>
#include <stdexcept>
#include <utility>
#include <vector>

#include "mercury_common.h"

namespace merc {

enum OpType { OP_COPY, OP_FILL, OP_SETV, OP_WALLF };

// one operation of one field (or of fields sharing an index list) in one
// phase of a group's program; host lists only
struct SyncOp {
    OpType type;
    int phase = 0;
    std::vector<int> slots;
    std::vector<double> fillv;  // FILL: a value per slot; WALLF of Na+: the ghosts' state
    int is_na = 0;  // WALLF: species (0 H+, 1 Na+, 2 He++)
    std::vector<int> hidx;     // pairs for COPY, (first, deeper, ghosts) for WALLF
    std::vector<double> hval;  // SETV values
};

// Turns the phases of a field's sync into as few launches as can be.  It follows
// the ops in order, symbolically: what each value is after them, in terms of the
// values before the first: a copy of one, a constant, or a wall state made of the
// cell behind the wall's first layer.  A launch then writes every changed value
// from there, whatever the number of phases (three to six launches of about 5 us
// each before, one behind the other).
//
// Threads of a launch run in no order, so a value that others read must not be
// written in the same launch.  The one exception is an aliased value, which ghosts
// copy before its owner's value replaces it: one thread makes those copies and
// then the replacement (a chain).  Where the ops cannot be joined under these
// rules, the longest run of them that can makes a launch and the rest follow.
class SyncPlan {
public:
    explicit SyncPlan(long long nvalues) : sym(nvalues, {NONE, 0}) {}
    // appends one field's sync: ops in program order that touch slots slot ..
    // slot + ncomp - 1; launch n of every field goes to the same kernel launch
    // keep: the values to write (all of them without it)
    void add(const std::vector<const SyncOp *> &ops, int slot, int ncomp, int g, const std::function<bool(int)> &keep = nullptr) {
        // where a launch may end: not between the components of one set of values
        std::vector<size_t> ends;
        for (size_t n = 0; n < ops.size(); ++n) {
            if (ops[n]->type == OP_SETV) n += ncomp - 1;
            ends.push_back(n + 1);
        }
        size_t at = 0, launch = 0;
        for (size_t u = 0; u < ends.size();) {
            size_t last = ends.size() - 1;
            while (!(follow(ops, at, ends[last], slot, ncomp, g) && (last + 1 < ends.size() || !keep || drop(keep)) && joins())) {
                // an op by itself can: no destination of it is a source of it
                if (last == u) throw std::logic_error("sync plan: an op reads what it sets");
                --last;
            }
            emit(launch++, slot, ncomp);
            at = ends[last];
            u = last + 1;
        }
    }
    struct Host {
        std::vector<SyncWave> waves;
        std::vector<int> ent;
        std::vector<double> val;
        // appends the waves of another group's launch
        void append(const Host &o) {
            const int e0 = (int)(ent.size() / 2), v0 = (int)val.size();
            ent.insert(ent.end(), o.ent.begin(), o.ent.end());
            val.insert(val.end(), o.val.begin(), o.val.end());
            for (SyncWave w : o.waves) {
                w.first += e0;
                if (w.kind == SYNC_CONST || w.kind == SYNC_CHAIN_CONST)
                    for (int l = 0; l < 64; ++l) ent[2 * ((size_t)w.first + l) + 1] += v0;
                waves.push_back(w);
            }
        }
    };
    std::vector<Host> out;

private:
    enum { NONE = 0, RAW, CST, WALL_FIRST, WALL_GHOST };
    struct Sym {
        int type, a;
    };
    std::vector<Sym> sym;  // per value index: what it is after the ops followed so far
    std::vector<int> touched;
    std::vector<double> rows;  // constants, ncomp each
    int wall_species = 0;
    std::vector<std::pair<int, int>> chain;  // (aliased value, a ghost that copies it)
    static constexpr size_t kWaveEntries = 64;

    void set(int d, Sym v) {
        if (sym[d].type == NONE) touched.push_back(d);
        sym[d] = v;
    }
    Sym value_of(int s) const { return sym[s].type == NONE ? Sym{RAW, s} : sym[s]; }
    int row(const double *v, int ncomp) {
        if (rows.size() < (size_t)ncomp || std::memcmp(rows.data() + rows.size() - ncomp, v, sizeof(double) * ncomp) != 0)
            rows.insert(rows.end(), v, v + ncomp);
        return (int)rows.size() - ncomp;
    }
    void reset() {
        for (int d : touched) sym[d] = {NONE, 0};
        touched.clear();
        rows.clear();
    }
    // false: a wall op needs the value of a cell that an op before it changes
    bool follow(const std::vector<const SyncOp *> &ops, size_t b, size_t e, int slot, int ncomp, int g) {
        reset();
        for (size_t n = b; n < e; ++n) {
            const SyncOp &o = *ops[n];
            const size_t c0 = std::find(o.slots.begin(), o.slots.end(), slot) - o.slots.begin();
            if (o.type == OP_FILL) {
                for (int d : o.hidx) set(d, {CST, row(o.fillv.data() + c0, ncomp)});
            } else if (o.type == OP_SETV) {
                // values of their own per entry, one op per component over the same entries
                std::vector<double> v(ncomp);
                for (size_t t = 0; t < o.hidx.size(); ++t) {
                    for (int c = 0; c < ncomp; ++c) v[c] = ops[n + c]->hval[t];
                    set(o.hidx[t], {CST, row(v.data(), ncomp)});
                }
                n += ncomp - 1;
            } else if (o.type == OP_WALLF) {
                wall_species = o.is_na;
                for (size_t t = 0; t + 2 + g <= o.hidx.size(); t += 2 + g) {
                    const int *w = &o.hidx[t];
                    if (o.is_na == 1) {  // Na+: a floor state in the ghosts
                        for (int l = 0; l < g; ++l) set(w[2 + l], {CST, row(o.fillv.data(), ncomp)});
                        continue;
                    }
                    if (sym[w[1]].type != NONE) return false;
                    set(w[0], {WALL_FIRST, w[1]});
                    for (int l = 0; l < g; ++l) set(w[2 + l], {WALL_GHOST, w[1]});
                }
            } else {
                for (size_t t = 0; t + 1 < o.hidx.size(); t += 2) set(o.hidx[t], value_of(o.hidx[t + 1]));
            }
        }
        return true;
    }
    // drops the values that need not be written (in the last launch of a field, so
    // that no later op reads them)
    bool drop(const std::function<bool(int)> &keep) {
        size_t n = 0;
        for (int d : touched) {
            if (keep(d)) touched[n++] = d;
            else sym[d] = {NONE, 0};
        }
        touched.resize(n);
        return true;
    }
    // whether the values can be written in one launch; collects the chains
    bool joins() {
        chain.clear();
        for (int d : touched) {
            const Sym v = sym[d];
            if (v.type == CST || sym[v.a].type == NONE || (v.type == RAW && v.a == d)) continue;
            if (v.type != RAW) return false;  // a wall state of a value that is written
            chain.push_back({v.a, d});
        }
        std::sort(chain.begin(), chain.end());
        auto read = [&](int x) {
            const auto it = std::lower_bound(chain.begin(), chain.end(), std::make_pair(x, INT_MIN));
            return it != chain.end() && it->first == x;
        };
        for (const auto &p : chain) {
            const Sym v = sym[p.first];
            // the value read is replaced by an unchanged one or a constant, and the reader is read by nobody
            if ((v.type != CST && (v.type != RAW || sym[v.a].type != NONE)) || read(p.second)) return false;
        }
        return true;
    }
    void emit(size_t launch, int slot, int ncomp) {
        if (out.size() <= launch) out.resize(launch + 1);
        Host &H = out[launch];
        std::vector<int> part[SYNC_CHAIN];
        const int base = (int)H.val.size();
        H.val.insert(H.val.end(), rows.begin(), rows.end());
        for (int d : touched) {
            const Sym v = sym[d];
            if (!chain.empty()) {
                const auto it = std::lower_bound(chain.begin(), chain.end(), std::make_pair(d, INT_MIN));
                if (it != chain.end() && it->first == d) continue;  // the end of a chain
            }
            if (v.type == RAW) {
                if (v.a == d || sym[v.a].type != NONE) continue;  // unchanged, or a reader in a chain
                part[SYNC_COPY].insert(part[SYNC_COPY].end(), {d, v.a});
            } else if (v.type == CST) {
                part[SYNC_CONST].insert(part[SYNC_CONST].end(), {d, base + v.a});
            } else {
                std::vector<int> &q = part[v.type == WALL_FIRST ? SYNC_WALL1 : SYNC_WALL2];
                q.insert(q.end(), {d, v.a});
            }
        }
        for (int kind = 0; kind < SYNC_CHAIN; ++kind)
            for (size_t t = 0; t < part[kind].size(); t += 2 * kWaveEntries) {
                H.waves.push_back(SyncWave{kind, slot, ncomp, (int)(H.ent.size() / 2), wall_species, 0});
                const size_t n = std::min(2 * kWaveEntries, part[kind].size() - t);
                H.ent.insert(H.ent.end(), part[kind].begin() + t, part[kind].begin() + t + n);
                H.ent.resize(H.ent.size() + 2 * kWaveEntries - n, -1);
            }
        // chains, 64 a wave: (aliased value, owner), then the ghosts that read it
        for (int kind : {SYNC_CHAIN, SYNC_CHAIN_CONST}) {
            std::vector<std::pair<int, int>> lane;  // (number of ghosts, first in chain), the short ones first
            for (size_t t = 0, u; t < chain.size(); t = u) {
                for (u = t + 1; u < chain.size() && chain[u].first == chain[t].first;) ++u;
                if ((sym[chain[t].first].type == CST) == (kind == SYNC_CHAIN_CONST)) lane.push_back({(int)(u - t), (int)t});
            }
            std::sort(lane.begin(), lane.end());
            for (size_t t = 0; t < lane.size(); t += kWaveEntries) {
                const size_t n = std::min(kWaveEntries, lane.size() - t);
                const int np = (lane[t + n - 1].first + 1) / 2;
                H.waves.push_back(SyncWave{kind, slot, ncomp, (int)(H.ent.size() / 2), 0, np});
                const size_t e0 = H.ent.size();
                H.ent.resize(e0 + 2 * kWaveEntries * (1 + np), -1);
                for (size_t l = 0; l < n; ++l) {
                    const auto &c = lane[t + l];
                    const int x = chain[c.second].first;
                    H.ent[e0 + 2 * l] = x;
                    H.ent[e0 + 2 * l + 1] = sym[x].a + (kind == SYNC_CHAIN_CONST ? base : 0);
                    for (int u = 0; u < c.first; ++u) H.ent[e0 + 2 * (kWaveEntries * (1 + u / 2) + l) + u % 2] = chain[c.second + u].second;
                }
            }
        }
        reset();
        chain.clear();
    }
};

}  // namespace merc
