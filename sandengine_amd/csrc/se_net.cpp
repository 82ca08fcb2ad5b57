#include "se_net.hpp"

#include <algorithm>
#include <cstdio>

namespace se {

Net::Lit Net::make(Kind k, Lit a, Lit b, Lit c) {
    auto key = std::make_tuple((int)k, a, b, c);
    auto it = unique_.find(key);
    if (it != unique_.end()) return 2 * it->second;
    nodes_.push_back({k, {a, b, c}});
    unique_[key] = (int)nodes_.size() - 1;
    return 2 * ((int)nodes_.size() - 1);
}

Net::Lit Net::land(Lit a, Lit b) {
    if (a > b) std::swap(a, b);
    if (a == kZero || a == inv(b)) return kZero;
    if (a == kOne || a == b) return b;
    return make(And, a, b, 0);
}

Net::Lit Net::lxor(Lit a, Lit b) {
    const Lit flip = (a & 1) ^ (b & 1);
    a &= ~1;
    b &= ~1;
    if (a > b) std::swap(a, b);
    if (a == b) return flip;
    if (a == kZero) return b ^ flip;
    return make(Xor, a, b, 0) ^ flip;
}

Net::Lit Net::mux(Lit s, Lit a, Lit b) {
    if (s == kOne || a == b) return a;
    if (s == kZero) return b;
    if (s & 1) {
        s ^= 1;
        std::swap(a, b);
    }
    if (a == inv(b)) return inv(lxor(s, a));
    if (a == kOne || a == s) return lor(s, b);
    if (a == kZero || a == inv(s)) return land(inv(s), b);
    if (b == kZero || b == s) return land(s, a);
    if (b == kOne || b == inv(s)) return lor(inv(s), a);
    const Lit flip = a & 1;
    return make(Mux, s, a ^ flip, b ^ flip) ^ flip;
}

Net::Lit Net::func(const std::vector<Lit>& vars, const std::vector<char>& tt) {
    bool any0 = false, any1 = false;
    for (char v : tt) {
        any0 |= v == 0;
        any1 |= v == 1;
    }
    if (!any1) return kZero;
    if (!any0) return kOne;
    const size_t n = vars.size();
    auto half = [&](size_t v, int bit, size_t i) {  // entry i of the cofactor vars[v] = bit
        const size_t lo = i & ((1u << v) - 1), hi = i >> v;
        return tt[(hi << (v + 1)) | ((size_t)bit << v) | lo];
    };
    auto without = [&](size_t v) {
        std::vector<Lit> r = vars;
        r.erase(r.begin() + (long)v);
        return r;
    };
    const size_t m = tt.size() / 2;
    for (size_t v = 0; v < n; v++) {  // a variable that need not matter, or enters by exclusive or
        bool same = true, opposite = true;
        for (size_t i = 0; i < m; i++) {
            const char a = half(v, 0, i), b = half(v, 1, i);
            if (a == 2 || b == 2) continue;
            same &= a == b;
            opposite &= a != b;
        }
        if (!same && !opposite) continue;
        std::vector<char> g(m);
        for (size_t i = 0; i < m; i++) {
            const char a = half(v, 0, i), b = half(v, 1, i);
            g[i] = a != 2 ? a : b == 2 ? 2 : same ? b : (char)(1 - b);
        }
        const Lit f = func(without(v), g);
        return same ? f : lxor(vars[v], f);
    }
    // the variable whose cofactors depend on the fewest others
    size_t best = 0;
    int best_score = 1 << 20;
    for (size_t v = 0; v < n; v++) {
        int score = 0;
        for (int bit = 0; bit < 2; bit++) {
            bool c0 = false, c1 = false;
            for (size_t i = 0; i < m; i++) {
                c0 |= half(v, bit, i) == 0;
                c1 |= half(v, bit, i) == 1;
            }
            if (!c0 || !c1) continue;
            for (size_t u = 0; u + 1 < n; u++) {
                bool dep = false;
                for (size_t i = 0; i < m; i++) {
                    if (i & (1u << u)) continue;
                    const char a = half(v, bit, i), b = half(v, bit, i | (1u << u));
                    dep |= a != 2 && b != 2 && a != b;
                }
                score += dep ? 1 : 0;
            }
        }
        if (score < best_score) {
            best_score = score;
            best = v;
        }
    }
    std::vector<char> f0(m), f1(m);
    for (size_t i = 0; i < m; i++) {
        f0[i] = half(best, 0, i);
        f1[i] = half(best, 1, i);
    }
    const std::vector<Lit> rest = without(best);
    const Lit a = func(rest, f1), b = func(rest, f0);
    return mux(vars[best], a, b);
}

void Net::eval(const std::vector<uint32_t>& in, const std::vector<Lit>& outs, std::vector<uint32_t>& out) const {
    std::vector<uint32_t> v(nodes_.size(), 0u);
    for (size_t i = 0; i < inputs_.size(); i++) v[inputs_[i]] = in[i];
    auto val = [&](Lit l) { return (l & 1) ? ~v[l >> 1] : v[l >> 1]; };
    for (size_t i = 0; i < nodes_.size(); i++) {
        const Node& n = nodes_[i];
        if (n.kind == And) v[i] = val(n.in[0]) & val(n.in[1]);
        else if (n.kind == Xor) v[i] = val(n.in[0]) ^ val(n.in[1]);
        else if (n.kind == Mux) v[i] = (val(n.in[0]) & val(n.in[1])) | (~val(n.in[0]) & val(n.in[2]));
    }
    out.resize(outs.size());
    for (size_t i = 0; i < outs.size(); i++) out[i] = val(outs[i]);
}

namespace {
struct Cut {
    int n = 0;
    int leaf[3] = {0, 0, 0};
    uint8_t tt = 0;  // over (leaf 0, leaf 1, leaf 2) = (0xf0, 0xcc, 0xaa)
    double cost = 0;
    bool operator==(const Cut& o) const {
        return n == o.n && leaf[0] == o.leaf[0] && leaf[1] == o.leaf[1] && leaf[2] == o.leaf[2];
    }
};
const uint8_t kVar[3] = {0xf0, 0xcc, 0xaa};

// The function of cut c over the leaves of the larger cut u.
uint8_t widen(const Cut& c, const Cut& u) {
    int at[3] = {0, 0, 0};
    for (int i = 0; i < c.n; i++)
        for (int j = 0; j < u.n; j++)
            if (u.leaf[j] == c.leaf[i]) at[i] = j;
    uint8_t r = 0;
    for (int m = 0; m < 8; m++) {
        int idx = 0;
        for (int i = 0; i < c.n; i++)
            if ((kVar[at[i]] >> m) & 1) idx |= 4 >> i;
        if ((c.tt >> idx) & 1) r |= (uint8_t)(1 << m);
    }
    return r;
}

bool join(const Cut& a, const Cut& b, Cut& u) {
    int all[6], n = 0;
    for (int i = 0; i < a.n; i++) all[n++] = a.leaf[i];
    for (int i = 0; i < b.n; i++) all[n++] = b.leaf[i];
    std::sort(all, all + n);
    n = (int)(std::unique(all, all + n) - all);
    if (n > 3) return false;
    u = Cut();
    u.n = n;
    for (int i = 0; i < n; i++) u.leaf[i] = all[i];
    return true;
}
}  // namespace

// Cover by cuts of at most three leaves: the cheapest cut of each node by area
// flow (a table's cost shared over its fanouts), repeated with the fanouts of the
// cover found before, which favours tables that others use anyway.
int Net::emit(const std::vector<Lit>& outs, const std::vector<std::string>& in_names,
              const std::vector<std::string>& out_names, const std::string& indent, std::string& code) const {
    const size_t N = nodes_.size();
    std::vector<double> refs(N, 0.0);
    for (auto& n : nodes_)
        for (int i = 0; i < (n.kind == Mux ? 3 : n.kind == And || n.kind == Xor ? 2 : 0); i++) refs[n.in[i] >> 1] += 1;
    for (Lit o : outs) refs[o >> 1] += 1;
    std::vector<Cut> best(N), kept;
    std::vector<char> used(N, 0), kept_used;
    int best_count = 1 << 30;
    for (int pass = 0; pass < 8; pass++) {
        std::vector<std::vector<Cut>> cuts(N);
        std::vector<double> flow(N, 0.0);
        for (size_t i = 1; i < N; i++) {
            const Node& n = nodes_[i];
            Cut self;
            self.n = 1;
            self.leaf[0] = (int)i;
            self.tt = 0xf0;
            if (n.kind == Input) {
                cuts[i].push_back(self);
                continue;
            }
            const int k = n.kind == Mux ? 3 : 2;
            std::vector<Cut> found;
            auto flip = [&](Lit l, uint8_t t) { return (uint8_t)((l & 1) ? ~t : t); };
            auto add = [&](const Cut& u) {
                for (auto& c : found)
                    if (c == u) return;
                found.push_back(u);
            };
            const auto& A = cuts[n.in[0] >> 1];
            const auto& B = cuts[n.in[1] >> 1];
            for (auto& a : A)
                for (auto& b : B) {
                    Cut u;
                    if (!join(a, b, u)) continue;
                    if (k == 2) {
                        const uint8_t x = flip(n.in[0], widen(a, u)), y = flip(n.in[1], widen(b, u));
                        u.tt = n.kind == And ? (x & y) : (x ^ y);
                        add(u);
                        continue;
                    }
                    for (auto& c : cuts[n.in[2] >> 1]) {
                        Cut w;
                        if (!join(u, c, w)) continue;
                        const uint8_t s = flip(n.in[0], widen(a, w)), x = flip(n.in[1], widen(b, w)),
                                      y = flip(n.in[2], widen(c, w));
                        w.tt = (uint8_t)((s & x) | (~s & y));
                        add(w);
                    }
                }
            for (auto& c : found) {
                c.cost = 1;
                for (int j = 0; j < c.n; j++) c.cost += flow[c.leaf[j]];
            }
            std::stable_sort(found.begin(), found.end(), [](const Cut& x, const Cut& y) { return x.cost < y.cost; });
            best[i] = found[0];
            flow[i] = found[0].cost / std::max(1.0, refs[i]);
            if (found.size() > 24) found.resize(24);
            cuts[i] = found;
            cuts[i].push_back(self);
        }
        std::fill(used.begin(), used.end(), 0);
        std::vector<double> now(N, 0.0);
        for (Lit o : outs) {
            now[o >> 1] += 1;
            used[o >> 1] = 1;
        }
        int count = 0;
        for (size_t i = N; i-- > 1;) {
            if (!used[i] || nodes_[i].kind == Input) continue;
            count++;
            for (int j = 0; j < best[i].n; j++) {
                used[best[i].leaf[j]] = 1;
                now[best[i].leaf[j]] += 1;
            }
        }
        if (count < best_count) {
            best_count = count;
            kept = best;
            kept_used = used;
        }
        for (size_t i = 0; i < N; i++) refs[i] = 0.5 * (refs[i] + std::max(now[i], 0.1));
    }
    // tables read by other tables or by an output as they are; an output that is the
    // complement of a node gets the complemented table
    std::vector<char> plain(N, 0);
    for (size_t i = 1; i < N; i++)
        if (kept_used[i] && nodes_[i].kind != Input)
            for (int j = 0; j < kept[i].n; j++) plain[kept[i].leaf[j]] = 1;
    for (Lit o : outs)
        if (!(o & 1)) plain[o >> 1] = 1;
    std::vector<std::string> name(N);
    for (size_t i = 0; i < inputs_.size(); i++) name[inputs_[i]] = in_names[i];
    auto table = [&](size_t i, bool invert) {
        const Cut& c = kept[i];  // absent leaves repeat the first: the table does not depend on them
        char tt[16];
        snprintf(tt, sizeof tt, "0x%02x", invert ? (uint8_t)~c.tt : c.tt);
        const std::string a = name[c.leaf[0]];
        return std::string("se_lut3<") + tt + ">(" + a + ", " + (c.n > 1 ? name[c.leaf[1]] : a) + ", " +
               (c.n > 2 ? name[c.leaf[2]] : a) + ")";
    };
    for (size_t i = 1; i < N; i++) {
        if (!kept_used[i] || nodes_[i].kind == Input || !plain[i]) continue;
        name[i] = "t" + std::to_string(i);
        code += indent + "const unsigned int " + name[i] + " = " + table(i, false) + ";\n";
    }
    for (size_t i = 0; i < outs.size(); i++) {
        const size_t n = (size_t)(outs[i] >> 1);
        std::string v;
        if (n == 0) v = (outs[i] & 1) ? "~0u" : "0u";
        else if (!(outs[i] & 1)) v = name[n];
        else v = nodes_[n].kind == Input ? "~" + name[n] : table(n, true);
        code += indent + out_names[i] + " = " + v + ";\n";
    }
    return best_count;
}

}  // namespace se
