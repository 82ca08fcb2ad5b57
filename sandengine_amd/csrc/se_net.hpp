// Boolean networks over machine words and their covering by three-input lookup
// tables: the sliced form of a rule set (se_hipgen.cpp) is one such network, and
// v_bitop3_b32 evaluates any function of three words in one instruction.
#pragma once
#include <cstdint>
#include <map>
#include <string>
#include <tuple>
#include <vector>

namespace se {

class Net {
public:
    using Lit = int;  // 2 * node + complement
    static constexpr Lit kZero = 0, kOne = 1;

    Net() { nodes_.push_back({Const, {0, 0, 0}}); }

    Lit input() {
        nodes_.push_back({Input, {0, 0, 0}});
        inputs_.push_back((int)nodes_.size() - 1);
        return 2 * inputs_.back();
    }
    static Lit inv(Lit a) { return a ^ 1; }
    Lit land(Lit a, Lit b);
    Lit lor(Lit a, Lit b) { return inv(land(inv(a), inv(b))); }
    Lit lxor(Lit a, Lit b);
    Lit mux(Lit s, Lit a, Lit b);  // s ? a : b
    // The function of `vars` whose value on assignment i (variable j = bit j of i)
    // is tt[i]: 0, 1, or 2 where it does not matter.
    Lit func(const std::vector<Lit>& vars, const std::vector<char>& tt);

    size_t inputs() const { return inputs_.size(); }
    // Values of `outs` for 32 assignments at a time (in[i]: the words of input i).
    void eval(const std::vector<uint32_t>& in, const std::vector<Lit>& outs, std::vector<uint32_t>& out) const;

    // Straight-line code computing `outs` into the lvalues out_names from in_names,
    // one statement per table; returns the number of tables.
    int emit(const std::vector<Lit>& outs, const std::vector<std::string>& in_names,
             const std::vector<std::string>& out_names, const std::string& indent, std::string& code) const;

private:
    enum Kind { Const, Input, And, Xor, Mux };
    struct Node {
        Kind kind;
        Lit in[3];
    };
    std::vector<Node> nodes_;
    std::vector<int> inputs_;
    std::map<std::tuple<int, Lit, Lit, Lit>, int> unique_;
    Lit make(Kind k, Lit a, Lit b, Lit c);
};

}  // namespace se
