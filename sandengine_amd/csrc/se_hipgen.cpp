#include "se_hipgen.hpp"

#include "se_net.hpp"

#include <algorithm>
#include <array>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <set>
#include <sstream>

namespace se {

static const char* kKernelTemplates =
#include "se_kernels_src.inc"
    ;
static const char* kSlicedTemplates =
#include "se_sliced_src.inc"
    ;

namespace {

constexpr uint64_t kTableMaxBytes = 48 * 1024;  // transition table staged in LDS
constexpr uint64_t kCTableMaxBytes = 64 * 1024;  // coded table: D^4 u8 entries staged in LDS

[[noreturn]] void gen_error(const std::string& m) { throw LangError("NotRecognized", "(HIP codegen) " + m); }

// ------------------------------------------------------------------ expressions
enum class Ty { Bool, Num, Mat };

struct Ex {
    enum K { Num, Bool, CellMat, MatConst, Dens, MatId, TypeId, IsType, Rand, Cmp, And, Or, Not, Neg } k;
    Ty ty = Ty::Bool;
    int op = 0;  // Cmp: 0 <, 1 <=, 2 >, 3 >=, 4 ==, 5 !=
    float num = 0;
    bool bval = false;
    int cell = 0, mat = 0, type = 0, lane = 0;
    std::unique_ptr<Ex> a, b;
};
using ExP = std::unique_ptr<Ex>;

struct Ctx {
    std::map<std::string, int> mats;   // name -> id
    std::map<std::string, int> types;  // name -> id
    std::vector<int> mat_type;         // material id -> type id
    std::vector<float> dens;           // material id -> density
    std::vector<std::array<float, 4>> color, emission;  // material id -> RGBA
    std::vector<std::vector<int>> type_members;  // type id -> {type id} + children type ids
    int nmat = 0;
};

int cell_index(const std::string& n) {
    if (n == "self") return 0;
    if (n == "right") return 1;
    if (n == "down") return 2;
    if (n == "downright") return 3;
    if (n == "left" || n == "downleft")
        gen_error("cell '" + n + "' is not declared in the generated rule functions (only self, right, down, "
                  "downright are)");
    gen_error("unknown cell '" + n + "'");
}

struct Tok {
    int kind;  // 0 num, 1 id, 2 op
    std::string s;
};

std::vector<Tok> tokenize(const std::string& s) {
    std::vector<Tok> out;
    size_t i = 0;
    while (i < s.size()) {
        char c = s[i];
        if (std::isspace((unsigned char)c)) { i++; continue; }
        if (std::isdigit((unsigned char)c) || (c == '.' && i + 1 < s.size() && std::isdigit((unsigned char)s[i + 1]))) {
            size_t j = i;
            while (j < s.size() && std::isdigit((unsigned char)s[j])) j++;
            if (j < s.size() && s[j] == '.') { j++; while (j < s.size() && std::isdigit((unsigned char)s[j])) j++; }
            if (j < s.size() && (s[j] == 'e' || s[j] == 'E')) {
                size_t k = j + 1;
                if (k < s.size() && (s[k] == '+' || s[k] == '-')) k++;
                if (k < s.size() && std::isdigit((unsigned char)s[k])) {
                    j = k;
                    while (j < s.size() && std::isdigit((unsigned char)s[j])) j++;
                }
            }
            std::string num = s.substr(i, j - i);
            if (j < s.size() && (s[j] == 'f' || s[j] == 'F')) j++;
            out.push_back({0, num});
            i = j;
            continue;
        }
        if (std::isalpha((unsigned char)c) || c == '_') {
            size_t j = i;
            while (j < s.size() && (std::isalnum((unsigned char)s[j]) || s[j] == '_')) j++;
            out.push_back({1, s.substr(i, j - i)});
            i = j;
            continue;
        }
        static const char* two[] = {"&&", "||", "==", "!=", "<=", ">="};
        bool got = false;
        for (auto* t : two)
            if (s.compare(i, 2, t) == 0) { out.push_back({2, t}); i += 2; got = true; break; }
        if (got) continue;
        if (std::strchr("<>!().-", c)) { out.push_back({2, std::string(1, c)}); i++; continue; }
        gen_error("unsupported character '" + std::string(1, c) + "' in condition '" + s + "'");
    }
    return out;
}

class ExprParser {
public:
    ExprParser(const std::string& src, const Ctx& ctx) : src_(src), t_(tokenize(src)), ctx_(ctx) {}

    ExP parse() {
        ExP e = orx();
        if (i_ != t_.size()) gen_error("unexpected '" + t_[i_].s + "' in condition '" + src_ + "'");
        if (e->ty != Ty::Bool) gen_error("condition is not boolean: '" + src_ + "'");
        return e;
    }

private:
    std::string src_;
    std::vector<Tok> t_;
    size_t i_ = 0;
    const Ctx& ctx_;

    bool peek_op(const char* o) const { return i_ < t_.size() && t_[i_].kind == 2 && t_[i_].s == o; }
    Tok take() {
        if (i_ >= t_.size()) gen_error("unexpected end of condition '" + src_ + "'");
        return t_[i_++];
    }
    void expect_op(const char* o) {
        if (!peek_op(o)) gen_error(std::string("expected '") + o + "' in condition '" + src_ + "'");
        i_++;
    }
    std::string expect_id() {
        Tok t = take();
        if (t.kind != 1) gen_error("expected identifier in condition '" + src_ + "'");
        return t.s;
    }
    static ExP mk(Ex::K k, Ty ty) {
        ExP e(new Ex());
        e->k = k;
        e->ty = ty;
        return e;
    }
    ExP bin(Ex::K k, ExP a, ExP b) {
        if (a->ty != Ty::Bool || b->ty != Ty::Bool) gen_error("&&/|| on non-boolean in '" + src_ + "'");
        ExP e = mk(k, Ty::Bool);
        e->a = std::move(a);
        e->b = std::move(b);
        return e;
    }
    ExP orx() {
        ExP e = andx();
        while (peek_op("||")) { i_++; e = bin(Ex::Or, std::move(e), andx()); }
        return e;
    }
    ExP andx() {
        ExP e = eqx();
        while (peek_op("&&")) { i_++; e = bin(Ex::And, std::move(e), eqx()); }
        return e;
    }
    ExP cmp(int op, ExP a, ExP b) {
        if (op >= 4) {
            if (a->ty != b->ty) gen_error("== / != between different types in '" + src_ + "'");
        } else if (a->ty != Ty::Num || b->ty != Ty::Num) {
            gen_error("relational comparison of non-numbers in '" + src_ + "'");
        }
        ExP e = mk(Ex::Cmp, Ty::Bool);
        e->op = op;
        e->a = std::move(a);
        e->b = std::move(b);
        return e;
    }
    ExP eqx() {
        ExP e = relx();
        for (;;) {
            if (peek_op("==")) { i_++; e = cmp(4, std::move(e), relx()); }
            else if (peek_op("!=")) { i_++; e = cmp(5, std::move(e), relx()); }
            else return e;
        }
    }
    ExP relx() {
        ExP e = unary();
        for (;;) {
            int op = -1;
            if (peek_op("<")) op = 0;
            else if (peek_op("<=")) op = 1;
            else if (peek_op(">")) op = 2;
            else if (peek_op(">=")) op = 3;
            if (op < 0) return e;
            i_++;
            e = cmp(op, std::move(e), unary());
        }
    }
    ExP unary() {
        if (peek_op("!")) {
            i_++;
            ExP a = unary();
            if (a->ty != Ty::Bool) gen_error("! on non-boolean in '" + src_ + "'");
            ExP e = mk(Ex::Not, Ty::Bool);
            e->a = std::move(a);
            return e;
        }
        if (peek_op("-")) {
            i_++;
            ExP a = unary();
            if (a->ty != Ty::Num) gen_error("unary - on non-number in '" + src_ + "'");
            ExP e = mk(Ex::Neg, Ty::Num);
            e->a = std::move(a);
            return e;
        }
        return primary();
    }
    ExP primary() {
        Tok t = take();
        if (t.kind == 0) {
            ExP e = mk(Ex::Num, Ty::Num);
            e->num = std::strtof(t.s.c_str(), nullptr);
            return e;
        }
        if (t.kind == 2 && t.s == "(") {
            ExP e = orx();
            expect_op(")");
            return e;
        }
        if (t.kind != 1) gen_error("unexpected '" + t.s + "' in condition '" + src_ + "'");
        const std::string& id = t.s;
        if (id == "true" || id == "false") {
            ExP e = mk(Ex::Bool, Ty::Bool);
            e->bval = id == "true";
            return e;
        }
        if (id.rfind("isType_", 0) == 0) {
            std::string tn = id.substr(7);
            auto it = ctx_.types.find(tn);
            if (it == ctx_.types.end()) gen_error("unknown type '" + tn + "'");
            expect_op("(");
            std::string c = expect_id();
            expect_op(")");
            ExP e = mk(Ex::IsType, Ty::Bool);
            e->cell = cell_index(c);
            e->type = it->second;
            return e;
        }
        if (id.rfind("MAT_", 0) == 0) {
            auto it = ctx_.mats.find(id.substr(4));
            if (it == ctx_.mats.end()) gen_error("unknown material '" + id + "'");
            ExP e = mk(Ex::MatConst, Ty::Mat);
            e->mat = it->second;
            return e;
        }
        if (id.rfind("TYPE_", 0) == 0) {
            auto it = ctx_.types.find(id.substr(5));
            if (it == ctx_.types.end()) gen_error("unknown type '" + id + "'");
            ExP e = mk(Ex::Num, Ty::Num);
            e->num = (float)it->second;
            return e;
        }
        if (id == "rand") {
            expect_op(".");
            std::string sw = expect_id();
            static const char* lanes = "xyzw";
            static const char* lanes2 = "rgba";
            if (sw.size() != 1) gen_error("rand swizzle '" + sw + "' unsupported");
            const char* p = std::strchr(lanes, sw[0]);
            const char* q = std::strchr(lanes2, sw[0]);
            if (!p && !q) gen_error("rand swizzle '" + sw + "' unsupported");
            ExP e = mk(Ex::Rand, Ty::Num);
            e->lane = p ? (int)(p - lanes) : (int)(q - lanes2);
            return e;
        }
        int cell = cell_index(id);
        expect_op(".");
        std::string f = expect_id();
        if (f != "mat") gen_error("only '.mat' is supported on cells (got '" + f + "')");
        if (peek_op(".")) {
            i_++;
            std::string fld = expect_id();
            ExP e;
            if (fld == "density") e = mk(Ex::Dens, Ty::Num);
            else if (fld == "id") e = mk(Ex::MatId, Ty::Num);
            else if (fld == "type") e = mk(Ex::TypeId, Ty::Num);
            else gen_error("material field '" + fld + "' unsupported in conditions");
            e->cell = cell;
            return e;
        }
        ExP e = mk(Ex::CellMat, Ty::Mat);
        e->cell = cell;
        return e;
    }
};

// ------------------------------------------------------------------ analysis and folding
unsigned cells_used(const Ex& e) {
    unsigned m = 0;
    switch (e.k) {
        case Ex::CellMat: case Ex::Dens: case Ex::MatId: case Ex::TypeId: case Ex::IsType: m = 1u << e.cell; break;
        default: break;
    }
    if (e.a) m |= cells_used(*e.a);
    if (e.b) m |= cells_used(*e.b);
    return m;
}
bool uses_rand(const Ex& e) {
    if (e.k == Ex::Rand) return true;
    return (e.a && uses_rand(*e.a)) || (e.b && uses_rand(*e.b));
}

struct Env {
    int c[4];
    float r[4];
};

float eval_num(const Ex& e, const Env& v, const Ctx& ctx);
int eval_mat(const Ex& e, const Env& v) { return e.k == Ex::CellMat ? v.c[e.cell] : e.mat; }
bool eval_bool(const Ex& e, const Env& v, const Ctx& ctx) {
    switch (e.k) {
        case Ex::Bool: return e.bval;
        case Ex::IsType: {
            int ty = ctx.mat_type[v.c[e.cell]];
            for (int t : ctx.type_members[e.type])
                if (t == ty) return true;
            return false;
        }
        case Ex::And: return eval_bool(*e.a, v, ctx) && eval_bool(*e.b, v, ctx);
        case Ex::Or: return eval_bool(*e.a, v, ctx) || eval_bool(*e.b, v, ctx);
        case Ex::Not: return !eval_bool(*e.a, v, ctx);
        case Ex::Cmp: {
            if (e.a->ty == Ty::Mat) {
                bool eq = eval_mat(*e.a, v) == eval_mat(*e.b, v);
                return e.op == 4 ? eq : !eq;
            }
            if (e.a->ty == Ty::Bool) {
                bool eq = eval_bool(*e.a, v, ctx) == eval_bool(*e.b, v, ctx);
                return e.op == 4 ? eq : !eq;
            }
            float x = eval_num(*e.a, v, ctx), y = eval_num(*e.b, v, ctx);
            switch (e.op) {
                case 0: return x < y;
                case 1: return x <= y;
                case 2: return x > y;
                case 3: return x >= y;
                case 4: return x == y;
                default: return x != y;
            }
        }
        default: gen_error("internal: not a boolean node");
    }
}
float eval_num(const Ex& e, const Env& v, const Ctx& ctx) {
    switch (e.k) {
        case Ex::Num: return e.num;
        case Ex::Dens: return ctx.dens[v.c[e.cell]];
        case Ex::MatId: return (float)v.c[e.cell];
        case Ex::TypeId: return (float)ctx.mat_type[v.c[e.cell]];
        case Ex::Rand: return v.r[e.lane];
        case Ex::Neg: return -eval_num(*e.a, v, ctx);
        default: gen_error("internal: not a numeric node");
    }
}

// rand = RNE_f32(u) * 2^-32, monotone in u.  thr(c, le): max u with rand(u) (<=|<) c, or -1.
float rnd_of(uint64_t u) { return (float)(uint32_t)u * 0x1p-32f; }
int64_t rand_threshold(float c, bool le) {
    auto ok = [&](uint64_t u) { return le ? rnd_of(u) <= c : rnd_of(u) < c; };
    if (!ok(0)) return -1;
    uint64_t lo = 0, hi = 0xFFFFFFFFull;
    while (lo < hi) {
        uint64_t mid = (lo + hi + 1) / 2;
        if (ok(mid)) lo = mid;
        else hi = mid - 1;
    }
    return (int64_t)lo;
}

std::string hex_u32(uint64_t v) {
    char b[32];
    snprintf(b, sizeof b, "0x%08llxu", (unsigned long long)(v & 0xFFFFFFFFull));
    return b;
}
std::string hex_u64(uint64_t v) {
    char b[40];
    snprintf(b, sizeof b, "0x%016llxull", (unsigned long long)v);
    return b;
}
std::string flit(float f) {
    if (std::isnan(f)) return "__builtin_nanf(\"\")";
    if (std::isinf(f)) return f > 0 ? "__builtin_inff()" : "(-__builtin_inff())";
    char b[64];
    snprintf(b, sizeof b, "%af", (double)f);
    return b;
}
const char* kCell[4] = {"c0", "c1", "c2", "c3"};

class Emitter {
public:
    explicit Emitter(const Ctx& ctx) : ctx_(ctx) {}

    // material bitmask as a device expression testing id `c`
    std::string bit(const std::vector<bool>& m, const std::string& c) const {
        int n = ctx_.nmat;
        bool all = true, none = true;
        for (int i = 0; i < n; i++) { all &= (bool)m[i]; none &= !m[i]; }
        if (all) return "true";
        if (none) return "false";
        int ones = 0, one = -1;
        for (int i = 0; i < n; i++)
            if (m[i]) { ones++; one = i; }
        if (ones == 1) return "(" + c + " == " + std::to_string(one) + "u)";
        if (n <= 32) {
            uint64_t w = 0;
            for (int i = 0; i < n; i++)
                if (m[i]) w |= 1ull << i;
            return "(((" + hex_u32(w) + " >> " + c + ") & 1u) != 0u)";
        }
        std::string words[4];
        int nw = (n + 63) / 64;
        for (int k = 0; k < nw; k++) {
            uint64_t w = 0;
            for (int i = 0; i < 64 && k * 64 + i < n; i++)
                if (m[k * 64 + i]) w |= 1ull << i;
            words[k] = hex_u64(w);
        }
        if (nw == 1) return "(((" + words[0] + " >> " + c + ") & 1ull) != 0ull)";
        std::string sel = words[nw - 1];
        for (int k = nw - 2; k >= 0; k--) sel = "(" + c + " < " + std::to_string((k + 1) * 64) + "u ? " + words[k] + " : " + sel + ")";
        return "(((" + sel + " >> (" + c + " & 63u)) & 1ull) != 0ull)";
    }

    std::string emit_bool(const Ex& e) {
        unsigned cm = cells_used(e);
        bool r = uses_rand(e);
        if (!r && cm == 0) {
            Env v{};
            return eval_bool(e, v, ctx_) ? "true" : "false";
        }
        if (!r && (cm & (cm - 1)) == 0) {
            int k = __builtin_ctz(cm);
            std::vector<bool> m(ctx_.nmat);
            for (int mat = 0; mat < ctx_.nmat; mat++) {
                Env v{};
                v.c[k] = mat;
                m[mat] = eval_bool(e, v, ctx_);
            }
            return bit(m, kCell[k]);
        }
        switch (e.k) {
            case Ex::And: return "(" + emit_bool(*e.a) + " && " + emit_bool(*e.b) + ")";
            case Ex::Or: return "(" + emit_bool(*e.a) + " || " + emit_bool(*e.b) + ")";
            case Ex::Not: return "(!" + emit_bool(*e.a) + ")";
            case Ex::Cmp: return emit_cmp(e);
            default: gen_error("internal: unexpected boolean node");
        }
    }

    std::set<int> lanes_used;
    std::map<int, std::set<uint32_t>> thresholds;  // lane -> t for every "h <= t" / "h > t" emitted
    bool rand_float_used = false;                  // rand read as a float (no threshold form)
    bool rank_used = false, dens_used = false, type_used = false;

private:
    const Ctx& ctx_;

    static const char* opstr(int op) {
        static const char* s[] = {"<", "<=", ">", ">=", "==", "!="};
        return s[op];
    }

    std::string emit_cmp(const Ex& e) {
        if (e.a->ty == Ty::Mat) {
            std::string x = e.a->k == Ex::CellMat ? kCell[e.a->cell] : std::to_string(e.a->mat) + "u";
            std::string y = e.b->k == Ex::CellMat ? kCell[e.b->cell] : std::to_string(e.b->mat) + "u";
            return "(" + x + (e.op == 4 ? " == " : " != ") + y + ")";
        }
        if (e.a->ty == Ty::Bool)
            return "(" + emit_bool(*e.a) + (e.op == 4 ? " == " : " != ") + emit_bool(*e.b) + ")";
        // density of one cell against density of another: compare ranks
        if (e.a->k == Ex::Dens && e.b->k == Ex::Dens) {
            rank_used = true;
            return "(se_rank(" + std::string(kCell[e.a->cell]) + ") " + opstr(e.op) + " se_rank(" + kCell[e.b->cell] + "))";
        }
        // rand lane against a constant: integer threshold on the hash lane
        const Ex* rn = nullptr;
        const Ex* cst = nullptr;
        int op = e.op;
        if (e.a->k == Ex::Rand && !uses_rand(*e.b) && cells_used(*e.b) == 0) { rn = e.a.get(); cst = e.b.get(); }
        else if (e.b->k == Ex::Rand && !uses_rand(*e.a) && cells_used(*e.a) == 0) {
            rn = e.b.get(); cst = e.a.get();
            static const int flip[] = {2, 3, 0, 1, 4, 5};
            op = flip[op];
        }
        if (rn) {
            Env v{};
            float c = eval_num(*cst, v, ctx_);
            lanes_used.insert(rn->lane);
            std::string h = "h" + std::to_string(rn->lane);
            if (std::isnan(c)) return op == 5 ? "true" : "false";
            int64_t tle = rand_threshold(c, true), tlt = rand_threshold(c, false);
            const int lane = rn->lane;
            auto le = [&](int64_t t) -> std::string {  // h <= t
                if (t < 0) return "false";
                if (t >= 0xFFFFFFFFll) return "true";
                thresholds[lane].insert((uint32_t)t);
                return "(" + h + " <= " + hex_u32((uint64_t)t) + ")";
            };
            auto gt = [&](int64_t t) -> std::string {  // h > t
                if (t < 0) return "true";
                if (t >= 0xFFFFFFFFll) return "false";
                thresholds[lane].insert((uint32_t)t);
                return "(" + h + " > " + hex_u32((uint64_t)t) + ")";
            };
            switch (op) {
                case 0: return le(tlt);
                case 1: return le(tle);
                case 2: return gt(tle);
                case 3: return gt(tlt);
                case 4: return "(" + gt(tlt) + " && " + le(tle) + ")";
                default: return "(!(" + gt(tlt) + " && " + le(tle) + "))";
            }
        }
        return "(" + emit_num(*e.a) + " " + opstr(e.op) + " " + emit_num(*e.b) + ")";
    }

    std::string emit_num(const Ex& e) {
        switch (e.k) {
            case Ex::Num: return flit(e.num);
            case Ex::Dens: dens_used = true; return "se_dens(" + std::string(kCell[e.cell]) + ")";
            case Ex::MatId: return "((float)" + std::string(kCell[e.cell]) + ")";
            case Ex::TypeId: type_used = true; return "((float)se_type(" + std::string(kCell[e.cell]) + "))";
            case Ex::Rand:
                lanes_used.insert(e.lane);
                rand_float_used = true;
                return "((float)h" + std::to_string(e.lane) + " * 0x1p-32f)";
            case Ex::Neg: return "(-" + emit_num(*e.a) + ")";
            default: gen_error("internal: unexpected numeric node");
        }
    }
};

// ------------------------------------------------------------------ actions
std::string emit_actions(const std::string& text, const Ctx& ctx, const std::string& ind) {
    std::string out;
    std::istringstream is(text);
    std::string line;
    while (std::getline(is, line)) {
        size_t b = line.find_first_not_of(" \t"), e = line.find_last_not_of(" \t\r");
        if (b == std::string::npos) continue;
        line = line.substr(b, e - b + 1);
        if (line.rfind("swap(", 0) == 0) {
            size_t comma = line.find(", "), close = line.find(");");
            if (comma == std::string::npos || close == std::string::npos || close + 2 != line.size())
                gen_error("unrecognised action '" + line + "'");
            int a = cell_index(line.substr(5, comma - 5)), c = cell_index(line.substr(comma + 2, close - comma - 2));
            out += ind + "SE_GSWAP(" + kCell[a] + ", " + kCell[c] + ");\n";
            continue;
        }
        size_t eq = line.find(" = newCell(MAT_");
        if (eq != std::string::npos) {
            int a = cell_index(line.substr(0, eq));
            size_t s = eq + std::strlen(" = newCell(MAT_");
            size_t comma = line.find(", pos);", s);
            if (comma == std::string::npos || comma + 7 != line.size()) gen_error("unrecognised action '" + line + "'");
            std::string mat = line.substr(s, comma - s);
            auto it = ctx.mats.find(mat);
            if (it == ctx.mats.end())
                gen_error("SET to unknown material 'MAT_" + mat + "' (not declared in the generated GLSL either)");
            out += ind + kCell[a] + " = " + std::to_string(it->second) + "u;\n";
            continue;
        }
        gen_error("unrecognised action '" + line + "'");
    }
    return out;
}

Ctx build_ctx(const ParsingResult& r) {
    Ctx ctx;
    std::set<std::string> tnames, mnames;
    for (auto& t : r.types) {
        if (!tnames.insert(t.name).second) gen_error("type '" + t.name + "' is defined twice (TYPE_ redefinition)");
        ctx.types[t.name] = (int)t.id;
    }
    for (auto& m : r.materials) {
        if (!mnames.insert(m.name).second) gen_error("material '" + m.name + "' is defined twice (MAT_ redefinition)");
        ctx.mats[m.name] = (int)m.id;
    }
    ctx.nmat = (int)r.materials.size();
    if (ctx.nmat > 255) gen_error("more than 255 materials are not supported");
    ctx.mat_type.resize(ctx.nmat);
    ctx.dens.resize(ctx.nmat);
    ctx.color.resize(ctx.nmat);
    ctx.emission.resize(ctx.nmat);
    for (auto& m : r.materials) {
        auto it = ctx.types.find(m.mattype);
        if (it == ctx.types.end()) gen_error("material '" + m.name + "' has unknown type");
        ctx.mat_type[m.id] = it->second;
        ctx.dens[m.id] = m.density;
        for (int k = 0; k < 4; k++) {
            ctx.color[m.id][k] = m.color[k];
            ctx.emission[m.id][k] = m.emission[k];
        }
    }
    ctx.type_members.resize(r.types.size());
    for (auto& t : r.types) {
        ctx.type_members[t.id].push_back((int)t.id);
        for (auto& c : t.children) {
            auto it = ctx.types.find(c);
            if (it != ctx.types.end()) ctx.type_members[t.id].push_back(it->second);
        }
    }
    return ctx;
}

// rules.rs:47-73 pairing of the flattened if/do/probability lists.
struct Level {
    float p;
    std::string cond, act;
};
void levels_of(const SandRule& r, std::vector<Level>& lv, std::string* final_act, bool* has_final) {
    std::vector<std::string> ifs = r.if_conds, dos = r.do_actions;
    std::vector<float> ps = r.probabilities;
    *has_final = false;
    for (;;) {
        if (ifs.empty() && dos.empty()) break;
        if (ifs.empty()) { *final_act = dos[0]; *has_final = true; break; }
        if (dos.empty()) break;
        lv.push_back({ps[0], ifs[0], dos[0]});
        ifs.erase(ifs.begin());
        dos.erase(dos.begin());
        ps.erase(ps.begin());
    }
}

std::string emit_rule(const SandRule& r, const Ctx& ctx, Emitter& em) {
    std::ostringstream o;
    o << "    // rule " << r.name << "\n";
    std::string ind = "    ";
    bool guarded = false;
    {
        // every condition and action must translate (the GLSL would fail to compile
        // otherwise), even where folding later removes the code
        Emitter probe(ctx);
        std::vector<Level> lv0;
        std::string fin0;
        bool hf0;
        levels_of(r, lv0, &fin0, &hf0);
        for (auto& l : lv0) {
            std::string text = (l.p == 1.0f ? std::string() : "rand.y <= " + fmt_f32(l.p) + " && ") + l.cond;
            probe.emit_bool(*ExprParser(text, ctx).parse());
            emit_actions(l.act, ctx, "");
        }
        if (hf0) emit_actions(fin0, ctx, "");
    }
    if (r.precondition) {
        ExP pre = ExprParser(*r.precondition, ctx).parse();
        std::string c = em.emit_bool(*pre);
        if (c == "false") return o.str() + "    // (precondition never holds)\n";
        if (c != "true") {
            o << "    if (" << c << ") {\n";
            ind = "        ";
            guarded = true;
        }
    }
    std::vector<Level> lv;
    std::string fin;
    bool has_fin;
    levels_of(r, lv, &fin, &has_fin);
    int open = 0;
    for (size_t i = 0; i < lv.size(); i++) {
        std::string text = (lv[i].p == 1.0f ? std::string() : "rand.y <= " + fmt_f32(lv[i].p) + " && ") + lv[i].cond;
        ExP ce = ExprParser(text, ctx).parse();
        std::string c = em.emit_bool(*ce);
        std::string pad = ind + std::string(4 * open, ' ');
        o << pad << "if (" << c << ") {\n" << emit_actions(lv[i].act, ctx, pad + "    ") << pad << "} else {\n";
        open++;
    }
    if (has_fin) o << emit_actions(fin, ctx, ind + std::string(4 * open, ' '));
    for (int k = open - 1; k >= 0; k--) o << ind << std::string(4 * k, ' ') << "}\n";
    if (guarded) o << "    }\n";
    return o.str();
}

}  // namespace

std::string hip_rules_source(const ParsingResult& r, HipGenInfo* info, bool allow_ctable, uint64_t ct_x_words) {
    Ctx ctx = build_ctx(r);
    Emitter em(ctx);
    std::string mirrored, right;
    int nrules = 0;
    for (auto& rl : r.rules) {
        if (!rl.used) continue;
        nrules++;
        if (rl.ruletype == RuleType::Left)
            gen_error("rule '" + rl.name + "' is a Left rule; its generated call passes an undeclared 'left' cell");
        std::string body = emit_rule(rl, ctx, em);
        if (rl.ruletype == RuleType::Mirrored) mirrored += body;
        else right += body;
    }
    std::ostringstream o;
    const int n = ctx.nmat;
    o << "// ---- generated by the sandengine HIP backend: " << n << " materials, " << nrules << " rules\n";
    o << "#define SE_NMAT " << n << "u\n";
    // guarded swap refuses WALL/NULL-typed cells (operations.glsl:16-23)
    std::vector<bool> fixed(n);
    for (int i = 0; i < n; i++) fixed[i] = ctx.mat_type[i] == 1 || ctx.mat_type[i] == 2;
    o << "__device__ __forceinline__ bool se_fixed(unsigned int c) { return " << em.bit(fixed, "c") << "; }\n";
    // density ranks (equal densities share a rank; NaN densities are refused)
    {
        std::vector<float> d = ctx.dens;
        for (float x : d)
            if (std::isnan(x)) gen_error("NaN density is not supported by the HIP backend");
        std::vector<float> u = d;
        std::sort(u.begin(), u.end());
        u.erase(std::unique(u.begin(), u.end(), [](float a, float b) { return a == b; }), u.end());
        std::vector<int> rank(n);
        for (int i = 0; i < n; i++)
            rank[i] = (int)(std::lower_bound(u.begin(), u.end(), d[i]) - u.begin());
        int bits = 1;
        while ((1 << bits) < (int)u.size()) bits++;
        if (bits == 3) bits = 4;
        if (bits > 4 && bits < 8) bits = 8;
        o << "__device__ __forceinline__ unsigned int se_rank(unsigned int c) {\n";
        if (n * bits <= 32) {
            uint64_t w = 0;
            for (int i = 0; i < n; i++) w |= (uint64_t)rank[i] << (i * bits);
            o << "    return __builtin_amdgcn_ubfe(" << hex_u32(w) << ", c * " << bits << "u, " << bits << "u);\n";
        } else if (n * bits <= 64) {
            uint64_t w = 0;
            for (int i = 0; i < n; i++) w |= (uint64_t)rank[i] << (i * bits);
            o << "    return (unsigned int)(" << hex_u64(w) << " >> (c * " << bits << "u)) & " << ((1u << bits) - 1)
              << "u;\n";
        } else {
            o << "    const unsigned char t[" << n << "] = {";
            for (int i = 0; i < n; i++) o << (i ? ", " : "") << rank[i];
            o << "};\n    return t[c];\n";
        }
        o << "}\n";
    }
    // per-material tables in constant memory (a local array indexed by a
    // runtime id would be rebuilt in scratch memory at every use)
    o << "__constant__ float se_dens_tab[" << n << "] = {";
    for (int i = 0; i < n; i++) o << (i ? ", " : "") << flit(ctx.dens[i]);
    o << "};\n__device__ __forceinline__ float se_dens(unsigned int c) { return se_dens_tab[c]; }\n";
    o << "__constant__ unsigned int se_type_tab[" << n << "] = {";
    for (int i = 0; i < n; i++) o << (i ? ", " : "") << ctx.mat_type[i];
    o << "};\n__device__ __forceinline__ unsigned int se_type(unsigned int c) { return se_type_tab[c]; }\n";
    // render side-outputs (operations.glsl:99-170): material colour and emission,
    // and isLightObstacle (operations.glsl:68-70): no RGB emission and not of type EMPTY
    for (int k = 0; k < 2; k++) {
        const auto& tab = k == 0 ? ctx.color : ctx.emission;
        const char* nm = k == 0 ? "se_color" : "se_emission";
        o << "__constant__ float4 " << nm << "_tab[" << n << "] = {";
        for (int i = 0; i < n; i++)
            o << (i ? ", " : "") << "{" << flit(tab[i][0]) << ", " << flit(tab[i][1]) << ", " << flit(tab[i][2]) << ", "
              << flit(tab[i][3]) << "}";
        o << "};\n__device__ __forceinline__ float4 " << nm << "(unsigned int c) { return " << nm << "_tab[c]; }\n";
    }
    {
        int empty_type = -1;
        auto it = ctx.types.find("EMPTY");
        if (it != ctx.types.end()) empty_type = it->second;
        std::vector<bool> obst(n);
        for (int i = 0; i < n; i++)
            obst[i] = ctx.emission[i][0] == 0.0f && ctx.emission[i][1] == 0.0f && ctx.emission[i][2] == 0.0f &&
                      ctx.mat_type[i] != empty_type;
        o << "__device__ __forceinline__ bool se_light_obstacle(unsigned int c) { return " << em.bit(obst, "c")
          << "; }\n";
    }
    o << "__device__ __forceinline__ unsigned int se_lowbias(unsigned int h) {\n"
         "    h ^= h >> 16; h *= 0x7feb352du; h ^= h >> 15; h *= 0x846ca68bu; h ^= h >> 16;\n    return h;\n}\n";
    // guarded swap on register values (copies first: a conditional over lvalues
    // would select between addresses and keep the cells out of registers)
    o << "#define SE_GSWAP(a, b) do { const unsigned int _a = (a), _b = (b); "
         "const bool _ok = !se_fixed(_a) && !se_fixed(_b); (a) = _ok ? _b : _a; (b) = _ok ? _a : _b; } while (0)\n";
    // se_block_h: simulate() for one block (falling_sand.glsl:61-118) given the
    // four hash lanes of the block; se_block computes them from (origin, frame).
    int64_t tmirror = rand_threshold(0.5f, false);
    em.thresholds[0].insert((uint32_t)tmirror);
    static const unsigned mult[4] = {213u, 2131u, 21313u, 213132u};
    // The rule chain works on local copies, written back once at the end: stores
    // through the reference parameters inside the branches would be merged into
    // stores through pointer phis, which keeps the cells in scratch memory.
    o << "__device__ __forceinline__ void se_block_h(unsigned int& r0, unsigned int& r1, unsigned int& r2, "
         "unsigned int& r3, unsigned int h0, unsigned int h1, unsigned int h2, unsigned int h3) {\n";
    o << "    (void)h1; (void)h2; (void)h3;\n";
    o << "    unsigned int c0 = r0, c1 = r1, c2 = r2, c3 = r3;\n";
    o << "    if ((c0 | c1 | c2 | c3) == 0u) return;\n";
    o << "    const bool mirror = h0 <= " << hex_u32((uint64_t)tmirror) << ";\n";
    o << "    if (mirror) { SE_GSWAP(c0, c1); SE_GSWAP(c2, c3); }\n";
    o << mirrored;
    o << "    if (mirror) {\n        SE_GSWAP(c0, c1);\n        SE_GSWAP(c2, c3);\n    } else {\n";
    if (!right.empty()) {
        std::istringstream is(right);
        std::string ln;
        while (std::getline(is, ln)) o << "    " << ln << "\n";
    }
    o << "    }\n    r0 = c0; r1 = c1; r2 = c2; r3 = c3;\n}\n";
    // x = ox*461 + oy*2131 + frame*2131*2131 (math.glsl:74-79) and lane k hashes
    // x*m_k; the products are distributed so that the per-block terms use 24-bit
    // multiplies where the constant fits (|ox|, |oy| < 2^23; -1 stays -1).
    auto hash_expr = [&](int l) {
        uint32_t A = 461u * mult[l], B = 2131u * mult[l], Cf = 4541161u * mult[l];
        auto term = [](uint32_t k, const char* v) -> std::string {
            if (k < (1u << 23)) return "(unsigned int)__mul24((int)" + std::string(v) + ", " + std::to_string(k) + ")";
            return std::string(v) + " * " + std::to_string(k) + "u";
        };
        return "se_lowbias(" + term(A, "ox") + " + " + term(B, "oy") + " + frame * " + std::to_string(Cf) + "u)";
    };
    o << "__device__ __forceinline__ unsigned int se_hash_lane(int l, unsigned int ox, unsigned int oy, "
         "unsigned int frame) {\n";
    for (int l = 0; l < 4; l++) o << "    if (l == " << l << ") return " << hash_expr(l) << ";\n";
    o << "    return 0u;\n}\n";
    // the same hash split into a column term gx*ka, a row term gy*kb and a frame
    // term frame*kf (all mod 2^32), for kernels that keep the terms across blocks
    {
        const char* nm[3] = {"ka", "kb", "kf"};
        const uint32_t base[3] = {461u, 2131u, 4541161u};
        for (int k = 0; k < 3; k++) {
            o << "__device__ __forceinline__ unsigned int se_hash_" << nm[k] << "(int l) {\n";
            for (int l = 0; l < 4; l++) o << "    if (l == " << l << ") return " << (uint32_t)(base[k] * mult[l]) << "u;\n";
            o << "    return 0u;\n}\n";
        }
        o << "__device__ __forceinline__ bool se_hash_used(int l) {\n    return l == 0";
        for (int l = 1; l < 4; l++)
            if (em.lanes_used.count(l)) o << " || l == " << l;
        o << ";\n}\n";
    }
    o << "__device__ __forceinline__ void se_block(unsigned int& r0, unsigned int& r1, unsigned int& r2, "
         "unsigned int& r3, unsigned int ox, unsigned int oy, unsigned int frame) {\n";
    o << "    if ((r0 | r1 | r2 | r3) == 0u) return;\n";
    for (int l = 0; l < 4; l++) {
        if (l > 0 && !em.lanes_used.count(l)) o << "    const unsigned int h" << l << " = 0u;\n";
        else o << "    const unsigned int h" << l << " = " << hash_expr(l) << ";\n";
    }
    o << "    se_block_h(r0, r1, r2, r3, h0, h1, h2, h3);\n}\n";
    // Transition table: the block result is a function of the four ids and, per
    // hash lane, of which threshold interval the lane falls in (every use of a
    // lane is a compare against one of its thresholds).  Enumerated on the
    // device by se_build_table from se_block_h itself; used when it fits LDS.
    {
        uint64_t R = 1;
        std::vector<std::vector<uint32_t>> th(4);
        for (int l = 0; l < 4; l++) {
            th[l].assign(em.thresholds[l].begin(), em.thresholds[l].end());
            R *= th[l].size() + 1;
        }
        uint64_t tuples = (uint64_t)n * n * n * n;
        uint64_t bytes = tuples * R * 4;
        bool ok = !em.rand_float_used && bytes <= kTableMaxBytes;
        // Coded table, for rule sets whose full table does not fit: tuples of the
        // D = n - 2 materials other than NULL and WALL (blocks holding those run
        // the chain), the mirror factored out as a byte permutation (lane 0 only
        // decides the mirror and there are no Right rules), and per tuple a u8
        // naming its outcome vector over the classes of lanes 1..3.  Whether the
        // rule set fits that form is checked on the enumerated table when the rule
        // set is loaded; it is generated without it otherwise.
        const uint64_t D = (uint64_t)n - 2, Rc = R / 2;
        const uint64_t ct_bytes = D * D * D * D, t1_words = (ct_bytes + 15) / 16 * 4;
        const bool ct = allow_ctable && !ok && !em.rand_float_used && right.empty() && th[0].size() == 1 &&
                        n >= 3 && D <= 16 && ct_bytes <= kCTableMaxBytes;
        o << "#define SE_TBL " << (ok ? 1 : ct ? 2 : 0) << "\n";
        o << "#define SE_TBL_R " << R << "u\n";
        o << "#define SE_TBL_ENTRIES " << (ok ? tuples * R : 1) << "u\n";
        // u32 words of the table staged into LDS (the coded table's outcome vectors
        // are counted when the enumerated table has been compacted)
        o << "#define SE_TBL_WORDS " << (ok ? tuples * R : ct ? t1_words + ct_x_words : 0) << "u\n";
        if (ct) {
            o << "#define SE_CT_D " << D << "u\n";
            o << "#define SE_CT_R " << Rc << "u\n";
            o << "#define SE_CT_T1_WORDS " << t1_words << "u\n";
            o << "#define SE_CT_MIRROR_T " << hex_u32((uint64_t)tmirror) << "\n";
            o << "__device__ __forceinline__ unsigned int se_rclass_ct(unsigned int h1, unsigned int h2, "
                 "unsigned int h3) {\n    (void)h1; (void)h2; (void)h3;\n    unsigned int r = 0u;\n";
            uint64_t st = 1;
            for (int l = 1; l < 4; l++) {
                for (uint32_t t : th[l]) o << "    r += (h" << l << " > " << hex_u32(t) << ") ? " << st << "u : 0u;\n";
                st *= th[l].size() + 1;
            }
            o << "    return r;\n}\n";
        }
        // class index: lane l contributes (#thresholds below h) * stride_l
        o << "__device__ __forceinline__ unsigned int se_rclass(unsigned int h0, unsigned int h1, unsigned int h2, "
             "unsigned int h3) {\n    (void)h0; (void)h1; (void)h2; (void)h3;\n    unsigned int r = 0u;\n";
        uint64_t stride = 1;
        for (int l = 0; l < 4; l++) {
            for (uint32_t t : th[l]) o << "    r += (h" << l << " > " << hex_u32(t) << ") ? " << stride << "u : 0u;\n";
            stride *= th[l].size() + 1;
        }
        o << "    return r;\n}\n";
        // representative hash value of each interval (its upper end)
        o << "__device__ __forceinline__ unsigned int se_rclass_rep(int l, unsigned int idx) {\n";
        for (int l = 0; l < 4; l++) {
            o << "    if (l == " << l << ") {\n";
            for (size_t j = 0; j < th[l].size(); j++)
                o << "        if (idx == " << j << "u) return " << hex_u32(th[l][j]) << ";\n";
            o << "        return 0xffffffffu;\n    }\n";
        }
        o << "    return 0u;\n}\n";
        o << "__device__ __forceinline__ unsigned int se_rclass_count(int l) {\n";
        for (int l = 0; l < 4; l++) o << "    if (l == " << l << ") return " << th[l].size() + 1 << "u;\n";
        o << "    return 1u;\n}\n";
        if (info) {
            info->table = ok;
            info->table_R = (int)R;
            info->ctable = ct;
            info->ct_D = ct ? (int)D : 0;
            info->ct_R = ct ? (int)Rc : 0;
        }
    }
    if (info) {
        info->nmat = n;
        info->nrules = nrules;
        info->rand_lanes.assign(em.lanes_used.begin(), em.lanes_used.end());
    }
    return o.str();
}

// ------------------------------------------------------------------ sliced form
// The rule chain over bit planes: a cell is `planes` words whose bit i belongs to
// block i, a condition is a word, an action a select under that word.  One
// evaluation advances 32 blocks.
namespace {

constexpr int kSlicedMaxMaterials = 16, kSlicedMaxClasses = 8;

struct NotSliced {};  // the rule set reads something that has no word form

class Slicer {
public:
    // code: of a material; order: ascending with the density where rules compare it
    Slicer(const Ctx& ctx, int planes, const std::vector<int>& code, const std::vector<int>& order)
        : ctx_(ctx), K_(planes), code_(code), order_(order) {
        for (int c = 0; c < 4; c++)
            for (int k = 0; k < K_; k++) cell_[c].push_back(net.input());
    }
    Net net;
    std::vector<std::pair<int, uint32_t>> classes;  // inputs after the cells, in order of first use
    std::vector<Net::Lit> class_lit;

    Net::Lit below(int lane, int64_t t) {  // hash lane <= t
        if (t < 0) return Net::kZero;
        if (t >= 0xFFFFFFFFll) return Net::kOne;
        for (size_t i = 0; i < classes.size(); i++)
            if (classes[i] == std::make_pair(lane, (uint32_t)t)) return class_lit[i];
        // here and not after the chain: its last check goes through all class words
        if (classes.size() == (size_t)kSlicedMaxClasses) throw NotSliced();
        classes.push_back({lane, (uint32_t)t});
        class_lit.push_back(net.input());
        return class_lit.back();
    }

    // simulate() after the cell reads (falling_sand.glsl:61-118), as se_block_h
    std::vector<Net::Lit> chain(const ParsingResult& r) {
        std::vector<bool> fixed(ctx_.nmat);
        for (int i = 0; i < ctx_.nmat; i++) fixed[i] = ctx_.mat_type[i] == 1 || ctx_.mat_type[i] == 2;
        fixed_of_ = fixed;
        State in;
        for (int c = 0; c < 4; c++) {
            in.cell[c] = cell_[c];
            in.fixed[c] = holds(in.cell[c], fixed);
        }
        State s = in;
        const Net::Lit mirror = below(0, rand_threshold(0.5f, false));
        swap(s, 0, 1, mirror);
        swap(s, 2, 3, mirror);
        for (auto& rl : r.rules)
            if (rl.used && rl.ruletype == RuleType::Mirrored) rule(rl, Net::kOne, s);
        swap(s, 0, 1, mirror);
        swap(s, 2, 3, mirror);
        for (auto& rl : r.rules)
            if (rl.used && rl.ruletype != RuleType::Mirrored) rule(rl, Net::inv(mirror), s);
        std::vector<Net::Lit> out;
        for (int c = 0; c < 4; c++) out.insert(out.end(), s.cell[c].begin(), s.cell[c].end());
        // a block of four EMPTY cells stays as it is (falling_sand.glsl:77-79): kept
        // out of the network where the rules leave it alone anyway
        std::vector<uint32_t> words(net.inputs(), 0u), got;
        for (int c = 0; c < 4; c++)
            for (int k = 0; k < K_; k++) words[c * K_ + k] = (code_[0] >> k) & 1 ? ~0u : 0u;
        bool stays = true;
        for (uint32_t m = 0; m < (1u << classes.size()); m += 32) {
            for (size_t j = 0; j < classes.size(); j++) {
                uint32_t w = 0;
                for (uint32_t i = 0; i < 32; i++) w |= (((m + i) >> j) & 1u) << i;
                words[4 * K_ + j] = w;
            }
            net.eval(words, out, got);
            for (size_t i = 0; i < out.size(); i++) stays = stays && got[i] == words[i];
        }
        if (!stays) {
            std::vector<bool> empty(ctx_.nmat);
            empty[0] = true;
            Net::Lit all = Net::kOne;
            for (int c = 0; c < 4; c++) all = net.land(all, holds(in.cell[c], empty));
            for (int c = 0; c < 4; c++)
                for (int k = 0; k < K_; k++) out[c * K_ + k] = net.mux(all, in.cell[c][k], out[c * K_ + k]);
        }
        return out;
    }

private:
    using Cell = std::vector<Net::Lit>;
    struct State {
        Cell cell[4];
        Net::Lit fixed[4];  // the cell refuses swaps; a swap never moves such a cell
    };
    const Ctx& ctx_;
    int K_;
    std::vector<int> code_, order_;
    Cell cell_[4];
    std::vector<bool> fixed_of_;

    template <class F>  // f(material id) over the codes of one cell
    Net::Lit table(const Cell& c, F f) {
        std::vector<char> tt((size_t)1 << K_, 2);
        for (int m = 0; m < ctx_.nmat; m++) tt[code_[m]] = (char)f(m);
        return net.func(c, tt);
    }
    Net::Lit holds(const Cell& c, const std::vector<bool>& set) {
        return table(c, [&](int m) { return set[m] ? 1 : 0; });
    }
    // a cell's order with equal densities sharing the lowest of theirs
    Cell rank(const Cell& c) {
        Cell r;
        for (int k = 0; k < K_; k++)
            r.push_back(table(c, [&](int m) {
                int low = order_[m];
                for (int o = 0; o < ctx_.nmat; o++)
                    if (ctx_.dens[o] == ctx_.dens[m]) low = std::min(low, order_[o]);
                return (low >> k) & 1;
            }));
        return r;
    }
    Net::Lit less(const Cell& a, const Cell& b) {
        Net::Lit r = Net::kZero;
        for (int k = 0; k < K_; k++) r = net.mux(net.lxor(a[k], b[k]), b[k], r);
        return r;
    }
    Net::Lit equal(const Cell& a, const Cell& b) {
        Net::Lit r = Net::kOne;
        for (int k = 0; k < K_; k++) r = net.land(r, Net::inv(net.lxor(a[k], b[k])));
        return r;
    }

    Net::Lit cond(const Ex& e, const State& s) {
        const unsigned cm = cells_used(e);
        const bool rnd = uses_rand(e);
        if (!rnd && cm == 0) {
            Env v{};
            return eval_bool(e, v, ctx_) ? Net::kOne : Net::kZero;
        }
        if (!rnd && (cm & (cm - 1)) == 0) {
            const int k = __builtin_ctz(cm);
            return table(s.cell[k], [&](int m) {
                Env v{};
                v.c[k] = m;
                return eval_bool(e, v, ctx_) ? 1 : 0;
            });
        }
        switch (e.k) {
            case Ex::And: { const Net::Lit a = cond(*e.a, s); return net.land(a, cond(*e.b, s)); }
            case Ex::Or: { const Net::Lit a = cond(*e.a, s); return net.lor(a, cond(*e.b, s)); }
            case Ex::Not: return Net::inv(cond(*e.a, s));
            case Ex::Cmp: return compare(e, s);
            default: gen_error("internal: unexpected boolean node");
        }
    }
    Net::Lit compare(const Ex& e, const State& s) {
        if (e.a->ty == Ty::Bool) {
            const Net::Lit x = cond(*e.a, s), d = net.lxor(x, cond(*e.b, s));
            return e.op == 4 ? Net::inv(d) : d;
        }
        if (e.a->ty == Ty::Mat) {  // two cells (a cell against a constant is a table of one cell)
            const Net::Lit q = equal(s.cell[e.a->cell], s.cell[e.b->cell]);
            return e.op == 4 ? q : Net::inv(q);
        }
        if (e.a->k == Ex::Dens && e.b->k == Ex::Dens) {
            const Cell a = rank(s.cell[e.a->cell]), b = rank(s.cell[e.b->cell]);
            switch (e.op) {
                case 0: return less(a, b);
                case 1: return Net::inv(less(b, a));
                case 2: return less(b, a);
                case 3: return Net::inv(less(a, b));
                case 4: return equal(a, b);
                default: return Net::inv(equal(a, b));
            }
        }
        if (!uses_rand(e)) {  // any other compare of two cells' numbers: a table over both codes
            const unsigned cm = cells_used(e);
            const int x = __builtin_ctz(cm), y = 31 - __builtin_clz(cm);
            if (__builtin_popcount(cm) != 2) throw NotSliced();
            Cell both = s.cell[x];
            both.insert(both.end(), s.cell[y].begin(), s.cell[y].end());
            std::vector<char> tt((size_t)1 << (2 * K_), 2);
            for (int a = 0; a < ctx_.nmat; a++)
                for (int b = 0; b < ctx_.nmat; b++) {
                    Env v{};
                    v.c[x] = a;
                    v.c[y] = b;
                    tt[(size_t)code_[a] | ((size_t)code_[b] << K_)] = eval_bool(e, v, ctx_) ? 1 : 0;
                }
            return net.func(both, tt);
        }
        const Ex* rn = nullptr;
        const Ex* cst = nullptr;
        int op = e.op;
        if (e.a->k == Ex::Rand && !uses_rand(*e.b) && cells_used(*e.b) == 0) { rn = e.a.get(); cst = e.b.get(); }
        else if (e.b->k == Ex::Rand && !uses_rand(*e.a) && cells_used(*e.a) == 0) {
            rn = e.b.get(); cst = e.a.get();
            static const int flip[] = {2, 3, 0, 1, 4, 5};
            op = flip[op];
        }
        if (!rn) throw NotSliced();
        Env v{};
        const float c = eval_num(*cst, v, ctx_);
        if (std::isnan(c)) return op == 5 ? Net::kOne : Net::kZero;
        const int64_t tle = rand_threshold(c, true), tlt = rand_threshold(c, false);
        const int l = rn->lane;
        switch (op) {
            case 0: return below(l, tlt);
            case 1: return below(l, tle);
            case 2: return Net::inv(below(l, tle));
            case 3: return Net::inv(below(l, tlt));
            case 4: return net.land(Net::inv(below(l, tlt)), below(l, tle));
            default: return Net::inv(net.land(Net::inv(below(l, tlt)), below(l, tle)));
        }
    }

    // guarded swap (operations.glsl:16-23) where `m` holds
    void swap(State& s, int a, int b, Net::Lit m) {
        const Net::Lit ok = net.land(m, net.land(Net::inv(s.fixed[a]), Net::inv(s.fixed[b])));
        for (int k = 0; k < K_; k++) {
            const Net::Lit x = s.cell[a][k], y = s.cell[b][k];
            s.cell[a][k] = net.mux(ok, y, x);
            s.cell[b][k] = net.mux(ok, x, y);
        }
    }
    void set(State& s, int a, int mat, Net::Lit m) {
        for (int k = 0; k < K_; k++)
            s.cell[a][k] = net.mux(m, (code_[mat] >> k) & 1 ? Net::kOne : Net::kZero, s.cell[a][k]);
        s.fixed[a] = net.mux(m, fixed_of_[mat] ? Net::kOne : Net::kZero, s.fixed[a]);
    }
    // the action lines of emit_actions, under the word m
    void actions(const std::string& text, State& s, Net::Lit m) {
        std::istringstream is(emit_actions(text, ctx_, ""));
        std::string line;
        while (std::getline(is, line)) {
            int a = 0, b = 0;
            if (std::sscanf(line.c_str(), "SE_GSWAP(c%d, c%d);", &a, &b) == 2) swap(s, a, b, m);
            else if (std::sscanf(line.c_str(), "c%d = %du;", &a, &b) == 2) set(s, a, b, m);
            else gen_error("internal: action '" + line + "'");
        }
    }
    // One rule where `on` holds.  The levels exclude each other, so every level's
    // condition reads the cells as the rule found them.
    void rule(const SandRule& r, Net::Lit on, State& s) {
        const State in = s;
        Net::Lit rest = on;
        if (r.precondition) rest = net.land(rest, cond(*ExprParser(*r.precondition, ctx_).parse(), in));
        std::vector<Level> lv;
        std::string fin;
        bool has_fin;
        levels_of(r, lv, &fin, &has_fin);
        for (auto& l : lv) {
            const std::string text = (l.p == 1.0f ? std::string() : "rand.y <= " + fmt_f32(l.p) + " && ") + l.cond;
            const Net::Lit c = cond(*ExprParser(text, ctx_).parse(), in);
            actions(l.act, s, net.land(rest, c));
            rest = net.land(rest, Net::inv(c));
        }
        if (has_fin) actions(fin, s, rest);
    }
};

}  // namespace

std::string hip_sliced_source(const ParsingResult& r, SlicedInfo& out) {
    out = SlicedInfo();
    const Ctx ctx = build_ctx(r);
    const int n = ctx.nmat;
    if (n > kSlicedMaxMaterials || n < 3) return "";
    for (float d : ctx.dens)
        if (std::isnan(d)) return "";
    int K = 1;
    while ((1 << K) < n) K++;
    // Codes ascend with the density (ties by id) where rules compare it, so that
    // comparing densities compares codes, up to an exclusive or that makes WALL 0:
    // the planes that come in from outside a tile are then 0, which the wave shifts
    // give for nothing.
    Emitter em(ctx);
    for (auto& rl : r.rules)
        if (rl.used) emit_rule(rl, ctx, em);
    std::vector<int> by(n), order(n), code(n), id_of(16, 2);
    for (int i = 0; i < n; i++) by[i] = i;
    if (em.rank_used)
        std::stable_sort(by.begin(), by.end(), [&](int a, int b) { return ctx.dens[a] < ctx.dens[b]; });
    for (int i = 0; i < n; i++) order[by[i]] = i;
    for (int i = 0; i < n; i++) {
        code[i] = order[i] ^ order[2];
        id_of[code[i]] = i;
    }
    Slicer sl(ctx, K, code, order);
    std::vector<Net::Lit> outs;
    try {
        outs = sl.chain(r);
    } catch (const NotSliced&) {
        return "";
    }
    const int P = (int)sl.classes.size();
    // does any block change a WALL cell?  (every tuple of codes, every class word)
    bool kept = true;
    {
        std::vector<uint32_t> in(sl.net.inputs()), got;
        for (int t = 0; t < n * n * n * n && kept; t++) {
            const int id[4] = {t % n, t / n % n, t / n / n % n, t / n / n / n};
            bool wall = false;
            for (int c = 0; c < 4; c++) {
                wall |= id[c] == 2;
                for (int k = 0; k < K; k++) in[c * K + k] = (code[id[c]] >> k) & 1 ? ~0u : 0u;
            }
            if (!wall) continue;
            for (uint32_t m = 0; m < (1u << P); m += 32) {
                for (int j = 0; j < P; j++) {
                    uint32_t w = 0;
                    for (uint32_t i = 0; i < 32; i++) w |= (((m + i) >> j) & 1u) << i;
                    in[4 * K + j] = w;
                }
                sl.net.eval(in, outs, got);
                for (int c = 0; c < 4; c++)
                    for (int k = 0; k < K && id[c] == 2; k++) kept = kept && got[c * K + k] == in[c * K + k];
            }
        }
    }
    // ids whose uniform block no class word changes, as codes
    for (int i = 0; i < n; i++) {
        std::vector<uint32_t> in(sl.net.inputs()), got;
        bool stays = true;
        for (int c = 0; c < 4; c++)
            for (int k = 0; k < K; k++) in[c * K + k] = (code[i] >> k) & 1 ? ~0u : 0u;
        for (uint32_t m = 0; m < (1u << P) && stays; m += 32) {
            for (int j = 0; j < P; j++) {
                uint32_t w = 0;
                for (uint32_t b = 0; b < 32; b++) w |= (((m + b) >> j) & 1u) << b;
                in[4 * K + j] = w;
            }
            sl.net.eval(in, outs, got);
            for (int c = 0; c < 4 * K; c++) stays = stays && got[c] == in[c];
        }
        if (stays) out.stable |= 1u << code[i];
    }
    out.ok = true;
    out.planes = K;
    out.code = code;
    out.classes = sl.classes;
    out.wall_kept = kept;
    std::vector<std::string> in_names, out_names;
    for (int c = 0; c < 4; c++)
        for (int k = 0; k < K; k++) {
            in_names.push_back("c" + std::to_string(c) + "[" + std::to_string(k) + "]");
            out_names.push_back("n" + std::to_string(c) + "_" + std::to_string(k));
        }
    for (int j = 0; j < P; j++) in_names.push_back("h[" + std::to_string(j) + "]");
    std::string body;
    out.tables = sl.net.emit(outs, in_names, [&] {
        std::vector<std::string> decl;
        for (auto& o : out_names) decl.push_back("const unsigned int " + o);
        return decl;
    }(), "    ", body);
    std::ostringstream o;
    o << "// ---- sliced form: " << K << " bit planes per cell, " << P << " hash planes, " << out.tables
      << " tables per 32 blocks\n";
    o << "template <int TT>\n__device__ __forceinline__ unsigned int se_lut3(unsigned int a, unsigned int b, unsigned int "
         "c) {\n    return __builtin_amdgcn_bitop3_b32(a, b, c, TT);\n}\n";
    o << "#define SE_SL_K " << K << "\n#define SE_SL_P " << P << "\n#define SE_SL_KEEP " << (kept ? 1 : 0) << "\n";
    // code of id i and id of code i as bytes of four words
    for (int dir = 0; dir < 2; dir++) {
        uint32_t w[4] = {0, 0, 0, 0};
        for (int i = 0; i < 16; i++) {
            const int v = dir == 0 ? (i < n ? code[i] : code[1]) : id_of[i];
            w[i / 4] |= (uint32_t)v << (8 * (i & 3));
        }
        for (int j = 0; j < 4; j++) o << "#define SE_SL_" << (dir == 0 ? "CODE" : "ID") << j << " " << hex_u32(w[j]) << "\n";
    }
    // hash planes: the lane and the threshold of each
    for (int part = 0; part < 2; part++) {
        o << "__device__ __forceinline__ constexpr unsigned int se_sliced_class_" << (part == 0 ? "lane" : "max")
          << "(int p) {\n    return ";
        for (int j = 0; j + 1 < P; j++)
            o << "p == " << j << " ? " << (part == 0 ? std::to_string(sl.classes[j].first) + "u" : hex_u32(sl.classes[j].second))
              << " : ";
        o << (part == 0 ? std::to_string(sl.classes[P - 1].first) + "u" : hex_u32(sl.classes[P - 1].second)) << ";\n}\n";
    }
    o << "__device__ __forceinline__ constexpr bool se_sliced_lane(int l) {\n    return false";
    for (int l = 0; l < 4; l++)
        for (auto& c : sl.classes)
            if (c.first == l) { o << " || l == " << l; break; }
    o << ";\n}\n";
    o << "__device__ __forceinline__ void se_sliced_block(unsigned int* c0, unsigned int* c1, unsigned int* c2, "
         "unsigned int* c3, const unsigned int* h) {\n" << body;
    for (int c = 0; c < 4; c++)
        for (int k = 0; k < K; k++) o << "    " << in_names[c * K + k] << " = " << out_names[c * K + k] << ";\n";
    o << "}\n";
    return o.str();
}

std::string lds_kernel_name(const LdsVariant& v) {
    return "se_step_lds_" + std::to_string(v.tw) + "x" + std::to_string(v.th) + "_h" + std::to_string(v.hb) + "_t" +
           std::to_string(v.nt);
}

std::string hip_program_source(const ParsingResult& r, const std::vector<LdsVariant>& lds, bool allow_ctable,
                               uint64_t ct_x_words, SlicedInfo* sliced) {
    HipGenInfo form;
    std::string s = hip_rules_source(r, &form, allow_ctable, ct_x_words);
    s += "\n";
    s += kKernelTemplates;
    s += "\n";
    for (auto& v : lds)
        s += "SE_LDS_KERNEL(" + std::to_string(v.tw) + ", " + std::to_string(v.th) + ", " + std::to_string(v.hb) + ", " +
             std::to_string(v.nt) + ")\n";
    if (!lds.empty()) {  // not in the small module that only enumerates the coded table
        SlicedInfo local;
        SlicedInfo& sl = sliced ? *sliced : local;
        const std::string rules = hip_sliced_source(r, sl);
        // A network this large is never the faster one beside a transition table, whose
        // cost does not grow with the rules (se_sliced.cpp: 1661 tables, 4096^2, 64 steps 920 us
        // and 586 by the table), and takes seconds to compile.
        if (sl.ok && (form.table || form.ctable) && sl.tables > 1000) sl = SlicedInfo();
        if (sl.ok) s += rules + kSlicedTemplates;
    }
    return s;
}

}  // namespace se
