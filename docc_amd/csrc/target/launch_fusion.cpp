// RocmLaunchFusionPass: launches that take several of the scheduled nodes. It runs on the copy of the SDFG that host code is
// generated from, so the scheduled form keeps one node per operation (which is what it is inspected, serialised and
// instrumented by) and only the generated calls change:
//   * a GEMM and the elementwise block that alone reads its result - bias, activation, rounding to bf16, residual - become
//     docc_rocm_linear, which has the chain in the product's store;
//   * a convolution and the elementwise block that alone reads its result - residual, ReLU - become docc_rocm_conv2d_f32_chain;
//   * an upload, a softmax and the download of its result become docc_rocm_softmax_host, which has the copies of different rows beside each other;
//   * Mean, centre and square, Mean, scale and shift (how a layer norm is spelled with tensor nodes), with the casts around
//     them for bf16, become docc_rocm_layer_norm, and with a layer on a few rows behind it docc_rocm_norm_linear.
// A transformer's feed-forward block of nine to eleven launches is three calls this way. The reference stops at fusing Maps
// with Maps (python/bindings/py_structured_sdfg.cpp:258-260); its products and reductions stay apart.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <set>

#include "map_form.h"

namespace sdfg::rocm {

namespace blas = math::blas;
namespace tensor = math::tensor;
using data_flow::LibraryNode;

namespace {

// ---- the nodes that exist between this pass and code generation -----------------------------------

bool is_offloading(const Block& b) { return b.node->code() == LibraryNodeType_ROCM_Offloading; }

bool floating16(P t) { return t == P::Float || t == P::BFloat; }

int type_code(P t) { return t == P::BFloat ? 1 : 2; }   // DOCC_ROCM_TYPE_BF16 / _F32

class LaunchNode : public LibraryNode {
public:
    LaunchNode(std::string code, std::vector<std::string> inputs)
        : LibraryNode(std::move(code), {"_y"}, std::move(inputs), false, ImplementationType_ROCMWithoutTransfers) {}
    void to_json(json::Value&) const override { throw InvalidSDFGException(code() + ": a node of code generation has no serialised form"); }
    Expression connector_bytes(const std::string&) const override { return "0"; }   // never copied by a dispatcher
};

class LinearLaunch : public LaunchNode {
public:
    LinearLaunch(std::vector<std::string> inputs) : LaunchNode(LibraryNodeType_ROCM_Linear, std::move(inputs)) {}
    bool trans_a = false, trans_b = false;
    Expression m, n, k, lda, ldb;
    P type = P::Float, bias_type = P::Float, residual_type = P::Float, y_type = P::Float;
    bool has_bias = false, has_residual = false;
    int activation = -1, rounding = 0;
};

// both of them in one call; the result of the norm is its scratch
class NormLinearLaunch : public LaunchNode {
public:
    NormLinearLaunch(std::vector<std::string> inputs) : LaunchNode(LibraryNodeType_ROCM_NormLinear, std::move(inputs)) {}
    Expression m, n, k, ldb, eps;
    P type = P::Float, bias_type = P::Float, residual_type = P::Float, y_type = P::Float;
    bool has_weight = false, has_norm_bias = false, has_bias = false, has_residual = false;
    int activation = -1, rounding = 0;
};

class ConvChainLaunch : public LaunchNode {
public:
    ConvChainLaunch(std::vector<std::string> inputs) : LaunchNode(LibraryNodeType_ROCM_ConvChain, std::move(inputs)) {}
    std::string extents;
    Expression group;
    bool has_bias = false, has_residual = false;
    int activation = -1;
};

class SoftmaxHostLaunch : public LaunchNode {
public:
    SoftmaxHostLaunch() : LaunchNode(LibraryNodeType_ROCM_SoftmaxHost, {"_x"}) {}
    Expression outer, extent, inner;
    bool fp64 = false, rows = false;   // rows: over the last axis of floats
};

class LayerNormLaunch : public LaunchNode {
public:
    LayerNormLaunch(std::vector<std::string> inputs) : LaunchNode(LibraryNodeType_ROCM_LayerNorm, std::move(inputs)) {}
    Expression rows, cols, eps;
    P type = P::Float;
    bool has_weight = false, has_bias = false;
};

// ---- reading a form -----------------------------------------------------------------------------

// The values of a form by name. Names of statements, loads and scalar operands are unique within it.
class Values {
public:
    explicit Values(const MapForm& f) : form_(f) {
        for (auto& s : f.statements) statements_[s.out] = &s;
        for (auto& r : f.reads) reads_[r.value] = &r;
        for (auto& s : f.scalars) scalars_[s.value] = &s;
    }
    const Statement* statement(const std::string& v, const char* op) const {
        auto it = statements_.find(v);
        return it != statements_.end() && it->second->op == op ? it->second : nullptr;
    }
    const MapForm::Read* read(const std::string& v) const {
        auto it = reads_.find(v);
        return it == reads_.end() ? nullptr : it->second;
    }
    // the text of a literal or of a scalar operand that is a constant
    std::string constant(const std::string& v) const {
        if (!v.empty() && v[0] == '#') return v.substr(1);
        auto it = scalars_.find(v);
        return it != scalars_.end() && it->second->source.is_constant ? it->second->source.data : "";
    }
    // the value of a constant that is a plain number; other text (FLT_MAX, an expression) is compiled as it stands and says nothing here
    bool number(const std::string& v, double* value) const {
        const std::string text = constant(v);
        char* end = nullptr;
        *value = std::strtod(text.c_str(), &end);
        if (end != text.c_str() && (*end == 'f' || *end == 'F')) end++;
        return end != text.c_str() && *end == 0;
    }
    bool is(const std::string& v, double value) const {
        double got = 0;
        return number(v, &got) && std::fabs(got - value) <= 1e-7 * std::fabs(value);
    }
    bool is_zero(const std::string& v) const {   // +0: the larger of x and -0 is another zero
        double got = 0;
        return number(v, &got) && got == 0.0 && !std::signbit(got);
    }
    // `v` without the conversions it passed through; *rounded: one of them was to bf16
    std::string through_casts(std::string v, bool* rounded) const {
        while (const Statement* s = statement(v, "assign")) {
            if (s->type == P::BFloat) *rounded = true;
            v = s->args[0];
        }
        return v;
    }
    // the other operand of op(a, b) when `pick` accepts one of them; "" if it accepts neither
    template <typename F>
    std::string other(const std::string& v, const char* op, F pick) const {
        const Statement* s = statement(v, op);
        if (!s) return "";
        if (pick(s->args[1])) return s->args[0];
        if (pick(s->args[0])) return s->args[1];
        return "";
    }
    // float arithmetic with conversions to and from bf16, nothing else
    bool plain_float() const {
        for (auto& s : form_.statements)
            if (s.type != P::Float && !(s.type == P::BFloat && s.op == "assign")) return false;
        return true;
    }

private:
    const MapForm& form_;
    std::map<std::string, const Statement*> statements_;
    std::map<std::string, const MapForm::Read*> reads_;
    std::map<std::string, const MapForm::Scalar*> scalars_;
};

// strides of a dense operand over the loops [from, end) that is repeated along the others, as Converter spells them
std::vector<Expression> dense_strides(const std::vector<Expression>& bounds, size_t from, size_t end) {
    std::vector<Expression> s(bounds.size(), "0");
    Expression run = "1";
    for (size_t l = end; l-- > from;) {
        s[l] = run;
        run = run == "1" ? bounds[l] : "(" + bounds[l] + ")*" + run;
    }
    return s;
}

bool same_strides(const std::vector<Expression>& a, const std::vector<Expression>& b) {
    if (a.size() != b.size()) return false;
    for (size_t l = 0; l < a.size(); l++)
        if (!symbolic::equal(a[l], b[l])) return false;
    return true;
}

// sigmoid(x) = 1 / (1 + exp(-x)): x, or ""
std::string sigmoid_of(const Values& v, const std::string& name) {
    const Statement* div = v.statement(name, "fp_div");
    if (!div || !v.is(div->args[0], 1.0)) return "";
    const std::string e = v.other(div->args[1], "fp_add", [&](const std::string& a) { return v.is(a, 1.0); });
    const Statement* ex = e.empty() ? nullptr : v.statement(e, "exp");
    const Statement* neg = ex ? v.statement(ex->args[0], "fp_neg") : nullptr;
    return neg ? neg->args[0] : "";
}

// x of x * c
std::string scaled(const Values& v, const std::string& name, double c) {
    return v.other(name, "fp_mul", [&](const std::string& a) { return v.is(a, c); });
}

// The activation that makes `name` (its code in *act) and what it is of; `name` itself and -1 where it is none of them.
std::string activation_of(const Values& v, const std::string& name, int* act) {
    *act = -1;
    if (const Statement* s = v.statement(name, "fabs")) return *act = 0, s->args[0];
    if (const Statement* s = v.statement(name, "tanh")) return *act = 5, s->args[0];
    const std::string r = v.other(name, "fmax", [&](const std::string& a) { return v.is_zero(a); });
    if (!r.empty()) return *act = 2, r;
    const std::string sg = sigmoid_of(v, name);
    if (!sg.empty()) return *act = 3, sg;
    const Statement* mul = v.statement(name, "fp_mul");
    if (!mul) return name;
    for (int side = 0; side < 2; side++) {
        const std::string a = mul->args[side], b = mul->args[1 - side];
        if (sigmoid_of(v, b) == a) return *act = 18, a;                                             // x sigmoid(x)
        const std::string x = scaled(v, a, 0.5);
        const std::string gate = x.empty() ? "" : v.other(b, "fp_add", [&](const std::string& one) { return v.is(one, 1.0); });
        if (gate.empty()) continue;
        if (const Statement* erf = v.statement(gate, "erf"))                                        // 0.5 x (1 + erf(x / sqrt 2))
            if (scaled(v, erf->args[0], 0.7071067811865476) == x) return *act = 16, x;
        if (const Statement* th = v.statement(gate, "tanh")) {                                      // 0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3)))
            const std::string inner = scaled(v, th->args[0], 0.7978845608028654);
            const std::string cube = inner.empty() ? "" : v.other(inner, "fp_add", [&](const std::string& t) { return t == x; });
            const std::string x3 = cube.empty() ? "" : scaled(v, cube, 0.044715);
            const std::string x2 = x3.empty() ? "" : v.other(x3, "fp_mul", [&](const std::string& t) { return t == x; });
            const Statement* sq = x2.empty() ? nullptr : v.statement(x2, "fp_mul");
            if (sq && sq->args[0] == x && sq->args[1] == x) return *act = 17, x;
        }
    }
    return name;
}

class LaunchFusion {
public:
    explicit LaunchFusion(StructuredSDFG& sdfg) : sdfg_(sdfg), blocks_(sdfg.blocks()), convert_(sdfg) {}

    bool run() {
        take_lifetimes();
        bool applied = false;
        for (bool changed = true; changed;) {
            changed = false;
            for (size_t j = 0; j < blocks_.size() && !changed; j++) changed = layer_norm(j) || linear(j) || conv_chain(j) || softmax_host(j);
            applied = applied || changed;
        }
        // (when nothing is left that becomes a layer norm or a linear layer)
        for (bool changed = true; changed;) {
            changed = false;
            for (size_t j = 0; j < blocks_.size() && !changed; j++) changed = norm_linear(j);
            applied = applied || changed;
        }
        restore_lifetimes(applied);
        return applied;
    }

private:
    // ---- lifetimes ---------------------------------------------------------------------------------
    // Blocks that only allocate or only free a container say where it is first and last used; they are set aside while
    // launches are merged and put back around the uses that are left.
    struct Lifetime {
        size_t at;        // where the block stood
        bool alloc;
        std::string name;
        Block block;
    };

    void take_lifetimes() {
        std::map<std::string, int> allocs, frees;
        for (auto& b : blocks_)
            if (is_offloading(b)) {
                const auto& n = static_cast<const ROCMDataOffloadingNode&>(*b.node);
                if (n.is_alloc()) allocs[b.outputs[0].data]++;
                if (n.is_free()) frees[b.inputs[0].data]++;
            }
        std::vector<Block> rest;
        for (size_t i = 0; i < blocks_.size(); i++) {
            Block& b = blocks_[i];
            bool movable = false, alloc = false;
            std::string name;
            if (is_offloading(b)) {
                const auto& n = static_cast<const ROCMDataOffloadingNode&>(*b.node);
                alloc = n.is_alloc();
                if (!n.is_h2d() && !n.is_d2h() && (n.is_alloc() != n.is_free())) {
                    name = alloc ? b.outputs[0].data : b.inputs[0].data;
                    movable = allocs[name] <= 1 && frees[name] <= 1;
                }
            }
            if (movable) lifetimes_.push_back({i, alloc, name, std::move(b)});
            else rest.push_back(std::move(b));
        }
        blocks_ = std::move(rest);
    }

    void restore_lifetimes(bool applied) {
        if (!applied) {   // exactly as it was
            for (auto& l : lifetimes_) blocks_.insert(blocks_.begin() + (long) l.at, std::move(l.block));
            return;
        }
        for (bool alloc : {false, true})
            for (auto& l : lifetimes_) {
                if (l.alloc != alloc || !sdfg_.exists(l.name)) continue;
                long first = -1, last = -1;
                for (size_t i = 0; i < blocks_.size(); i++)
                    if (touches(blocks_[i], l.name)) {
                        if (first < 0) first = (long) i;
                        last = (long) i;
                    }
                if (first < 0) continue;
                blocks_.insert(blocks_.begin() + (alloc ? first : last + 1), std::move(l.block));
            }
    }

    static bool touches(const Block& b, const std::string& name) {
        for (auto& in : b.inputs)
            if (!in.is_constant && in.data == name) return true;
        for (auto& out : b.outputs)
            if (out.data == name) return true;
        return false;
    }

    // ---- what may move -------------------------------------------------------------------------------
    bool ours(size_t i) const { return blocks_[i].node->implementation_type() == ImplementationType_ROCMWithoutTransfers; }

    // whether what stands between two blocks writes `name` or releases it (a download that frees its buffer has stayed in place)
    bool lost_between(const std::string& name, size_t from, size_t to) const {
        for (size_t i = from + 1; i < to; i++) {
            const Block& b = blocks_[i];
            for (auto& out : b.outputs)
                if (out.data == name) return true;
            if (!is_offloading(b) || !static_cast<const ROCMDataOffloadingNode&>(*b.node).is_free()) continue;
            for (auto& in : b.inputs)
                if (!in.is_constant && in.data == name) return true;
        }
        return false;
    }

    // a transient that no block but those of `users` touches: it goes away with them
    bool private_to(const std::string& name, const std::set<size_t>& users) const {
        const Container& c = sdfg_.container(name);
        if (c.is_argument || !c.transient || name == sdfg_.return_container()) return false;
        for (size_t i = 0; i < blocks_.size(); i++)
            if (!users.count(i) && touches(blocks_[i], name)) return false;
        return true;
    }

    // the only block that writes `name`, if it stands before `before`
    long writer_of(const std::string& name, size_t before) const {
        long w = -1;
        for (size_t i = 0; i < blocks_.size(); i++)
            for (auto& out : blocks_[i].outputs)
                if (out.data == name) {
                    if (w >= 0) return -1;
                    w = (long) i;
                }
        return w >= 0 && (size_t) w < before ? w : -1;
    }

    static ConnectorBinding bind(const std::string& connector, const std::string& data) {
        ConnectorBinding b;
        b.connector = connector;
        b.data = data;
        return b;
    }

    // `node` in place of block j; the blocks of `gone` and the containers of `links` go
    void install(size_t j, std::unique_ptr<LaunchNode> node, std::vector<ConnectorBinding> inputs, const std::string& result, std::set<size_t> gone,
                 const std::set<std::string>& links) {
        node->set_element_id(blocks_[j].node->element_id());
        blocks_[j].node = std::move(node);
        blocks_[j].inputs = std::move(inputs);
        blocks_[j].outputs = {bind("_y", result)};
        for (auto it = gone.rbegin(); it != gone.rend(); ++it) blocks_.erase(blocks_.begin() + (long) *it);
        for (auto& name : links) sdfg_.remove_container(name);
    }

    // ---- a product and the block behind it -------------------------------------------------------------
    bool linear(size_t j) {
        if (!ours(j)) return false;
        std::optional<MapForm> f = convert_.form_of(blocks_[j]);
        if (!f || f->results.size() != 1 || !floating16(f->results[0].element)) return false;
        const Values v(*f);
        if (!v.plain_float()) return false;
        const std::vector<Expression> whole = dense_strides(f->bounds, 0, f->bounds.size()),
                                      row = dense_strides(f->bounds, f->bounds.size() - 1, f->bounds.size());
        if (!same_strides(f->results[0].strides, whole)) return false;
        for (auto& candidate : f->reads) {
            const std::string link = candidate.data;
            const long w = writer_of(link, j);
            if (w < 0 || !ours((size_t) w) || candidate.element != P::Float || !same_strides(candidate.strides, whole)) continue;
            const size_t i = (size_t) w;
            const auto* g = dynamic_cast<const blas::GEMMNode*>(blocks_[i].node.get());
            if (!g || (g->precision() != blas::s && g->precision() != blas::b) || g->ldc() != g->n() || g->reads("__C", blocks_[i].inputs)) continue;
            if (g->trans_a() == blas::ConjTrans || g->trans_b() == blas::ConjTrans) continue;
            if (!g->epilogue_activation().empty() && g->epilogue_activation() != "ml::ReLU" && g->epilogue_activation() != "ml::Abs") continue;
            if (!private_to(link, {i, j})) continue;
            // the loops are [m as its leading extents, n] ([n] when m is 1)
            if (!symbolic::equal(f->bounds.back(), g->n()) ||
                !symbolic::equal(symbolic::product(f->bounds, 0, f->bounds.size() - 1), g->m()))
                continue;
            if (chain(i, j, *g, *f, v, link, whole, row)) return true;
        }
        return false;
    }

    bool chain(size_t i, size_t j, const blas::GEMMNode& g, const MapForm& f, const Values& v, const std::string& link, const std::vector<Expression>& whole,
               const std::vector<Expression>& row) {
        const MapForm::Read *bias = nullptr, *residual = nullptr;
        auto is_link = [&](const std::string& name) {
            const MapForm::Read* r = v.read(name);
            return r && r->data == link;
        };
        // an addend that is loaded: by strides the residual (whole) or a bias row; casts of it to float do not matter
        auto addend = [&](const std::string& name, const std::vector<Expression>& strides) -> const MapForm::Read* {
            bool rounded = false;
            const MapForm::Read* r = v.read(v.through_casts(name, &rounded));
            return r && !rounded && r->data != link && floating16(r->element) && same_strides(r->strides, strides) ? r : nullptr;
        };
        bool store_rounds = false, after = false, before = false;
        std::string top = v.through_casts(f.results[0].value, &store_rounds);
        if (store_rounds != (f.results[0].element == P::BFloat)) return false;
        const std::string base = v.other(top, "fp_add", [&](const std::string& a) { return addend(a, whole) != nullptr; });
        if (!base.empty() && f.bounds.size() + (g.m() == "1" ? 1 : 0) > 1 && !(g.m() == "1" && !g.epilogue_bias() && is_link(base))) {
            const Statement* add = v.statement(top, "fp_add");
            residual = addend(add->args[0] == base ? add->args[1] : add->args[0], whole);
            top = v.through_casts(base, &after);
        }
        int act = -1;
        const std::string of = activation_of(v, top, &act);
        std::string inner = v.through_casts(of, &before);
        if (act < 0) {   // one rounding, between product and residual
            after = after || before;
            before = false;
        }
        const std::string sum = v.other(inner, "fp_add", [&](const std::string& a) { return addend(a, row) != nullptr; });
        if (!sum.empty()) {
            const Statement* add = v.statement(inner, "fp_add");
            bias = addend(add->args[0] == sum ? add->args[1] : add->args[0], row);
            bool rounded = false;
            inner = v.through_casts(sum, &rounded);
            if (rounded) return false;   // rounded before the bias: not a chain of the store
        }
        if (!is_link(inner)) return false;
        std::string bias_name = bias ? bias->data : "";
        P bias_type = bias ? bias->element : P::Float;
        const Block& product = blocks_[i];
        if (g.has_epilogue()) {
            if (bias) return false;
            if (!g.epilogue_activation().empty()) {
                if (act >= 0) return false;
                act = g.epilogue_activation() == "ml::ReLU" ? 2 : 0;
            }
            if (g.epilogue_bias()) bias_name = product.input("__bias")->data;
        }
        // without a residual a rounding behind the activation is the store's own
        if (!residual && after && f.results[0].element != P::BFloat) return false;
        const std::string result = f.results[0].data, a = product.input("__A")->data, b = product.input("__B")->data;
        // what the product reads it now reads where block j stands; what block j reads of its own it reads there already
        for (const std::string& name : {a, b, bias ? std::string() : bias_name})
            if (!name.empty() && lost_between(name, i, j)) return false;
        if (result == a || result == b || result == bias_name) return false;
        const ConnectorBinding alpha = *product.input("__alpha");
        if (!alpha.is_constant && lost_between(alpha.data, i, j)) return false;

        std::vector<std::string> connectors{"_a", "_b", "__alpha"};
        std::vector<ConnectorBinding> inputs{bind("_a", a), bind("_b", b), alpha};
        if (!bias_name.empty()) connectors.push_back("_bias"), inputs.push_back(bind("_bias", bias_name));
        if (residual) connectors.push_back("_residual"), inputs.push_back(bind("_residual", residual->data));
        auto node = std::make_unique<LinearLaunch>(connectors);
        node->trans_a = g.trans_a() == blas::Trans;
        node->trans_b = g.trans_b() == blas::Trans;
        node->m = g.m(), node->n = g.n(), node->k = g.k(), node->lda = g.lda(), node->ldb = g.ldb();
        node->type = g.precision() == blas::b ? P::BFloat : P::Float;
        node->has_bias = !bias_name.empty();
        node->bias_type = bias_type;
        node->has_residual = residual != nullptr;
        if (residual) node->residual_type = residual->element;
        node->activation = act;
        node->rounding = (act >= 0 && before ? 1 : 0) | (residual && after ? 2 : 0);
        node->y_type = f.results[0].element;
        install(j, std::move(node), std::move(inputs), result, {i}, {link});
        return true;
    }

    // ---- a convolution and the block behind it ---------------------------------------------------------
    bool conv_chain(size_t j) {
        if (!ours(j)) return false;
        std::optional<MapForm> f = convert_.form_of(blocks_[j]);
        if (!f || f->results.size() != 1 || f->results[0].element != P::Float) return false;
        const Values v(*f);
        for (auto& s : f->statements)
            if (s.type != P::Float) return false;
        const std::vector<Expression> whole = dense_strides(f->bounds, 0, f->bounds.size());
        if (!same_strides(f->results[0].strides, whole)) return false;
        int act = -1;
        const std::string inner = activation_of(v, f->results[0].value, &act);
        if (act != -1 && act != 2) return false;
        auto dense = [&](const std::string& name) -> const MapForm::Read* {
            const MapForm::Read* r = v.read(name);
            return r && r->element == P::Float && same_strides(r->strides, whole) ? r : nullptr;
        };
        // what the activation is of: the convolution's result, or its sum with a tensor of the same extents - either operand of which may be it
        const Statement* sum = v.statement(inner, "fp_add");
        if (!sum) return act != -1 && dense(inner) && conv_chain(j, *f, dense(inner), nullptr, act);
        const MapForm::Read *a = dense(sum->args[0]), *b = dense(sum->args[1]);
        return a && b && a->data != b->data && (conv_chain(j, *f, a, b, act) || conv_chain(j, *f, b, a, act));
    }

    bool conv_chain(size_t j, const MapForm& f, const MapForm::Read* link, const MapForm::Read* residual, int act) {
        const long w = writer_of(link->data, j);
        if (w < 0 || !ours((size_t) w)) return false;
        const size_t i = (size_t) w;
        const auto* c = dynamic_cast<const tensor::ConvNode*>(blocks_[i].node.get());
        if (!c || c->element() != P::Float || c->shape().size() != 4) return false;
        const Expression whole = symbolic::mul(symbolic::mul(c->shape()[0], c->output_channels()), symbolic::mul(c->output_dim(0), c->output_dim(1)));
        if (!symbolic::equal(symbolic::product(f.bounds, 0, f.bounds.size()), whole) || !private_to(link->data, {i, j})) return false;
        // what the convolution reads it now reads where block j stands; the result overlaps none of it, nor the residual
        std::vector<std::string> connectors{"X", "W"};
        if (c->has_bias()) connectors.push_back("B");
        std::vector<ConnectorBinding> inputs;
        for (auto& name : connectors) {
            inputs.push_back(*blocks_[i].input(name));
            if (inputs.back().is_constant || lost_between(inputs.back().data, i, j) || inputs.back().data == f.results[0].data) return false;
        }
        if (residual) {
            if (residual->data == f.results[0].data) return false;
            connectors.push_back("_residual"), inputs.push_back(bind("_residual", residual->data));
        }
        auto node = std::make_unique<ConvChainLaunch>(connectors);
        node->extents = conv_launch_extents(*c);
        node->group = c->group();
        node->has_bias = c->has_bias();
        node->has_residual = residual != nullptr;
        node->activation = act;
        install(j, std::move(node), std::move(inputs), f.results[0].data, {i}, {link->data});
        return true;
    }

    // ---- a layer norm and the layer on a few rows behind it ---------------------------------------------
    bool norm_linear(size_t j) {
        const auto* l = dynamic_cast<const LinearLaunch*>(blocks_[j].node.get());
        if (!l || l->trans_a || !l->trans_b) return false;
        const std::string link = blocks_[j].input("_a")->data;
        const long w = writer_of(link, j);
        const auto* norm = w < 0 ? nullptr : dynamic_cast<const LayerNormLaunch*>(blocks_[(size_t) w].node.get());
        if (!norm || norm->type != l->type || !symbolic::equal(norm->rows, l->m) || !symbolic::equal(norm->cols, l->k) || !symbolic::equal(l->lda, l->k)) return false;
        const size_t i = (size_t) w;
        // up to 16 rows of a line of 128 bytes and more: what the launcher has a kernel for
        int64_t m = 0, k = 0;
        if (!symbolic::is_integer(l->m, &m) || !symbolic::is_integer(l->k, &k) || m > 16 || k * (l->type == P::BFloat ? 2 : 4) < 128) return false;
        if (!private_to(link, {i, j})) return false;
        for (auto& in : blocks_[j].inputs)      // the rows as residual, weights or bias as well: the one launch does not store them
            if (in.connector != "_a" && !in.is_constant && in.data == link) return false;
        std::vector<std::string> connectors{"_x"};
        std::vector<ConnectorBinding> inputs{bind("_x", blocks_[i].input("_x")->data)};
        for (const char* name : {"_weight", "_bias"}) {
            if (!(name[1] == 'w' ? norm->has_weight : norm->has_bias)) continue;
            connectors.push_back(name[1] == 'w' ? "_weight" : "_norm_bias");
            inputs.push_back(bind(connectors.back(), blocks_[i].input(name)->data));
        }
        const std::string result = blocks_[j].outputs[0].data;
        for (auto& in : inputs)      // read where block j stands, by every work-group
            if (lost_between(in.data, i, j) || in.data == result) return false;
        for (auto& in : blocks_[j].inputs) {
            connectors.push_back(in.connector == "_a" ? "_scratch" : in.connector);
            inputs.push_back(in);
            inputs.back().connector = connectors.back();
        }
        auto node = std::make_unique<NormLinearLaunch>(connectors);
        node->m = l->m, node->n = l->n, node->k = l->k, node->ldb = l->ldb, node->eps = norm->eps;
        node->type = l->type, node->bias_type = l->bias_type, node->residual_type = l->residual_type, node->y_type = l->y_type;
        node->has_weight = norm->has_weight, node->has_norm_bias = norm->has_bias, node->has_bias = l->has_bias, node->has_residual = l->has_residual;
        node->activation = l->activation, node->rounding = l->rounding;
        install(j, std::move(node), std::move(inputs), result, {i}, {});
        return true;
    }

    // ---- a softmax between its operand's upload and its result's download ------------------------------
    bool softmax_host(size_t j) {
        const auto* n = dynamic_cast<const tensor::SoftmaxNode*>(blocks_[j].node.get());
        if (!n || !ours(j)) return false;
        const std::string x = blocks_[j].input("X")->data, y = blocks_[j].outputs[0].data;
        const long w = writer_of(x, j);
        if (w < 0 || !is_offloading(blocks_[(size_t) w])) return false;
        const size_t i = (size_t) w;
        const auto& up = static_cast<const ROCMDataOffloadingNode&>(*blocks_[i].node);
        size_t l = j + 1;
        while (l < blocks_.size() && !touches(blocks_[l], y)) l++;
        if (l == blocks_.size() || !is_offloading(blocks_[l])) return false;
        const auto& down = static_cast<const ROCMDataOffloadingNode&>(*blocks_[l].node);
        if (!up.is_h2d() || !up.is_alloc() || !down.is_d2h() || !down.is_free() || !private_to(x, {i, j}) || !private_to(y, {j, l})) return false;
        if (!symbolic::equal(up.size(), n->connector_bytes("X")) || !symbolic::equal(down.size(), n->connector_bytes("Y"))) return false;
        int64_t bytes = 0;
        if (symbolic::is_integer(up.size(), &bytes) && bytes < (int64_t(16) << 20)) return false;   // copied as a whole anyway
        // the upload moves to where the download stands: nothing in between writes its source or touches the result
        const std::string from = blocks_[i].inputs[0].data, to = blocks_[l].outputs[0].data;
        if (lost_between(from, i, l)) return false;
        for (size_t k = i + 1; k < l; k++)
            if (k != j && touches(blocks_[k], to)) return false;
        auto node = std::make_unique<SoftmaxHostLaunch>();
        node->outer = n->outer(), node->extent = n->extent(), node->inner = n->inner();
        node->fp64 = n->element() == P::Double;
        node->rows = n->last_axis_only() && n->element() == P::Float;
        if (node->rows) node->outer = n->rows(), node->extent = n->cols();
        install(l, std::move(node), {bind("_x", from)}, to, {i, j}, {x, y});
        return true;
    }

    // ---- layer norm ------------------------------------------------------------------------------------
    // the Mean over the trailing loops from `trailing` on whose result a form of loops `bounds` loads once per row
    const tensor::ReduceNode* row_mean(const std::string& name, size_t before, size_t* at) const {
        const long w = writer_of(name, before);
        if (w < 0 || !ours((size_t) w)) return nullptr;
        const auto* r = dynamic_cast<const tensor::ReduceNode*>(blocks_[(size_t) w].node.get());
        if (!r || r->code() != "ml::Mean" || r->element() != P::Float || !r->adjacent_axes() || r->inner() != "1") return nullptr;
        *at = (size_t) w;
        return r;
    }

    bool layer_norm(size_t q) {
        if (!ours(q)) return false;
        std::optional<MapForm> f = convert_.form_of(blocks_[q]);
        if (!f || f->results.size() != 1 || !floating16(f->results[0].element)) return false;
        const Values v(*f);
        if (!v.plain_float()) return false;
        const size_t loops = f->bounds.size();
        const std::vector<Expression> whole = dense_strides(f->bounds, 0, loops);
        if (!same_strides(f->results[0].strides, whole)) return false;
        bool out16 = false;
        std::string top = v.through_casts(f->results[0].value, &out16);
        if (out16 != (f->results[0].element == P::BFloat)) return false;

        // [(centred / sqrt(var + eps)) * weight] + bias, weight and bias optional
        const MapForm::Read *weight = nullptr, *bias = nullptr;
        auto loaded = [&](const std::string& name) -> const MapForm::Read* {
            bool rounded = false;
            const MapForm::Read* r = v.read(v.through_casts(name, &rounded));
            return r && !rounded && floating16(r->element) ? r : nullptr;
        };
        auto peel = [&](const char* op, const MapForm::Read** operand) {
            const std::string rest = v.other(top, op, [&](const std::string& a) { return loaded(a) != nullptr; });
            if (rest.empty()) return;
            const Statement* s = v.statement(top, op);
            *operand = loaded(s->args[0] == rest ? s->args[1] : s->args[0]);
            top = rest;
        };
        peel("fp_add", &bias);
        peel("fp_mul", &weight);
        const Statement* div = v.statement(top, "fp_div");
        if (!div) return false;
        // sqrt(var + eps): in this block, or - a single row has no loop the map fusion could place it in - in one of its own
        std::set<size_t> gone;
        std::set<std::string> links;
        std::string var_data, eps;
        std::vector<Expression> var_strides;
        auto root_of = [&](const Values& in, const std::string& name) {
            const Statement* root = in.statement(name, "sqrt");
            const std::string value = root ? in.other(root->args[0], "fp_add", [&](const std::string& a) { return in.constant(a) != ""; }) : "";
            const MapForm::Read* var = value.empty() ? nullptr : in.read(value);
            if (!var || var->element != P::Float) return false;
            const Statement* plus = in.statement(root->args[0], "fp_add");
            eps = in.constant(plus->args[0] == value ? plus->args[1] : plus->args[0]);
            var_data = var->data;
            var_strides = var->strides;
            return true;
        };
        const MapForm::Read *centred = v.read(div->args[0]), *scale = v.read(div->args[1]);
        if (!centred || centred->element != P::Float || !same_strides(centred->strides, whole)) return false;
        if (scale) {
            const long w5 = writer_of(scale->data, q);
            std::optional<MapForm> f5 = w5 >= 0 && ours((size_t) w5) ? convert_.form_of(blocks_[(size_t) w5]) : std::nullopt;
            if (!f5 || f5->results.size() != 1 || f5->results[0].element != P::Float || f5->bounds != std::vector<Expression>{"1"}) return false;
            const Values v5(*f5);
            if (scale->element != P::Float || !v5.plain_float() || !root_of(v5, f5->results[0].value)) return false;
            var_strides = scale->strides;
            gone.insert((size_t) w5);
            links.insert(scale->data);
        } else if (!root_of(v, div->args[1])) {
            return false;
        }

        size_t i3, i1;
        const tensor::ReduceNode* mean2 = row_mean(var_data, q, &i3);
        if (!mean2) return false;
        const std::string squares = blocks_[i3].input("X")->data;
        const long w2 = writer_of(squares, i3);
        if (w2 < 0 || !ours((size_t) w2) || writer_of(centred->data, q) != w2) return false;
        const size_t i2 = (size_t) w2;
        std::optional<MapForm> f2 = convert_.form_of(blocks_[i2]);
        if (!f2 || f2->results.size() != 2 || f2->bounds != f->bounds) return false;
        const Values v2(*f2);
        if (!v2.plain_float()) return false;
        std::string c_value, s_value;
        for (auto& r : f2->results) {
            if (!same_strides(r.strides, whole) || r.element != P::Float) return false;
            if (r.data == centred->data) c_value = r.value;
            if (r.data == squares) s_value = r.value;
        }
        const Statement *sq = v2.statement(s_value, "fp_mul"), *sub = v2.statement(c_value, "fp_sub");
        if (!sq || !sub || sq->args[0] != c_value || sq->args[1] != c_value) return false;
        const MapForm::Read *x = v2.read(sub->args[0]), *mean = v2.read(sub->args[1]);
        if (!x || !mean || x->element != P::Float || mean->element != P::Float || !same_strides(x->strides, whole)) return false;
        const tensor::ReduceNode* mean1 = row_mean(mean->data, i2, &i1);
        if (!mean1 || mean1->shape() != mean2->shape() || mean1->sorted_axes() != mean2->sorted_axes() || blocks_[i1].input("X")->data != x->data) return false;

        // which loops are the reduced ones, and that the rows' values and weight and bias are laid out by that
        size_t split = loops;
        Expression extent = "1";
        while (split > 0 && !symbolic::equal(extent, mean1->extent())) extent = symbolic::mul(f->bounds[--split], extent);
        if (!symbolic::equal(extent, mean1->extent()) || !symbolic::equal(symbolic::product(f->bounds, 0, split), mean1->outer())) return false;
        const std::vector<Expression> per_row = dense_strides(f->bounds, 0, split), per_column = dense_strides(f->bounds, split, loops);
        if (!same_strides(var_strides, per_row) || !same_strides(mean->strides, per_row)) return false;
        for (auto* r : {weight, bias})
            if (r && !same_strides(r->strides, per_column)) return false;

        // float32 throughout, or bf16 rows, weight, bias and result around it
        gone.insert({i1, i2, i3});
        links.insert({mean->data, centred->data, squares, var_data});
        std::string source = x->data;
        const P type = out16 ? P::BFloat : P::Float;
        if (out16) {
            const long w0 = writer_of(x->data, i1);
            const auto* cast = w0 < 0 ? nullptr : dynamic_cast<const tensor::CastNode*>(blocks_[(size_t) w0].node.get());
            if (!cast || !ours((size_t) w0) || cast->element() != P::BFloat || cast->target_type() != P::Float) return false;
            source = blocks_[(size_t) w0].input("X")->data;
            gone.insert((size_t) w0);
            links.insert(x->data);
        }
        for (auto* r : {weight, bias})
            if (r && r->element != type) return false;
        std::set<size_t> users = gone;
        users.insert(q);
        for (auto& name : links)
            if (!private_to(name, users)) return false;
        const std::string result = f->results[0].data;
        if (lost_between(source, *gone.begin(), q)) return false;
        for (auto* r : {weight, bias})   // (X in place is fine: a row is read before it is written)
            if (r && r->data == result) return false;

        std::vector<std::string> connectors{"_x"};
        std::vector<ConnectorBinding> inputs{bind("_x", source)};
        if (weight) connectors.push_back("_weight"), inputs.push_back(bind("_weight", weight->data));
        if (bias) connectors.push_back("_bias"), inputs.push_back(bind("_bias", bias->data));
        auto node = std::make_unique<LayerNormLaunch>(connectors);
        node->rows = mean1->outer(), node->cols = mean1->extent(), node->eps = eps;
        node->type = type;
        node->has_weight = weight != nullptr;
        node->has_bias = bias != nullptr;
        install(q, std::move(node), std::move(inputs), result, gone, links);
        return true;
    }

    StructuredSDFG& sdfg_;
    std::vector<Block>& blocks_;
    Converter convert_;
    std::vector<Lifetime> lifetimes_;
};

// ---- dispatchers ---------------------------------------------------------------------------------------

class LaunchDispatcher : public codegen::LibraryNodeDispatcher {
public:
    using LibraryNodeDispatcher::LibraryNodeDispatcher;

    void dispatch_code(codegen::PrettyPrinter& s, codegen::PrettyPrinter& globals, codegen::CodeSnippetFactory&) override {
        emit_runtime_preamble(globals, function_);
        if (const auto* l = dynamic_cast<const LinearLaunch*>(&node_)) {
            // an empty product is not launched, as the GEMM's dispatcher has it (a leading dimension of 0 is an error to the launcher)
            s << "if ((" << l->m << ") != 0 && (" << l->n << ") != 0) DOCC_ROCM_CHECK(docc_rocm_linear(nullptr, " << type_code(l->type) << ", " << (l->trans_a ? 112 : 111) << ", " << (l->trans_b ? 112 : 111)
              << ", " << l->m << ", " << l->n << ", " << l->k << ", (float) __alpha, _a, " << l->lda << ", _b, " << l->ldb << ", "
              << (l->has_bias ? "_bias" : "nullptr") << ", " << type_code(l->bias_type) << ", " << l->activation << ", "
              << (l->has_residual ? "_residual" : "nullptr") << ", " << type_code(l->residual_type) << ", " << l->rounding << ", _y, " << type_code(l->y_type)
              << "));" << std::endl;
        } else if (const auto* l = dynamic_cast<const NormLinearLaunch*>(&node_)) {
            s << "if ((" << l->m << ") != 0 && (" << l->n << ") != 0) DOCC_ROCM_CHECK(docc_rocm_norm_linear(nullptr, " << type_code(l->type) << ", " << l->m << ", " << l->n << ", "
              << l->k << ", (float) (" << l->eps << "), _x, " << (l->has_weight ? "_weight" : "nullptr") << ", " << (l->has_norm_bias ? "_norm_bias" : "nullptr")
              << ", (float) __alpha, _b, " << l->ldb << ", " << (l->has_bias ? "_bias" : "nullptr") << ", " << type_code(l->bias_type) << ", " << l->activation << ", "
              << (l->has_residual ? "_residual" : "nullptr") << ", " << type_code(l->residual_type) << ", " << l->rounding << ", _scratch, _y, " << type_code(l->y_type) << "));"
              << std::endl;
        } else if (const auto* c = dynamic_cast<const ConvChainLaunch*>(&node_)) {
            s << "{" << std::endl;
            s.setIndent(s.indent() + 4);
            int64_t group = 0;
            const bool whole = symbolic::is_integer(c->group, &group) && group == 1;   // grouped convolutions take no workspace
            s << "const int64_t __ws_bytes = " << (whole ? conv_launch_workspace(c->extents, "W") : std::string("0")) << ";" << std::endl;
            s << "void *__ws = nullptr;" << std::endl;
            s << "if (__ws_bytes > 0) DOCC_ROCM_CHECK(docc_rocm_malloc_async(&__ws, (size_t) __ws_bytes, nullptr));" << std::endl;
            s << "DOCC_ROCM_CHECK(docc_rocm_conv2d_f32_chain(nullptr, " << c->extents << ", (int64_t) (" << c->group << "), X, W, " << (c->has_bias ? "B" : "nullptr") << ", "
              << (c->has_residual ? "_residual" : "nullptr") << ", " << c->activation << ", _y, __ws, __ws_bytes));" << std::endl;
            s << "if (__ws) DOCC_ROCM_CHECK(docc_rocm_free_async(__ws, nullptr));" << std::endl;
            s.setIndent(s.indent() - 4);
            s << "}" << std::endl;
        } else if (const auto* h = dynamic_cast<const SoftmaxHostLaunch*>(&node_)) {
            if (h->rows) s << "DOCC_ROCM_CHECK(docc_rocm_softmax_f32_host(nullptr, " << h->outer << ", " << h->extent << ", _x, _y));" << std::endl;
            else s << "DOCC_ROCM_CHECK(docc_rocm_softmax_host(nullptr, " << (h->fp64 ? 64 : 32) << ", " << h->outer << ", " << h->extent << ", " << h->inner
              << ", _x, _y));" << std::endl;
        } else if (const auto* n = dynamic_cast<const LayerNormLaunch*>(&node_)) {
            s << "DOCC_ROCM_CHECK(docc_rocm_layer_norm(nullptr, " << type_code(n->type) << ", " << n->rows << ", " << n->cols << ", (float) (" << n->eps
              << "), _x, " << (n->has_weight ? "_weight" : "nullptr") << ", " << (n->has_bias ? "_bias" : "nullptr") << ", _y));" << std::endl;
        }
    }
};

} // namespace

bool RocmLaunchFusionPass::run_pass(builder::StructuredSDFGBuilder& builder, analysis::AnalysisManager&) { return LaunchFusion(builder.subject()).run(); }

void register_launch_dispatchers(codegen::LibraryNodeDispatcherRegistry& reg) {
    for (auto& code : {LibraryNodeType_ROCM_Linear, LibraryNodeType_ROCM_NormLinear, LibraryNodeType_ROCM_ConvChain, LibraryNodeType_ROCM_SoftmaxHost, LibraryNodeType_ROCM_LayerNorm})
        reg.register_library_node_dispatcher(code + "::" + ImplementationType_ROCMWithoutTransfers,
                                             [](codegen::LanguageExtension& le, const Function& f, const data_flow::DataFlowGraph& b, const LibraryNode& n) {
                                                 return std::make_unique<LaunchDispatcher>(le, f, b, n);
                                             });
}

} // namespace sdfg::rocm
