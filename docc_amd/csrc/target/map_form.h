// Blocks of elementwise kind as loops over a shape (MapForm): what the passes that merge them work on - the map fusion pass
// (map_fusion.cpp) and the launch fusion at code generation (launch_fusion.cpp).
#pragma once

#include <map>
#include <optional>

#include "rocm_target.h"

namespace sdfg::rocm {

using data_flow::ConnectorBinding;
using structured_control_flow::Block;
namespace tensor = math::tensor;
using Statement = ROCMMapNode::Statement;
using P = types::PrimitiveType;

inline bool is_rocm_map_type(const std::string& impl) {
    return impl == ImplementationType_ROCMWithTransfers || impl == ImplementationType_ROCMWithoutTransfers;
}

// A block of elementwise kind written as loops over a shape: loads, statements on values, one store. Values carry
// names that are unique within the pass; the node built from the form renames them.
struct MapForm {
    struct Read {
        std::string data;
        std::vector<Expression> strides;
        Expression extent;
        P element;
        std::string value;
    };
    struct Scalar {
        ConnectorBinding source;   // a scalar container or a constant
        P element;
        std::string value;
    };
    std::vector<Expression> bounds;
    std::vector<Read> reads;
    std::vector<Scalar> scalars;
    struct Result {
        std::string value, data;
        std::vector<Expression> strides;
        Expression extent;
        P element;
    };
    std::vector<Statement> statements;
    std::vector<Result> results;   // the tensor nodes have one; a nest that was imported, or merged, may store several
    P element = P::Float;          // of the statements a tensor node becomes
};

class Converter {
public:
    explicit Converter(const StructuredSDFG& sdfg) : sdfg_(sdfg) {}

    // nullopt: the block is not of elementwise kind (or uses an operation the statements cannot spell)
    std::optional<MapForm> form_of(const Block& blk) {
        if (!is_rocm_map_type(blk.node->implementation_type()) || blk.outputs.empty()) return std::nullopt;
        std::optional<MapForm> f;
        if (auto* m = dynamic_cast<const ROCMMapNode*>(blk.node.get())) f = from_map(blk, *m);
        else if (auto* e = dynamic_cast<const tensor::ElementWiseNode*>(blk.node.get())) f = from_elementwise(blk, *e);
        else if (auto* fe = dynamic_cast<const ROCMFusedElementWiseNode*>(blk.node.get())) f = from_fused(blk, *fe);
        else if (auto* b = dynamic_cast<const tensor::BroadcastNode*>(blk.node.get())) f = from_broadcast(blk, *b);
        else if (auto* c = dynamic_cast<const tensor::CastNode*>(blk.node.get())) f = from_cast(blk, *c);
        if (f && f->bounds.size() > 6) return std::nullopt;   // a ROCMMap node holds at most six loops
        return f;
    }

    std::string fresh(const char* kind) { return std::string(kind) + std::to_string(counter_++); }

private:
    // loops: the dimensions of `shape` that are not literally 1 (a single loop of one iteration if none is left)
    static std::vector<size_t> kept_dims(const std::vector<Expression>& shape) {
        std::vector<size_t> kept;
        for (size_t d = 0; d < shape.size(); d++)
            if (shape[d] != "1") kept.push_back(d);
        return kept;
    }

    // Strides of a dense row-major operand of shape `own` (same rank as `shape` after right alignment; an extent of 1
    // where `shape` has more repeats the operand) along the loops, in the spelling the kernel planner merges loops by.
    static bool layout(const std::vector<Expression>& shape, std::vector<Expression> own, std::vector<Expression>* strides, Expression* extent) {
        if (own.size() > shape.size()) return false;
        own.insert(own.begin(), shape.size() - own.size(), "1");
        const std::vector<size_t> kept = kept_dims(shape);
        std::vector<Expression> per(kept.empty() ? 1 : kept.size(), "0");
        Expression run = "1";
        for (size_t k = kept.size(); k-- > 0;) {
            const size_t d = kept[k];
            if (own[d] == "1") continue;          // repeated along this loop
            if (own[d] != shape[d]) return false;
            per[k] = run;
            run = run == "1" ? own[d] : "(" + own[d] + ")*" + run;
        }
        *strides = per;
        *extent = run;
        return true;
    }

    static std::vector<Expression> bounds_of(const std::vector<Expression>& shape) {
        std::vector<Expression> b;
        for (size_t d : kept_dims(shape)) b.push_back(shape[d]);
        if (b.empty()) b.push_back("1");
        return b;
    }

    // a connector's value: a load (array), a kernel argument (scalar container or constant)
    bool operand(MapForm& f, const Block& blk, const std::string& connector, const std::vector<Expression>& shape,
                 const std::vector<Expression>& own_shape, std::string* value, std::optional<P> loaded_as = std::nullopt) {
        const ConnectorBinding* in = blk.input(connector);
        if (!in) return false;
        if (in->is_constant || !sdfg_.container(in->data).is_pointer) {
            // passed by value as the host code holds it: the local of the connector has the constant's or the container's type
            const P held = in->is_constant ? in->type : sdfg_.container(in->data).element;
            if (!floating(held)) return false;
            MapForm::Scalar s{*in, held, fresh("s")};
            *value = s.value;
            f.scalars.push_back(std::move(s));
            return true;
        }
        MapForm::Read r;
        r.data = in->data;
        r.element = loaded_as.value_or(f.element);
        if (!layout(shape, own_shape, &r.strides, &r.extent)) return false;
        r.value = fresh("r");
        *value = r.value;
        f.reads.push_back(std::move(r));
        return true;
    }

    bool result(MapForm& f, const Block& blk, const std::vector<Expression>& shape, const std::string& value) {
        MapForm::Result r;
        r.data = blk.outputs[0].data;
        r.value = value;
        r.element = f.element;
        if (!layout(shape, shape, &r.strides, &r.extent)) return false;
        f.results.push_back(std::move(r));
        return true;
    }

    std::string emit(MapForm& f, const std::string& op, std::vector<std::string> args) {
        Statement st{fresh("t"), f.element, op, std::move(args)};
        f.statements.push_back(st);
        return st.out;
    }

    // the operations of elementwise_ops.h as statements; empty: not spelled here
    std::string unary(MapForm& f, const std::string& code, const std::string& x) {
        static const std::map<std::string, std::string> calls = {{"ml::Abs", "fabs"}, {"ml::Exp", "exp"}, {"ml::Sqrt", "sqrt"},
                                                                 {"ml::Tanh", "tanh"}, {"ml::Erf", "erf"}};
        auto c = calls.find(code);
        if (c != calls.end()) return emit(f, c->second, {x});
        if (code == "ml::ReLU") return emit(f, "fmax", {x, "#0.0"});
        if (code == "ml::Sigmoid") {
            const std::string e = emit(f, "exp", {emit(f, "fp_neg", {x})});
            return emit(f, "fp_div", {"#1.0", emit(f, "fp_add", {"#1.0", e})});
        }
        return "";
    }

    std::string binary(MapForm& f, const std::string& code, const std::string& a, const std::string& b) {
        static const std::map<std::string, std::string> ops = {{"ml::Add", "fp_add"}, {"ml::Sub", "fp_sub"}, {"ml::Mul", "fp_mul"},
                                                               {"ml::Div", "fp_div"}, {"ml::Maximum", "fmax"}, {"ml::Minimum", "fmin"},
                                                               {"ml::Pow", "pow"}};
        auto o = ops.find(code);
        return o == ops.end() ? "" : emit(f, o->second, {a, b});
    }

    static bool floating(P t) { return t == P::Float || t == P::Double; }

    std::optional<MapForm> from_elementwise(const Block& blk, const tensor::ElementWiseNode& e) {
        if (!floating(e.element()) || e.shape().empty()) return std::nullopt;
        MapForm f;
        f.element = e.element();
        f.bounds = bounds_of(e.shape());
        std::string y;
        if (e.is_binary()) {
            std::string a, b;
            if (!operand(f, blk, "A", e.shape(), e.shape(), &a) || !operand(f, blk, "B", e.shape(), e.shape(), &b)) return std::nullopt;
            y = binary(f, e.code(), a, b);
        } else {
            std::string x;
            if (!operand(f, blk, "X", e.shape(), e.shape(), &x)) return std::nullopt;
            y = unary(f, e.code(), x);
        }
        if (y.empty() || !result(f, blk, e.shape(), y)) return std::nullopt;
        return f;
    }

    std::optional<MapForm> from_fused(const Block& blk, const ROCMFusedElementWiseNode& n) {
        if (!floating(n.element()) || n.shape().empty()) return std::nullopt;
        MapForm f;
        f.element = n.element();
        f.bounds = bounds_of(n.shape());
        std::string y;
        if (!operand(f, blk, "A", n.shape(), n.a_shape(), &y)) return std::nullopt;
        if (n.has_b()) {
            std::string b;
            if (!operand(f, blk, "B", n.shape(), n.b_shape(), &b)) return std::nullopt;
            y = binary(f, n.binary(), y, b);
            if (y.empty()) return std::nullopt;
        }
        for (auto& code : n.post()) {
            y = unary(f, code, y);
            if (y.empty()) return std::nullopt;
        }
        if (f.statements.empty()) y = emit(f, "assign", {y});
        if (!result(f, blk, n.shape(), y)) return std::nullopt;
        return f;
    }

    std::optional<MapForm> from_broadcast(const Block& blk, const tensor::BroadcastNode& b) {
        if (!floating(b.element()) || b.output_shape().empty()) return std::nullopt;
        MapForm f;
        f.element = b.element();
        f.bounds = bounds_of(b.output_shape());
        std::string x;
        if (!operand(f, blk, "X", b.output_shape(), b.input_shape(), &x)) return std::nullopt;
        if (!result(f, blk, b.output_shape(), emit(f, "assign", {x}))) return std::nullopt;
        return f;
    }

    // between float, double and bf16 (a bf16 tensor widened for the float32 nodes, their result rounded to bf16: the
    // compiler's conversions, to nearest even): the conversion is the assignment's
    std::optional<MapForm> from_cast(const Block& blk, const tensor::CastNode& c) {
        auto convertible = [](P t) { return floating(t) || t == P::BFloat; };
        if (!convertible(c.element()) || !convertible(c.target_type()) || c.shape().empty()) return std::nullopt;
        if (c.element() == P::BFloat && c.target_type() == P::BFloat) return std::nullopt;
        MapForm f;
        f.element = c.target_type();
        f.bounds = bounds_of(c.shape());
        std::string x;
        const ConnectorBinding* in = blk.input("X");
        if (!in || in->is_constant || !sdfg_.container(in->data).is_pointer) return std::nullopt;
        if (!operand(f, blk, "X", c.shape(), c.shape(), &x, c.element())) return std::nullopt;
        if (!result(f, blk, c.shape(), emit(f, "assign", {x}))) return std::nullopt;
        return f;
    }

    std::optional<MapForm> from_map(const Block& blk, const ROCMMapNode& m) {
        MapForm f;
        f.bounds = m.bounds();
        f.element = m.writes()[0].element;
        std::map<std::string, std::string> names;   // the node's names -> values of the pass
        for (auto& r : m.reads()) {
            const ConnectorBinding* in = blk.input(r.connector);
            if (!in || in->is_constant) return std::nullopt;
            names[r.connector] = fresh("r");
            f.reads.push_back({in->data, r.strides, r.extent, r.element, names[r.connector]});
        }
        for (auto& s : m.scalars()) {
            const ConnectorBinding* in = blk.input(s.connector);
            if (!in) return std::nullopt;
            names[s.connector] = fresh("s");
            f.scalars.push_back({*in, s.element, names[s.connector]});
        }
        auto renamed = [&](const std::string& name) { return name[0] == '#' ? name : names.at(name); };
        for (auto& st : m.statements()) {
            Statement out{fresh("t"), st.type, st.op, {}};
            for (auto& a : st.args) out.args.push_back(renamed(a));
            names[st.out] = out.out;
            f.statements.push_back(std::move(out));
        }
        for (auto& w : m.writes()) {
            const ConnectorBinding* out = blk.output(w.connector);
            if (!out) return std::nullopt;
            f.results.push_back({renamed(w.value), out->data, w.strides, w.extent, w.element});
        }
        return f;
    }

    const StructuredSDFG& sdfg_;
    size_t counter_ = 0;
};

} // namespace sdfg::rocm
