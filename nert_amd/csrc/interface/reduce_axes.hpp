#pragma once
// Stand-in for NERT's reduce-axes helpers (see nert/graph.hpp beside it):
// ReduceMean, ReduceMax and ReduceL2 take their axes from an input since
// version 18 of the operator set, from an attribute before.

#include "axes_form.hpp"

namespace nert {

enum class ReduceAxesForm { Attribute, Input };

struct ReduceAxes {
    ReduceAxesForm form = ReduceAxesForm::Input;
    const Attribute* axes_attribute = nullptr;
    bool noop_with_empty_axes = false;
};

inline const std::vector<int64_t>* ReduceAttributeIntList(const Attribute* attr) { return NodeAttributeIntList(attr); }

inline int64_t ReduceAxesElementCount(const std::vector<int64_t>& dims, const std::string& context) {
    return AxesElementCount(dims, context);
}

inline ReduceAxes ResolveReduceAxes(const Node& node) {
    const Attribute* axes = NodeAttribute(node, "axes");
    if (TakesAttribute(node, axes, 18)) {
        return {ReduceAxesForm::Attribute, axes, false};
    }
    const Attribute* noop = NodeAttribute(node, "noop_with_empty_axes");
    const int64_t* flag = noop == nullptr ? nullptr : std::get_if<int64_t>(&noop->value);
    return {ReduceAxesForm::Input, nullptr, flag != nullptr && *flag != 0};
}

} // namespace nert
