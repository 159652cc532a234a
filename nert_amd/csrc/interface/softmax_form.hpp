#pragma once
// Stand-in for NERT's softmax-form helper (see nert/graph.hpp beside it):
// before version 13 Softmax coerces its input to 2-D at `axis` (default 1);
// since then it works along one axis (default -1).

#include "axes_form.hpp"

namespace nert {

enum class SoftmaxForm { SingleAxis, LegacyCoerce2D };

inline SoftmaxForm ResolveSoftmaxForm(const Node& node) {
    return node.schema_version > 0 && node.schema_version < 13 ? SoftmaxForm::LegacyCoerce2D : SoftmaxForm::SingleAxis;
}

inline int64_t SoftmaxAxis(const Node& node, SoftmaxForm form, const std::string& context) {
    const Attribute* attr = NodeAttribute(node, "axis");
    if (attr == nullptr) {
        return form == SoftmaxForm::LegacyCoerce2D ? 1 : -1;
    }
    const int64_t* axis = std::get_if<int64_t>(&attr->value);
    if (axis == nullptr) {
        throw InferenceException(context + ": attribute 'axis' must be an integer");
    }
    return *axis;
}

} // namespace nert
