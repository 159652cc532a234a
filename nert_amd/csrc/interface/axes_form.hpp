#pragma once
// Stand-in for NERT's axes-form helpers (see nert/graph.hpp beside it): where
// Squeeze, Unsqueeze, ReduceSum and Split take their axes or sizes from. The
// ONNX operators moved them from an attribute to an input at version 13; an
// unversioned node with the attribute and no such input keeps the attribute.

#include "nert/device.hpp"

#include <string>
#include <vector>

namespace nert {

enum class AxesSource { Attribute, Input };

inline const Attribute* NodeAttribute(const Node& node, const char* name) {
    for (const Attribute& attr : node.attributes) {
        if (attr.name == name) {
            return &attr;
        }
    }
    return nullptr;
}

inline const std::vector<int64_t>* NodeAttributeIntList(const Attribute* attr) {
    return attr == nullptr ? nullptr : std::get_if<std::vector<int64_t>>(&attr->value);
}

// Elements of a 1-D axes tensor; a negative extent is an error.
inline int64_t AxesElementCount(const std::vector<int64_t>& dims, const std::string& context) {
    int64_t count = 1;
    for (const int64_t dim : dims) {
        if (dim < 0) {
            throw InferenceException(context + ": negative dimension");
        }
        count *= dim;
    }
    return count;
}

inline bool TakesAttribute(const Node& node, const Attribute* attr, int64_t input_since) {
    if (node.schema_version > 0) {
        return node.schema_version < input_since;
    }
    const bool has_input = node.inputs.size() > 1 && !node.inputs[1].empty();
    return attr != nullptr && !has_input;
}

struct AxesForm {
    AxesSource source = AxesSource::Input;
    const Attribute* axes_attribute = nullptr;
};

inline AxesForm ResolveAxesForm(const Node& node) {
    const Attribute* axes = NodeAttribute(node, "axes");
    if (TakesAttribute(node, axes, 13)) {
        return {AxesSource::Attribute, axes};
    }
    return {};
}

struct SplitForm {
    AxesSource source = AxesSource::Input;
    const Attribute* split_attribute = nullptr;
};

inline SplitForm ResolveSplitForm(const Node& node) {
    const Attribute* split = NodeAttribute(node, "split");
    if (TakesAttribute(node, split, 13)) {
        return {AxesSource::Attribute, split};
    }
    return {};
}

// Sizes of a Split without explicit sizes: equal parts, the last one smaller
// where num_outputs (version 18) allows it.
inline std::vector<int64_t> DefaultSplitParts(const Node& node, int64_t dim, size_t outputs, bool parts_supplied,
                                              const std::string& context) {
    const Attribute* given = NodeAttribute(node, "num_outputs");
    const int64_t count = static_cast<int64_t>(outputs);
    if (given != nullptr) {
        const int64_t* n = std::get_if<int64_t>(&given->value);
        if (n == nullptr) {
            throw InferenceException(context + ": attribute 'num_outputs' must be an integer");
        }
        if (*n != count) {
            throw InferenceException(context + ": Split num_outputs must match the output count");
        }
    }
    if (parts_supplied) {
        return {};
    }
    const int64_t part = given != nullptr ? (dim + count - 1) / count : dim / count;
    if (given == nullptr && part * count != dim) {
        throw InferenceException(context + ": Split axis must divide evenly");
    }
    std::vector<int64_t> parts(outputs, part);
    if (!parts.empty()) {
        parts.back() = dim - part * (count - 1);
        if (parts.back() < 0) {
            throw InferenceException(context + ": Split split sizes must be non-negative");
        }
    }
    return parts;
}

} // namespace nert
