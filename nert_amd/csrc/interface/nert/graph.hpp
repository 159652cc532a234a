#pragma once
// Stand-in for NERT's graph types, for building this library without a NERT
// checkout: just the declarations the rows use, written from their use in
// this repository. A build with a checkout (NERT_REF) takes NERT's own
// headers instead; a library that is to be linked with NERT's executor has to
// be built that way, since only NERT's headers fix the C++ ABI of the seam.

#include <cstdint>
#include <stdexcept>
#include <string>
#include <utility>
#include <variant>
#include <vector>

namespace nert {

// What a row throws; the message names the op and the node.
class InferenceException : public std::runtime_error {
  public:
    using std::runtime_error::runtime_error;
};

enum class DataType { Float32, Int64, Bool, Unknown };

// One node attribute. The alternatives are in the order of nert_attr_kind.
struct Attribute {
    using Value = std::variant<int64_t, float, std::string, std::vector<int64_t>, std::vector<float>, bool>;

    Attribute(std::string attr_name, Value attr_value) : name(std::move(attr_name)), value(std::move(attr_value)) {}

    std::string name;
    Value value;
};

struct Node {
    std::string op_type;
    std::string name;
    std::vector<std::string> inputs; // an empty name is an omitted operand
    std::vector<std::string> outputs;
    std::vector<Attribute> attributes;
    int64_t schema_version = 0; // operator set version of the node; 0 when unversioned
};

} // namespace nert
