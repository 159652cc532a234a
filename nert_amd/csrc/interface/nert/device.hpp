#pragma once
// Stand-in for NERT's device seam (see graph.hpp beside it).

#include "nert/graph.hpp"

#include <cstdint>
#include <string>
#include <vector>

namespace nert {

// A borrowed dense tensor; the default value marks an omitted operand.
struct TensorView {
    void* data = nullptr;
    DataType dtype = DataType::Unknown;
    std::vector<int64_t> dims;
};

using KernelFn = void (*)(const Node&, const std::vector<TensorView>&, const std::vector<TensorView>&);

class Allocator {
  public:
    virtual ~Allocator() = default;
    virtual void* allocate(int64_t bytes) = 0;
    virtual void release(void* buffer) = 0;
};

class Transfer {
  public:
    virtual ~Transfer() = default;
    virtual void host_to_device(void* dst, const void* src, int64_t bytes) = 0;
    virtual void device_to_host(void* dst, const void* src, int64_t bytes) = 0;
};

class KernelTable {
  public:
    virtual ~KernelTable() = default;
    virtual KernelFn find(const std::string& op_type) const = 0;
};

class Device {
  public:
    virtual ~Device() = default;
    virtual const char* name() const = 0;
    virtual Allocator& allocator() = 0;
    virtual Transfer& transfer() = 0;
    virtual const KernelTable& kernels() const = 0;
    virtual bool is_host() const = 0;
    virtual bool supports_arena_offsets() const { return true; }
};

const Device& HipDevice();

} // namespace nert
