// The names of XLA's FFI API that bux_amd/xla/xla_ffi.cc uses, with just enough behind them
// to call its handlers as functions on buffers a test makes up. A handler's registration
// expands to nothing.
#pragma once

#include <cstddef>
#include <cstdint>
#include <string>
#include <utility>
#include <vector>

namespace xla::ffi {

enum class DataType { U8, S32, BF16, F32 };
enum class ErrorCode { kOk, kInvalidArgument, kInternal };

class Error {
 public:
  Error(ErrorCode code, std::string message) : code_(code), message_(std::move(message)) {}
  static Error Success() { return Error(ErrorCode::kOk, ""); }
  bool success() const { return code_ == ErrorCode::kOk; }
  ErrorCode errc() const { return code_; }
  const std::string& message() const { return message_; }

 private:
  ErrorCode code_;
  std::string message_;
};

class AnyBuffer {
 public:
  AnyBuffer(DataType type, std::vector<int64_t> dims, void* data = nullptr)
      : type_(type), dims_(std::move(dims)), data_(data) {}
  DataType element_type() const { return type_; }
  const std::vector<int64_t>& dimensions() const { return dims_; }
  size_t element_count() const {
    size_t n = 1;
    for (int64_t d : dims_) n *= static_cast<size_t>(d);
    return n;
  }
  size_t size_bytes() const {
    return element_count() * (type_ == DataType::U8 ? 1 : type_ == DataType::BF16 ? 2 : 4);
  }
  void* untyped_data() const { return data_; }

 private:
  DataType type_;
  std::vector<int64_t> dims_;
  void* data_;
};

template <typename T>
class Result {
 public:
  Result(T value) : value_(std::move(value)) {}
  T* operator->() { return &value_; }
  T& operator*() { return value_; }

 private:
  T value_;
};

template <typename T>
struct PlatformStream {};

}  // namespace xla::ffi

#define XLA_FFI_DEFINE_HANDLER_SYMBOL(name, impl, binding)
