// Calls two XLA FFI handlers on made-up buffers, the library's entry points replaced by
// ones that say they were reached. Prints a line a case: the error code, then the calls.
#include "../bux_amd/xla/xla_ffi.cc"

#include <cstdio>

static int calls = 0;
static int32_t word = 0;
static bool listed = false;

extern "C" const char* bux_last_error() { return ""; }
extern "C" int bux_moe_permute_layer(const int32_t*, int64_t, int32_t, const void*,
                                     int32_t weight_bytes, int32_t*, int32_t*, int32_t*, int32_t*,
                                     void*, void* list, size_t, int64_t, int64_t, void*, size_t,
                                     void*) {
  ++calls;
  word = weight_bytes;
  listed = list != nullptr;
  return 0;
}
extern "C" int bux_mx_grouped_rows_biased(const uint8_t*, const uint8_t*, const uint8_t*,
                                          const uint8_t*, void*, size_t, int32_t, int64_t, int64_t,
                                          int64_t, int64_t, int out_dtype, const void*, void*,
                                          void*) {
  ++calls;
  word = out_dtype;
  return 0;
}

using ffi::DataType;
static char memory[64];
static In buffer(DataType type, std::vector<int64_t> dims) { return In(type, std::move(dims), memory); }

static void sorted(DataType type, std::vector<int64_t> weights, DataType out_type, int64_t out,
                   int64_t list_bytes) {
  calls = 0;
  const In idx = buffer(DataType::S32, {10, 2});
  const Out ints = buffer(DataType::S32, {20});
  const ffi::Error e = MoePermuteLayer(nullptr, idx, buffer(type, std::move(weights)), 4, 128, 20,
                                       ints, ints, ints, ints, buffer(out_type, {out}),
                                       buffer(DataType::U8, {list_bytes}), buffer(DataType::U8, {64}));
  std::printf("%d %d %d %d\n", static_cast<int>(e.errc()), calls, word, static_cast<int>(listed));
}

static void biased(DataType type, std::vector<int64_t> bias, DataType out) {
  calls = 0;
  const In a = buffer(DataType::U8, {4, 128, 64}), b = buffer(DataType::U8, {3, 4, 96, 64});
  const ffi::Error e = MxRowsBiased(nullptr, a, a, b, b, buffer(DataType::U8, {512}),
                                    buffer(type, std::move(bias)), buffer(out, {128, 96}));
  std::printf("%d %d %d\n", static_cast<int>(e.errc()), calls, word);
}

int main() {
  sorted(DataType::BF16, {10, 2}, DataType::BF16, 20, 512);
  sorted(DataType::F32, {20}, DataType::F32, 20, 0);
  sorted(DataType::BF16, {9, 2}, DataType::BF16, 20, 512);
  sorted(DataType::BF16, {11, 2}, DataType::BF16, 20, 512);
  sorted(DataType::S32, {10, 2}, DataType::S32, 20, 512);
  sorted(DataType::BF16, {10, 2}, DataType::F32, 20, 512);
  sorted(DataType::BF16, {10, 2}, DataType::BF16, 19, 512);
  biased(DataType::BF16, {3, 96}, DataType::BF16);
  biased(DataType::F32, {3, 48, 2}, DataType::F32);
  biased(DataType::BF16, {2, 96}, DataType::BF16);
  biased(DataType::F32, {3, 96}, DataType::BF16);
  return 0;
}
