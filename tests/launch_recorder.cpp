// Stand-in for the HIP runtime that records kernel launches instead of making them.  Loaded with RTLD_GLOBAL in front of the
// library, it answers every HIP call the library's host code makes, so that what a call would launch can be looked at on a
// machine without a GPU (tests/test_dispatch_cpu.py, in a process of its own).
#include <hip/hip_runtime.h>

#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "../cute-examples_amd/csrc/gemm_launch.h"

namespace {
struct Launch {
  std::string name;
  int64_t v[12];
};
std::map<const void*, std::string>& names() { static std::map<const void*, std::string> m; return m; }
std::vector<Launch>& launches() { static std::vector<Launch> l; return l; }
dim3 pushed_grid, pushed_block;
}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) { static void* module; return &module; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names()[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t) {
  pushed_grid = grid;
  pushed_block = block;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
  *grid = pushed_grid;
  *block = pushed_block;
  *shared = 0;
  *stream = nullptr;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDevice(int* device) { *device = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* value, hipDeviceAttribute_t, int) { *value = 256; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** address, const void*) { *address = (void*)(uintptr_t)(1u << 30); return hipSuccess; }

// v: of the GEMM kernels M, N, K, lda, ldb, ldc, A, B, C, c_ragged, splits, tail_tiles; of the repack kernel, for the first and
// then the second operand, rows, row stride in bytes, source, destination, destination's row stride, workgroups; of the others
// nothing.
hipError_t hipLaunchKernel(const void* function, dim3 grid, dim3, void** args, size_t, hipStream_t) {
  Launch l = {names()[function], {}};
  const auto has = [&](const char* part) { return l.name.find(part) != std::string::npos; };
  if (has("gemm_tn_")) {
    const mi355::GemmArgs& g = *(const mi355::GemmArgs*)args[0];
    const int64_t v[12] = {g.M, g.N, g.K, g.lda, g.ldb, g.ldc, (int64_t)g.A, (int64_t)g.B, (int64_t)g.C, g.c_ragged, g.splits, g.tail_tiles};
    std::memcpy(l.v, v, sizeof v);
  } else if (has("repack_rows")) {
    const uint32_t first_blocks = *(const uint32_t*)args[3];
    for (int i = 0; i < 2; ++i) {
      const mi355::RepackOperand& o = *(const mi355::RepackOperand*)args[i];
      const int64_t v[6] = {o.rows, o.src_ld, (int64_t)o.src, (int64_t)o.dst, o.dst_ld, i == 0 ? first_blocks : grid.x - first_blocks};
      std::memcpy(l.v + 6 * i, v, sizeof v);
    }
  }
  launches().push_back(l);
  return hipSuccess;
}

int recorded() { return (int)launches().size(); }
void forget() { launches().clear(); }
const char* recorded_name(int i) { return launches()[i].name.c_str(); }
const int64_t* recorded_values(int i) { return launches()[i].v; }

}  // extern "C"
