// fake_hip.h -- the HIP runtime's entry points that libcuot_amd.so calls, as
// stand-ins of a program with two imaginary devices: device memory is host memory,
// launches are written down and not run.  A program that defines them and links
// the library checks on the CPU what the library asks the runtime for.
#pragma once

#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>
#include <utility>
#include <vector>

struct Dim3 {
  uint32_t x, y, z;
};

struct Launch {
  std::string kernel;  // mangled name
  int device;
  Dim3 grid, block;
  size_t lds;
  void* stream;
};

static int g_device = 0;
static std::vector<Launch> g_launches;
static std::map<std::pair<int, std::string>, int> g_lds_limit;  // (device, kernel) -> dynamic LDS allowed
static std::map<std::pair<int, const void*>, int> g_symbol_uploads;

static std::map<const void*, std::string>& kernel_names() {
  static std::map<const void*, std::string> m;  // filled before main
  return m;
}

extern "C" {
void** __hipRegisterFatBinary(const void*) {
  static void* handle[1];
  return handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
  kernel_names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}

static thread_local struct {
  Dim3 grid, block;
  size_t lds;
  void* stream;
} t_config;
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void* stream) {
  t_config = {grid, block, lds, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** stream) {
  *grid = t_config.grid;
  *block = t_config.block;
  *lds = t_config.lds;
  *stream = t_config.stream;
  return 0;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void**, size_t lds, void* stream) {
  g_launches.push_back({kernel_names()[f], g_device, grid, block, lds, stream});
  return 0;
}

int hipGetDeviceCount(int* n) {
  *n = 2;
  return 0;
}
int hipGetDevice(int* d) {
  *d = g_device;
  return 0;
}
int hipSetDevice(int d) {
  g_device = d;
  return 0;
}
int hipFuncSetAttribute(const void* f, int, int value) {
  g_lds_limit[{g_device, kernel_names()[f]}] = value;
  return 0;
}
int hipMemcpyToSymbol(const void* symbol, const void*, size_t, size_t, int) {
  g_symbol_uploads[{g_device, symbol}]++;
  return 0;
}
int hipGetSymbolAddress(void** p, const void*) {
  static char area[1 << 16];
  *p = area;
  return 0;
}
int hipMalloc(void** p, size_t n) {
  *p = calloc(1, n);
  return *p ? 0 : 2;
}
int hipFree(void* p) {
  free(p);
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
  memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) {
  memcpy(d, s, n);
  return 0;
}
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "fake"; }
int hipDeviceSynchronize() { return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = malloc(1);
  return 0;
}
int hipStreamDestroy(void* s) {
  free(s);
  return 0;
}
int hipStreamSynchronize(void*) { return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipEventCreateWithFlags(void** e, unsigned) {
  *e = malloc(1);
  return 0;
}
int hipEventDestroy(void* e) {
  free(e);
  return 0;
}
int hipEventRecord(void*, void*) { return 0; }
}
