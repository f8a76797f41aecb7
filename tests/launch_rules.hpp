// What the objects of test_launch_rules.py need to load without a device: a source of kernels compiled for the host alone refers to its device image and to the
// runtime's launch calls. Nothing is launched.
#pragma once
#include "../ferric_amd/csrc/common.hpp"

#include <stdarg.h>
#include <stdio.h>

extern "C" {
char __hip_fatbin[4096];
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, dim3*, dim3*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipErrorNoDevice; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipErrorNoDevice; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipErrorNoDevice; }
hipError_t hipGetLastError() { return hipErrorNoDevice; }
}
namespace fhip {
int device_cus() { return 256; }
int set_error(int code, const char*, ...) { return code; }
int check_hip(hipError_t e, const char*) { return e == hipSuccess ? FHIP_OK : FHIP_ERR_HIP; }
}  // namespace fhip
