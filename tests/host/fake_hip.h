// Interface of fake_hip.cpp.
#pragma once
#include <hip/hip_runtime_api.h>

struct FakeLaunch {
    const char* name;    // mangled kernel name
    dim3 grid, block;
    size_t lds;
    void** args;
};

extern long long fake_free_bytes;   // device memory there is
extern long long fake_used_bytes;   // of which allocated
extern void (*fake_on_launch)(const FakeLaunch&);
