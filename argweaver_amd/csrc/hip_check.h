// hip_check.h -- errors of HIP calls.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdio>

// reports an error and returns 1 from the caller
#define HIP_OK(x)                                                                       \
    do {                                                                                \
        hipError_t e_ = (x);                                                            \
        if (e_ != hipSuccess) {                                                         \
            fprintf(stderr, "argweaver_amd: HIP error %s at %s:%d\n", hipGetErrorString(e_), \
                    __FILE__, __LINE__);                                                \
            return 1;                                                                   \
        }                                                                               \
    } while (0)
