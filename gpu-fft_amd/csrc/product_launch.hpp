// Launches of the fused FP64 product kernels (product.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

namespace gfa {

// Entries of the merged root table: 2^n roots and, of split products, 4^SB
// residue powers.
constexpr size_t product_table_entries(int n, int SB)
{
    return ((size_t)1 << n) + (SB > 0 ? (size_t)1 << (2 * SB) : 0);
}

// Compute units of the current device.
inline int device_cus()
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 64)
        cus = 256;
    return cus;
}

// Workgroups of a persistent launch of which `resident` share a CU: what the
// CUs hold at once, if there is as much work.
inline int persistent_grid(long long items, int resident)
{
    return (int)std::min<long long>(items, (long long)device_cus() * resident);
}

int launch_product_table(void* w, int n, int SB, hipStream_t st, const char* who);
// Products of 2^n complex points in 2^SB sub-problems of 2^S: into out
// (SB = 0) or the sub-results in scratch.
int launch_product_f64(int n, int S, int SB, int batch, const void* w, const double* a, const double* b,
                       double* out, void* scratch, hipStream_t st, const char* who);
// The top SB inverse stages from scratch to out.
int launch_combine_f64(int n, int S, int SB, int batch, const void* w, const void* scratch, double* out,
                       hipStream_t st, const char* who);

}  // namespace gfa
