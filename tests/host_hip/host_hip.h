// A HIP runtime for the library's host code on a machine without a GPU: device
// memory is host memory, kernels do nothing, and streams and events keep vector
// clocks, so that a test can ask what a stream's later work comes after.
// Allocations, launches and graph launches can be made to fail from the n-th on
// (once), from the host.
#pragma once
#include <cstddef>

namespace host_hip {
// the n-th call from now fails (0: the next one; -1: none)
void fail_malloc(long n);        // hipMalloc: out of memory
void fail_launch(long n);        // kernels, graphs
void fail_new(long n);           // operator new: std::bad_alloc
bool all_used();                 // every armed failure has happened
void clear_error();              // the last error is forgotten
size_t live();                   // device allocations not freed
// work launched on any stream that neither the host has waited for nor `stream`
// comes after
size_t outstanding(void *stream);
}  // namespace host_hip
