// Controls of the stand-in HIP runtime (hip_stub.cpp).
#pragma once
#include <cstddef>

int stub_faults();                       // objections so far
void stub_set_memory(std::size_t bytes);  // device memory from now on
std::size_t stub_memory_held();
std::size_t stub_memory_peak();          // since stub_reset_peak
void stub_reset_peak();
long stub_launches();                     // kernel launches so far
long stub_graphs();                       // graphs that exist
// The n-th kernel launch from now on fails (0: none); an executable's
// instantiation counts as one.
void stub_fail_launch(long n);
