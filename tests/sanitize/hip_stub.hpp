// Controls of the stand-in HIP runtime (hip_stub.cpp).
#pragma once
#include <cstddef>
#include <string>
#include <vector>

int stub_faults();                       // objections so far
bool stub_inside();                       // a call of the stand-in is running
void stub_set_memory(std::size_t bytes);  // device memory from now on
std::size_t stub_memory_held();
std::size_t stub_memory_peak();          // since stub_reset_peak
void stub_reset_peak();
long stub_launches();                     // kernel launches so far
// The (mangled) names of the kernels launched since the last call, in order.
std::vector<std::string> stub_take_launches();
long stub_graphs();                       // graphs that exist
// The n-th kernel launch from now on fails (0: none); an executable's
// instantiation counts as one.
void stub_fail_launch(long n);
