// launch_check.cpp -- the launch shapes that the host plan code
// (splinegrids.jl_amd/csrc/sg_plan_host.hip) chooses, on the CPU under the
// address and undefined-behaviour sanitizers: what a launch may ask of the
// runtime, at sizes no test allocates.  The argument names the check; prints
// "launch_check ok <name>" and exits 0, or names the first failure.
#include <cstdio>
#include <cstdlib>
#include <string>

#include "sg_plan_host.hpp"

using namespace sg;

namespace {

void require(bool ok, const std::string& what) {
  if (!ok) {
    std::fprintf(stderr, "launch_check FAILED: %s\n", what.c_str());
    std::exit(1);
  }
}

// The general adjoint: blocks of max(G, 256) threads over outputs * G threads
// stay below 2^32 for every number of outputs that one thread each can take.
void check_csr_limit() {
  const double entries[] = {1, 48, 49, 100, 300, 1000, 1025, 4096, 4097, 6000, 1e5, 1e7};
  for (long long outputs = 1; outputs < (1LL << 32) - 512; outputs = outputs * 9 / 8 + 1)
    for (double e : entries) {
      const int g = csr_threads(outputs, e);
      require(g == 1 || g == kLanes || g == kCsrBlock, "threads per control point");
      const long long block = g > 256 ? g : 256;
      const long long threads = (outputs * g + block - 1) / block * block;
      require(threads < (1LL << 32), std::to_string(outputs) + " outputs of " + std::to_string(e) +
                                         " entries: " + std::to_string(threads) + " threads");
    }
  // cubic volumes of 120^3 control points x 3 with 4.5 samples per control
  // point and dimension, unsorted; quadratic 4-D grids of 64^4 points x 4
  require(csr_threads(3LL * 120 * 120 * 120, 18.0 * 18 * 18) == kLanes, "5 million outputs");
  require(csr_threads(4LL << 24, 81.0) == 1, "67 million outputs");
}

}  // namespace

int main(int argc, char** argv) {
  const std::string name = argc > 1 ? argv[1] : "";
  if (name == "csr_limit")
    check_csr_limit();
  else
    require(false, "no check named '" + name + "'");
  std::printf("launch_check ok %s\n", name.c_str());
  return 0;
}
