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
    for (int k = 0; k < 12 * 4; ++k) {
      const double e = entries[k / 4];
      const int g = csr_threads(outputs, e, 1 + k % 4);
      require(g == 1 || g == kLanes || g == kCsrBlock, "threads per control point");
      const long long block = g > 256 ? g : 256;
      const long long threads = (outputs * g + block - 1) / block * block;
      require(threads < (1LL << 32), std::to_string(outputs) + " outputs of " + std::to_string(e) +
                                         " entries: " + std::to_string(threads) + " threads");
    }
  // cubic volumes of 120^3 control points x 3 with 4.5 samples per control
  // point and dimension, unsorted; quadratic 4-D grids of 64^4 points x 4
  require(csr_threads(3LL * 120 * 120 * 120, 18.0 * 18 * 18, 3) == kLanes, "5 million outputs");
  require(csr_threads(4LL << 24, 81.0, 4) == 1, "67 million outputs");
}

// Where many outputs fill the chip a thread walks each list: shapes on which a
// wave each took two to three times as long.
void check_csr_many() {
  require(csr_threads(995328, 52.8, 4) == 1, "24^4 x 3 linear control points");
  require(csr_threads(270000, 66.7, 2) == 1, "300^2 x 3 control points of degree 6");
  require(csr_threads(128000, 50.0, 3) == 1, "64 000 x 2 control points of degree 6");
  // and the waves and workgroups that pay
  require(csr_threads(600000, 52.0, 1) == kLanes, "a curve of 200 000 x 3 control points");
  require(csr_threads(131072, 410.0, 3) == kLanes, "131 072 outputs of 410 entries");
  require(csr_threads(11858, 6000.0, 2) == kLanes, "11 858 outputs of 6 000 entries");
  require(csr_threads(1458, 6000.0, 2) == kCsrBlock, "1 458 outputs of 6 000 entries");
  require(csr_threads(20, 8000.0, 1) == kCsrBlock, "20 outputs of 8 000 entries");
}

// A launch of launch_groups(t) parts of t threads is below 2^32, and one more
// part would not be.
void check_groups() {
  for (long long t = 64; t < (1LL << 32); t = t * 3 / 2 + 64) {
    const long long n = launch_groups(t);
    require(n >= 1 && n * t < (1LL << 32) && (n + 1) * t >= (1LL << 32),
            "parts of " + std::to_string(t) + " threads");
  }
}

}  // namespace

int main(int argc, char** argv) {
  const std::string name = argc > 1 ? argv[1] : "";
  if (name == "csr_limit")
    check_csr_limit();
  else if (name == "csr_many")
    check_csr_many();
  else if (name == "groups")
    check_groups();
  else
    require(false, "no check named '" + name + "'");
  std::printf("launch_check ok %s\n", name.c_str());
  return 0;
}
