// K ping-pong GEMM (128 x 128 and 256 x 128 tiles) for bf16 (kernel template: mfma_kpp.hpp).
#include "mfma_kpp.hpp"

namespace mb {
namespace m16 {
hipError_t launch_bf16_kpp(bool ktail, int bm, bool a_kc, bool b_kc, const GemmArgs &g, dim3 grid, hipStream_t st) {
    return launch_kpp<bf16_t>(ktail, bm, a_kc, b_kc, g, grid, st);
}
}  // namespace m16
}  // namespace mb
