// prompt_q40.hip - the prompt GEMM's Q4_0 kernels (prompt_gemm.hpp).
#include "prompt_gemm.hpp"

namespace aljabr {

int prompt_launch_q40(const PgArgs &a, int mt, hipStream_t s) {
    return mt == 4 ? pg::launch<kPgQ40, 2, 4, 2, 2>(a, s) : pg::launch<kPgQ40, 2, 2, 2, 2>(a, s);
}

}  // namespace aljabr
