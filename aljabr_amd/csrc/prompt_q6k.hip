// prompt_q6k.hip - the prompt GEMM's Q6_K kernels (prompt_gemm.hpp).
#include "prompt_gemm.hpp"

namespace aljabr {

int prompt_launch_q6k(const PgArgs &a, int mt, hipStream_t s) {
    return mt == 4 ? pg::launch<kPgQ6K, 2, 4, 2, 2>(a, s) : pg::launch<kPgQ6K, 2, 2, 2, 2>(a, s);
}

}  // namespace aljabr
