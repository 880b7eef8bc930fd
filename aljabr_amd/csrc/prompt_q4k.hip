// prompt_q4k.hip - the prompt GEMM's Q4_K kernels (prompt_gemm.hpp).
#include "prompt_gemm.hpp"

namespace aljabr {

int prompt_launch_q4k(const PgArgs &a, int xp, int mt, hipStream_t s) {
    if (xp == 1)
        return mt == 4 ? pg::launch<kPgQ4K, 1, 4, 2, 4>(a, s) : pg::launch<kPgQ4K, 1, 2, 2, 4>(a, s);
    return mt == 4 ? pg::launch<kPgQ4K, 2, 4, 2, 2>(a, s) : pg::launch<kPgQ4K, 2, 2, 2, 2>(a, s);
}

}  // namespace aljabr
