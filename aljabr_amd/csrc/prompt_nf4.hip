// prompt_nf4.hip - the prompt GEMM's NF4 kernels (prompt_gemm.hpp).
#include "prompt_gemm.hpp"

namespace aljabr {

int prompt_launch_nf4(const PgArgs &a, int xp, int mt, hipStream_t s) {
    if (xp == 1)
        return mt == 4 ? pg::launch<kPgNF4, 1, 4, 2, 2>(a, s) : pg::launch<kPgNF4, 1, 2, 2, 2>(a, s);
    return mt == 4 ? pg::launch<kPgNF4, 2, 4, 2, 2>(a, s) : pg::launch<kPgNF4, 2, 2, 2, 2>(a, s);
}

}  // namespace aljabr
