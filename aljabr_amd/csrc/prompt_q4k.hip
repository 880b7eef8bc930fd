// prompt_q4k.hip - the prompt GEMM's Q4_K kernels (prompt_gemm.hpp).
#include "prompt_gemm.hpp"

namespace aljabr {

template <> void prompt_pack<kPgQ4K>(const PgArgs &a, hipStream_t s) { pg::pack_weights<kPgQ4K>(a, s); }

template <> void prompt_multiply<kPgQ4K>(const PgArgs &a, int xp, int mt, hipStream_t s) {
    if (xp == 1) return mt == 4 ? pg::launch<kPgQ4K, 1, 4, 2, 4>(a, s) : pg::launch<kPgQ4K, 1, 2, 2, 4>(a, s);
    mt == 4 ? pg::launch<kPgQ4K, 2, 4, 2, 2>(a, s) : pg::launch<kPgQ4K, 2, 2, 2, 2>(a, s);
}

}  // namespace aljabr
