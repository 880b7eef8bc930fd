// prompt_q6k.hip - the prompt GEMM's Q6_K kernels (prompt_gemm.hpp).
#include "prompt_gemm.hpp"

namespace aljabr {

template <> void prompt_pack<kPgQ6K>(const PgArgs &a, hipStream_t s) { pg::pack_weights<kPgQ6K>(a, s); }

template <> void prompt_multiply<kPgQ6K>(const PgArgs &a, int , int mt, hipStream_t s) {
    mt == 4 ? pg::launch<kPgQ6K, 2, 4, 2, 2>(a, s) : pg::launch<kPgQ6K, 2, 2, 2, 2>(a, s);
}

}  // namespace aljabr
