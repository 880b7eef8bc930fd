// prompt_q40.hip - the prompt GEMM's Q4_0 kernels (prompt_gemm.hpp).
#include "prompt_gemm.hpp"

namespace aljabr {

template <> void prompt_pack<kPgQ40>(const PgArgs &a, hipStream_t s) { pg::pack_weights<kPgQ40>(a, s); }

template <> void prompt_multiply<kPgQ40>(const PgArgs &a, int , int mt, hipStream_t s) {
    mt == 4 ? pg::launch<kPgQ40, 2, 4, 2, 2>(a, s) : pg::launch<kPgQ40, 2, 2, 2, 2>(a, s);
}

}  // namespace aljabr
