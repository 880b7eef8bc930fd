// prompt_nf4.hip - the prompt GEMM's NF4 kernels (prompt_gemm.hpp).
#include "prompt_gemm.hpp"

namespace aljabr {

template <> void prompt_pack<kPgNF4>(const PgArgs &a, hipStream_t s) { pg::pack_weights<kPgNF4>(a, s); }

template <> void prompt_multiply<kPgNF4>(const PgArgs &a, int xp, int mt, hipStream_t s) {
    if (xp == 1) return mt == 4 ? pg::launch<kPgNF4, 1, 4, 2, 2>(a, s) : pg::launch<kPgNF4, 1, 2, 2, 2>(a, s);
    mt == 4 ? pg::launch<kPgNF4, 2, 4, 2, 2>(a, s) : pg::launch<kPgNF4, 2, 2, 2, 2>(a, s);
}

}  // namespace aljabr
