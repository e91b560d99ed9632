// shake256-128f / shake256-192f / shake256-256f mixed batches, their WOTS chains in one
// launch; FORS leaves per lane as in each set's own batches
#include "family_impl.hpp"

using F128 = spx::Params<spx::kShake, 16, 66, 22, 6, 33>;
using F192 = spx::Params<spx::kShake, 24, 66, 22, 8, 33>;
using F256 = spx::Params<spx::kShake, 32, 68, 17, 9, 35>;
SPX_REGISTER_FAMILY(cuspx_family_shake256_f, F128, 2, 7, F192, 2, 9, F256, 3, 11)
