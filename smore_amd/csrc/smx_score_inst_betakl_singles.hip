// BetaE rows a float per lane and step, see beta_singles.
#include "smx_score_impl.h"

namespace smx {

int beta_singles_dispatch(hipStream_t st, const ScoreArgs& A, int nit, bool forward) {
  switch (nit) {
    case 1: return launch_beta_singles<1>(st, A, forward);
    case 2: return launch_beta_singles<2>(st, A, forward);
    case 3: return launch_beta_singles<3>(st, A, forward);
    case 5: return launch_beta_singles<5>(st, A, forward);
    case 6: return launch_beta_singles<6>(st, A, forward);
    default: return launch_beta_singles<7>(st, A, forward);
  }
}

}  // namespace smx
