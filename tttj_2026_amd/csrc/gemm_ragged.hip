// MFMA GEMM launches for widths that are multiples of 8 but not of 64 (d_model 32, 96, 160, ...): the
// register-path tiles of gemm_tile.hpp and the narrow tiles of gemm_narrow.hpp in their RAG form.
#include "gemm_narrow.hpp"
#include "gemm_tile.hpp"

namespace tt {

template <int MODE>
static int run_ragged_mode(RaggedTile tile, const half* x, const half* w, int m, int n, int k,
                           const EpiArgs& ep, hipStream_t stream) {
  switch (tile) {
    case RaggedTile::k128x128: return run_tile<128, 128, MODE, 1, 4, true>(x, w, m, n, k, ep, stream);
    case RaggedTile::k64x64: return run_tile<64, 64, MODE, 1, 4, true>(x, w, m, n, k, ep, stream);
    case RaggedTile::kNarrowStaged: return launch_narrow_mode<MODE, true, true>(x, w, m, n, k, ep, stream);
    default: return launch_narrow_mode<MODE, true>(x, w, m, n, k, ep, stream);
  }
}

int run_ragged(RaggedTile tile, const half* x, const half* w, int m, int n, int k, const EpiArgs& ep,
               hipStream_t stream) {
  switch (ep.mode) {
    case TT_EPI_BIAS: return run_ragged_mode<TT_EPI_BIAS>(tile, x, w, m, n, k, ep, stream);
    case TT_EPI_BIAS_GELU: return run_ragged_mode<TT_EPI_BIAS_GELU>(tile, x, w, m, n, k, ep, stream);
    case TT_EPI_RESID_MASKED: return run_ragged_mode<TT_EPI_RESID_MASKED>(tile, x, w, m, n, k, ep, stream);
    case TT_EPI_MASKED_RESID: return run_ragged_mode<TT_EPI_MASKED_RESID>(tile, x, w, m, n, k, ep, stream);
    default: return run_ragged_mode<TT_EPI_QKV>(tile, x, w, m, n, k, ep, stream);
  }
}

}  // namespace tt
