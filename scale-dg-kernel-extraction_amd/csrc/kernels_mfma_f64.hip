// The FP64 form's instantiations (HIP, tile candidates) of the stage kernels of
// stage_aug.hpp.
#include "stage_aug.hpp"

namespace dgk {

int prepare_tile_f64(int Nq) {
#define DGK_CALL(N) prepare_nq_all<PrecF64, N>()
  DGK_NQ_SWITCH(Nq, DGK_CALL)
#undef DGK_CALL
}

int launch_tile_f64(int Nq, int cand, const StageArgs &a, hipStream_t s) {
  if (a.Ne < 1) return DGK_OK;
#define DGK_CALL(N) launch_nq_cand<PrecF64, N>(cand, a, s)
  DGK_NQ_SWITCH(Nq, DGK_CALL)
#undef DGK_CALL
}

int tile_f64_shapes(int Nq, int *epb, int n) {
  if (Nq < kMinNq || Nq > kMaxNq || !epb || n < kKinds) return 0;
#define DGK_CALL(N) shapes_of<PrecF64, N>(epb)
  DGK_NQ_SWITCH(Nq, DGK_CALL)
#undef DGK_CALL
}

}  // namespace dgk
