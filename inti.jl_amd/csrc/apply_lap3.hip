// Direct-sum kernels instantiated for one (PDE, dimension): INTI_LAPLACE, 3D.
#include "apply_kernel.hpp"
#include "apply_sym.hpp"

namespace inti {
ApplyFn apply_pick_lap3(int kind, int mixed, int nr) { return apply_pick_pd<INTI_LAPLACE, 3>(kind, mixed, nr); }
RowFn row_pick_lap3(int kind, int mixed, int nr) { return row_pick_pd<INTI_LAPLACE, 3>(kind, mixed, nr); }
BatchFn batch_pick_lap3(int kind, int mixed, int nr) { return batch_pick_pd<INTI_LAPLACE, 3>(kind, mixed, nr); }
SymFn sym_pick_lap3(int kind, int mixed, int tile, int G) { return sym_pick_pd<INTI_LAPLACE, 3>(kind, mixed, tile, G); }
SymFn sym_trans_pick_lap3(int kind, int tile, int G) { return sym_trans_pick_pd<INTI_LAPLACE, 3>(kind, tile, G); }
ApplyFn apply_trans_pick_lap3(int kind) { return apply_trans_pick_pd<INTI_LAPLACE, 3>(kind); }
}  // namespace inti
