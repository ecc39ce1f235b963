// Many-step kernel instantiations: PrecF32C.
#include "pml_fdm_deep.h"

namespace pml {
Deep fdm_deep_f32c(int eq, int integ, int ndim) { return deep_table<PrecF32C>(eq, integ, ndim); }
}  // namespace pml
