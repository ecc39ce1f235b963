// Many-step kernel instantiations: PrecF32.
#include "pml_fdm_deep.h"

namespace pml {
Deep fdm_deep_f32(int eq, int integ, int ndim) { return deep_table<PrecF32>(eq, integ, ndim); }
}  // namespace pml
