// Many-step kernel instantiations: PrecF64.
#include "pml_fdm_deep.h"

namespace pml {
Deep fdm_deep_f64(int eq, int integ, int ndim) { return deep_table<PrecF64>(eq, integ, ndim); }
}  // namespace pml
