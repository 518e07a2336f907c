// One (x form, sources) of the skinny GPTQ kernel (i4xs.hpp), a translation
// unit of its own so that they compile in parallel.
#include "i4xs.hpp"

namespace st {
namespace xs {
template int launch<X_F32, 1>(st_context *, const Args &, int, int, bool);
}  // namespace xs
}  // namespace st
