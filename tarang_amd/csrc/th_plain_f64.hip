// th_plain_f64.hip -- the plain steppers of th_plain.hpp in FP64.
#include <algorithm>
#include "th_plain.hpp"

namespace th {
template int plain_step<double>(th_plan*, int, int, cplx<double>* const*, double, double, double, const ForceBand*, const ForceBand*,
                            cplx<double>* const*);
}  // namespace th
