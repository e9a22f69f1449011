// th_plain_f32.hip -- the plain steppers of th_plain.hpp in FP32.
#include <algorithm>
#include "th_plain.hpp"

namespace th {
template int plain_step<float>(th_plan*, int, int, cplx<float>* const*, double, double, double, const ForceBand*, const ForceBand*,
                            cplx<float>* const*);
}  // namespace th
