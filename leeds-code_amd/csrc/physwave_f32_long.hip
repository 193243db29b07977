// Instantiations of the wave form of the physical-space pass (physwave.h).
// Points per lane grow to 18 here (one wave per SIMD).  FP64 would need more
// than the register file, so its lengths past 512 stay on the workgroup form.
#include "physwave.h"

namespace lsd {

int physwave_f32_long(Ctx& c, PwArgs<float>& a, bool cfl) {
    switch (c.Ph) {
    PW_CASE(float, 576, 16, 4, 9, 0);
    PW_CASE(float, 648, 18, 3, 12, 0);
    PW_CASE(float, 768, 16, 4, 12, 0);
    PW_CASE(float, 864, 18, 3, 16, 0);
    PW_CASE(float, 972, 18, 3, 18, 0);
    PW_CASE(float, 1024, 16, 4, 16, 0);
    default: return 1;
    }
}

}  // namespace lsd
