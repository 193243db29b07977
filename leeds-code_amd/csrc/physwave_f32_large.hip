// Instantiations of the wave form of the physical-space pass (physwave.h).
#include "physwave.h"

namespace lsd {

int physwave_f32_large(Ctx& c, PwArgs<float>& a, bool cfl) {
    switch (c.Ph) {
    PW_LARGE(float);
    default: return 1;
    }
}

}  // namespace lsd
