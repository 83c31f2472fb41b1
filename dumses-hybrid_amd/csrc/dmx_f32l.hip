// float32-bulk engine of contexts with the learned limiter (slope_type 4): the
// float32 engine with the fields of both faces of a cell in the trace summary
// (DMX_BOTH_FACES, dmx_kernels.h), without the batch.
#define DMX_T float
#define DMX_NS f32l
#define DMX_BOTH_FACES 1
#include "dmx_step.inc"

namespace dmx {
Engine* make_engine_f32l(const dmx_params& p, int* rc)
{
    f32l::EngineT* e = new f32l::EngineT();
    *rc = e->init(p);
    if (*rc) {
        delete e;
        return nullptr;
    }
    return e;
}
} // namespace dmx
