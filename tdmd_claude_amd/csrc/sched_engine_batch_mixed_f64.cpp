#include "sched_engine.hpp"

namespace tdmd_hip {

EngineBase* make_engine_batch_mixed_f64(tdmd_sched* s) { return new Engine<float, sched::ManyBoxes<sched::MirrorF64>>(s); }

}  // namespace tdmd_hip
