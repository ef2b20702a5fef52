#include "sched_engine.hpp"

namespace tdmd_hip {

EngineBase* make_engine_fp64(tdmd_sched* s) { return new Engine<double, sched::MirrorF64>(s); }

}  // namespace tdmd_hip
