#include "sched_engine.hpp"

namespace tdmd_hip {

EngineBase* make_engine_fixed(tdmd_sched* s) { return new Engine<float, sched::MirrorFixed>(s); }

}  // namespace tdmd_hip
