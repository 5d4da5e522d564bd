// pf_sweep_list.hip — listed-cell instances of the phase-field sweep (both forms) and the copy-cell
// classification that builds their list.  Kernel definitions: pf_sweep_impl.h.
#include "pf_sweep_impl.h"

namespace pfamd {
PF_INST_SWEEP_LIST(FormF64, 4, 2, false)
PF_INST_SWEEP_LIST(FormF64, 4, 3, false)
PF_INST_SWEEP_LIST(FormF64, 6, 2, false)
PF_INST_SWEEP_LIST(FormF64, 6, 3, false)
PF_INST_SWEEP_LIST(FormMixed, 4, 2, false)
PF_INST_SWEEP_LIST(FormMixed, 4, 3, false)
PF_INST_SWEEP_LIST(FormMixed, 6, 2, false)
PF_INST_SWEEP_LIST(FormMixed, 6, 3, false)
PF_INST_SWEEP_LIST(FormF64, 6, 2, true)
PF_INST_SWEEP_LIST(FormF64, 6, 3, true)
// FP64, K = 4 lists: the register path with its overflow list, then the general path over it
#define PF_INST_SWEEP_SPLIT(F, P, ISO)                     \
  PF_INST_SWEEP_M(F, 4, P, 4, false, ISO, true, 1)         \
  PF_INST_SWEEP_M(F, 4, P, 6, false, ISO, true, 1)         \
  PF_INST_SWEEP_M(F, 4, P, 6, true, ISO, true, 1)          \
  PF_INST_SWEEP_M(F, 4, P, 4, false, ISO, true, 2)         \
  PF_INST_SWEEP_M(F, 4, P, 6, false, ISO, true, 2)         \
  PF_INST_SWEEP_M(F, 4, P, 6, true, ISO, true, 2)
PF_INST_SWEEP_SPLIT(FormF64, 2, false)
PF_INST_SWEEP_SPLIT(FormF64, 3, false)
PF_INST_SWEEP_SPLIT(FormF64, 2, true)
PF_INST_SWEEP_SPLIT(FormF64, 3, true)
PF_INST_SWEEP_CLASSIFY(FormF64, 4, false)
PF_INST_SWEEP_CLASSIFY(FormF64, 6, false)
PF_INST_SWEEP_CLASSIFY(FormMixed, 4, false)
PF_INST_SWEEP_CLASSIFY(FormMixed, 6, false)
PF_INST_SWEEP_CLASSIFY(FormF64, 4, true)
PF_INST_SWEEP_CLASSIFY(FormF64, 6, true)
}  // namespace pfamd
