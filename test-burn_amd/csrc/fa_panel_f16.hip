// Panel kernels for 16-bit weights.
#include "fa_panel_impl.h"

template fa_status fa_panel::launch<16>(FaLaunchScope &, bool, bool, bool, uint32_t, uint32_t, uint32_t, dim3, const PanelDev &);
