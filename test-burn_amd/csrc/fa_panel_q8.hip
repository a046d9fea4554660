// Panel kernels for 8-bit weights.
#include "fa_panel_impl.h"

template fa_status fa_panel::launch<8>(FaLaunchScope &, bool, bool, const Plan &, const PanelDev &);
