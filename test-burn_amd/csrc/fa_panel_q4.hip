// Panel kernels for 4-bit weights.
#include "fa_panel_impl.h"

template fa_status fa_panel::launch<4>(FaLaunchScope &, bool, bool, const Plan &, const PanelDev &);
