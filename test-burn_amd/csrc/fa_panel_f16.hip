// Panel kernels for 16-bit weights.
#include "fa_panel_impl.h"

template fa_status fa_panel::launch<16>(FaLaunchScope &, bool, bool, const Plan &, const PanelDev &);
