#include "fa_tile.h"
fa_status fa_tile::launch_f16(fa_ctx *ctx, FaLaunchScope &scope, TileShape shape, GemmDev &a, bool canonical) {
    return canonical ? launch_tile<16, true>(ctx, scope, shape, a) : launch_tile<16, false>(ctx, scope, shape, a);
}
