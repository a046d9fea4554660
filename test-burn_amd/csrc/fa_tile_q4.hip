#include "fa_tile.h"
fa_status fa_tile::launch_q4(fa_ctx *ctx, FaLaunchScope &scope, TileShape shape, GemmDev &a, bool canonical) {
    return canonical ? launch_tile<4, true>(ctx, scope, shape, a) : launch_tile<4, false>(ctx, scope, shape, a);
}
