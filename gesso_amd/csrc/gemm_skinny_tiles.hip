// The weight-streaming products reading the tile-major copy of the weight.
#include "gemm_skinny_impl.h"

// The same for weights loaded non-temporally (gemm_skinny_once.hip).
void gs_skinny_plain_tiles_once(const SkinnyCall& c);
void gs_skinny_gated_tiles_once(const SkinnyCall& c);
void gs_skinny_plain_half_tiles_once(const SkinnyCall& c);
void gs_skinny_residual_tiles_once(const SkinnyCall& c);
void gs_skinny_residual_half_tiles_once(const SkinnyCall& c);
void gs_skinny_conv_tiles_once(const SkinnyCall& c);
void gs_skinny_conv_half_tiles_once(const SkinnyCall& c);
void gs_skinny_parts_tiles_once(const SkinnyCall& c, int parts);

void gs_skinny_plain_tiles(const SkinnyCall& c) { skinny_once(c.N, c.K) ? gs_skinny_plain_tiles_once(c) : skinny_plain<1>(c); }
void gs_skinny_gated_tiles(const SkinnyCall& c) { skinny_once(c.N, c.K) ? gs_skinny_gated_tiles_once(c) : skinny_gated<1>(c); }
void gs_skinny_plain_half_tiles(const SkinnyCall& c) { skinny_once(c.N, c.K) ? gs_skinny_plain_half_tiles_once(c) : skinny_plain_halves<2>(c); }
void gs_skinny_residual_tiles(const SkinnyCall& c) { skinny_once(c.N, c.K) ? gs_skinny_residual_tiles_once(c) : skinny_residual<1>(c); }
void gs_skinny_residual_half_tiles(const SkinnyCall& c) { skinny_once(c.N, c.K) ? gs_skinny_residual_half_tiles_once(c) : skinny_residual<2>(c); }
void gs_skinny_conv_tiles(const SkinnyCall& c) { skinny_once(c.N, c.K) ? gs_skinny_conv_tiles_once(c) : skinny_conv<1>(c); }
void gs_skinny_conv_half_tiles(const SkinnyCall& c) { skinny_once(c.N, c.K) ? gs_skinny_conv_half_tiles_once(c) : skinny_conv<2>(c); }
void gs_skinny_parts_tiles(const SkinnyCall& c, int parts) { skinny_once(c.N, c.K) ? gs_skinny_parts_tiles_once(c, parts) : skinny_parts<1>(c, parts); }
