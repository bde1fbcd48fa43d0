// The weight-streaming products reading the tile-major copy of a large weight, non-temporally.
#include "gemm_skinny_impl.h"

void gs_skinny_plain_tiles_once(const SkinnyCall& c) { skinny_plain<1 | SKINNY_ONCE>(c); }
void gs_skinny_gated_tiles_once(const SkinnyCall& c) { skinny_gated<1 | SKINNY_ONCE>(c); }
void gs_skinny_plain_half_tiles_once(const SkinnyCall& c) { skinny_plain_halves<2 | SKINNY_ONCE>(c); }
void gs_skinny_residual_tiles_once(const SkinnyCall& c) { skinny_residual<1 | SKINNY_ONCE>(c); }
void gs_skinny_residual_half_tiles_once(const SkinnyCall& c) { skinny_residual<2 | SKINNY_ONCE>(c); }
void gs_skinny_conv_tiles_once(const SkinnyCall& c) { skinny_conv<1 | SKINNY_ONCE>(c); }
void gs_skinny_conv_half_tiles_once(const SkinnyCall& c) { skinny_conv<2 | SKINNY_ONCE>(c); }
void gs_skinny_parts_tiles_once(const SkinnyCall& c, int parts) { skinny_parts<1 | SKINNY_ONCE>(c, parts); }
