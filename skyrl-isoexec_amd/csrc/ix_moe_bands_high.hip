// The expert GEMMs in bands of 192 rows (pipeline G).
#include "ix_moe_bands.h"

int ix_moe_experts_bands_high(IX_MOE_BANDS_ARGS) {
  if (BM == 192)
    return ix_moe_experts_bands<6, true>(x, ldx, T, rows, sorted_token, permuted_prob, W1, W2, meta, max_tiles, inter, out,
                                                Hd, F, st);
  return IX_ERR_ARG;
}
