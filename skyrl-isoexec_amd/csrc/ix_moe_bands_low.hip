// The expert GEMMs in bands of 96 and 160 rows (pipeline G).
#include "ix_moe_bands.h"

int ix_moe_experts_bands_low(IX_MOE_BANDS_ARGS) {
  if (BM == 96)
    return ix_moe_experts_bands<3, false>(x, ldx, T, rows, sorted_token, permuted_prob, W1, W2, meta, max_tiles, inter, out,
                                                Hd, F, st);
  if (BM == 160)
    return ix_moe_experts_bands<5, true>(x, ldx, T, rows, sorted_token, permuted_prob, W1, W2, meta, max_tiles, inter, out,
                                                Hd, F, st);
  return IX_ERR_ARG;
}
