// Dense products in bands of 128, 160, 192 or 224 rows (pipeline G).
#include "ix_gemm_dense.h"

template <int MI>
struct IxBand {
  template <bool ONCE>
  using Cfg = IxBandCfg<MI, ONCE>;
};

int ix_gemm_bf16_bands_launch(int mi, const bf16_t* A, long lda, const bf16_t* W, long ldw, bf16_t* C, long ldc, long M, long N,
                              long K, float* parts, long parts_ld, hipStream_t st) {
  switch (mi) {
    case 4: return ix_gemm_bf16_stream_launch<IxBand<4>::Cfg>(A, lda, W, ldw, C, ldc, M, N, K, parts, parts_ld, st);
    case 5: return ix_gemm_bf16_stream_launch<IxBand<5>::Cfg>(A, lda, W, ldw, C, ldc, M, N, K, parts, parts_ld, st);
    case 6: return ix_gemm_bf16_stream_launch<IxBand<6>::Cfg>(A, lda, W, ldw, C, ldc, M, N, K, parts, parts_ld, st);
    case 7: return ix_gemm_bf16_stream_launch<IxBand<7>::Cfg>(A, lda, W, ldw, C, ldc, M, N, K, parts, parts_ld, st);
    default: return IX_ERR_ARG;
  }
}
