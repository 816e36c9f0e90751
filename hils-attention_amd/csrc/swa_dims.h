// Shape of a sliding-window attention call, shared by the tile kernel (swa.hip) and the row kernel (swa_rows.hip).
#pragma once
#include "common.h"
#include "../../include/hils_amd.h"

struct SwaDims {
  int Lq, Lk, HQ, H, window, chunk, mask_lmk, expand, kv_start, chunk_pow2;
  float sm_scale;
  long k_batch, v_batch;  // elements from a sequence's keys / values to the next one's
};

// Is the row kernel the faster one for this shape?
bool hils_swa_rows_better(int B, int D, int Dv, const SwaDims& dm);
int hils_swa_fwd_rows(int B, hipStream_t st, const void* q, const void* k, const void* v, void* o, float* lse, int D,
                      int Dv, const SwaDims& dm);
