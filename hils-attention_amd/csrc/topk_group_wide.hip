// The one-pass selection kernel for queries that see 513 to 1024 chunks: 64 logits per lane and head row, one
// wavefront per SIMD (512 registers).  A file of its own: these instantiations take longer to compile than
// all the others together.
#include "topk_group_kernel.h"

void tg_launch_wide(int GM, int D, bool perq, bool half, bool exp, dim3 grid, hipStream_t st, const TgArgs& a) {
  tg_dispatch(GM, D, a.bias != nullptr, perq, half, [&](auto gm, auto ks, auto bi, auto pq, auto hf) {
    if (exp) tg_call<gm.value, ks.value, 64, true, bi.value, pq.value, hf.value>(grid, st, a);
    else tg_call<gm.value, ks.value, 64, false, bi.value, pq.value, hf.value>(grid, st, a);
  });
}
