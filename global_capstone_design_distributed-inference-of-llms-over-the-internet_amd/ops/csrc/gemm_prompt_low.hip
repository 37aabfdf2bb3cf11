// Prompt products whose tiles are 128, 160, 192 or 224 rows high and 256 weight rows wide: what gemm_prompt.hip asks for where they
// fill rounds of 256 CUs, or the last tile's rows, better than tiles of 256 rows.  A wave has 4 to 7 fragments of rows to the eight of
// weights, loads as many pieces of rows, and needs no half tile.  Bound as those are, by MFMA issue and power; with 4 fragments by LDS,
// whose reads and loads into it take 1280 of a stage's cycles to 1024 of MFMAs.  A stage's time, 256 tiles of K 8192 (128 stages
// and their ends): 1.36 us of 256 rows, 1.21 of 224, 1.06 of 192, 0.92 of 160, 0.77 of 128.
#include "gemm_prompt.h"

namespace mp {

template <int EPI>
static void launch_low(const GemmPrompt& a, hipStream_t stream) {
  if (a.frags == 4) launch_prompt<EPI, 4>(a, stream);
  else if (a.frags == 5) launch_prompt<EPI, 5>(a, stream);
  else if (a.frags == 6) launch_prompt<EPI, 6>(a, stream);
  else launch_prompt<EPI, 7>(a, stream);
}

}  // namespace mp

extern "C" void mp_gemm_prompt_low(const mp::GemmPrompt* a, int epi, hipStream_t stream) {
  using namespace mp;
  if (epi == 0) launch_low<0>(*a, stream);
  else if (epi == 1) launch_low<1>(*a, stream);
  else if (epi == 4) launch_low<4>(*a, stream);
  else launch_low<GW_COLUMNS>(*a, stream);
}
