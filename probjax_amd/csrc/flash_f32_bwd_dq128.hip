// float32 dQ at head dim 128: the instances of flash_f32_bwd.h and their choice.
#include "flash_f32_bwd.h"

namespace pjx {

int run_dq_f32_128(const FlashBwdArgs& a, hipStream_t s) {
  const FlashArgs& f = a.f;
  return with_ext(a, [&](auto ext) {
    constexpr int EX = decltype(ext)::value;
    const bool few = (f.Lq + 127L) / 128 * f.B * f.Hq <= 256;  // 128-row tiles: at most one per CU
    auto go = [&](auto bias) {
      constexpr int BI = decltype(bias)::value;
      if constexpr (EX == 0) {
        if (!few) return launch_dq_planes<128, 4, 1, 1, 1, BI, EX>(a, s);
      }
      return launch_dq_planes<128, 2, 2, 1, 1, BI, EX>(a, s);
    };
    if (a.dbias) return go(std::integral_constant<int, 2>{});
    return f.bias ? go(std::integral_constant<int, 1>{}) : go(std::integral_constant<int, 0>{});
  });
}

}  // namespace pjx
