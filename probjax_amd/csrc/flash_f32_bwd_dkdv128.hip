// float32 dK / dV at head dim 128: the instances of flash_f32_bwd.h and their choice.
#include "flash_f32_bwd.h"

namespace pjx {

int run_dkdv_f32_128(const FlashBwdArgs& a, hipStream_t s) {
  const FlashArgs& f = a.f;
  return with_ext(a, [&](auto ext) {
    constexpr int EX = decltype(ext)::value;
    const bool few = (f.Lk + 127L) / 128 * f.B * f.Hkv <= 256;  // 128-key blocks: at most one per CU
    auto go = [&](auto bias) {
      constexpr bool HB = decltype(bias)::value;
      if constexpr (EX == 0) {
        if (!few) return launch_dkdv_planes<128, 4, 1, 1, true, HB, EX>(a, s);
      }
      return launch_dkdv_planes<128, 2, 2, 1, true, HB, EX>(a, s);
    };
    return f.bias ? go(std::true_type{}) : go(std::false_type{});
  });
}

}  // namespace pjx
