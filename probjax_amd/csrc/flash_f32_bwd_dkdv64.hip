// float32 dK / dV at head dim 64: the instances of flash_f32_bwd.h and their choice.
#include "flash_f32_bwd.h"

namespace pjx {

int run_dkdv_f32_64(const FlashBwdArgs& a, hipStream_t s) {
  const FlashArgs& f = a.f;
  return with_ext(a, [&](auto ext) {
    constexpr int EX = decltype(ext)::value;
    const bool few = (f.Lk + 127L) / 128 * f.B * f.Hkv <= 256;  // 128-key blocks: at most one per CU
    auto go = [&](auto bias) {
      constexpr bool HB = decltype(bias)::value;
      if constexpr (!HB && EX == 0) {
        if ((f.Lk + 31L) / 32 * f.B * f.Hkv <= 256) return launch_dkdv_planes<64, 1, 4, 1, false, HB, EX>(a, s);
      }
      if constexpr (EX == 0) {
        if (!few) return launch_dkdv_planes<64, 4, 2, 2, false, HB, EX>(a, s);
      }
      return launch_dkdv_planes<64, 2, 4, 2, false, HB, EX>(a, s);
    };
    return f.bias ? go(std::true_type{}) : go(std::false_type{});
  });
}

}  // namespace pjx
