// k_fft_fixed.hip -- one direction and precision of the compiled-in transforms: the
// makefile compiles this file once for each, side by side.
#include "fft_fixed.hpp"

#include <utility>

#ifndef PLL_FFT_T
#define PLL_FFT_T double
#endif
#ifndef PLL_FFT_PASS
#define PLL_FFT_PASS FftPass::x_fwd
#endif

namespace pll {
namespace {

using Launch = int (*)(pll_context*, bool);

// The y length ny is even.
template <typename T, FftPass PASS, int L>
constexpr Launch entry() {
  constexpr bool kX = PASS == FftPass::x_fwd || PASS == FftPass::x_bwd;
  if constexpr (!fixed_length(L) || (!kX && L % 2))
    return nullptr;
  else if constexpr (PASS == FftPass::x_fwd)
    return launch_xf<T, L>;
  else if constexpr (PASS == FftPass::x_bwd)
    return launch_xb<T, L>;
  else
    return launch_y<T, L, PASS == FftPass::y_fwd>;
}

template <typename T, FftPass PASS, int... L>
Launch lookup(int n, std::integer_sequence<int, L...>) {
  static constexpr Launch table[] = {entry<T, PASS, L>()...};
  return table[n];
}

}  // namespace

template <typename T, FftPass PASS>
int fft_fixed(pll_context* c, int n, bool step) {
  const Launch f = n < 0 || n > kFixedMax
                       ? nullptr
                       : lookup<T, PASS>(n, std::make_integer_sequence<int, kFixedMax + 1>{});
  return f ? f(c, step) : fail(PLL_ERR_STATE, "no compiled-in transform of this length");
}
template int fft_fixed<PLL_FFT_T, PLL_FFT_PASS>(pll_context*, int, bool);

}  // namespace pll
