// rows_plan.h — which convolution layers the row kernel (denoise.hip) takes. Host code only.
#pragma once
#include <cstdint>

namespace gdn {

// The 16-channel output fragments a wave of the row kernel's instance makes for a layer from ca channels at half
// resolution and cb at full resolution to cout; 0: the layer takes k_conv. grad: the data gradient, whose input is the
// layer's output gradient.
inline int rows_frags(int ca, int cb, int cout, bool grad) {
  switch (ca * 1000 + cb) {
    case 16: return 2;
    case 32: return cout == 48 ? 3 : cout > 32 && cout % 80 == 0 ? 5 : 2;
    case 48: return cout == 48 ? 3 : 2;
    case 64: return 2;
    case 80: return cout == 32 && !grad ? 2 : 0;
    case 96: return 2;
    case 48032: return cout == 32 ? 2 : 0;
    case 64032: return 2;
    case 64048: return 3;
    case 96064: return 2;
    default: return 0;
  }
}

}  // namespace gdn
