#pragma once

namespace mi {

struct ConvGeom {
  int batch, in_h, in_w, in_c, out_h, out_w, out_c;
  int kernel_h, kernel_w, stride_h, stride_w, dilation_h, dilation_w, pad_u, pad_l;
};

}  // namespace mi
