// Host object of the learned surrogate network (fp_surrogate): master weights and optimiser state
// on the device, the device training set and the training workspace; plus the packing of the
// inference kernel's LDS image.
#pragma once

#include <vector>

#include "host_util.hpp"
#include "surrogate.hpp"

struct fp_surrogate {
  fp_surrogate_config cfg{};
  hipStream_t stream = nullptr;
  fph::DBuf<float> p, g, m, v;  // f32 master weights, gradient, Adam moments (kParams each)
  fph::DBuf<__bf16> wb, wbt;    // bf16 copies read by the training kernels: natural, W2 and W3 transposed
  uint64_t adam_t = 0;
  // training set: features (bf16 [count][72]) and targets (f32 [count][3], output units)
  fph::DBuf<__bf16> X;
  fph::DBuf<float> T;
  uint64_t count = 0;
  // training workspace (see TrainBatch): the transposed operands, the weight gradients' slices, the
  // workgroups' losses, the losses of a train call; and a gradient call's own rows and outputs
  int pitch = 0;
  fph::DBuf<__bf16> tr, Xb;
  fph::DBuf<float> part, loss_part, lossv, loss, Xf, Tb, Y;

  ~fp_surrogate() {
    if (stream) (void)hipStreamSynchronize(stream);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace fph {

// The inference kernel's LDS image (kImgBytes) from the f32 parameter vector.
std::vector<uint8_t> pack_image(const std::vector<float>& params);

}  // namespace fph
