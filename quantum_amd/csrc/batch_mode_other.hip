// Instantiates the batch kernel for kModeState, kModeSamples, kModeSampledExpectation, kModeInnerProduct.
#include "batch_kernel_impl.h"

namespace tfqx {
namespace {

template <int MODE>
const void* KernelPtr(int variant) {
  switch (variant) {
    case kVariantWide: return reinterpret_cast<const void*>(&batch_kernel<MODE, kVariantWide>);
    case kVariantLds: return reinterpret_cast<const void*>(&batch_kernel<MODE, kVariantLds>);
    case kVariantEngine: return reinterpret_cast<const void*>(&batch_kernel<MODE, kVariantEngine>);
    default: return reinterpret_cast<const void*>(&batch_kernel<MODE, kVariantAny>);
  }
}

}  // namespace

const void* BatchKernelOther(int mode, int variant) {
  switch (mode) {
    case kModeState: return KernelPtr<kModeState>(variant);
    case kModeSamples: return KernelPtr<kModeSamples>(variant);
    case kModeSampledExpectation: return KernelPtr<kModeSampledExpectation>(variant);
    default: return KernelPtr<kModeInnerProduct>(variant);
  }
}

}  // namespace tfqx
