// Instantiates the batch kernel for kModeInnerProductGrad.
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

const void* BatchKernelInnerProductGrad(int mode, int variant) {
  switch (mode) {
    default: return KernelPtr<kModeInnerProductGrad>(variant);
  }
}

}  // namespace tfqx
