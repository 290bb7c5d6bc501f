// Packed Hermitian stage kernels, FP32 bulk precision (stage 0 reads the
// FP64 state).
#include "heom_packed.h"

namespace phi {

hipError_t LaunchRk4PackedF32(const RhsArgs& a, int stage, const void* in, double* rho,
                              const void* kk, void* yout, double dt, hipStream_t s) {
  const double* x = (const double*)in;
  const float* v = (const float*)in;
  const float* k = (const float*)kk;
  float* y = (float*)yout;
  switch (stage) {
    case 0: return LaunchPacked<float>(a, x, dev::PkIncr<float, 0>{rho, k, y, dt}, s);
    case 1: return LaunchPacked<float>(a, v, dev::PkIncr<float, 1>{rho, k, y, dt}, s);
    case 2: return LaunchPacked<float>(a, v, dev::PkIncr<float, 2>{rho, k, y, dt}, s);
    default: return LaunchPacked<float>(a, v, dev::PkIncr<float, 3>{rho, k, y, dt}, s);
  }
}

hipError_t LaunchRkf45PackedF32(const RhsArgs& a, int stage, const void* in, const double* rho,
                                const Rkf45Bufs<float>& b, const Rkf45Coefs& c, hipStream_t s) {
  const double* x = (const double*)in;
  const float* v = (const float*)in;
  switch (stage) {
    case 0: return LaunchPacked<float>(a, x, dev::PkRkf45<float, 0>{b, rho, c}, s);
    case 1: return LaunchPacked<float>(a, v, dev::PkRkf45<float, 1>{b, rho, c}, s);
    case 2: return LaunchPacked<float>(a, v, dev::PkRkf45<float, 2>{b, rho, c}, s);
    case 3: return LaunchPacked<float>(a, v, dev::PkRkf45<float, 3>{b, rho, c}, s);
    case 4: return LaunchPacked<float>(a, v, dev::PkRkf45<float, 4>{b, rho, c}, s);
    default: return LaunchPacked<float>(a, v, dev::PkRkf45<float, 5>{b, rho, c}, s);
  }
}

}  // namespace phi
