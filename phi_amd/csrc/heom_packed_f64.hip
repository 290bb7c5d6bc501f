// Packed Hermitian stage kernels, FP64 bulk precision.
#include "heom_packed.h"

namespace phi {

hipError_t LaunchRk4PackedF64(const RhsArgs& a, int stage, const void* in, double* rho,
                              const void* kk, void* yout, double dt, hipStream_t s) {
  const double* x = (const double*)in;
  const double* k = (const double*)kk;
  double* y = (double*)yout;
  switch (stage) {
    case 0: return LaunchPacked<double>(a, x, dev::PkIncr<double, 0>{rho, k, y, dt}, s);
    case 1: return LaunchPacked<double>(a, x, dev::PkIncr<double, 1>{rho, k, y, dt}, s);
    case 2: return LaunchPacked<double>(a, x, dev::PkIncr<double, 2>{rho, k, y, dt}, s);
    default: return LaunchPacked<double>(a, x, dev::PkIncr<double, 3>{rho, k, y, dt}, s);
  }
}

hipError_t LaunchRkf45PackedF64(const RhsArgs& a, int stage, const void* in, const double* rho,
                                const Rkf45Bufs<double>& b, const Rkf45Coefs& c, hipStream_t s) {
  const double* x = (const double*)in;
  switch (stage) {
    case 0: return LaunchPacked<double>(a, x, dev::PkRkf45<double, 0>{b, rho, c}, s);
    case 1: return LaunchPacked<double>(a, x, dev::PkRkf45<double, 1>{b, rho, c}, s);
    case 2: return LaunchPacked<double>(a, x, dev::PkRkf45<double, 2>{b, rho, c}, s);
    case 3: return LaunchPacked<double>(a, x, dev::PkRkf45<double, 3>{b, rho, c}, s);
    case 4: return LaunchPacked<double>(a, x, dev::PkRkf45<double, 4>{b, rho, c}, s);
    default: return LaunchPacked<double>(a, x, dev::PkRkf45<double, 5>{b, rho, c}, s);
  }
}

}  // namespace phi
