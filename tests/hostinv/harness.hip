// Host build of the divsteps inversion, for tests/test_inverse.py.
#include "../../era-bellman-cuda_amd/csrc/inverse.cuh"

extern "C" void hostinv(int base_field, const uint32_t *a, uint32_t *out) {
  bc::fe x;
  for (int i = 0; i < 8; i++)
    x.v[i] = a[i];
  const bc::fe r = base_field ? bc::inverse<bc::FqParams>(x) : bc::inverse<bc::FrParams>(x);
  for (int i = 0; i < 8; i++)
    out[i] = r.v[i];
}
