// prints the FP32 coefficients of the complex-symmetric polynomial (tests/test_symcoef.py)
#include <cstdio>
#include "../../ctemsoft_amd/csrc/ctem_symcoef.h"

int main() {
  const ctem::SymPoly k = ctem::sym_poly();
  for (const float* v : {k.c, k.d1, k.d2, k.r, k.e1, k.g}) printf("%a %a\n", v[0], v[1]);
}
