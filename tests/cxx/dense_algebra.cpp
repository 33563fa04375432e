// The analysis' dense algebra for tests/test_dense_algebra.py: body 0 runs on
// any x86-64 processor, body 1 with AVX2 and FMA.
#include "../../adamantine_amd/csrc/adm_dense.hpp"

extern "C" {

int has_body(int body) { return body == 0 || adm::has_avx2() ? 1 : 0; }

int lu(int body, int m, double *A, int nrhs, double *B) {
  return (body ? adm::lu_avx2 : adm::lu_plain)(m, A, nrhs, B) ? 1 : 0;
}

void gram(int body, int m, int p, const double *X, int q, const double *Y,
          double *C) {
  (body ? adm::gram_avx2 : adm::gram_plain)(m, p, X, q, Y, C);
}

int is_diagonal(int m, const double *R) {
  return adm::is_diagonal(m, R) ? 1 : 0;
}

}
