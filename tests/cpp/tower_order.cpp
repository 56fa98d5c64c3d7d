// The tower order of autopas_amd/csrc/ljg_order.h for the host's tests.
#include "../../autopas_amd/csrc/ljg_order.h"

extern "C" {

// out[i * n + j] = 1 if particle i comes before particle j (slots are the indices).
void tower_before_matrix(int n, const double *z, const int64_t *id, unsigned char *out) {
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) out[i * n + j] = ljg::tower_before(z[i], id[i], i, z[j], id[j], j);
}

void tower_keys32(int n, const double *z, float *out) {
  for (int i = 0; i < n; ++i) out[i] = ljg::tower_key32(z[i]);
}

}  // extern "C"
