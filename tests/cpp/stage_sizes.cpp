// The staging sizes of autopas_amd/csrc/ljg_stage.h for the host's tests.
#include "../../autopas_amd/csrc/ljg_stage.h"

extern "C" {
size_t stage_capacity(size_t wanted, size_t had) { return ljg::stage_capacity(wanted, had); }
size_t download_chunk(size_t total) { return ljg::download_chunk(total); }
size_t ring_bytes() { return ljg::kRingBytes; }
}
