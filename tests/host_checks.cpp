// Host-side rules of the library behind C names, for tests/test_host_rules.py: they decide which kernel a call runs, and
// none of them touches a GPU.  Compiled for the host and linked with the library's objects.
#include "../ffn_kernel_amd/csrc/launch.hpp"
#include "../ffn_kernel_amd/csrc/tile_table.hpp"

using namespace ffnk;

extern "C" {

int hc_direct_ok(int64_t K, int64_t gathered_rows, int64_t lda, int64_t ldb) { return direct_ok(K, gathered_rows, lda, ldb); }

}  // extern "C"
