// Which row kernel launch_row_best (csrc/mlstm_kernels.h) takes, compiled for the host only and run on the CPU, with launches that note their kernel.
// A forward whose row kernel is to form the gates by itself (RowArgs::gate_F) reads arrays that nobody else writes: it goes to roww_kernel or nowhere,
// whatever the process-wide switches say by the time of the launch.
#include <cstdio>
#include <string>
#include "mlstm_kernels.h"

namespace mlstm {
bool g_force_generic = false;
int g_col_variant = 0;
static std::string launched;
static int roww_rc = 0;
static int note(const char* what, int rc = 0) { launched += what; return rc; }
int launch_row_kernel(int, int, int, const RowArgs&, hipStream_t) { return note("row "); }
int launch_row8_kernel(int, int, int, const RowArgs&, hipStream_t) { return note("row8 "); }
int launch_roww_kernel(int, int, int, const RowArgs&, hipStream_t) { return note("roww ", roww_rc); }
int launch_rowx_kernel(int, int, int, const RowArgs&, hipStream_t) { return note("rowx "); }
}  // namespace mlstm

using namespace mlstm;

int main() {
    int failures = 0;
    const int value = 0;
    for (int D : {128, 256})
        for (bool gates : {false, true})
            for (int turned : {0, 1, 2, 3}) {   // nothing; the generic kernels; a bound on the wait; a launch that fails
                RowArgs a{};
                a.BH = 2; a.S = 640; a.NG = 10;
                a.spin_limit = DEFAULT_SPIN_LIMIT;
                g_force_generic = false;
                if (!roww_serves(MLSTM_BF16, D, a)) { failures++; std::printf("roww_kernel does not serve D = %d\n", D); }
                if (gates) a.gate_F = a.gate_I = &value;
                g_force_generic = turned == 1;
                if (turned == 2) a.spin_limit = 1;
                roww_rc = turned == 3 ? MLSTM_ESHAPE : 0;
                launched.clear();
                const int rc = launch_row_best(0, MLSTM_BF16, D, a, nullptr);
                const char* const plain[] = {"roww ", "row ", "row8 ", "roww row8 "};
                const std::string want = gates ? "roww " : plain[turned];
                if (launched != want || rc != (gates ? roww_rc : 0)) {
                    failures++;
                    std::printf("D = %d, gates %d, switch %d: launched %s(rc %d), expected %s\n", D, gates, turned, launched.c_str(), rc, want.c_str());
                }
            }
    std::printf(failures ? "row_dispatch: %d failures\n" : "row_dispatch: ok\n", failures);
    return failures != 0;
}
