// Which column kernel the library takes for 16-bit types at D = 128 and 256 (colw_serves, csrc/mlstm_kernels.h), compiled for the host only and run on the
// CPU: at sizes where one of the two was measured to be clearly the faster one (5 % or more), it is the one that is taken.
#include <cstdio>
#include "mlstm_kernels.h"

namespace mlstm {
bool g_force_generic = false;
int g_col_variant = 0;
}
using namespace mlstm;

struct Point { int dtype, D, precise, heads, S, colw; };
static const Point points[] = {
    {MLSTM_BF16, 256, 0, 768, 64, 1}, {MLSTM_BF16, 256, 0, 160, 200, 0}, {MLSTM_BF16, 256, 0, 103, 320, 0}, {MLSTM_BF16, 256, 0, 64, 512, 1}, {MLSTM_BF16, 256, 0, 96, 512, 0},
    {MLSTM_BF16, 256, 0, 58, 640, 0}, {MLSTM_BF16, 256, 0, 32, 1000, 1}, {MLSTM_BF16, 256, 0, 36, 1000, 1}, {MLSTM_BF16, 256, 0, 44, 1000, 0}, {MLSTM_BF16, 256, 0, 48, 1000, 0},
    {MLSTM_BF16, 256, 0, 33, 1100, 0}, {MLSTM_BF16, 256, 0, 40, 1025, 0}, {MLSTM_BF16, 256, 0, 25, 1536, 0}, {MLSTM_BF16, 256, 0, 12, 4096, 1}, {MLSTM_F16, 256, 0, 153, 320, 1},
    {MLSTM_F16, 256, 0, 41, 1100, 1}, {MLSTM_F16, 256, 0, 12, 4096, 1}, {MLSTM_BF16, 256, 1, 36, 1000, 1}, {MLSTM_BF16, 256, 1, 48, 1000, 0}, {MLSTM_BF16, 256, 1, 33, 1100, 0},
    {MLSTM_BF16, 256, 1, 12, 4096, 1}, {MLSTM_F16, 256, 1, 64, 640, 1}, {MLSTM_BF16, 128, 0, 192, 200, 0}, {MLSTM_F16, 128, 0, 128, 300, 0}, {MLSTM_BF16, 128, 0, 96, 384, 1},
    {MLSTM_BF16, 128, 0, 107, 384, 0}, {MLSTM_BF16, 128, 0, 110, 448, 0}, {MLSTM_BF16, 128, 0, 96, 512, 1}, {MLSTM_BF16, 128, 0, 48, 1000, 1}, {MLSTM_BF16, 128, 0, 29, 1100, 1},
    {MLSTM_BF16, 128, 0, 42, 1100, 0}, {MLSTM_BF16, 128, 0, 32, 1536, 1}, {MLSTM_BF16, 128, 0, 24, 2048, 1}, {MLSTM_BF16, 128, 1, 768, 64, 1}, {MLSTM_BF16, 128, 1, 103, 320, 0},
    {MLSTM_BF16, 128, 1, 32, 1000, 1}, {MLSTM_BF16, 128, 1, 48, 1000, 0}, {MLSTM_F16, 128, 1, 48, 1000, 0}, {MLSTM_BF16, 128, 1, 33, 1100, 0}, {MLSTM_BF16, 128, 1, 12, 4096, 1},
};

int main() {
    int failures = 0;
    for (const Point& p : points) {
        ColArgs a{};
        a.BH = p.heads; a.S = p.S; a.NG = (p.S + 63) / 64; a.precise = p.precise;
        a.chunk_len = p.S >= 1024 ? 512 : 0;
        if (colw_serves(p.dtype, p.D, a) == (p.colw != 0)) continue;
        failures++;
        std::printf("type %d, D = %d, split mode %d, %d heads x %d: %s taken\n", p.dtype, p.D, p.precise, p.heads, p.S, p.colw ? "cold_kernel" : "colw_kernel");
    }
    std::printf(failures ? "col_dispatch: %d failures\n" : "col_dispatch: ok\n", failures);
    return failures != 0;
}
