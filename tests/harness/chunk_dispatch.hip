// Which kernels launch_chunk_states (csrc/mlstm_chunk.hip) takes, compiled for the host only and run on the CPU: the runtime's entry points are stand-ins
// that note a launch and say of a kernel what the test wants said.  A one-pass kernel that a compiler gave scratch memory is not launched: where the library
// chose it, the two kernels of the same bits take its place; where the caller named it, the call is refused.
#include <map>
#include <set>
#include <string>
#include <cstdio>
#include "mlstm_chunk.hip"

namespace mlstm {
bool g_force_generic = false;
}
static std::set<std::string> launched;
static std::map<const void*, std::string> names;
static bool scratch_at_256 = false;

extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* module; return &module; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* stub, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { names[stub] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes* attr, const void* kernel) {
    *attr = {};
    attr->localSizeBytes = scratch_at_256 && names[kernel].find("Li256E") != std::string::npos ? 4 : 0;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* kernel, dim3, dim3, void**, size_t, hipStream_t) {
    for (const char* short_name : {"chunk_seq", "chunk_sum", "chunk_carry"})
        if (names[kernel].find(short_name) != std::string::npos) launched.insert(short_name);
    return hipSuccess;
}
}

using namespace mlstm;

int main(int argc, char**) {
    scratch_at_256 = argc > 1;   // (a kernel is asked about once per process)
    const std::set<std::string> one{"chunk_seq"}, two{"chunk_sum", "chunk_carry"};
    static char memory[64];
    int failures = 0, cases = 0;
    for (int dtype : {MLSTM_BF16, MLSTM_F16})
        for (int D : {128, 256})
            for (int precise : {0, 1})
                for (int states : {0, 1, 2, 3})   // key-major; value-major; both; value-major with the contraction
                    for (int form : {0, 1, 2})
                        for (int heads : {1, 64}) {   // (an eighth of a round of workgroups at the most, and whole rounds)
                            ChunkArgs a{};
                            a.BH = heads; a.S = 2048; a.NG = 32; a.L = 512; a.NCS = 3; a.precise = precise;
                            a.Cst = states == 0 || states == 2 ? memory : nullptr;
                            a.CstT = states != 0 ? memory : nullptr;
                            a.Cst_lo = precise ? a.Cst : nullptr;
                            a.CstT_lo = precise ? a.CstT : nullptr;
                            if (states == 3) { a.dot_part = reinterpret_cast<float*>(memory); a.dot_with = memory; a.dot_with_lo = precise ? memory : nullptr; }
                            launched.clear();
                            set_state_kernel(form);
                            const int rc = launch_chunk_states(dtype, D, a, nullptr);
                            const bool serves = (D == 256 || !precise) && (form == 2 || (form == 0 && heads == 64)), spilled = scratch_at_256 && D == 256;
                            const int want_rc = serves && spilled && form == 2 ? MLSTM_EBUILD : 0;
                            const auto want = want_rc ? std::set<std::string>{} : serves && !spilled ? one : two;
                            cases++;
                            if (rc == want_rc && launched == want) continue;
                            failures++;
                            std::printf("type %d, D = %d, split mode %d, states %d, form %d, %d heads: rc %d, expected %d; launched", dtype, D, precise, states, form, heads, rc, want_rc);
                            for (const auto& name : launched) std::printf(" %s", name.c_str());
                            std::printf("\n");
                        }
    std::printf(failures ? "chunk_dispatch: %d failures\n" : "chunk_dispatch: %d cases ok\n", failures ? failures : cases);
    return failures != 0;
}
