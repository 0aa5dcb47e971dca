"""Pinned memory that the host reads while a kernel writes it is asked for as coherent, and blocks of one kind are never handed out as another:
the pool's own source in a host program whose runtime is a stub (no GPU)."""
import os
import subprocess

MAIN = r"""
#include "pool.h"
#include <cstdio>
#include <cstdlib>
#include <map>
static std::map<void *, unsigned> flags; // of the blocks of pinned memory there are
extern "C" {
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return *p = malloc(n), hipSuccess; }
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { return *p = malloc(n), flags[*p] = f, hipSuccess; }
hipError_t hipHostFree(void *p) { return flags.erase(p), free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *p, unsigned) { return *d = p, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }
hipError_t hipStreamCreateWithFlags(hipStream_t *, unsigned) { return hipErrorUnknown; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
}
void evt_set_error(const char *, ...) {}
void models_trim() {}
int main() {
    for (int round = 0; round < 3; round++) { // the second round's blocks are the first's, kept
        void *c = coherent_take(5000), *p = pinned_take(5000), *d = dev_take(5000);
        if (flags.at(c) != (hipHostMallocPortable | hipHostMallocCoherent) || flags.at(p) != hipHostMallocPortable || flags.count(d)) return printf("round %d\n", round), 1;
        if (flags.size() != 2) return printf("round %d: %zu blocks\n", round, flags.size()), 2;
        pinned_give(p), coherent_give(c), dev_give(d);
        if (round == 1 && (evt_trim() != EVT_OK || flags.size())) return printf("%zu blocks after evt_trim\n", flags.size()), 3;
    }
    return 0;
}
"""


def test_coherent_blocks_stay_apart(evt, tmp_path):
    csrc = os.path.join(os.path.dirname(evt.__file__), "csrc")
    (tmp_path / "main.hip").write_text(MAIN)
    objs = []
    for src in (os.path.join(csrc, "pool.hip"), str(tmp_path / "main.hip")):
        objs.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.run(["hipcc", "--offload-host-only", "-O0", "-fPIC", "-std=c++17", "-I", csrc, "-c", src, "-o", objs[-1]], check=True)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-o", exe] + objs, check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
    with open(os.path.join(csrc, "api.hip")) as f:  # the slots that finished trees are written to are of that kind, taken and given back
        api = f.read()
    assert "coherent_take(2 * c->h_stage_bytes" in api and "coherent_give(c->h_stage_base)" in api
