"""Small uploads through a context's pinned ring (csrc/gpi_util.hip: copy_h2d), in the CPU build with
the allocation of pinned memory counted or refused: a shot runs without pinned memory, and the entry
point that allocates nothing does not allocate the ring either."""
import os
import subprocess

from test_kept_buffers import EMU, run

SHIM = r"""
#include <dlfcn.h>
#include <cstddef>
#include <cstdlib>
extern "C" { int pinned_calls = 0; int pinned_refuse = 0; }
int host_malloc(void** p, size_t bytes, unsigned flags) __asm__("_Z13hipHostMallocPPvmj");
int host_malloc(void** p, size_t bytes, unsigned flags)
{
    ++pinned_calls;
    if (pinned_refuse) return 2;   // hipErrorOutOfMemory
    void* lib = dlopen(getenv("PINNED_NEXT"), RTLD_LAZY | RTLD_NOLOAD);   // the CPU build's own
    return ((int (*)(void**, size_t, unsigned))dlsym(lib, "_Z13hipHostMallocPPvmj"))(p, bytes, flags);
}
"""

SCRIPT = r"""
import os
shim = C.CDLL(os.environ["LD_PRELOAD"])
calls, refuse = (C.c_int.in_dll(shim, k) for k in ("pinned_calls", "pinned_refuse"))
# no strips and arrays above the ring's size limit: the model's creation uploads nothing small
def big(ctx):
    return experiment(layered_acoustic(nz=300, nx=290), nt=5, npml=0, pml_faces=[], nr=9, rfields=("p",), ctx=ctx)

refuse.value = 1
a = _lib.Context(0)
want = [shot(a, 40).run_shot(0)[0]["p"].copy(), big(a).run_shot(0)[0]["p"].copy()]
refuse.value = 0
b = _lib.Context(0)
p = big(b)
p._ensure_model()
n = calls.value
got = p.run_shot(0, static=True)[0]["p"].copy()
assert calls.value == n, "pinned memory allocated in a call that allocates nothing"
assert np.array_equal(got, want[1])
assert np.array_equal(shot(b, 40).run_shot(0)[0]["p"], want[0])
assert calls.value == n + 1, (calls.value, n)   # the ring, once, in the first call that may
print("uploads agree")
"""


def test_uploads_without_pinned_memory(tmp_path):
    src, lib = tmp_path / "shim.cpp", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-shared", "-fPIC", "-o", str(lib), str(src), "-ldl"], check=True)
    run(SCRIPT, "uploads agree", env=dict(LD_PRELOAD=str(lib), EMU_THREADS="2",
                                           PINNED_NEXT=os.path.join(EMU, "_build", "libgpi_emu.so")))
