"""The kernels that a piece of work launches, by name: run in a second process, in which the library's launches are noted on their way to the runtime."""
import os
import subprocess
import sys

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
#include <mutex>
#include <string>
struct dim { unsigned x, y, z; };
static std::mutex mu;
static std::string seen;
static void *next(const char *name) {
    void *runtime = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    return runtime ? dlsym(runtime, name) : nullptr;
}
extern "C" {
int hipLaunchKernel(const void *f, dim g, dim b, void **a, size_t l, void *s) {
    static const auto to = (int (*)(const void *, dim, dim, void **, size_t, void *))next("hipLaunchKernel");
    static const auto name = (const char *(*)(const void *, void *))next("hipKernelNameRefByPtr");
    {
        std::lock_guard<std::mutex> lk(mu);
        const char *n = name ? name(f, nullptr) : nullptr;
        seen += std::string(n ? n : "?") + "\n";
    }
    return to ? to(f, g, b, a, l, s) : 999;
}
const char *names(void) { /* since the last call */
    static std::string out;
    std::lock_guard<std::mutex> lk(mu);
    out.swap(seen);
    seen.clear();
    return out.c_str();
}
}
"""

HEAD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)        # before the library: its launches come here first
shim.names.restype = ctypes.c_char_p
sys.path.insert(0, sys.argv[2])


def launches(be, f, *a, **kw):
    '''The names of the kernels that f launches on `be`.'''
    be.sync()
    shim.names()
    f(*a, **kw)
    be.sync()
    return shim.names().decode().split()


"""


def run(tmp_path, program, timeout=100):
    """Runs `program` behind HEAD; it has to end with the line "done"."""
    here = os.path.dirname(os.path.abspath(__file__))
    (tmp_path / "shim.cpp").write_text(SHIM)
    (tmp_path / "program.py").write_text(HEAD + program)
    subprocess.check_call(["g++", "-shared", "-fPIC", "-o", str(tmp_path / "shim.so"), str(tmp_path / "shim.cpp"), "-ldl"])
    r = subprocess.run([sys.executable, str(tmp_path / "program.py"), str(tmp_path / "shim.so"), here], env=dict(os.environ, PYTHONPATH=os.path.dirname(here)),
                       capture_output=True, text=True, timeout=timeout)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0 and r.stdout.endswith("done\n")
