"""A stand-in for the HIP runtime, for tests of the library's host code without
a GPU: a host program defines the runtime's functions on host memory, and its
symbols come before those of the runtime when it loads the library. No kernel
runs; the launches are listed by name, and any of them can be made to fail."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

RUNTIME = r"""
#include <dlfcn.h>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include "vct.h"

struct dim3 { unsigned x, y, z; };
static std::map<const void*, std::string> names;
static std::string launched;  // the names of the kernels launched, a blank after each
static std::string failing;   // a launch of a kernel with this in its name fails
static int last_error = 0, capturing = 0;
static int waits = 0;                    // waits of the host for the stream
static unsigned long long counted = 0;   // what every 8-byte read from the device finds
static dim3 grid_, block_;
static size_t shared_;
static void* stream_;
extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, void* s)
{
    grid_ = g;
    block_ = b;
    shared_ = m;
    stream_ = s;
    return 0;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, void** s)
{
    *g = grid_;
    *b = block_;
    *m = shared_;
    *s = stream_;
    return 0;
}
int hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, void*)
{
    const std::string& n = names[f];
    if (!failing.empty() && n.find(failing) != std::string::npos) return last_error = 1;
    launched += n + ' ';
    return 0;
}
int hipGetLastError()
{
    const int e = last_error;
    last_error = 0;
    return e;
}
const char* hipGetErrorString(int) { return "error"; }
int hipMalloc(void** p, size_t n) { return (*p = calloc(1, n)) ? 0 : 2; }
int hipFree(void* p)
{
    free(p);
    return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
int hipHostFree(void* p) { return hipFree(p); }
int hipMemset(void* p, int v, size_t n)
{
    memset(p, v, n);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*)
{
    memcpy(d, kind == 2 && n == 8 ? &counted : s, n);
    return 0;
}
int hipGetDevice(int* d) { return *d = 0; }
int hipGetStreamDeviceId(void*) { return 0; }
int hipDeviceGetAttribute(int* v, int, int)
{
    *v = 64;
    return 0;
}
int hipGetDevicePropertiesR0600(void* p, int)
{
    memset(p, 0, 1472);  // the size of the properties
    return 0;
}
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void*)
{
    ++waits;
    return 0;
}
int hipGetSymbolAddress(void** p, const void*)
{
    static char c;
    *p = &c;
    return 0;
}
int hipStreamIsCapturing(void*, int* s)
{
    *s = capturing;
    return 0;
}
}

// the library's function `name`, from the handle `lib`
#define CALL(name) ((decltype(&name))dlsym(lib, #name))
"""


def build(directory: Path, main: str) -> str:
    """Compiles `main` (a C++ program that includes nothing of the above) behind
    the stand-in; returns the executable's path."""
    (directory / "main.cpp").write_text(RUNTIME + main)
    exe = str(directory / "host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-rdynamic", f"-I{ROOT / 'include'}", str(directory / "main.cpp"),
                    "-ldl", "-o", exe], check=True)
    return exe
