"""Build the unpopped-hip host library in-tree.

Produces ``unpopped_amd/libunpopped_hip.so`` from ``unpopped_amd/csrc``: the device template
library (``csrc/kernels/unp_device.hip``) is embedded as a string (the emitter writes it into
every kernel source), the host code is compiled with g++ against the HIP headers, the one HIP
source (``csrc/scratch.hip``, the no-allocation launch's static device array) with hipcc, and all
of it linked to libamdhip64 and libhiprtc.  ``check_device`` also compiles sample instantiations of every
device template for gfx950 with hipcc, so a device-side error shows at build time rather than
at the first hipRTC compile on a GPU box.
"""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
BUILD = HERE / "_build"
LIB = HERE / "libunpopped_hip.so"
SYNTH_LIB = HERE / "libunpopped_synth.so"
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))

HOST_SOURCES = ["emit_hip.cpp", "compile_rtc.cpp", "runtime.cpp", "kernel_ir.cpp", "lifts.cpp"]

HIPCC_DEVICE_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _run(cmd: list[str]) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"build step failed: {' '.join(cmd[:3])} ...")


def embed_device_library() -> Path:
    """Write the device library as a C++ string constant."""
    BUILD.mkdir(exist_ok=True)
    text = (CSRC / "kernels" / "unp_device.hip").read_bytes()
    out = BUILD / "embedded_device.cpp"
    parts = ", ".join(str(b) for b in text)
    out.write_text(
        "// generated by unpopped_amd/build.py from csrc/kernels/unp_device.hip\n"
        "namespace unp {\n"
        f"static const char kDeviceLibraryBytes[] = {{{parts}, 0}};\n"
        "extern const char* const kDeviceLibrary = kDeviceLibraryBytes;\n"
        "}\n"
    )
    return out


def build_host() -> Path:
    embedded = embed_device_library()
    objs = []
    for src in HOST_SOURCES + [str(embedded)]:
        path = Path(src) if os.path.isabs(src) else CSRC / src
        obj = BUILD / (path.stem + ".o")
        _run([
            "g++", "-std=c++17", "-O2", "-fPIC", "-Wall", "-Wno-unused-function",
            "-D__HIP_PLATFORM_AMD__", f"-I{ROCM / 'include'}", "-c", str(path), "-o", str(obj),
        ])
        objs.append(str(obj))
    # The static scratch of the no-allocation launch is device memory of this library's own code
    # object, so its one source is compiled as HIP.
    # The view packers (staged storage images) are kernels of the library's own code object too.
    for hip_src in ("scratch.hip", "views.hip"):
        hip_obj = BUILD / (Path(hip_src).stem + ".o")
        _run([str(ROCM / "bin" / "hipcc"), *HIPCC_DEVICE_FLAGS, "-fPIC", "-Wall", f"-I{CSRC}", "-c",
              str(CSRC / hip_src), "-o", str(hip_obj)])
        objs.append(str(hip_obj))
    tmp = LIB.with_suffix(".so.tmp")
    _run([
        "g++", "-shared", "-o", str(tmp), *objs, f"-L{ROCM / 'lib'}", "-lamdhip64", "-lhiprtc",
        f"-Wl,-rpath,{ROCM / 'lib'}",
    ])
    os.replace(tmp, LIB)
    return LIB


CHECK_INSTANTIATIONS = r"""
#include "unp_device.hip"
#define KB __launch_bounds__(256)
// The descriptors the host passes by value (runtime.cpp asserts the same sizes for its images).
static_assert(sizeof(unp::red_axes) == 61 * 8, "red_axes");
static_assert(sizeof(unp::red_view) == 44 * 8, "red_view");
static_assert(sizeof(unp::scan_view) == 29 * 8, "scan_view");
static_assert(sizeof(unp::gather_view) == 35 * 8, "gather_view");
static_assert(sizeof(unp::ew_tile_view) == 114 * 8, "ew_tile_view");
extern "C" __global__ void KB c_rr(const float* a, float* b, float* c, long long r, long long n) { unp::rowreduce<float, unp::OP_SUM, unp::OP_MAX, 2, 4, 256, 4, true>(a, b, c, r, n); }
extern "C" __global__ void KB c_rw(const float* a, float* b, float* c, long long r, long long n) { unp::rowreduce_wave<float, unp::OP_SUM, unp::OP_MAX, 2, 4, 256, 8, true>(a, b, c, r, n); }
extern "C" __global__ void KB c_rri(const long long* a, long long* b, long long* c, long long r, long long n) { unp::rowreduce<long long, unp::OP_PROD, unp::OP_MIN, 2, 2, 256, 8, false>(a, b, c, r, n); }
extern "C" __global__ void KB c_ra(const double* a, double* b, long long n, unsigned long long* p, unsigned* k, unsigned e, unp::waits w) { unp::reduce_all<double, unp::OP_MEAN, 2, 256, 4>(a, b, n, p, k, e, w); }
extern "C" __global__ void KB c_rn(const float* a, float* b, float* c, long long r, long long n) { unp::rowreduce_wave<float, unp::OP_MAXNUM, unp::OP_MINNUM, 2, 4, 256, 8, false>(a, b, c, r, n); }
extern "C" __global__ void KB c_rx(const int* a, int* b, long long n, unsigned long long* p, unsigned* k, unsigned e, unp::waits w) { unp::reduce_all<int, unp::OP_XOR, 4, 256, 4>(a, b, n, p, k, e, w); }
extern "C" __global__ void __launch_bounds__(512) c_rb(const long long* a, long long* b, unsigned long long* p, unsigned* k, unsigned e, unp::waits w, unp::red_axes d) { const long long* in[1] = {a}; unp::xreduce_inner<long long, 1, unp::OP_AND, unp::plain_ops<long long, unp::OP_AND>, 2, 8, 512, 8>(in, b, p, k, e, w, d); }
extern "C" __global__ void __launch_bounds__(512) c_ro(const float* a, float* b, unsigned long long* p, unsigned* k, unsigned e, unp::waits w, unp::red_axes d) { const float* in[1] = {a}; unp::xreduce_outer<float, 1, unp::OP_SUM, unp::plain_ops<float, unp::OP_SUM>, 4, 512, 8>(in, b, p, k, e, w, d); }
extern "C" __global__ void __launch_bounds__(512) c_rs(const double* a, double* b, unp::red_axes d) { const double* in[1] = {a}; unp::xreduce_outer_wave<double, 1, unp::OP_SUM, unp::plain_ops<double, unp::OP_SUM>, 2, 512, 8>(in, b, d); }
extern "C" __global__ void __launch_bounds__(512) c_rz(const int* a, int* b, unp::red_axes d) { const int* in[1] = {a}; unp::xreduce_outer_alone<int, 1, unp::OP_MAX, unp::plain_ops<int, unp::OP_MAX>, 1, 512, 8>(in, b, d); }
extern "C" __global__ void KB c_rl(const float* a, float* b, unp::red_axes d) { const float* in[1] = {a}; unp::xreduce_lanes<float, 1, unp::OP_SUM, unp::plain_ops<float, unp::OP_SUM>, 4, true, 256>(in, b, d); }
extern "C" __global__ void KB c_rm(const double* a, double* b, unp::red_axes d) { const double* in[1] = {a}; unp::xreduce_lanes<double, 1, unp::OP_MAX, unp::plain_ops<double, unp::OP_MAX>, 2, false, 256>(in, b, d); }
extern "C" __global__ void KB c_rq(const float* a, float* b, unp::red_view d) { unp::reduce_serial<float, unp::OP_MAXNUM, 256>(a, b, d); }
extern "C" __global__ void KB c_rq2(const long long* a, long long* b, unp::red_view d) { unp::reduce_serial<long long, unp::OP_XOR, 256>(a, b, d); }
extern "C" __global__ void KB c_rv(const float* a, float* b, unp::red_view d) { unp::reduce_strided<float, unp::OP_SUM, 256>(a, b, d); }
extern "C" __global__ void __launch_bounds__(576) c_sc(const double* a, double* b, long long S, long long B, long long n, long long c, int wide) { __shared__ __attribute__((aligned(16))) unsigned char ring[9 * 16384]; if (wide) unp::scan_cols<double, unp::OP_MEAN, true, true, true, 8>(a, b, S, B, n, c, ring); else unp::scan_cols<double, unp::OP_MEAN, true, true, false, 8>(a, b, S, B, n, c, ring); }
extern "C" __global__ void KB c_sv(const double* a, double* b, unp::scan_view v) { unp::scan_strided<double, unp::OP_MEAN, true, true>(a, b, v); }
extern "C" __global__ void KB c_gv(const unsigned short* t, const long long* i, unsigned short* o, unp::gather_view v, long long x) { unp::gather_strided<unsigned short, long long, unp::OOB_ZEROFILL>(t, i, o, v, x); }
extern "C" __global__ void KB c_si(const int* a, int* b, long long r, long long c, unsigned long long* s, unsigned* k, unsigned t, unsigned e, unp::waits w) { unp::scan_lookback<int, unp::OP_SUM, true, true, 4, 16, 4, 32>(a, b, r, c, s, k, t, e, w); }
extern "C" __global__ void __launch_bounds__(448) c_ss(const int* a, int* b, long long r, long long c, unsigned long long* s, unsigned* k, unsigned t, unsigned e, unp::waits w) { unp::scan_staged<int, unp::OP_MAX, true, true, 4, 12, 6, 32>(a, b, r, c, s, k, t, e, w); }
extern "C" __global__ void __launch_bounds__(320) c_sf(const float* a, float* b, long long r, long long c, unsigned long long* s, unsigned* k, unsigned t, unsigned e, unp::waits w) { unp::scan_staged<float, unp::OP_SUM, false, false, 4, 18, 4, 32>(a, b, r, c, s, k, t, e, w); }
extern "C" __global__ void __launch_bounds__(320) c_sff(const float* a, float* b, long long r, long long c, unsigned long long* s, unsigned* k, unsigned t, unsigned e, unp::waits w) { unp::scan_staged<float, unp::OP_SUM, true, true, 4, 18, 4, 32, true>(a, b, r, c, s, k, t, e, w); }
extern "C" __global__ void KB c_sif(const double* a, double* b, long long r, long long c, unsigned long long* s, unsigned* k, unsigned t, unsigned e, unp::waits w) { unp::scan_lookback<double, unp::OP_MAX, false, false, 1, 16, 4, 32, true>(a, b, r, c, s, k, t, e, w); }
extern "C" __global__ void __launch_bounds__(320) c_sd(const double* a, double* b, long long r, long long c, unsigned long long* s, unsigned* k, unsigned t, unsigned e, unp::waits w) { unp::scan_staged<double, unp::OP_MIN, false, true, 2, 18, 4, 32>(a, b, r, c, s, k, t, e, w); }
struct c_xops { typedef double arg; typedef double acc; static constexpr bool has_post = true; static __device__ double pre(const double* x) { return x[0] * x[1]; } static __device__ double post(const double* r, const double* x) { return r[0] - x[0]; } };
struct c_iops { typedef long long arg; typedef long long acc; static constexpr bool has_post = false; static __device__ long long pre(const long long* x) { return unp::xi::div<long long>(x[0], x[1]); } static __device__ long long post(const long long* r) { return r[0]; } };
extern "C" __global__ void KB c_xi(const long long* a, const long long* b, long long* o, long long n, unsigned long long* p, unsigned* k, unsigned e, unp::waits w) { const long long* in[2] = {a, b}; unp::xreduce_all<long long, 2, unp::OP_PROD, c_iops, 2, 256, 8>(in, o, n, p, k, e, w); }
extern "C" __global__ void KB c_xq(const float* a, const float* b, float* o, long long A, long long S, long long B) { const float* in[2] = {a, b}; unp::xscan_seq<float, 2, unp::OP_MEAN, c_xops, true, true>(in, o, A, S, B); }
extern "C" __global__ void __launch_bounds__(512) c_xs(const double* a, const double* b, double* o, long long r, long long c, unsigned long long* s, unsigned* k, unsigned t, unsigned e, unp::waits w) { const double* in[2] = {a, b}; unp::xscan_lookback<double, 2, unp::OP_MAX, c_xops, false, true, 8, 8, 32>(in, o, r, c, s, k, t, e, w); }
extern "C" __global__ void KB c_g(const unsigned char* t, const unsigned* i, unsigned char* o, long long n, long long b, unsigned x) { unp::gather_rows<unsigned, unp::OOB_CLAMP, 2, 256, 16, 2>(t, i, o, n, b, x); }
extern "C" __global__ void KB c_d(const unsigned char* q, const unsigned short* s, const unsigned char* z, unsigned short* o, long long r, long long c) { unp::dequant4_bf16<true, true, 64, 256, 8>(q, s, z, o, r, c); }
"""


def check_device() -> None:
    BUILD.mkdir(exist_ok=True)
    src = BUILD / "check_instantiations.hip"
    src.write_text(CHECK_INSTANTIATIONS)
    hipcc = str(ROCM / "bin" / "hipcc")
    _run([hipcc, *HIPCC_DEVICE_FLAGS, "--genco", f"-I{CSRC / 'kernels'}", str(src), "-o",
          str(BUILD / "check_instantiations.co")])


def build_synth() -> Path:
    """The seeded input generator (host C, OpenMP)."""
    tmp = SYNTH_LIB.with_suffix(".so.tmp")
    _run(["gcc", "-std=c11", "-O2", "-fPIC", "-fopenmp", "-shared", str(CSRC / "synth.c"), "-o", str(tmp), "-lm"])
    os.replace(tmp, SYNTH_LIB)
    return SYNTH_LIB


def build(check: bool = True) -> Path:
    if check:
        check_device()
    build_synth()
    return build_host()


if __name__ == "__main__":
    print(build())
