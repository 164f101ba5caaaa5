"""Build the gfx950 HIP library race_attention_amd/librace_attention.so and the
autograd calls over it, race_attention_amd/_race_torch.so.

The library is one translation unit (csrc/race_capi.hip, which includes the
kernel sources) compiled with hipcc for gfx950 only.  Packed-fp32 instruction
selection is disabled (-packed-fp32-ops) for all device code.  The autograd
calls (csrc/race_torch.cpp) are host code against torch's C++ API.
"""
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "csrc", "race_capi.hip")
OUT = os.path.join(HERE, "librace_attention.so")
TORCH_SRC = os.path.join(HERE, "csrc", "race_torch.cpp")
TORCH_OUT = os.path.join(HERE, "_race_torch.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-shared", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
]


# host-side sanitizer build (device code unchanged): -fsanitize applies to the
# host compilation only, through -Xarch_host
SAN_OUT = os.path.join(HERE, "_san", "librace_attention_asan.so")
SAN_FLAGS = ["-g", "-fno-omit-frame-pointer", "-Xarch_host", "-fsanitize=address",
             "-Xarch_host", "-fsanitize=undefined"]


def _torch_cmd(out: str):
    import torch
    root = os.path.dirname(torch.__file__)
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           sysconfig.get_paths()["include"], "/opt/rocm/include"]
    return (["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__=1",
             f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"] + ["-I" + i for i in inc] +
            [TORCH_SRC, "-o", out, "-L" + os.path.join(root, "lib")] +
            ["-l" + x for x in ("torch", "torch_cpu", "torch_hip", "c10", "c10_hip", "torch_python")])


def build(verbose: bool = True, sanitize: bool = False) -> str:
    """Both libraries (sanitize: the operator library alone), built side by side."""
    out = SAN_OUT if sanitize else OUT
    host = None
    if not sanitize:
        host = subprocess.Popen(_torch_cmd(TORCH_OUT + ".tmp"), stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                                text=True)
    if sanitize:
        os.makedirs(os.path.dirname(out), exist_ok=True)
    cmd = [HIPCC] + FLAGS + (SAN_FLAGS if sanitize else []) + [SRC, "-o", out + ".tmp"]
    if verbose:
        print("build:", " ".join(cmd), flush=True)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0 and host is not None:
        host.kill()
        host.wait()
    msgs = [ln for ln in proc.stdout.splitlines() if "packed-fp32-ops" not in ln]
    if proc.returncode != 0:
        print("\n".join(msgs), file=sys.stderr)
        raise RuntimeError("hipcc failed building librace_attention.so")
    if verbose and msgs:
        print("\n".join(msgs))
    os.replace(out + ".tmp", out)
    if host is not None:
        text = host.communicate()[0]
        if host.returncode != 0:
            print(text, file=sys.stderr)
            raise RuntimeError("g++ failed building _race_torch.so")
        os.replace(TORCH_OUT + ".tmp", TORCH_OUT)
    return out


if __name__ == "__main__":
    build(sanitize="--sanitize" in sys.argv)
