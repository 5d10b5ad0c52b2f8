"""Builds the C++ test programs into tests/cpp/_build: sampling_mirror, the
driver of the C++ operator mirror, against the in-tree libjf_sampler.so, and
launch_plan, the library's host objects over recording launchers (build the
library first)."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(os.path.dirname(HERE))
LIBDIR = os.path.join(REPO, "justfit-llm_amd", "jf_sampler")
OBJ = os.path.join(REPO, "justfit-llm_amd", "_build")
OUT = os.path.join(HERE, "_build", "sampling_mirror")
PLAN = os.path.join(HERE, "_build", "launch_plan")


def _compile(source, out, link, verbose):
    cmd = [os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-O2", "-std=c++20",
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-I" + os.path.join(REPO, "include"),
           "-I" + os.path.join(REPO, "justfit-llm_amd", "csrc"),
           os.path.join(HERE, source)] + link + ["-o", out]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in res.stderr.splitlines()
                    if "'-packed-fp32-ops' is not a recognized feature" not in l)
    if res.returncode != 0:
        sys.stderr.write(err + "\n")
        raise RuntimeError(f"building {source} failed")


def build(verbose=True):
    os.makedirs(os.path.dirname(OUT), exist_ok=True)
    _compile("sampling_mirror.cpp", OUT,
             ["-L" + LIBDIR, "-ljf_sampler",
              "-Wl,-rpath,$ORIGIN/../../../justfit-llm_amd/jf_sampler"], verbose)
    _compile("launch_plan.cpp", PLAN,
             ["-x", "none"] + [os.path.join(OBJ, n + ".o")
                               for n in ("jf_sampler.cpp", "jf_host.cpp")], verbose)
    return OUT


if __name__ == "__main__":
    print(build())
