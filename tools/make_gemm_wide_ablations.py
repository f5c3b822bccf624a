#!/usr/bin/env python3
"""make_gemm_wide_ablations.py — the timing-only variants of csrc/gemm_wide.hip that tools/gpu_wide_ablate.sh times .

Each variant is the shipped source with ONE part of the K loop compiled out (results are WRONG on purpose) or one load hint
changed (`plain`: right results), built as csrc/libswiftllm_hip_gw<name>.so next to the product library (it travels to the
GPU box with the snapshot; delete the files afterwards):

    python tools/make_gemm_wide_ablations.py            # writes /tmp/gw_<name>.hip and builds every variant
    gpurun -- 'bash tools/gpu_wide_ablate.sh'

  plain   W without the non-temporal hint
  nox     every slice of x is the first one (L1 hits)
  nolds   x fragments taken from the weight fragments instead of LDS
  wcache  every slice of W is the first one (cache hits instead of the HBM stream)
  nomfma  one fma per fragment pair instead of the MFMA"""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "swiftllm_amd", "csrc", "gemm_wide.hip")

EDITS = {
    "plain": [("global_load_lds_dwordx4 %1, %2 nt", "global_load_lds_dwordx4 %1, %2")],
    "nox": [("*xs = xsrc + static_cast<int64_t>(st) * kWT * 2;", "*xs = xsrc;")],
    "nolds": [("xf[set][b] = *reinterpret_cast<const vec8_t<T> *>(s + b * 4096 + frag[e]);", "xf[set][b] = wf[set][b & 1];")],
    "wcache": [("wsrc + static_cast<int64_t>(st) * 4096", "wsrc")],
    "nomfma": [("acc[a][b] = mfma_w(wf[set][a], xf[set][b], acc[a][b]);", "acc[a][b][0] += to_f(wf[set][a][0]) * to_f(xf[set][b][0]);")],
}


def main():
    src = open(SRC).read()
    names = sys.argv[1:] or list(EDITS)
    for name in names:
        text = src
        for old, new in EDITS[name]:
            assert text.count(old) == 1, f"{name}: pattern not found exactly once — the kernel moved on: {old[:60]}"
            text = text.replace(old, new)
        path = f"/tmp/gw_{name}.hip"
        open(path, "w").write(text)
        subprocess.run([sys.executable, "-m", "swiftllm_amd.csrc.build", "--tag", f"gw{name}", "--swap",
                        f"gemm_wide.hip={path}"], cwd=ROOT, check=True)


if __name__ == "__main__":
    main()
