"""The pair term's block of assembly writes the sums of its first targets before
it reads the inputs of its last ones.  Compiled with sums that start from the
targets' and the source's own values, no sum may lie in a register that is also
an input."""
import importlib.util
import re
import subprocess
from pathlib import Path

import pytest

PKG = Path(__file__).resolve().parent.parent / "cuda-to-sycl-nbody_amd"

KERNEL = """
#include "nb_pair_block.hpp"
extern "C" __global__ void pairs(const float *in, float *out, float eps) {{
  constexpr int U = {U}, SRC = {SRC}, ACC = {ACC};
  in += threadIdx.x;
  out += threadIdx.x;
  float s[SRC], t[U][SRC], a[U][ACC], r[ACC];
  for (int c = 0; c < SRC; ++c) s[c] = in[64 * c];
  for (int k = 0; k < U; ++k)
    for (int c = 0; c < SRC; ++c) t[k][c] = in[64 * (SRC * (k + 1) + c)];
  for (int k = 0; k < U; ++k)
    for (int c = 0; c < ACC; ++c) a[k][c] = t[U - 1 - k][c % SRC];
  for (int c = 0; c < ACC; ++c) r[c] = s[c % SRC];
  nb::{name}<U>(s, t, a, r, eps);
  for (int k = 0; k < U; ++k)
    for (int c = 0; c < ACC; ++c) out[64 * (ACC * k + c)] = a[k][c];
  for (int c = 0; c < ACC; ++c) out[64 * (ACC * U + c)] = r[c];
}}
"""


def _build():
    spec = importlib.util.spec_from_file_location("nb_pkg_build", PKG / "build.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.mark.parametrize("name, src, acc", [("force_block", 3, 3), ("adjoint_block", 6, 3),
                                            ("fused_block", 6, 6), ("kahan_block", 3, 6)])
def test_sums_and_inputs_are_apart(tmp_path, name, src, acc):
    b = _build()
    if not Path(b.HIPCC).exists():
        pytest.skip("no hipcc")
    (tmp_path / "k.hip").write_text(KERNEL.format(U=4, SRC=src, ACC=acc, name=name))
    subprocess.run([b.HIPCC, *b.HIP_FLAGS, "--cuda-device-only", "-S", "k.hip", "-o", "k.s"],
                   cwd=tmp_path, check=True, capture_output=True)
    text = (tmp_path / "k.s").read_text()
    body = re.search(r";;#ASMSTART(.*?);;#ASMEND", text, re.S).group(1)
    written, inputs = set(), set()
    for line in body.splitlines():
        m = re.match(r"\s*v_(\w+) (.*)", line)
        if not m:
            continue
        regs = [int(x) for x in re.findall(r"\bv(\d+)\b", m.group(2))]
        if m.group(1).startswith("sub") and not written & set(regs[1:]):
            inputs.update(regs[1:])  # s - t of positions and cotangents
        written.add(regs[0])
    assert len(inputs) == src * 5 and not inputs & written, (sorted(inputs & written))
