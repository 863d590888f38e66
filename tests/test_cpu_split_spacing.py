"""The f16 hi + lo split of the MFMA linears (lm_split4): an instruction that
writes the high half of a register must not be followed at once by one that
reads it, which the compiler does not see to for inline assembly.  Checked on
the assembly of a kernel that splits side by side with other work."""
import os
import re
import shutil

import pytest

from qtpytorch_amd.csrc import build as b
from qtpytorch_amd.csrc import check_lgkm as ck

STUB = """
#include "mxk_linear_mfma.h"
template <bool F32>
__global__ void k_split(const uint32_t* c, const float* s, uint32_t* o) {
  uint32_t cc[4], r[8];
  float ss[4];
  for (int i = 0; i < 4; ++i) { cc[i] = c[threadIdx.x + 64 * i]; ss[i] = s[threadIdx.x + 64 * i]; }
  mxk::lm_split4<F32>(cc, ss, r[0], r[1], r[2], r[3]);
  for (int i = 0; i < 4; ++i) ss[i] *= 3.0f;
  mxk::lm_split4<F32>(cc, ss, r[4], r[5], r[6], r[7]);
  for (int i = 0; i < 8; ++i) o[threadIdx.x + 64 * i] = r[i] ^ 5u;
}
template __global__ void k_split<true>(const uint32_t*, const float*, uint32_t*);
template __global__ void k_split<false>(const uint32_t*, const float*, uint32_t*);
"""


def _followers(asm):
    """(writes of a high half, those that the next instruction reads)"""
    n, bad, owed = 0, [], set()
    for line in asm.splitlines():
        text = line.split(";")[0].strip()
        if not text or text.startswith(".") or text.endswith(":"):
            continue
        op, _, rest = text.partition(" ")
        args = rest.split(",")
        reads = {int(r) for a in args[1:] for r in re.findall(r"\bv(\d+)\b", a)}
        for lo, hi in re.findall(r"v\[(\d+):(\d+)\]", ",".join(args[1:])):
            reads.update(range(int(lo), int(hi) + 1))
        if owed & reads:
            bad.append(text)
        owed = {int(r) for r in re.findall(r"\bv(\d+)\b", args[0])} if op == "v_fma_mixhi_f16" else set()
        n += bool(owed)
    return n, bad


def test_planted_reader_is_found():
    hi = "\tv_fma_mixhi_f16 v3, v1, v2, 0\n"
    assert _followers(hi + "\tv_xor_b32_e32 v4, 5, v3\n") == (1, ["v_xor_b32_e32 v4, 5, v3"])
    assert _followers(hi + "\tglobal_store_dwordx2 v9, v[2:3], s[0:1]\n")[1]
    assert _followers(hi + "\ts_nop 0\n\tv_xor_b32_e32 v4, 5, v3\n") == (1, [])


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="needs hipcc")
def test_split_keeps_its_distance(tmp_path):
    src = tmp_path / "split.hip"
    src.write_text(STUB)
    asm = ck.compile_asm(str(src), b.hipcc(), b.HIPCC_FLAGS + ["-I", b.HERE])
    n, bad = _followers(asm)
    assert n == 16 and bad == []
    # each split is one statement: nothing can move into it
    blocks = re.findall(r";;#ASMSTART\n(.*?);;#ASMEND", asm, re.S)
    assert sorted(t.count("v_fma_mix") for t in blocks if "v_fma_mix" in t) == [8] * 4
