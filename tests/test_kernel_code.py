"""What the compiler makes of a kernel whose waits are counted by hand: the decode attention's order of loads and waits, read from
its assembly (compiled here; no GPU)."""

from __future__ import annotations

import re
import shutil
import subprocess
from pathlib import Path

import pytest

from miniserve_amd.kernels import build


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not (shutil.which("hipcc") or Path("/opt/rocm/bin/hipcc").exists()):
        pytest.skip("needs hipcc")
    out = tmp_path_factory.mktemp("code") / "attention_decode.s"
    flags = [f for f in build.HIP_FLAGS if f != "-fPIC"]
    subprocess.run([build._hipcc(), *flags, "-S", "--cuda-device-only", str(build.CSRC / "attention_decode.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    found = {}
    for text in re.split(r"\n(?=_Z\d+attn_decode_split_kernel)", out.read_text())[1:]:
        key = re.match(r"_Z\d+attn_decode_split_kernelILi(\d+)ELb([01])E", text)
        found.setdefault((int(key[1]), key[2] == "1"), []).append(text.split("s_endpgm")[0])
    return found


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("d", [64, 128])
def test_decode_attention_keeps_two_chunks_under_way(kernels, d, fused):
    """Keys go into LDS ahead of the chunk's values, which the counted wait for them relies on; and between a chunk's loads and its
    products no wait is for more than what the products need, so that the next chunk stays under way."""
    loads, values = d // 16, d // 16  # a chunk's loads of 1 KB: keys into LDS, values into registers
    ring = rf"s_waitcnt vmcnt\({loads + 2 * values}\)"
    assert kernels[d, fused]
    for text in kernels[d, fused]:
        code = [x.strip() for x in text.splitlines()]
        memory = [x for x in code if re.match(r"(global|buffer|flat|scratch)_(load|store|atomic)", x)]
        assert not any(x.startswith(("scratch", "flat")) for x in memory)
        into_lds = [i for i, x in enumerate(memory) if re.search(r"\blds\b|_lds_", x)]
        starts = [i for i in into_lds if i - 1 not in into_lds]
        assert len(starts) >= 2
        for i in starts:
            assert all(j in into_lds for j in range(i, i + loads)) and i + loads not in into_lds
            assert all(re.match(r"global_load_dwordx4 .* nt$", x) for x in memory[i + loads : i + loads + values]), memory[i + loads : i + loads + values]
        kept = 0
        for i in (i for i, x in enumerate(code) if re.match(ring, x)):  # from the last load of the next chunk to the last product of this one
            products = [j for j in range(i, len(code)) if code[j].startswith("v_mfma")][: d // 16 + values]
            waits = [int(m[1]) for x in code[i + 1 : products[-1]] if (m := re.match(r"s_waitcnt.*vmcnt\((\d+)\)", x))]
            kept += all(w >= loads + values for w in waits)
        assert kept >= 2  # the loop's two halves (behind it, the wait for the last chunk may stand among the products of the one before)
