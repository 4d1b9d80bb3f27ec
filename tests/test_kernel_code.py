"""What needs no GPU to be seen of the kernels: the order of loads and waits of the decode attention, which are counted by hand, and of
the float32 products of few rows, read from their assembly (compiled here); and the rules by which a product of few rows picks its form and its splits."""

from __future__ import annotations

import ctypes
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from miniserve_amd.kernels import build


def assembly(source, folder):
    if not (shutil.which("hipcc") or Path("/opt/rocm/bin/hipcc").exists()):
        pytest.skip("needs hipcc")
    out = folder / f"{source}.s"
    flags = [f for f in build.HIP_FLAGS if f != "-fPIC"]
    subprocess.run([build._hipcc(), *flags, "-S", "--cuda-device-only", str(build.CSRC / f"{source}.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    return out.read_text()


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    found = {}
    for text in re.split(r"\n(?=_Z\d+attn_decode_split_kernel)", assembly("attention_decode", tmp_path_factory.mktemp("code")))[1:]:
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


def test_float32_products_of_few_rows_ask_for_everything_at_once(tmp_path):
    """Where the weights come through LDS, the activations of all slabs are asked for ahead of the first wait for a load."""
    found = re.split(r"\n_Z\d+gemm_f32_few_kernelILi1ELi(\d)ELb[01]ELb1ELb1EE\w+:", assembly("gemm_f32", tmp_path))
    assert len(found) == 1 + 2 * 4
    for slabs, text in zip(found[1::2], found[2::2]):
        code = [x.strip() for x in text.split("s_endpgm")[0].splitlines()]
        ahead = code[: next(i for i, x in enumerate(code) if x.startswith("s_waitcnt") and "vmcnt" in x)]
        assert sum(x.startswith("global_load_dwordx4") for x in ahead) == 2 * int(slabs)  # 8 k of a row a slab and lane
        assert sum(x.startswith("global_load_lds_dwordx4") for x in ahead) == 2 * int(slabs)
        assert not any(re.match(r"(global|flat|scratch)_load_dwordx4", x) for x in code[len(ahead) :])


@pytest.mark.parametrize("m,n,k,splits,tiles", [
    (8, 10304, 2048, 8, False), (9, 10304, 2048, 5, True), (9, 16384, 1024, 4, False), (9, 12288, 1536, 4, True),  # 16 M to 20 M weights
    (8, 12272, 2048, 8, False), (8, 12288, 2048, 4, True), (4, 12288, 2048, 8, False),  # 24 M
    (16, 8192, 4096, 8, True), (17, 8192, 4096, 6, True), (8, 4096, 8192, 16, True), (16, 5120, 8192, 8, True), (16, 24576, 4096, 4, True),  # even slices
    (16, 8192, 4160, 6, True), (1, 151937, 4096, 1, True),
    (16, 16411, 4096, 4, True), (17, 16411, 4096, 4, True), (32, 16411, 4096, 4, True), (33, 16411, 4096, 3, True)])  # 128 MB
def test_products_of_few_rows_pick_their_form_and_splits(m, n, k, splits, tiles):
    lib = ctypes.CDLL(str(build.build_kernels()))
    assert lib.ms_gemm_bf16_small_splits(m, n, k) == splits
    assert (lib.ms_gemm_bf16_small_ring(m, n, k) != 0) == (tiles and lib.ms_gemm_bf16_small_tile_cols(n, k) == 64)
