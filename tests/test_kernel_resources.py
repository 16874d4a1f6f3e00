"""Registers of the built kernels, read from the library's own code objects: the decode GEMV's speed rests
on how many of its workgroups a CU holds (512 registers per lane of a SIMD, handed out in eights)."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "mlx-gen_amd", "mlxq", "libmlxq_hip.so")
LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> (VGPRs, spilled VGPRs) of every kernel built here."""
    if not os.path.exists(os.path.join(LLVM, "llvm-readelf")):
        pytest.skip("no LLVM tools")
    d = tmp_path_factory.mktemp("co")
    subprocess.run([f"{LLVM}/llvm-objcopy", "--dump-section", f".hip_fatbin={d}/fat", LIB, f"{d}/copy.so"], check=True)
    data = open(d / "fat", "rb").read()
    out = {}
    for m in re.finditer(rb"__CLANG_OFFLOAD_BUNDLE__", data):
        p = m.start()
        count, q = struct.unpack("<Q", data[p + 24:p + 32])[0], p + 32
        for _ in range(count):
            off, size, n = struct.unpack("<QQQ", data[q:q + 24])
            name, q = data[q + 24:q + 24 + n], q + 24 + n
            if b"gfx950" not in name or size == 0:
                continue
            (d / "co").write_bytes(data[p + off:p + off + size])
            notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", d / "co"], capture_output=True, text=True, check=True).stdout
            for k in notes.split("- .agpr_count:")[1:]:
                num = lambda f: int(re.search(rf"\.{f}:\s+(\d+)", k).group(1))  # noqa: E731
                out[re.search(r"\.symbol:\s+(\S+)\.kd", k).group(1)] = num("vgpr_count"), num("vgpr_spill_count")
    names = subprocess.run(["c++filt"], input="\n".join(out), capture_output=True, text=True, check=True).stdout.split("\n")
    return dict(zip(names, out.values()))


def _gemv(kernels):
    """(bits, gs, steps, rows, matrices, rounds, several tiles) -> (VGPRs, spills)."""
    found = {}
    for name, v in kernels.items():
        m = re.search(r"(qmv|swiglu)_mfma_kernel<(\d+), (\d+), (\d+), (\d+), (\d+), (true|false)>", name)
        if m:
            n = [int(t) for t in m.groups()[1:6]]
            found[(*n[:4], 1 if m.group(1) == "qmv" else 2, n[4], m.group(7) == "true")] = v
    assert len(found) > 200
    return found


# The forms whose one-tile kernel has at most 64 registers, so that two 16-wave workgroups share a CU: most
# load steps per (bits, group size), and where fewer rows are the condition, (steps, most rows).
TWO_PER_CU = {(8, 32): [(3, 8), (4, 2)], (8, 64): [(4, 8), (6, 2)], (8, 128): [(4, 8), (6, 2)],
              (4, 32): [(1, 8)], (4, 64): [(2, 8), (3, 2)], (4, 128): [(4, 8)]}


def test_one_tile_gemv_keeps_two_workgroups_per_cu(kernels):
    seen = 0
    for (bits, gs, steps, rows, nmat, ring, multi), (vgpr, _) in _gemv(kernels).items():
        two = any(steps <= st and rows <= r for st, r in TWO_PER_CU[bits, gs]) or (bits, gs, steps, rows) == (4, 32, 2, 2)
        if two and ring == 1 and not multi:
            seen += 1
            assert vgpr <= 64, (bits, gs, steps, rows, nmat, vgpr)
    assert seen > 100


# Pointers are two dwords, sizes one; the first 14 dwords of arguments are preloaded into registers.
NEEDED_FIRST = {  # what a workgroup needs for its loads and its result, in this order
    "qmv_mfma_kernel": ["x", "M", "K", "wq", "scales", "biases", "N", "rows", "y"],
    "qmv_row_kernel": ["x", "wq", "scales", "biases", "K", "N", "y"],
}


def test_gemv_arguments_are_preloaded(kernels):
    """A short launch waits for each argument that its first loads need and that is not in registers when
    it starts: those come before the epilogue's and the stacked launch's, which SwiGLU does not have."""
    seen = set()
    for name in kernels:
        m = re.search(r"mlxq::(qmv_mfma_kernel|qmv_row_kernel|swiglu_mfma_kernel|swiglu_row_kernel)<.*>\((.*)\)", name)
        if not m:
            continue
        seen.add(m.group(1))
        args = [t.strip() for t in m.group(2).split(",")]
        first = NEEDED_FIRST.get(m.group(1))
        if first is None:
            assert len(args) == (12 if "mfma" in m.group(1) else 10) and "QmmBatch" not in m.group(2), name
            continue
        assert [t == "int" for t in args[:len(first)]] == [len(f) == 1 and f.isupper() or f == "rows" for f in first], name
        assert sum(1 if t == "int" else 2 for t in args[:len(first)]) <= 14, name
    assert len(seen) == 4


def test_gemv_does_not_spill(kernels):
    """Spills double a short launch's time; every form that would spill is left out of the dispatch."""
    assert not {k: v for k, v in _gemv(kernels).items() if v[1]}
    assert not [n for n, v in kernels.items() if re.search("(qmv|swiglu)_row_kernel<", n) and v[1]]
