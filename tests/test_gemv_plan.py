"""The decode GEMV's launch plans, on the host: the sizes at which a plan is chosen for a reason that a
result does not show (how the activations are staged, when a workgroup walks several tiles)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    if not (os.path.exists(HIPCC) or shutil.which("hipcc")):
        pytest.skip("no hipcc")
    exe = str(tmp_path_factory.mktemp("plan") / "gemv_plan")
    subprocess.run([HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O0", os.path.join(HERE, "host_cpp", "gemv_plan.hip"),
                    "-o", exe], check=True, capture_output=True, timeout=110)

    def query(cases):
        r = subprocess.run([exe], input="\n".join(" ".join(map(str, c)) for c in cases), capture_output=True, text=True, check=True)
        return [None if line == "none" else tuple(map(int, line.split())) for line in r.stdout.split("\n") if line]

    return query


# A lane stages up to 8 chunks of activations at once.  Plans that need a second batch make every wave wait
# for memory twice before its first product, and are for problems that no other plan fits.
@pytest.mark.parametrize("M,K,N,gs,bits,nmat", [
    (8, 7808, 880, 128, 4, 1), (4, 16000, 2328, 128, 4, 1), (4, 14720, 21116, 128, 4, 1), (7, 3968, 7936, 128, 4, 2),
    (6, 7808, 21900, 128, 4, 1), (5, 7872, 643, 64, 8, 1), (6, 4096, 3328, 128, 8, 2), (6, 7360, 782, 64, 8, 1),
])
def test_activations_staged_in_one_batch(plans, M, K, N, gs, bits, nmat):
    (waves, steps, ring, rows, staged, _), = plans([(M, K, N, gs, bits, nmat)])
    assert rows == M and staged <= 8, (waves, steps, ring, staged)


def test_long_rows_keep_one_launch(plans):
    """Rows that fit only with two batches still go out in one launch, rows past the LDS in launches of four."""
    five, eight = plans([(5, 11008, 4096, 64, 4, 1), (8, 14336, 4096, 64, 4, 1)])
    assert five[3] == 5 and five[4] == 16 and eight[3] == 4


# Short chains per tile take more rows before a workgroup walks several tiles; longer ones keep 32.
@pytest.mark.parametrize("M,K,N,gs,bits,nmat,several", [
    (1, 1024, 11136, 32, 4, 2, False), (1, 1024, 13184, 32, 4, 2, False), (1, 1024, 16384, 32, 4, 2, True),
    (2, 1664, 8196, 64, 4, 1, False), (2, 960, 28817, 64, 8, 1, True), (2, 2048, 8704, 32, 4, 2, False),
    (2, 3072, 8064, 128, 8, 2, False), (2, 9728, 10101, 128, 4, 1, True), (2, 6528, 12017, 64, 4, 1, True),
    (2, 3872, 9269, 32, 8, 1, True), (2, 4000, 8762, 32, 8, 1, False),
    (2, 3072, 12288, 128, 8, 2, True), (1, 3968, 10240, 128, 8, 2, True),
    (3, 640, 28426, 128, 4, 1, False), (5, 1024, 8576, 128, 4, 2, False), (8, 1024, 8576, 128, 4, 2, True),
    (3, 1280, 9373, 128, 4, 1, True), (5, 4096, 11008, 64, 4, 2, True), (1, 4096, 14336, 64, 8, 1, True),
    (8, 2560, 9728, 128, 4, 1, True), (2, 3072, 8192, 64, 4, 2, False),
])
def test_several_tiles_where_they_pay(plans, M, K, N, gs, bits, nmat, several):
    (waves, steps, ring, _, _, rows), = plans([(M, K, N, gs, bits, nmat)])
    assert (rows > 0) == several, (waves, steps, ring, rows)
