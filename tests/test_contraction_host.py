"""The arithmetic of the long contractions on the matrix cores (stwo-gpu_amd/csrc/mfma_m31.hpp) built for the
host, against Python integers: limb sums at their bound of 2^29 (8192 columns of 4 digits) joined mod P,
and the operand rows of weights."""
import itertools
import os
import random
import shutil
import struct
import subprocess

import pytest

P = (1 << 31) - 1
HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    if not (os.path.exists(HIPCC) or shutil.which("hipcc")):
        pytest.skip("hipcc not found")
    out = str(tmp_path_factory.mktemp("contraction") / "contraction_host_check")
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-O2", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I" + os.path.join(ROOT, "stwo-gpu_amd", "csrc"),
                    os.path.join(HERE, "contraction_host_check.cpp"), "-o", out], check=True, capture_output=True)

    def run(rows):
        got = subprocess.run([out], input=b"".join(struct.pack("<4i", *r) for r in rows), capture_output=True,
                             check=True).stdout
        assert len(got) == 68 * len(rows)
        return list(struct.iter_unpack("<17I", got))

    return run


def test_join_of_extreme_sums(ask):
    rng = random.Random(0x5EED)
    bound = 1 << 29  # 8192 columns x 4 digits x 128 x 128
    rows = list(itertools.product((-bound, -bound + 1, -1, 0, 1, bound - 1, bound), repeat=4))
    rows += [tuple(rng.randint(-bound, bound) for _ in range(4)) for _ in range(5000)]
    for a, (joined, *_) in zip(rows, ask(rows)):
        assert joined == sum(v << (8 * i) for i, v in enumerate(a)) % P, a


def test_operand_rows_of_weights(ask):
    """Row 4 k + i holds, in byte j, limb i of c[k] 2^(8j): four signed limbs make the residue again."""
    rng = random.Random(0xC0DE)
    edge = [0, 1, P - 1, P // 2, P // 2 + 1, 1 << 30, 0x7F7F7F7F, 0x00808080]
    rows = [tuple(rng.choice(edge) for _ in range(4)) for _ in range(200)]
    rows += [tuple(rng.randrange(P) for _ in range(4)) for _ in range(2000)]
    signed = lambda w, j: ((w >> (8 * j)) & 0xFF) - 256 * ((w >> (8 * j + 7)) & 1)
    for c, (_, *words) in zip(rows, ask(rows)):
        for k in range(4):
            for j in range(4):
                limbs = [signed(words[4 * k + i], j) for i in range(4)]
                assert sum(v << (8 * i) for i, v in enumerate(limbs)) % P == (c[k] << (8 * j)) % P, (c, k, j)
