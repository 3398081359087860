"""The arithmetic of the matrix-core maps (stwo-gpu_amd/csrc/mfma_m31.hpp) built for the host: 16
products and their sum mod P through signed byte digits, limb sums and the join, against Python
integers, at values whose digits are all extreme and at random ones."""
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
def binary(tmp_path_factory):
    if not (os.path.exists(HIPCC) or shutil.which("hipcc")):
        pytest.skip("hipcc not found")
    out = str(tmp_path_factory.mktemp("mfma") / "mfma_host_check")
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-O2", "-I" + os.path.join(ROOT, "stwo-gpu_amd", "csrc"),
                    os.path.join(HERE, "mfma_host_check.cpp"), "-o", out], check=True, capture_output=True)
    return out


def from_digits(d):
    return sum(v << (8 * j) for j, v in enumerate(d)) % P


def test_map_by_digits(binary):
    rng = random.Random(0x5EED)
    edge = [0, 1, 2, P - 1, P - 2, 1 << 30, (1 << 30) - 1, P // 2, P // 2 + 1]
    edge += [from_digits(d) for d in itertools.product((-128, 127, 0), repeat=4)]
    # a digit operand may be any 32-bit value below 2^32 - 2^24 (what a join leaves unreduced)
    big = edge + [P, P + 1, (1 << 32) - (1 << 24) - 1, (1 << 31) + (1 << 30)]
    rows = [([x] * 16, [e] * 16) for x in big for e in edge]
    rows += [([rng.choice(big) for _ in range(16)], [rng.choice(edge) for _ in range(16)]) for _ in range(3000)]
    rows += [([rng.randrange(P) for _ in range(16)], [rng.randrange(P) for _ in range(16)]) for _ in range(3000)]
    data = b"".join(struct.pack("<32I", *x, *e) for x, e in rows)
    got = subprocess.run([binary], input=data, capture_output=True, check=True).stdout
    assert len(got) == 16 * len(rows)
    for (x, e), (canon, dig, want_dig, in_bounds) in zip(rows, struct.iter_unpack("<4I", got)):
        want = sum(a * b for a, b in zip(x, e)) % P
        assert canon == want and in_bounds
        # the digit word of the unreduced value stands for the same residue, top byte included
        s = [((dig >> (8 * j)) & 0xFF) - 256 * ((dig >> (8 * j + 7)) & 1) for j in range(4)]
        assert from_digits(s) == want
        t = [((want_dig >> (8 * j)) & 0xFF) - 256 * ((want_dig >> (8 * j + 7)) & 1) for j in range(4)]
        assert from_digits(t) == want
