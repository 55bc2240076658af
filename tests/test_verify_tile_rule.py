"""verify_tiles.verify_tile (what the GPU tests name their tiles by) is the rule of
csrc/verify.hip: the C++ function, compiled for the host, gives the same tile for
random launches and at its lines."""

import os
import random
import re
import shutil
import subprocess

import pytest

from gdn_recoverssm_ascend._build import CSRC_DIR
from verify_tiles import verify_tile


def test_restated_rule(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    with open(os.path.join(CSRC_DIR, "verify.hip")) as f:
        body = re.search(r"^static int verify_tile\(.*?^}\n", f.read(), re.S | re.M).group(0)
    (tmp_path / "rule.cpp").write_text(
        "#include <cstdint>\n#include <cstdio>\n" + body +
        "int main() { long r, h, K, V; int f, q, d; while (scanf(\"%ld %ld %ld %ld %d %d %d\", &r, &h, &K, &V, &f, &q, &d) "
        "== 7) printf(\"%d\\n\", verify_tile(r, h, K, V, f, q, d)); }\n")
    exe = str(tmp_path / "rule")
    subprocess.run([cxx, "-O1", "-std=c++17", str(tmp_path / "rule.cpp"), "-o", exe], check=True)
    rng = random.Random(5)
    cases = []
    for _ in range(20000):
        rows = int(2 ** rng.uniform(0, 12))
        cases.append((rows, rng.choice([1, 2, 4, 8, 12, 16, 32, 64]), rng.choice([8, 64, 96, 128, 136, 256]),
                      rng.choice([1, 16, 17, 32, 33, 48, 64, 65, 96, 127, 128, 129, 160, 192, 193, 256, 1000]),
                      rng.randrange(2), rng.choice([1, 2, 4, 8]), rng.randrange(2)))
    text = "\n".join(" ".join(map(str, c)) for c in cases)
    got = subprocess.run([exe], input=text.encode(), check=True, stdout=subprocess.PIPE).stdout.split()
    assert [int(x) for x in got] == [verify_tile(*c) for c in cases]
    assert {(c[6], int(x)) for c, x in zip(cases, got)} == {(0, 16), (0, 64), (0, 128), (1, 16), (1, 32), (1, 64)}
