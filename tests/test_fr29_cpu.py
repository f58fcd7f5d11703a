"""Fr29 (signed 29-bit limbs of the transforms' butterflies) against Python
integers, on the CPU through a host driver built here (fr29_host_check.cpp):
chains as long as a pass runs without reducing, random and extreme operands."""

import os
import random
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
R = 0x30644E72E131A029B85045B68181585D2833E84879B9709143E1F593F0000001
INV256 = pow(1 << 256, -1, R)


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    hipcc = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
    if not os.path.exists(hipcc):
        hipcc = shutil.which("hipcc")
    if not hipcc:
        pytest.skip("hipcc is not installed")
    exe = str(tmp_path_factory.mktemp("fr29") / "fr29_host_check")
    src = os.path.join(HERE, "fr29_host_check.cpp")
    subprocess.run([hipcc, "-O2", "-std=c++17", "-x", "hip", "--offload-arch=gfx950", src, "-o", exe],
                   check=True, capture_output=True)
    return exe


@pytest.mark.parametrize("stages", [1, 2, 5, 11])
def test_butterfly_chains(driver, stages):
    rng = random.Random(stages)
    edge = [0, 1, R - 1, (1 << 256) % R, (R + 1) // 2, (1 << 253) - 1]

    def pick():
        return rng.choice(edge) if rng.random() < 0.3 else rng.randrange(R)

    chains = [(pick(), pick(), [pick() for _ in range(stages)]) for _ in range(400)]
    chains += [(a, b, [w] * stages) for a in edge for b in edge for w in edge]
    text = "".join(f"chain {a:064x} {b:064x} {len(ws)}\n" + "".join(f"{w:064x}\n" for w in ws) for a, b, ws in chains)
    r = subprocess.run([driver], input=text, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    lines = iter(r.stdout.split("\n"))
    for a, b, ws in chains:
        for i, w in enumerate(ws):
            t = b * w * INV256 % R
            a, b = ((a - t) % R, (a + t) % R) if i & 1 else ((a + t) % R, (a - t) % R)
            ga, gb, ok = next(lines).split()
            for got, want in ((int(ga, 16), a), (int(gb, 16), b)):
                assert got % R == want
                assert got < R + R // 5000  # reduce() ends below 1.0002 r
            assert ok == "1", "a limb left its bound"


def test_inverse(driver):
    rng = random.Random(5)
    xs = [0, 1, 2, R - 1, R - 2, (1 << 253), (1 << 256) % R, pow(2, -1, R), pow(2, -253, R)]
    xs += [rng.randrange(R) for _ in range(3000)]
    r = subprocess.run([driver], input="".join(f"inv {x:064x}\n" for x in xs), capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    for x, line in zip(xs, r.stdout.split("\n")):
        want = pow(x, -1, R) * (1 << 512) % R if x else 0
        assert [int(h, 16) % R for h in line.split()] == [want, want]
