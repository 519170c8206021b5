"""The kick walk's tile over a batch of isothermal and adiabatic members does not
depend on their order, and a batch of one kind has one tile for all (host code:
tests/cpp/tile_rules)."""
import os
import random
import subprocess

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "tile_rules.bin")


def _tiles(members):
    if not os.path.exists(EXE):
        from fargocpt_amd import build
        build.build_host_check()
    out = subprocess.run([EXE, *(str(v) for m in members for v in m)], capture_output=True, text=True, check=True)
    return [tuple(map(int, line.split())) for line in out.stdout.splitlines()]


def test_order():
    rng = random.Random(1)
    for _ in range(40):
        members = [(rng.randint(8, 512), rng.randint(4, 1536), rng.randint(0, 1)) for _ in range(rng.randint(2, 24))]
        tiles = _tiles(members)
        assert len({t for pair in tiles for t in pair}) == 1, (members, tiles)
