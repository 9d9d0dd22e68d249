"""CPU: the rules that give a call its kernels (loki_amd/csrc/launch_rules.h), compiled as they are and checked over the sizes
that the entry points take."""
import ctypes
import os
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "loki_amd", "csrc", "launch_rules.h")
NS = sorted(set(list(range(1, 70)) + [n + d for n in (96, 128, 256, 400, 512, 1024, 2048, 4096, 65536) for d in (-1, 0, 1)]))
NEXPS = (8, 16, 31, 32, 33, 40, 64, 65, 96, 128, 160, 255, 256)


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, so = d / "rules.cpp", d / "rules.so"
    src.write_text('#include "%s"\n' % HEADER +
                   'extern "C" int parts(int n, int ne, int K) { return lk::router_parts(n, ne, K); }\n'
                   'extern "C" int split(int n, int P, int ne) { return lk::pf_split(n, P, ne); }\n'
                   'extern "C" int shared_tok(int n, int P) { return lk::split_shared_tok(n, P); }\n'
                   'extern "C" int few() { return lk::FEW_TOK; }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


def test_router_parts_fill_the_device(rules):
    """A split tile's parts depend on the number of 32 x 32 tiles, so a router of few experts runs on as many workgroups as
    one of 256 experts with the same number of tiles: at least 128 of them or the finest split. The parts' scratch stays
    within 8 MiB."""
    by_tiles = {}
    for ne in NEXPS:
        for n in NS:
            p = rules.parts(n, ne, 7168)
            tiles = -(-n // 32) * -(-ne // 32)
            assert p in (0, 2, 4, 8) and rules.parts(n, ne, 4096) == 0
            assert p * n * ne * 8 <= 8 << 20, (n, ne)
            if n < 21 or tiles > 512:
                assert p == 0, (n, ne)
                continue
            assert p == 8 or (p > 0 and p * tiles >= 128), (n, ne, p)
            assert by_tiles.setdefault(tiles, p) == p, (n, ne, p)


def test_split_tables_fit_their_scan(rules):
    """A split table's three totals share one 32-bit word (k_pf_cols): columns of 8 slots (11 bits), columns of 32 (11 bits) and
    experts of few slots (10 bits). The line between the tables goes by pairs and experts, so more experts never narrow it,
    a batch below it stays below with fewer pairs, and the shared expert's rows do not move it."""
    few = rules.few()
    for ne in NEXPS:
        inside = [P for P in range(1, 6000) if rules.split(0, P, ne)]
        assert inside == list(range(1, len(inside) + 1))
        top = inside[-1]
        assert top // few + ne < 1 << 11 and ne < 1 << 10, ne
        assert all(rules.split(n, top, ne) and not rules.split(n, top + 1, ne) for n in (0, 1, 500, 65536))
        assert ne == NEXPS[0] or rules.split(0, last, ne)
        last = top
    assert rules.split(300, 600, 256) and not rules.split(512, 4096, 256)   # 2 picks a row split, 8 not, whatever the rows
    for n in NS:
        assert rules.shared_tok(n, 0) in (8, 16, 32) and rules.shared_tok(n, 8 * n) == 32
