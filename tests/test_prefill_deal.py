"""The dealing of pieces to the prefill queues (pf_dealt of mi_prefill_kernel.h), compiled for the host.

Every (piece, kv-head) pair must lie in exactly one place of one queue, and a
queue's pieces must come in list order, which is heaviest first.
"""

import ctypes
import re
import subprocess
from pathlib import Path

import pytest

KERNEL = Path(__file__).resolve().parents[1] / "mstar_amd" / "csrc" / "mi_prefill_kernel.h"


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    text = KERNEL.read_text()
    parts = [re.search(r"__host__ __device__ (inline \w+ %s\(.*?\n})" % name, text, re.S).group(1)
             for name in ("pf_dealt_len", "pf_dealt")]
    tmp = tmp_path_factory.mktemp("deal")
    (tmp / "deal.cpp").write_text("\n".join(parts) + """
extern "C" int len(int np, int nkv, int x) { return pf_dealt_len(np, nkv, x); }
extern "C" int at(int nkv, int x, int i) { int p, h; pf_dealt(nkv, x, i, p, h); return h << 20 | p; }
""")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", tmp / "deal.so", tmp / "deal.cpp"], check=True)
    return ctypes.CDLL(str(tmp / "deal.so"))


@pytest.mark.parametrize("nkv", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 16, 20, 24, 32, 40])
def test_every_piece_of_every_head_is_dealt_once(deal, nkv):
    for np_ in [*range(0, 40), 63, 64, 65, 255, 1000, 1033]:
        seen = []
        for x in range(8):
            n = deal.len(np_, nkv, x)
            queue = [deal.at(nkv, x, i) for i in range(n)]
            pieces = [q & 0xFFFFF for q in queue]
            assert pieces == sorted(pieces), (np_, nkv, x)
            seen += queue
        assert sorted(seen) == [h << 20 | p for h in range(nkv) for p in range(np_)], (np_, nkv)
