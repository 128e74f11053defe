"""One tile table: the library's indices (kTileCfgs), its kernel dispatch, the
interface's description and the benchmark's list name the same shapes, and
the shapes of earlier tables that survive keep their index."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _read(*p):
    with open(os.path.join(ROOT, *p)) as f:
        return f.read()


def _table():
    body = re.search(r"kTileCfgs\[\] = \{(.*?)\};", _read("emergence_amd", "csrc", "em_pass.h"), re.S).group(1)
    return [tuple(map(int, m)) for m in re.findall(r"\{(\d+), (\d+), (\d+)\}", body)]


def test_dispatch_header_and_benchmark_agree():
    table = _table()
    calls = re.findall(r"case (\d+): return CALL\((\d+), (\d+), (\d+)\);", _read("emergence_amd", "csrc", "em_pass.hip"))
    assert [tuple(map(int, c)) for c in calls] == [(i,) + t for i, t in enumerate(table)]
    names = re.search(r"axis x pencils (.*?)\)", _read("include", "em_hip.h"), re.S).group(1)
    assert re.findall(r"(\d+)x(\d+)", names) == [(str(t), str(p)) for t, p, _ in table]
    ns = {}
    exec(re.search(r"^TILE_SHAPES = \[.*?\]", _read("bench.py"), re.S | re.M).group(0), ns)
    assert ns["TILE_SHAPES"] == table
    for name, t, p, i in re.findall(r"(TILE_(\d+)x(\d+)) = (\d+)", _read("emergence_amd", "csrc", "em_pass.h")):
        assert table[int(i)][:2] == (int(t), int(p)), name


def test_surviving_shapes_keep_their_index():
    table = _table()
    assert table[4] == (27, 8, 256) and table[5] == (59, 4, 256) and table[8] == (123, 4, 512)
    assert table[1][:2] == (64, 8)
