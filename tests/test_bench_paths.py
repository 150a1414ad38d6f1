"""bench.py names the engine's path from the library's counts (no GPU needed)."""
import importlib.util
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


class _Ctx:
    def __init__(self, after):
        self.after = after

    def pair_paths(self):
        return self.after


@pytest.mark.parametrize("before,after,want", [((1, 0, 0), (4, 0, 0), "walk"), ((1, 0, 0), (1, 5, 0), "strips"),
                                               ((0, 2, 0), (0, 2, 1), "region tiles"), ((3, 1, 0), (3, 1, 0), "tile kernel"),
                                               ((0, 0, 0), (1, 1, 0), "walk and strips")])
def test_path_name(before, after, want):
    spec = importlib.util.spec_from_file_location("bench", ROOT / "bench.py")
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    assert bench.path_since(_Ctx(after), before) == want
