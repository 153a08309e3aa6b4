"""The tuning cache serves choices among the present kernels only (no GPU calls)."""
import numpy as np

from gf2_amd import _lib, autotune


class _Qc:
    base_matrix = np.array([[0, 1, -1], [2, -1, 0]])

    def expansion_factor(self):
        return 8


class _Code:
    qc = _Qc()

    def n(self):
        return 24

    def m(self):
        return 16


class _Context:
    def __init__(self):
        self.calls = []

    def set_path(self, v):
        self.calls.append(("path", v))

    def set_tuning(self, k, v):
        self.calls.append((k, v))


def test_entries_of_earlier_kernels_are_not_applied(tmp_path):
    cache, ctx, code = autotune.TuningCache(str(tmp_path / "t.json")), _Context(), _Code()
    key = autotune.shape_key([code], 100, "single")
    before = "single:n24-m16-z8-e4-dc2-dv2:F128"  # as it was before the key named the kernels
    assert key.startswith(before + ":")
    cache.put(before, {"path": _lib.PATH_STATE, "lds_groups": 5}, 1.0, 2)
    assert autotune.apply_cached(ctx, [code], 100, cache=cache) is None and ctx.calls == []
    cache.put(key, {"frame_kernel": 1}, 1.0, 2)
    assert autotune.apply_cached(ctx, [code], 128, cache=cache) == {"frame_kernel": 1}
    assert ctx.calls == [(_lib.TUNE_FRAME_KERNEL, 1)]
