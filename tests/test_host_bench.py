"""The benchmark reads a stage left to the library's rule (-1, from the autotuner or --set) as unpinned."""
import pytest

from exciting_amd import autotune


class _Context:
    """Two variants a stage; the library's rule (-1) is as fast as the best of them."""

    def __init__(self):
        self.pinned = {}

    def num_variants(self, stage):
        return 2

    def set_variant(self, stage, v):
        self.pinned[stage] = v

    def set_timing(self, on):
        pass

    def read_timing(self):
        return {st: (1.0 if v == 1 else 2.0, 1) for st, v in self.pinned.items()}


def test_stage_left_to_the_rule_is_unpinned(monkeypatch):
    import bench
    import torch
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(autotune, "_whole", lambda *a: 1.0)
    ctx = _Context()
    tuned = autotune.tune(ctx, ["bmt", "crtgemm"], lambda: None, reps=1)
    assert tuned == {"bmt": -1, "crtgemm": -1} == ctx.pinned
    for stage in tuned:
        assert bench.pinned(tuned, stage) is None
    assert bench.pinned(None, "bmt") is None and bench.pinned({}, "bmt") is None and bench.pinned({"bmt": 0}, "bmt") == 0


@pytest.mark.parametrize("ngps,tuned,name", [([1200] * 8, {"crtgemm": -1}, "crt_gemm_pipe_kernel"),
                                             ([1200] * 8, None, "crt_gemm_pipe_kernel"),
                                             ([1200] * 8, {"crtgemm": 4}, "crt_gemm_kernel"),
                                             ([500] * 8, {"crtgemm": -1}, "crt_gemm_kernel"),
                                             ([500] * 8, {"crtgemm": 8}, "crt_gemm_pipe_kernel")])
def test_residue_gemm_named_by_the_rule(ngps, tuned, name):
    import bench
    assert bench.crt_gemm_name(ngps, bench.pinned(tuned, "crtgemm")) == name
