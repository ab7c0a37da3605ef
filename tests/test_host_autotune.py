"""The tuned table keeps no entry for a stage left to the library's rule (-1)."""
from exciting_amd import autotune


def test_save_takes_out_stages_left_to_the_rule(tmp_path):
    p = tmp_path / "t.json"
    autotune.save(p, "N256-naa8-natm1", {"bmt": 2, "olp": 3})
    autotune.save(p, "N256-naa8-natm1", {"bmt": -1, "bsplit": 1})
    assert autotune.load(p, "N256-naa8-natm1") == {"olp": 3, "bsplit": 1}
    autotune.save(p, "N256-naa8-natm1", {"olp": -1, "bsplit": -1})
    assert autotune.load(p, "N256-naa8-natm1") == {}
