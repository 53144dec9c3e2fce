"""The graph-tagged one-workgroup refinement is closed: a case with levels of up
to 16,384 vertices ended in a GPU fault of unknown cause. Its setting is still
accepted, and no kernel is left that it could reach."""
import os

import pytest

import jet_amd


@pytest.mark.parametrize("value", [0, 2048, 16384, 1 << 20])
def test_setting_is_accepted(value, tmp_path):
    old = jet_amd.tuning_get("batch_wg_max_n")
    with jet_amd.tuned(batch_wg_max_n=value):
        assert jet_amd.tuning_get("batch_wg_max_n") == value
    table = tmp_path / "table.txt"
    table.write_text(f"batch_wg_max_n {value}\n")
    jet_amd.tuning_load(str(table))
    assert jet_amd.tuning_get("batch_wg_max_n") == value
    jet_amd.tuning_set("batch_wg_max_n", old)


def test_no_tagged_kernel_in_the_library():
    path = os.path.join(os.path.dirname(os.path.dirname(jet_amd.__file__)), "libjet_amd.so")
    with open(path, "rb") as f:
        assert b"k_refine_wg" not in f.read()
