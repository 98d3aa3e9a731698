"""The device memory a server admits a search by (CPU): the looping path's
steps take the place of its programs' code, so a search asks for what it did
when that path interpreted the code itself (bytes planned then)."""
import os

import pytest

import gagp_amd
from _util import GOLDEN


@pytest.mark.parametrize("task,population,before", [
    ("let-sum", 8192, 66060288), ("list-sum", 1024, 7340032), ("list-sum", 8192, 66060288), ("list_count_gt_rev", 100, 1048576),
    ("list_count_gt_rev", 8192, 135266304), ("list_max_range", 1024, 15728640), ("list_range_nested", 8192, 135266304),
    ("list_sum_even", 100, 1048576), ("list_sum_even", 8192, 144179200), ("stmt_count_gt", 8192, 269484032), ("stmt_input", 1024, 15728640),
    ("stmt_sum_even", 8192, 278396928), ("polynomial", 8192, 66060288), ("quintic_wide", 8192, 282066944)])
def test_admission_is_what_it_was(task, population, before):
    batch = gagp_amd.Batch()
    planned = batch.planned_bytes(batch.add(os.path.join(GOLDEN, "tasks", task, "task.json"), None, population, 32, 1))
    assert planned == before
