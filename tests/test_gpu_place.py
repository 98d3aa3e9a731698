"""Placement takes up to 1024 draw groups at a time and settles their victims
together; a device search must place as the sequential rule does, restated
over the owner seam (test_gpu_owner.drive): one to 64 draws a group, groups
that place nothing, members taken several times in a chunk, more than one
chunk, and keys in LDS and in memory."""
import json
import os

import pytest

import gagp_amd
import test_gpu_owner
from _util import GOLDEN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("population,batch,draws,generations,task", [
    (2, 2, 1, 6, "polynomial"), (3, 3, 2, 5, "polynomial"), (64, 64, 1, 4, "polynomial"), (65, 65, 64, 3, "quintic"),
    (300, 100, 3, 3, "poly_c1"), (1024, 1024, 4, 2, "polynomial"), (2050, 1025, 2, 2, "polynomial"), (9000, 3000, 5, 1, "polynomial")])
def test_device_placement_is_the_sequential_rule(population, batch, draws, generations, task, tmp_path, monkeypatch):
    print("placement", population, batch, draws, task, flush=True)
    search = json.load(open(os.path.join(GOLDEN, "search", "steady_batch_rs3.json")))
    search.update(population_size=population, schedule={"mode": "steady_state", "replacement_size": draws, "batch": batch})
    config = tmp_path / "search.json"
    config.write_text(json.dumps(search))
    path = os.path.join(GOLDEN, "tasks", task, "task.json")
    b = gagp_amd.Batch()
    b.add(path, str(config), population, generations, 11)
    b.run()
    result = b.result(0)
    (tmp_path / "result.json").write_text(json.dumps(result))
    monkeypatch.setitem(test_gpu_owner.MANIFEST, str(tmp_path), {
        "population": population, "generations": generations, "seed": 11, "task": path, "search": str(config)})
    history, best = test_gpu_owner.drive(str(tmp_path))
    for got, want in zip(result["history"], history):
        assert {k: got[k] for k in want} == want
    assert result["best"]["program"] == best["program"]
