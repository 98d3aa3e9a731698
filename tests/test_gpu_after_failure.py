"""A call that a launch limit refuses fails alone: the next call in the process
is served as if there had been none."""
import json
import os

import pytest

import gagp_amd
from _util import GOLDEN, strip_timing

pytestmark = pytest.mark.gpu


def test_the_next_search_is_served(tmp_path):
    base = os.path.join(GOLDEN, "tasks", "stmt_sum_even")
    grammar = json.load(open(os.path.join(base, "grammar.json")))
    grammar["search_limits"]["max_depth"] = 60  # general VM stacks above a block's LDS
    (tmp_path / "grammar.json").write_text(json.dumps(grammar))
    doc = json.load(open(os.path.join(base, "task.json")))
    doc.update(grammar="grammar.json", train=os.path.join(base, doc["train"]), test=os.path.join(base, doc["test"]))
    (tmp_path / "task.json").write_text(json.dumps(doc))
    deep = gagp_amd.Batch()
    deep.add(str(tmp_path / "task.json"), None, 64, 2, 1)
    with pytest.raises(gagp_amd.GagpError):
        deep.run()
    del deep
    name = "polynomial_p100_g10_s5"
    m = json.load(open(os.path.join(GOLDEN, "runs", "manifest.json")))[name]
    b = gagp_amd.Batch()
    b.add(os.path.join(GOLDEN, m["task"]), None, m["population"], m["generations"], m["seed"])
    b.run()
    assert strip_timing(b.result(0)) == strip_timing(json.load(open(os.path.join(GOLDEN, "runs", name, "result.json"))))
