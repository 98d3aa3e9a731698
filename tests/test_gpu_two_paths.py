"""Programs of a search whose cases leave inputs out, and of a grammar whose
only list operations are len and index, scored by the owner seam twice: on the
task's cases, where the looping path runs them, and on the same cases repeated
to above 4096, where the general VM does. The draws do not read the cases, so
the programs are the same, and with integer losses every score and count is
the repetition's multiple. Initial population and one batch of children."""
import json
import os

import pytest

import gagp_amd
from _util import GOLDEN, strip_timing
from test_looping_grammar import reads_only

pytestmark = pytest.mark.gpu
REPEAT = 42  # 100 cases: two tiles, the second part full


def task_of(directory, name, edit):
    base = os.path.join(GOLDEN, "tasks", name)
    grammar = json.load(open(os.path.join(base, "grammar.json")))
    cases = json.load(open(os.path.join(base, "train.cases.json")))["cases"]
    cases = [json.loads(json.dumps(c)) for c in (cases * (100 // len(cases) + 1))[:100]]
    edit(grammar, cases)
    paths = []
    for repeat in (1, REPEAT):
        out = directory / ("x%d" % repeat)
        out.mkdir()
        (out / "grammar.json").write_text(json.dumps(grammar))
        (out / "cases.json").write_text(json.dumps({"format_version": "fitness-cases", "cases": cases * repeat}))
        doc = json.load(open(os.path.join(base, "task.json")))
        doc.update(grammar="grammar.json", train="cases.json", test="cases.json")
        (out / "task.json").write_text(json.dumps(doc))
        paths.append(str(out / "task.json"))
    return paths


def scores(path, population):
    owner = gagp_amd.Owner(path, None, population, 17)
    first = owner.evaluate()
    owner.begin_steady(population)
    order = sorted(range(population), key=lambda m: (-first[0][m], m))
    selection = [0.0] * population
    for rank, m in enumerate(order):
        selection[m] = float(population - rank)
    reuse = owner.make_batch(selection, 2, 0.4, 99)
    return first, reuse, owner.evaluate_batch()


def same_scores(short, long, population):
    looping, general = scores(short, population), scores(long, population)

    def compare(got, want, rows):
        wrong = [i for i in rows if (REPEAT * got[0][i], REPEAT * got[1][i], [REPEAT * c for c in got[2][i]]) !=
                 (want[0][i], want[1][i], want[2][i])]
        assert not wrong, (len(wrong), [(i, got[0][i], want[0][i], got[1][i], want[1][i], got[2][i], want[2][i]) for i in wrong[:4]])
    compare(looping[0], general[0], range(population))
    scored = [b for b, member in enumerate(looping[1]) if member < 0]
    assert len(scored) > population // 10
    assert scored == [b for b, member in enumerate(general[1]) if member < 0], "the children differ"
    compare(looping[2], general[2], scored)


def unset(name):
    def edit(grammar, cases):
        for k, case in enumerate(cases):
            if k % 3:
                case["inputs"].pop(name)
    return edit


@pytest.mark.parametrize("task,name,population", [("stmt_input", "x", 2000), ("list_sum_even", "xs", 300), ("stmt_sum_even", "xs", 300)])
def test_unset_inputs_score_as_in_the_general_vm(task, name, population, tmp_path):
    print("two paths", task, flush=True)
    same_scores(*task_of(tmp_path, task, unset(name)), population)


def reads(grammar, cases):
    grammar.clear()
    grammar.update(reads_only())


def test_list_reads_without_a_jump_score_as_in_the_general_vm(tmp_path):
    print("two paths reads", flush=True)
    short, long = task_of(tmp_path, "list_sum_even", reads)
    same_scores(short, long, 300)
    # Alone and beside a search with loops, straight and batched rounds publish the same.
    results = []
    for beside in (None, os.path.join(GOLDEN, "tasks", "list_sum_even", "task.json")):
        batch = gagp_amd.Batch()
        batch.add(short, None, 300, 6, 5)
        if beside:
            batch.add(beside, None, 300, 6, 5)
        batch.run()
        results.append(strip_timing(batch.result(0)))
    assert results[0] == results[1]
