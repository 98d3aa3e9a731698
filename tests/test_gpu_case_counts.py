"""Evaluation calls at the case counts where a block's LDS crosses 64 KB (the
scores of four programs beside their replay on the straight-line path, a
program's slots and scores on the looping one) and with more reduction lanes
than the replay holds at a time (512), against the oracle: discounted scores,
whose canonical totals are equal, bit for bit."""
import random

import pytest

import gagp_amd
from _util import oracle_fitness
from test_gpu_steps import ADD, GT, JF, JMP, LOAD, MUL, PUSH, RET, STORE, SUB

pytestmark = pytest.mark.gpu


def straight(rng):
    code = [(LOAD, rng.randrange(4), None)]
    for _ in range(rng.randrange(1, 6)):
        code += [(LOAD, rng.randrange(4), None), (rng.choice([ADD, SUB, MUL]), None, None)]
    return {"code": code + [(RET, None, None)], "consts": [], "n_locals": 4}


def branching(rng):
    code = [(LOAD, rng.randrange(4), None), (PUSH, 0, None), (GT, None, None), (JF, 6, None), (LOAD, rng.randrange(4), None), (JMP, 7, None),
            (LOAD, rng.randrange(4), None), (LOAD, rng.randrange(4), None), (rng.choice([ADD, SUB]), None, None), (RET, None, None)]
    return {"code": code, "consts": [rng.randrange(-9, 10)], "n_locals": 4}


@pytest.mark.parametrize("make,n_cases,lanes", [
    (straight, 1500, 512), (straight, 1520, 512), (straight, 1600, 513), (straight, 2048, 1500), (straight, 4096, 512),
    (branching, 3000, 512), (branching, 3300, 545), (branching, 3584, 1025), (branching, 4096, 512), (branching, 40, 1024)])
def test_case_counts_match_the_oracle(make, n_cases, lanes):
    print("case counts", make.__name__, n_cases, lanes, flush=True)
    rng = random.Random(n_cases + lanes)
    inputs = [[rng.randrange(-50, 51) for _ in range(4)] for _ in range(n_cases)]
    answers = [rng.randrange(-2000, 2000) for _ in range(n_cases)]
    programs = [make(rng) for _ in range(9)]
    want = oracle_fitness(programs, inputs, answers, fuel=1000, penalty=1000.0, lanes=lanes, proximity=1)
    got = gagp_amd.Session(inputs, answers, fuel=1000, lanes=lanes, penalty=1000.0, proximity=1).eval(programs)
    assert got == want


@pytest.mark.parametrize("depth,n_locals,n_cases", [(7, 5, 130), (17, 20, 64), (40, 25, 130), (40, 26, 130), (40, 27, 4096)])
def test_deep_stacks_beside_looping_programs(depth, n_locals, n_cases):
    # Stacks past the looping path run on the general VM in the launch of the
    # others, up to the LDS of a block (64 slots and locals) where each has its own.
    print("deep stacks", depth, n_locals, n_cases, flush=True)
    rng = random.Random(depth)
    deep = {"code": [(LOAD, 0, None), (STORE, n_locals - 1, None)] + [(LOAD, rng.randrange(4), None) for _ in range(depth)] +
            [(rng.choice([ADD, SUB]), None, None) for _ in range(depth - 1)] + [(LOAD, n_locals - 1, None), (ADD, None, None), (RET, None, None)],
            "consts": [], "n_locals": n_locals}
    inputs = [[rng.randrange(-50, 51) for _ in range(4)] for _ in range(n_cases)]
    answers = [rng.randrange(-200, 200) for _ in range(n_cases)]
    programs = [branching(rng) for _ in range(5)] + [deep] + [branching(rng) for _ in range(3)]
    want = oracle_fitness(programs, inputs, answers, fuel=1000, penalty=1000.0, lanes=512)
    session = gagp_amd.Session(inputs, answers, fuel=1000, lanes=512, penalty=1000.0)
    assert session.eval(programs) == want
    assert session.eval(programs[5:6]) == tuple(x[5:6] for x in want)
    assert session.eval(programs, allocate=False) == want
