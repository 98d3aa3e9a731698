"""A caller's looping programs on the decoded steps (gagp_session_eval with
jumps, hidden locals and IntList inputs) against the oracle: integers, counts
and canonical totals are equal, bit for bit. The programs fold a list with a
random body (if, mod, indexing that may fail, stores into the input), at case
counts on the edges of a 64-case tile and of a block's four tiles, with fuel
that runs out inside the loop, with unset inputs, with bodies above 64 steps,
and with programs outside the certificate in the same launch."""
import random

import pytest

import gagp_amd
from _util import oracle_fitness

pytestmark = pytest.mark.gpu

PUSH, LOAD, STORE, NEG, NOT, ADD, SUB, MUL, MOD, LT, GT, EQ, JMP, JF, JT, CALL, RET = (
    0, 1, 2, 3, 4, 5, 6, 7, 9, 10, 12, 14, 16, 17, 18, 19, 20)
MIN, MAX, CLIP, LEN, INDEX, IMOD0, NONNEG, CLAMPED = 1, 2, 3, 4, 7, 14, 30, 31
XS, Y, ACC, I, E = 0, 1, 2, 3, 4  # inputs xs, y; hidden acc, i, e


def expr(rng, depth, code, consts):
    def const(v):
        consts.append(v)
        code.append((PUSH, len(consts) - 1, None))
    if depth == 0:
        if rng.random() < 0.25:
            const(rng.choice([0, 1, 2, -1, 7, 2 ** 40, -(2 ** 63)]))
        else:
            code.append((LOAD, rng.choice([Y, ACC, I, E]), None))
        return
    kind = rng.randrange(9)
    if kind < 4:
        expr(rng, rng.randrange(depth), code, consts)
        expr(rng, rng.randrange(depth), code, consts)
        code.append((rng.choice([ADD, SUB, MUL, MOD]), None, None) if kind < 3 else (CALL, rng.choice([MIN, MAX, IMOD0]), 2))
    elif kind == 4:
        expr(rng, depth - 1, code, consts)
        code.append((NEG, None, None))
    elif kind == 5:  # an element by a computed index
        code.append((LOAD, XS, None))
        expr(rng, depth - 1, code, consts)
        code.append((CALL, rng.choice([CLAMPED, CLAMPED, INDEX, NONNEG]), 2))
    elif kind == 6:
        expr(rng, depth - 1, code, consts)
        const(-100)
        const(100)
        code.append((CALL, CLIP, 3))
    else:
        expr(rng, rng.randrange(depth), code, consts)
        expr(rng, rng.randrange(depth), code, consts)
        code.append((rng.choice([LT, GT, EQ]), None, None))
        if rng.random() < 0.3:
            code.append((NOT, None, None))
        jump = len(code)
        code.append(None)
        expr(rng, depth - 1, code, consts)
        end = len(code)
        code.append(None)
        code[jump] = (rng.choice([JF, JT]), len(code), None)
        expr(rng, depth - 1, code, consts)
        code[end] = (JMP, len(code), None)


def fold(rng, depth, boolean=False):
    code, consts = [(PUSH, 0, None), (STORE, ACC, None), (PUSH, 0, None), (STORE, I, None)], [0, 1]
    head = len(code)
    code += [(LOAD, I, None), (LOAD, XS, None), (CALL, LEN, 1), (LT, None, None)]
    leave = len(code)
    code += [None, (LOAD, XS, None), (LOAD, I, None), (CALL, INDEX, 2), (STORE, E, None)]
    expr(rng, depth, code, consts)
    code += [(STORE, ACC, None)]
    if rng.random() < 0.3:  # a store into an input: later loads read it
        code += [(LOAD, ACC, None), (STORE, Y, None)]
    code += [(LOAD, I, None), (PUSH, 1, None), (ADD, None, None), (STORE, I, None), (JMP, head, None)]
    code[leave] = (JF, len(code), None)
    code += [(LOAD, ACC, None)]
    if boolean:
        code += [(PUSH, 0, None), (GT, None, None)]
    return {"code": code + [(RET, None, None)], "consts": consts, "n_locals": 5}


@pytest.mark.parametrize("n_cases,fuel,proximity,unset", [
    (1, 4096, 0, False), (63, 4096, 0, False), (64, 600, 1, False), (65, 4096, 1, False), (257, 300, 0, False), (200, 4096, 0, True),
    (130, 9, 0, True)])
def test_looping_programs_match_the_oracle(n_cases, fuel, proximity, unset):
    rng = random.Random(n_cases * 31 + fuel)
    arena, inputs = [], []
    for _ in range(n_cases):
        n = rng.choice([0, 1, 2, 7, 30])
        inputs.append([("list", len(arena), n), rng.choice([0, 1, -1, rng.randrange(-10 ** 6, 10 ** 6)])])
        arena += [rng.randrange(-1000, 1001) for _ in range(n)]
    # Unset: y of every third case (None to the oracle).
    bound = [[True, k % 3 != 0] for k in range(n_cases)] if unset else None
    seen = [[xs, y if not unset or k % 3 else None] for k, (xs, y) in enumerate(inputs)]
    answers = [rng.randrange(-2000, 2000) for _ in range(n_cases)]
    programs = [fold(rng, rng.randrange(1, 6)) for _ in range(60)]
    programs += [fold(rng, 6) for _ in range(6)]  # most above 64 steps or outside the limits
    programs.append(dict(programs[0], n_locals=6))
    programs.append({"code": [(LOAD, E, None), (RET, None, None)], "consts": [], "n_locals": 5})  # an unset local: general VM
    want = oracle_fitness(programs, seen, answers, fuel=fuel, penalty=1000.0, lanes=512, proximity=proximity, arena=arena)
    s = gagp_amd.Session(inputs, answers, fuel=fuel, penalty=1000.0, proximity=proximity, arena=arena, input_set=bound)
    got = s.eval(programs)
    assert got[2] == want[2]
    assert got[1] == want[1]
    assert got[0] == want[0]
    assert s.eval(programs, allocate=False) == got
    # Programs that return Bools, against Bool answers.
    flags = [rng.random() < 0.5 for _ in range(n_cases)]
    bools = [fold(rng, rng.randrange(1, 4), boolean=True) for _ in range(20)]
    want = oracle_fitness(bools, seen, flags, fuel=fuel, penalty=1000.0, lanes=512, metric=2, arena=arena)
    s = gagp_amd.Session(inputs, flags, fuel=fuel, penalty=1000.0, metric=2, arena=arena, input_set=bound)
    assert tuple(s.eval(bools)) == tuple(want)
