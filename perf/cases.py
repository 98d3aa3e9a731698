"""The calls whose speed this repository is measured by.

Two boundaries of the library carry its users' work. `gagp_session_eval`
scores a caller's bytecode programs on a fixed case set (a host search loop's
fitness call), and `Batch` / `Server` run whole searches from task files, one
at a time, as one batch, or as a stream of requests. Inputs and results of
both live on the host, so a pass is the whole call: documents or program
tables in, scores or result documents out.

    listed()           the cases, with what each stands for
    draw(rng)          one more case of the same ranges
    prepare(case, s)   inputs of seed s: task files, programs, the session
    run(state)         one pass; returns the published numbers
    work(case)         bytes and VM operations one pass cannot do without
    exact(case, s)     evaluation results in 64 bits, without this library
"""
import ctypes
import json
import math
import os
import random
import tempfile

import numpy as np

import gagp_amd
from gagp_amd import workloads

# Bytecode opcodes and builtins (include/gagp_hip.h takes the ISA's numbers).
PUSH, LOAD, STORE, NEG, ADD, SUB, MUL, LT, GT, JMP, JIF, CALL, RET = 0, 1, 2, 3, 5, 6, 7, 10, 12, 16, 17, 19, 20
B_ABS, B_MIN, B_MAX, B_LEN, B_INDEX, B_IMOD0 = 0, 1, 2, 4, 7, 14
PENALTY = 1000.0
TEXT = 4096  # characters a published program's text is padded to


def listed():
    return [
        # A caller checks a handful of candidate formulas: latency and launches.
        dict(name="eval_few", kind="eval", programs=16, cases=21, inputs=1, nodes=15, lists=False, discounted=False),
        # One generation of a host-side search: a large ragged population.
        dict(name="eval_generation", kind="eval", programs=4001, cases=777, inputs=2, nodes=47, lists=False, discounted=False),
        # Fractional scores: totals in the canonical rounding order.
        dict(name="eval_discounted", kind="eval", programs=1000, cases=600, inputs=1, nodes=31, lists=False, discounted=True),
        # Programs with loops and branches over Int lists of uneven length.
        dict(name="eval_lists", kind="eval", programs=512, cases=200, inputs=1, nodes=21, lists=True, discounted=False),
        # A first try of a task: the smallest search anyone runs.
        dict(name="search_first_try", kind="search", task="poly", searches=1, population=100, generations=10, cases=21,
             discounted=False, schedule="steady"),
        # The reference's example size, a user's everyday search.
        dict(name="search_poly", kind="search", task="poly", searches=1, population=1024, generations=64, cases=21,
             discounted=False, schedule="steady"),
        # The larger symbolic regression of the benchmark.
        dict(name="search_quintic", kind="search", task="quintic", searches=1, population=4096, generations=128, cases=256,
             discounted=False, schedule="steady"),
        # The loop-heavy search: one traversal per program.
        dict(name="search_lists", kind="search", task="lists", searches=1, population=8192, generations=64, cases=200,
             discounted=False, schedule="steady"),
        # Statement programs (assignments, for_range, if) at an ordinary odd size.
        dict(name="search_statements", kind="search", task="statements", searches=1, population=1500, generations=48, cases=130,
             discounted=False, schedule="steady"),
        # The generational schedule with elites and discounted scores, many cases.
        dict(name="search_generational", kind="search", task="quintic", searches=1, population=1000, generations=40, cases=600,
             discounted=True, schedule="generational"),
        # Many independent searches of uneven size in one batch.
        dict(name="batch_mixed", kind="search", task="mixed", searches=64, population=4096, generations=64, cases=1024,
             discounted=False, schedule="steady"),
        # A burst of requests served with early exit.
        dict(name="serve_burst", kind="serve", searches=32, population=8192, generations=160, cases=1024),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["eval", "eval", "eval_lists", "poly", "quintic", "lists", "statements", "mixed", "serve"])
    if kind in ("eval", "eval_lists"):
        lists = kind == "eval_lists"
        return dict(kind="eval", programs=_log_int(rng, 8, 700 if lists else 4500), cases=_log_int(rng, 5, 400 if lists else 1200),
                    inputs=1 if lists else rng.choice([1, 2, 3]), nodes=rng.randint(7, 25 if lists else 60), lists=lists,
                    discounted=rng.random() < 0.3)
    if kind == "serve":
        return dict(kind="serve", searches=rng.randint(3, 20), population=_log_int(rng, 512, 8192),
                    generations=rng.randint(40, 160), cases=_log_int(rng, 32, 1024))
    if kind == "mixed":
        return dict(kind="search", task="mixed", searches=rng.randint(2, 40), population=_log_int(rng, 300, 4096),
                    generations=rng.randint(8, 64), cases=_log_int(rng, 20, 1024), discounted=False, schedule="steady")
    heavy = kind in ("lists", "statements")
    return dict(kind="search", task=kind, searches=1, population=_log_int(rng, 64, 6000 if heavy else 9000),
                generations=rng.randint(6, 64 if heavy else 100), cases=_log_int(rng, 10, 260 if heavy else 900),
                discounted=rng.random() < 0.3, schedule=rng.choice(["steady", "steady", "batches", "generational"]))


# ---- programs for the evaluation boundary ----
# A program is built as a tree, (op, children...) with leaves ("in", k),
# ("const", v), and inside a list fold ("acc",), ("elem",), ("index",); the
# tree gives both the bytecode and the 64-bit reference value.
def _tree(rng, size, leaves, branches):
    if size <= 1:
        return rng.choice(leaves)(rng)
    if size == 2:
        return (rng.choice(["neg", "abs"]), _tree(rng, 1, leaves, branches))
    if branches and size >= 7 and rng.random() < 0.3:
        a = rng.randint(1, size - 6)
        b = rng.randint(1, size - 5 - a)
        c = rng.randint(1, size - 4 - a - b)
        return ("if", _tree(rng, a, leaves, branches), _tree(rng, b, leaves, branches), _tree(rng, c, leaves, branches),
                _tree(rng, max(1, size - 2 - a - b - c), leaves, branches))
    op = rng.choices(["add", "sub", "mul", "min", "max", "mod"], [4, 4, 3, 1, 1, 1])[0]
    a = rng.randint(1, size - 2)
    return (op, _tree(rng, a, leaves, branches), _tree(rng, size - 1 - a, leaves, branches))


_BINARY = {"add": (ADD, None), "sub": (SUB, None), "mul": (MUL, None), "min": (CALL, B_MIN), "max": (CALL, B_MAX),
           "mod": (CALL, B_IMOD0)}


def _emit(t, code, consts, slots):
    """Appends the tree's instructions: (op, a, b), None where an operand is absent."""
    op = t[0]
    if op == "const":
        consts.append(t[1])
        code.append((PUSH, len(consts) - 1, None))
    elif op in slots:
        code.append((LOAD, slots[op], None))
    elif op == "in":
        code.append((LOAD, t[1], None))
    elif op in ("neg", "abs"):
        _emit(t[1], code, consts, slots)
        code.append((NEG, None, None) if op == "neg" else (CALL, B_ABS, 1))
    elif op == "if":  # if t1 > t2 then t3 else t4
        _emit(t[1], code, consts, slots)
        _emit(t[2], code, consts, slots)
        code.append((GT, None, None))
        at = len(code)
        code.append(None)
        _emit(t[3], code, consts, slots)
        out = len(code)
        code.append(None)
        code[at] = (JIF, len(code), None)
        _emit(t[4], code, consts, slots)
        code[out] = (JMP, len(code), None)
    else:
        _emit(t[1], code, consts, slots)
        _emit(t[2], code, consts, slots)
        o, b = _BINARY[op]
        code.append((o, b, 2) if o == CALL else (o, None, None))


def _fold_code(init, body):
    """fold(xs, init, body): a counted loop over the list input 0."""
    code, consts = [], [init, 0, 1]
    acc, i, e = 1, 2, 3
    code += [(PUSH, 0, None), (STORE, acc, None), (PUSH, 1, None), (STORE, i, None)]
    head = len(code)
    code += [(LOAD, i, None), (LOAD, 0, None), (CALL, B_LEN, 1), (LT, None, None)]
    exit_at = len(code)
    code += [None, (LOAD, 0, None), (LOAD, i, None), (CALL, B_INDEX, 2), (STORE, e, None)]
    _emit(body, code, consts, {"acc": acc, "index": i, "elem": e})
    code += [(STORE, acc, None), (LOAD, i, None), (PUSH, 2, None), (ADD, None, None), (STORE, i, None), (JMP, head, None)]
    code[exit_at] = (JIF, len(code), None)
    code += [(LOAD, acc, None), (RET, None, None)]
    return code, consts, 4


def _trees(case, seed):
    rng = random.Random(seed * 1000003 + 17)
    const = lambda r: ("const", r.randint(0, 9))  # noqa: E731
    if case["lists"]:
        leaves = [lambda r: ("acc",), lambda r: ("elem",), lambda r: ("elem",), lambda r: ("index",), const]
        return [(rng.choice([0, 1, -1001]), _tree(rng, rng.randint(3, case["nodes"]), leaves, True))
                for _ in range(case["programs"])]
    leaves = [(lambda k: lambda r: ("in", k))(k) for k in range(case["inputs"])] * 2 + [const]
    return [_tree(rng, rng.randint((case["nodes"] + 1) // 2, case["nodes"]), leaves, False) for _ in range(case["programs"])]


def _case_values(case, seed):
    """(scalar inputs [cases][inputs] or the lists, answers) of a seed."""
    rng = np.random.RandomState((seed * 31 + 7) % (1 << 32))
    n = case["cases"]
    if case["lists"]:
        xs = [rng.randint(-1000, 1001, rng.randint(0, 51)).astype(np.int64) for _ in range(n)]
        return xs, np.array([int(x[x % 2 == 0].sum()) for x in xs], dtype=np.int64)
    x = rng.randint(-50, 51, (n, case["inputs"])).astype(np.int64)
    return x, 3 * x[:, 0] ** 3 - 2 * x[:, -1] ** 2 + x[:, 0] - 7


class _Programs:
    """gagp_program table over numpy arrays laid out like the C structs."""

    INSTR = np.dtype([("op", "u1"), ("has_a", "u1"), ("has_b", "u1"), ("pad", "u1"), ("a", "i4"), ("b", "i4")])
    VALUE = np.dtype([("i", "i8"), ("b", "u1"), ("tag", "u1"), ("pad", "u1", 6)])

    def __init__(self, programs):
        self.n = len(programs)
        self.code = np.zeros(sum(len(c) for c, _, _ in programs), self.INSTR)
        self.code[:] = [(op, a is not None, b is not None, 0, a or 0, b or 0) for c, _, _ in programs for op, a, b in c]
        self.consts = np.zeros(sum(len(k) for _, k, _ in programs) + 1, self.VALUE)
        self.consts["i"][:-1] = [v for _, k, _ in programs for v in k]
        self.table = (gagp_amd.Program * self.n)()
        at = pool = 0
        for row, (c, k, n_locals) in zip(self.table, programs):
            row.code = ctypes.cast(self.code.ctypes.data + at * self.INSTR.itemsize, ctypes.POINTER(gagp_amd.Instr))
            row.code_len = len(c)
            row.consts = ctypes.cast(self.consts.ctypes.data + pool * self.VALUE.itemsize, ctypes.POINTER(gagp_amd.Value))
            row.n_consts, row.n_locals = len(k), n_locals
            at, pool = at + len(c), pool + len(k)


def _prepare_eval(case, seed):
    programs = []
    for t in _trees(case, seed):
        if case["lists"]:
            programs.append(_fold_code(*t))
        else:
            code, consts = [], []
            _emit(t, code, consts, {})
            programs.append((code + [(RET, None, None)], consts, case["inputs"]))
    x, answers = _case_values(case, seed)
    arena, inputs = [], []
    if case["lists"]:
        for v in x:
            inputs.append([("list", len(arena), len(v))])
            arena.extend(int(e) for e in v)
    else:
        inputs = [[int(v) for v in row] for row in x]
    session = gagp_amd.Session(inputs, [int(a) for a in answers], fuel=8192, arena=arena, penalty=PENALTY,
                               proximity=1 if case["discounted"] else 0)
    return {"kind": "eval", "session": session, "programs": _Programs(programs), "lib": gagp_amd.lib()}


def _run_eval(state):
    n = state["programs"].n
    fitness, wrong, counts = np.empty(n, np.float64), np.empty(n, np.uint32), np.empty((n, 3), np.uint32)
    status = state["lib"].gagp_session_eval(
        state["session"].h, state["programs"].table, n, fitness.ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
        wrong.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)), counts.ctypes.data_as(ctypes.POINTER(ctypes.c_uint32)))
    if status != gagp_amd.GAGP_OK:
        raise gagp_amd.GagpError(status, state["lib"].gagp_last_error().decode())
    return {"fitness": fitness, "wrong": wrong.astype(np.int64), "counts": counts.astype(np.int64)}


# ---- searches ----
def _int_cases(rng, coeffs, n, reach):
    out = []
    for _ in range(n):
        x = rng.randint(-reach, reach)
        out.append({"inputs": {"x": {"type": "int", "value": x}},
                    "expected": {"type": "int", "value": sum(c * x ** k for k, c in enumerate(coeffs))}})
    return out


def _task(directory, case, seed):
    """Writes the case's task documents; returns [(task, population)]."""
    rng = random.Random(seed * 7919 + 3)
    if case["task"] == "mixed":
        return workloads.mixed_searches(directory, n=case["searches"], seed=seed, p_range=(256, case["population"]),
                                        c_range=(16, case["cases"]), lists=True)
    if case["task"] in ("lists", "statements"):
        kind = "sum_even" if case["task"] == "lists" else "count_gt"
        task = workloads.list_task(directory, kind, seed, case["cases"], 2 * case["cases"], 50,
                                   fold="traverse" if case["task"] == "lists" else "statement")
    else:
        quintic = case["task"] == "quintic"
        coeffs = [rng.randint(-5, 5) for _ in range(5 if quintic else 3)] + [rng.choice([-2, -1, 1, 2])]
        reach = 50 if quintic else 10
        grammar = workloads.polynomial_grammar(range(10), 64, 12) if quintic else workloads.polynomial_grammar([1, 2], 31, 8)
        task = workloads.write_task(directory, case["task"], grammar, _int_cases(rng, coeffs, case["cases"], reach),
                                    _int_cases(rng, coeffs, 2 * case["cases"], 2 * reach))
    if case["discounted"]:
        doc = json.load(open(task))
        doc["fitness"] = {"metric": "absolute", "proximity": "discounted"}
        json.dump(doc, open(task, "w"))
    return [(task, case["population"])]


def _search_document(directory, case):
    """The search configuration file of a schedule (None: the built-in default)."""
    population = case["population"]
    if case["schedule"] == "steady":
        return None
    if case["schedule"] == "batches":  # four rounds per generation where the population divides, three draws per victim
        batch = population // 4 if population % 4 == 0 else population
        schedule = {"mode": "steady_state", "replacement_size": 3, "batch": batch}
    else:
        schedule = {"mode": "generational"}
    path = os.path.join(directory, "search.json")
    with open(path, "w") as f:
        json.dump({"format": "gagp-search-config-v1", "representation": "resident", "population_size": population,
                   "generations": case["generations"], "selection": {"method": "tournament", "size": 3}, "elitism": 3,
                   "crossover": {"probability": 0.9, "attempts": 4}, "mutation": {"probability": 0.4},
                   "sites": {"scope": "uniform_phase", "draw": "counted"}, "limits": {"site_depth": 7},
                   "ranking": {"tie_break": "ast_nodes"}, "schedule": schedule}, f)
    return path


def _prepare_search(case, seed):
    tmp = tempfile.TemporaryDirectory()
    return {"kind": "search", "tmp": tmp, "tasks": _task(tmp.name, case, seed), "generations": case["generations"],
            "search": _search_document(tmp.name, case), "seed": seed % (1 << 31)}


def _published(results, generations):
    """The result documents' numbers and program texts, one row per search."""
    n = len(results)
    out = {k: np.zeros((n, generations), np.float64) for k in ("best_fitness", "mean_fitness")}
    out.update({k: np.zeros((n, generations), np.int64) for k in ("best_wrong", "best_nodes")})
    out["best"] = np.zeros((n, 4), np.int64)
    out["fitness"], out["test_loss"] = np.zeros(n, np.float64), np.zeros(n, np.float64)
    out["text"] = np.zeros((n, TEXT), np.uint8)
    for i, r in enumerate(results):
        for g, row in enumerate(r["history"]):
            for k in ("best_fitness", "mean_fitness", "best_wrong", "best_nodes"):
                out[k][i, g] = row[k]
        best, test = r["best"], r["test"]
        out["best"][i] = int(best["wrong"]), int(best["nodes"]), int(test["correct"]), len(r["history"])
        out["fitness"][i], out["test_loss"][i] = best["fitness"], test["mean_loss"]
        text = np.frombuffer(best["text"].encode()[:TEXT], np.uint8)
        out["text"][i, :len(text)] = text
    return out


def _run_search(state):
    batch = gagp_amd.Batch()
    for i, (task, population) in enumerate(state["tasks"]):
        batch.add(task, state["search"], population, state["generations"], state["seed"] + i)
    batch.run()
    return _published([batch.result(i) for i in range(len(state["tasks"]))], state["generations"])


def _prepare_serve(case, seed):
    tmp = tempfile.TemporaryDirectory()
    requests = workloads.served_requests(tmp.name, n=case["searches"], seed=seed, p_range=(256, case["population"]),
                                         c_range=(16, case["cases"]), g_range=(32, case["generations"]), lists=True)
    return {"kind": "serve", "tmp": tmp, "requests": requests, "generations": case["generations"]}


def _run_serve(state):
    server = gagp_amd.Server()
    tickets = [server.submit(task, None, population, generations, seed, True, 0.0)
               for task, population, generations, seed, _ in state["requests"]]
    server.run()
    return _published([server.result(t) for t in tickets], state["generations"])


def prepare(case, seed):
    return {"eval": _prepare_eval, "search": _prepare_search, "serve": _prepare_serve}[case["kind"]](case, seed)


def run(state):
    return {"eval": _run_eval, "search": _run_search, "serve": _run_serve}[state["kind"]](state)


def work(case):
    """Bytes: the case set and the program or population rows read once, the
    scores or rows written once. Operations: VM instructions of the programs
    over the cases (a mean program of each grammar; a list program runs its
    body once per element of a mean list)."""
    if case["kind"] == "eval":
        length = case["nodes"] / 2 + 2 if case["lists"] else 0.75 * case["nodes"]
        executed = 25 * (length + 13) if case["lists"] else length
        values = case["cases"] * (26 if case["lists"] else case["inputs"] + 1)
        return {"bytes": 16 * values + case["programs"] * (12 * (length + 1) + 16 * length / 3 + 24),
                "flops": case["programs"] * case["cases"] * executed}
    # Uneven batches: log-uniform sizes have about a third of the range's top as their mean.
    scale = 1 / 3 if case["kind"] == "serve" or case["task"] == "mixed" else 1
    searches, members = case["searches"], case["population"] * scale
    cases, generations = case["cases"] * scale, case["generations"] * (0.4 if case["kind"] == "serve" else 1)
    nodes = 15 if case["kind"] == "search" and case["task"] == "poly" else 25
    loops = {"lists": 1, "statements": 1, "mixed": 0.5}.get(case.get("task"), 0) if case["kind"] == "search" else 0.5
    executed = nodes * (1 - loops) + 25 * nodes * loops
    # Rows (origin, site, constants) read and written once per child; a third of the children need scoring.
    return {"bytes": searches * (40 * cases + generations * members * 2 * 12 * nodes),
            "flops": searches * generations * members * cases * executed / 3}


# ---- the evaluation boundary in 64 bits ----
def _value(t, x, env):
    op = t[0]
    if op == "const":
        return np.int64(t[1])
    if op == "in":
        return x[:, t[1]]
    if op in env:
        return env[op]
    if op == "neg":
        return -_value(t[1], x, env)
    if op == "abs":
        return np.abs(_value(t[1], x, env))
    a, b = _value(t[1], x, env), _value(t[2], x, env)
    if op == "if":
        return np.where(a > b, _value(t[3], x, env), _value(t[4], x, env))
    if op == "mod":
        return np.where(b == 0, 0, np.mod(a, np.where(b == 0, 1, b)))
    return {"add": np.add, "sub": np.subtract, "mul": np.multiply, "min": np.minimum, "max": np.maximum}[op](a, b)


def exact(case, seed):
    if case["kind"] != "eval":
        return None  # a whole search on a host takes minutes
    x, answers = _case_values(case, seed)
    n = case["cases"]
    fitness, wrong = np.zeros(case["programs"]), np.zeros(case["programs"], np.int64)
    if case["lists"]:
        length = np.array([len(v) for v in x])
        padded = np.zeros((n, max(1, length.max())), np.int64)
        for i, v in enumerate(x):
            padded[i, :len(v)] = v
    with np.errstate(all="ignore"):
        for k, t in enumerate(_trees(case, seed)):
            if case["lists"]:
                y = np.full(n, t[0], np.int64)
                for i in range(int(length.max())):
                    env = {"acc": y, "index": np.full(n, i, np.int64), "elem": padded[:, i]}
                    y = np.where(i < length, _value(t[1], x, env), y)
            else:
                y = np.broadcast_to(_value(t, x, {}), (n,))
            hi, lo = np.maximum(y, answers), np.minimum(y, answers)
            gap = (hi.astype(np.uint64) - lo.astype(np.uint64)).astype(np.float64)
            score = gap / (1.0 + gap) if case["discounted"] else np.minimum(gap, PENALTY)
            fitness[k] = -math.fsum(score)
            wrong[k] = int((y != answers).sum())
    return {"fitness": fitness, "wrong": wrong, "counts": np.array([[n, 0, 0]] * case["programs"], dtype=np.int64)}
