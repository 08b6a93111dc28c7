"""The work that a user of this library has it do, as timed cases: sumcheck proofs (and their verification), LogUp-GKR
fraction trees, a domain's whole proof, commitments and their openings, each through the package's public entry points.

Sizes are the configured workloads' (sable_amd/workloads.py), the tests' and the benchmark's; draw() spreads over the
ranges between the smallest calls of each kind and those.  Everything is exact integer work, so outputs are compared
bit for bit.  Inputs are made on the GPU and handed over as wrapped device tables; a statement, the committed columns'
codewords and a domain's description are what a program holds before the call.
"""
import ctypes as C

import numpy as np
import torch

import sable_amd as sa
from sable_amd import domain as sd

P = sa.P

# (form, tables, constants): the configured statements, and the point reductions of an opening for one and two points
STATEMENTS = {
    "product": ("(* t0 t1)", ["t0", "t1"], []),
    "degree3": ("(+ (* alpha t0 t1 t2) (* 3 t1))", ["t0", "t1", "t2"], ["alpha"]),
    "degree4": ("(* (+ c0 3) (- c1 c0) c2 c3)", ["c0", "c1", "c2", "c3"], []),
    "points2": ("(+ (* e0 g0) (* e1 g1))", ["e0", "g0", "e1", "g1"], []),
}


def listed():
    return [
        # the smallest proofs of a protocol: a sumcheck over a thousand entries, one of hundreds in a larger proof
        dict(name="sumcheck_n10", kind="sumcheck", statement="product", n=10, d=4, ext=False, verify=False),
        # the configured small sumcheck, proved and verified
        dict(name="sumcheck_n16_verified", kind="sumcheck", statement="product", n=16, d=4, ext=False, verify=True),
        # the benchmark's headline: three base tables of 2^24, degree 3
        dict(name="sumcheck_n24", kind="sumcheck", statement="degree3", n=24, d=4, ext=False, verify=False),
        # the largest: four base tables of 2^26, degree 4, the degree-8 extension
        dict(name="sumcheck_n26_fp8", kind="sumcheck", statement="degree4", n=26, d=8, ext=False, verify=False),
        # the point reduction of an opening: tables that are extension elements from the start
        dict(name="points_n19", kind="sumcheck", statement="points2", n=19, d=4, ext=True, verify=False),
        # the configured lookup argument: 2^22 lookups into a table of 2^16, the two fraction trees side by side
        dict(name="gkr_n22_n16", kind="gkr_pair", n=22, m=16, d=4),
        # a domain's fraction trees: several blocks, several lookups proved together
        dict(name="gkr_n14_3_blocks", kind="gkr", n=14, blocks=3, lookups=2, d=4),
        # a whole domain proof: leaves, fraction tree, zerocheck, column claims
        dict(name="domain_n16", kind="domain", n=16, blocks=1, d=4),
        # the configured commitment: two columns of 2^23
        dict(name="commit_2_c23", kind="commit", c=23, ncols=2),
        # an ordinary commitment of many short columns (a leaf's hash is chained beyond 64 columns)
        dict(name="commit_70_c14", kind="commit", c=14, ncols=70),
        # the opening of the configured commitment, a second size class joining on the way
        dict(name="open_c23", kind="open", classes="19x1 23x2", queries=6, verify=False),
        # an opening of short columns in three size classes, proved and verified
        dict(name="open_c14_verified", kind="open", classes="10x2 13x1 14x2", queries=7, verify=True),
    ]


def draw(rng):
    kind = rng.choice(["sumcheck", "sumcheck", "sumcheck", "gkr", "gkr_pair", "domain", "commit", "commit", "open", "open"])
    if kind == "sumcheck":
        statement = rng.choice(["product", "degree3", "degree4", "points2"])
        if statement == "points2":
            return dict(kind=kind, statement=statement, n=rng.randint(8, 21), d=4, ext=True, verify=rng.random() < 0.3)
        if statement == "degree4":
            return dict(kind=kind, statement=statement, n=rng.randint(12, 25), d=8, ext=False, verify=rng.random() < 0.3)
        d = rng.choice([4, 4, 8]) if statement == "product" else 4
        return dict(kind=kind, statement=statement, n=rng.randint(8, 24), d=d, ext=False, verify=rng.random() < 0.3)
    if kind == "gkr":
        return dict(kind=kind, n=rng.randint(8, 17), blocks=rng.choice([1, 2, 3, 5]), lookups=rng.choice([1, 2, 3]), d=4)
    if kind == "gkr_pair":
        n = rng.randint(12, 22)
        return dict(kind=kind, n=n, m=rng.randint(10, min(n, 16)), d=4)
    if kind == "domain":
        return dict(kind=kind, n=rng.randint(8, 18), blocks=rng.choice([1, 1, 2, 3]), d=4)
    if kind == "commit":
        c = rng.randint(8, 23)
        most = min(130, 1 << (24 - c))  # no more than the configured commitment's elements
        return dict(kind=kind, c=c, ncols=max(1, round(most ** rng.random())))
    top = rng.randint(10, 23)
    below = sorted(rng.sample(range(6, top), rng.randint(0, 2)))
    classes = ["%dx%d" % (c, rng.choice([1, 2, 3, 5])) for c in below]
    return dict(kind=kind, classes=" ".join(classes + ["%dx%d" % (top, rng.choice([1, 2]))]), queries=rng.randint(4, 8),
                verify=rng.random() < 0.3)


# ------------------------------------------------------------------ inputs
class State:
    """What a program holds between calls; the tables' handles go with it."""

    def __init__(self, case):
        self.case, self.keep, self.owned = case, [], []

    def table(self, words, stride):
        """A device table over a tensor's memory."""
        words = words.to(torch.int32).contiguous()
        h = C.c_uint64()
        sa.check(sa.load().exh_table_wrap(C.c_void_p(words.data_ptr()), C.c_uint64(words.numel()), stride, C.byref(h)))
        self.keep.append(words)
        return self.own(sa.Table(h.value, words.numel(), stride))

    def own(self, table):
        self.owned.append(table)
        return table

    def __del__(self):
        for t in self.owned:
            t.free()


class Gpu:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        self.rng = np.random.default_rng(seed)

    def field(self, count):
        return torch.randint(0, P, (count,), dtype=torch.int32, device="cuda", generator=self.g)

    def integers(self, low, high, count):
        return torch.randint(low, high, (count,), dtype=torch.int64, device="cuda", generator=self.g)

    def host(self, *shape):
        return self.rng.integers(0, P, shape, dtype=np.uint32)


def _leaves(s, z, values, numerators):
    """A fraction tree's leaves numerators / (z - values) as device tables of degree-4 extension elements."""
    p = torch.zeros((len(values), 4), dtype=torch.int32, device="cuda")
    p[:, 0] = numerators
    q = torch.from_numpy(z.astype(np.int32)).cuda().repeat(len(values), 1)
    q[:, 0] = ((int(z[0]) - values) % P).to(torch.int32)
    return s.table(p, 4), s.table(q, 4)


def _classes(case):
    return [tuple(int(x) for x in part.split("x")) for part in case["classes"].split()]


def prepare(case, seed):
    sa.init()
    s, gpu, kind = State(case), Gpu(seed), case["kind"]
    if kind == "sumcheck":
        n, d = case["n"], case["d"]
        form, names, constants = STATEMENTS[case["statement"]]
        s.statement = sa.Statement(form, names, constants)
        stride = d if case["ext"] else 1
        s.tables = [s.table(gpu.field(stride << n), stride) for _ in names]
        # a point reduction's tables carry their eq weights themselves; every other proof is in eq mode
        s.eq = None if case["ext"] else gpu.host(n, d)
        s.constants = gpu.host(len(constants), d) if constants else None
        torch.cuda.synchronize()
        if case["verify"]:
            s.claim = sa.hypercube_sum(s.statement, n, s.tables, d, eq=s.eq, constants=s.constants)
    elif kind == "gkr_pair":
        n, m = case["n"], case["m"]
        z = gpu.host(4)
        values = gpu.integers(-128, 128, 1 << n)
        table = torch.arange(1 << m, dtype=torch.int64, device="cuda") - (1 << (m - 1))
        s.witness = _leaves(s, z, values, 1)
        s.lookup = _leaves(s, z, table, torch.bincount(values + (1 << (m - 1)), minlength=1 << m).to(torch.int32))
    elif kind == "gkr":
        z, count = gpu.host(4), case["blocks"] << case["n"]
        s.leaves = [_leaves(s, z, gpu.integers(-128, 128, count), 1) for _ in range(case["lookups"])]
    elif kind == "domain":
        # bits a, values b and their products c; a lookup of the pairs (a, b), a is a bit, c is the product
        count = case["blocks"] << case["n"]
        a, b = gpu.integers(0, 2, count), gpu.field(count).to(torch.int64)
        columns = [sd.Column(name, data=s.table(x, 1)) for name, x in (("a", a), ("b", b), ("c", a * b))]
        s.domain = sd.Domain("7.products", case["n"], columns, blocks=case["blocks"],
                             constraints=["(* a (- a 1))", "(- c (* a b))"], lookups=[{"tag": 5, "values": ["a", "b"]}])
        s.z, s.betas = gpu.host(4), gpu.host(2, 4)
    elif kind == "commit":
        s.columns = s.table(gpu.field(case["ncols"] << case["c"]), 1)
    else:
        s.keys = []
        nv = max(c for c, _ in _classes(case))
        s.nv, s.point, s.claim = nv, gpu.host(nv, 8), np.zeros(8, np.uint64)
        linear = sa.Statement("t0", ["t0"])
        for c, ncols in _classes(case):
            columns, coef = s.table(gpu.field(ncols << c), 1), gpu.host(ncols, 8)
            torch.cuda.synchronize()
            codewords = s.own(sa.encode(columns, ncols, c))
            levels, cap = sa.merkle_commit(codewords, ncols, c)
            s.own(levels)
            s.keys.append(dict(c=c, ncols=ncols, columns=columns, codewords=codewords, levels=levels, coef=coef, cap=cap))
            h = sa.combine_columns(columns, ncols, coef)
            s.claim = (s.claim + sa.hypercube_sum(linear, c, [h], 8, eq=s.point[nv - c:])) % P
            h.free()
        linear.free()
        s.claim = s.claim.astype(np.uint32)
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------ one pass
class _Device:
    """A device table that the library returned, for torch to read where it lies; freed with its last reader."""

    def __init__(self, table):
        self.table = table
        self.__cuda_array_interface__ = dict(shape=(table.n_u32,), typestr="<i4", data=(table.device_ptr(), False),
                                             version=2)

    def __del__(self):
        self.table.free()


def _tensor(table):
    return torch.as_tensor(_Device(table), device="cuda")


def _proof(tr):
    return np.frombuffer(tr.proof(), np.uint8)


def run(s):
    case, kind = s.case, s.case["kind"]
    if kind == "sumcheck":
        n, d = case["n"], case["d"]
        tr = sa.Transcript("sumcheck", d)
        challenges, finals, folded = sa.prove(tr, n, s.statement, s.tables, eq=s.eq, constants=s.constants)
        proof = tr.proof()
        out = [np.frombuffer(proof, np.uint8), challenges, finals, folded]
        if case["verify"]:
            check = sa.Transcript("sumcheck", d, proof=proof)
            at, reduced = sa.verify(check, n, s.statement, s.claim, eq=s.eq, constants=s.constants)
            out += [at, reduced, sa.check_final(reduced, s.statement, finals, constants=s.constants)]
        return out
    if kind == "gkr_pair":
        first, second = sa.Transcript("witness", 4), sa.Transcript("table", 4)
        claims = sa.prove_upper_pair((first, case["n"], 1, [s.witness]), (second, case["m"], 1, [s.lookup]))
        return [_proof(first), _proof(second), claims]
    if kind == "gkr":
        tr = sa.Transcript("gkr", 4)
        claims = sa.prove_upper(tr, case["n"], case["blocks"], s.leaves)
        return [_proof(tr), claims]
    if kind == "domain":
        tr = sa.Transcript("domain", 4)
        claims = sd.prove_domain(tr, s.domain, s.z, s.betas)
        return [_proof(tr), [(point, value) for _, point, value in claims]]
    if kind == "commit":
        tr = sa.Transcript("commit", 4)
        codewords, levels = sa.pcs_commit(tr, s.columns, case["ncols"], case["c"])
        return [_proof(tr), _tensor(codewords), _tensor(levels)]
    tr = sa.Transcript("open", 4)
    positions = sa.pcs_open(tr, s.nv, s.keys, s.point, s.claim, queries=case["queries"])
    proof = tr.proof()
    out = [np.frombuffer(proof, np.uint8), positions]
    if case["verify"]:
        check = sa.Transcript("open", 4, proof=proof)
        out.append(sa.pcs_verify_opening(check, s.nv, s.keys, s.point, s.claim, queries=case["queries"]))
    return out


# ------------------------------------------------------------------ what a pass cannot do without
# Operations are counted in 32-bit additions and multiplications of field words: a product of extension elements of
# degree d as d^2 products and d (d - 1) sums, a BLAKE3 compression as its 7 rounds of 8 mixing steps of 12 operations.
COMPRESSION = 7 * 8 * 12


def _ext(d):
    return 2 * d * d - d


def _sumcheck_work(n, blocks, tables, products, d, words):
    """A sumcheck's rounds over tables of blocks * 2^n entries of `words` words: the tables are read once; a pair
    costs `products` products of round values and a fold of each table (one product and two sums)."""
    pairs = blocks << n
    return 4 * words * tables * pairs, pairs * (products * _ext(d) + tables * (_ext(d) + 2 * d))


def _gkr_work(n, blocks, lookups, d):
    """A fraction tree: the leaves read once; a parent costs three products; a layer's sumcheck nine per pair and
    lookup (three products at three points)."""
    entries = lookups * blocks << n
    ops = entries * 3 * _ext(d)
    ops += sum(_sumcheck_work(l, blocks, 4 * lookups, 9 * lookups, d, d)[1] for l in range(1, n - 1))
    return 2 * 4 * d * entries, ops


def _tree_work(leaves, blocks_per_leaf):
    return 2 * 32 * leaves, (leaves * blocks_per_leaf + leaves) * COMPRESSION


def work(case):
    kind = case["kind"]
    if kind == "sumcheck":
        tables = len(STATEMENTS[case["statement"]][1])
        products = {"product": 4, "degree3": 12, "degree4": 20, "points2": 4}[case["statement"]]
        nbytes, ops = _sumcheck_work(case["n"], 1, tables, products, case["d"], case["d"] if case["ext"] else 1)
    elif kind == "gkr_pair":
        parts = [_gkr_work(case["n"], 1, 1, 4), _gkr_work(case["m"], 1, 1, 4)]
        nbytes, ops = sum(p[0] for p in parts), sum(p[1] for p in parts)
    elif kind == "gkr":
        nbytes, ops = _gkr_work(case["n"], case["blocks"], case["lookups"], 4)
    elif kind == "domain":
        nbytes = 3 * 4 * case["blocks"] << case["n"]
        ops = _gkr_work(case["n"], case["blocks"], 1, 4)[1] + _sumcheck_work(case["n"] - 1, case["blocks"], 6, 24, 4, 1)[1]
    elif kind == "commit":
        c, ncols = case["c"], case["ncols"]
        tree = _tree_work(1 << (c - 1), -(-16 * ncols // 64))
        nbytes = 4 * ncols * (3 << c) + tree[0]
        ops = ncols * (c << c) * 3 + tree[1]
    else:
        nbytes = ops = 0
        nv = max(c for c, _ in _classes(case))
        for c, ncols in _classes(case):  # the combinations of a class's columns and codewords
            nbytes += 4 * ncols * (3 << c)
            ops += ncols * (3 << c) * 8 * 2
        for i in range(max(0, nv - 5)):  # two sums and a fold of the table, a fold of the codeword, an oracle's tree
            ops += (3 << (nv - i)) * _ext(8) // 2 + (1 << (nv - i)) * 2 * _ext(8)
            if i % 2 == 1:
                ops += _tree_work(1 << (nv - i - 1), 2)[1]
    return {"bytes": nbytes, "flops": ops}


def tolerance(case):
    return "exact"
