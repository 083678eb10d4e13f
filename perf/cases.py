"""Cases of the block-tensor contraction path: what a correlated-methods program has the library do
in every iteration, through the public Python mirror of the C ABI.

Kinds (`kind` of a case; `occ` and `vir` list block sizes, for ladders per spin, `irr` the irrep of each virtual block):
  ring       C[ijab] = A[ikac] B[kjcb], no symmetry              btod_contract2.perform
  ladder     R[ijab] = T[ijcd] V[abcd], spin partitions, C2v labels, antisymmetric pairs   btod_contract2.perform
  ladder_add R += d (the same) into a tensor that holds data     btod_contract2.perform_add
  split      the ladder in split-precision mode (`slices` int8 slices), V immutable        btod_contract2.perform
  symm       the ladder symmetrized over (ij)(ab)                btod_symmetrize2.perform
  quadratic  D[ijab] = 1/4 (T[ijcd] T[klcd]) T[klab]             btod_contract3.perform
  update     R = c1 T + c2 P(U), then the scalar product <R, W>  btod_add, btod_dotprod
  dense      the ring on dense arrays                            tod_contract2
  permute    B = c P(A) on dense arrays                          tod_copy
"""
import itertools

import numpy as np
import torch

import libtensor_amd as lt
from libtensor_amd import workloads

_RING = ((1, 0), (3, 2))                 # contracted index pairs of ring and dense
_LADDER = ((2, 2), (3, 3))
_SWAP = (1, 0, 3, 2)                     # (ij)(ab)
_TABLE = {(p, q): p ^ q for p in range(4) for q in range(4)}     # C2v: the product of two irreps
_CTX = []


def _context():
    """One context for the process, as a program has it."""
    if not _CTX:
        _CTX.append(lt.Context(0))
        workloads.register_tables({"tables": [workloads.C2V]})
    return _CTX[0]


# ---------------------------------------------------------------------------
# cases

def listed():
    return [
        # the smallest call: one block, where launches and host work are what it costs
        {"name": "ring_small", "kind": "ring", "occ": "10", "vir": "40", "async": True},
        # a small molecule's ladder with all its symmetry: hundreds of blocks of a few elements each
        {"name": "ladder_small", "kind": "ladder", "occ": "3 2 2 1", "vir": "8 7 9 8", "irr": "0 1 2 3",
         "async": True},
        # a ladder term added into the residual; odd block sizes throughout
        {"name": "ladder_add", "kind": "ladder_add", "occ": "5 3 3 2", "vir": "13 11 17 9 15", "irr": "0 1 2 3 0"},
        # the particle-particle ladder of the benchmark (o = 40, v = 200), its iterations enqueued back to back
        {"name": "ladder_large", "kind": "ladder", "occ": "7 5 4 4", "vir": "18 16 16 14 12 24",
         "irr": "0 0 1 2 2 3", "async": True},
        # a ring of the serving mix: one block per dimension, odd extents (rows that no wide load is aligned to)
        {"name": "ring_odd", "kind": "ring", "occ": "29", "vir": "131"},
        # the largest: a ring over uneven blocks, gigabytes of operands
        {"name": "ring_large", "kind": "ring", "occ": "31 17", "vir": "83 41 72 44"},
        # emulated FP64 on the int8 matrix cores, integrals kept in an immutable tensor
        {"name": "ladder_split", "kind": "split", "occ": "7 5 4 4", "vir": "18 16 16 14 12 24",
         "irr": "0 0 1 2 2 3", "slices": 7},
        # a ladder whose result is symmetrized
        {"name": "ladder_symm", "kind": "symm", "occ": "6 4 3 3", "vir": "19 15 12 22 10", "irr": "0 1 2 3 0"},
        # the quadratic term: two contractions with the intermediate resident
        {"name": "quadratic", "kind": "quadratic", "occ": "7 5 4 4", "vir": "18 16 16 14 12 24",
         "irr": "0 0 1 2 2 3"},
        # amplitude update and its scalar product: bandwidth
        {"name": "update", "kind": "update", "occ": "17 15", "vir": "63 41 56"},
        # one dense contraction with all its index permutations, odd extents
        {"name": "dense", "kind": "dense", "occ": "15", "vir": "45"},
        # one dense permutation, odd extents
        {"name": "permute", "kind": "permute", "dims": "37 61 83 91", "perm": "2 0 3 1"},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _parts(rng, n, most):
    """n in at most `most` random parts."""
    k = rng.randint(1, max(1, min(most, n)))
    cut = sorted(rng.sample(range(1, n), k - 1)) if k > 1 else []
    return " ".join(str(b - a) for a, b in zip([0] + cut, cut + [n]))


def draw(rng):
    kind = rng.choice(["ring", "ring", "ladder", "ladder", "ladder_add", "split", "symm", "quadratic",
                       "update", "dense", "permute"])
    if kind == "permute":
        n = rng.randint(2, 6)
        total = _log(rng, 1 << 12, 1 << 24)
        dims = []
        for i in range(n):
            d = max(1, int(round(total ** (1.0 / (n - i)) * (0.4 + 1.2 * rng.random()))))
            dims.append(d)
            total = max(1, total // d)
        perm = list(range(n))
        rng.shuffle(perm)
        return {"kind": kind, "dims": " ".join(map(str, dims)), "perm": " ".join(map(str, perm))}
    if kind == "dense":
        return {"kind": kind, "occ": str(_log(rng, 3, 24)), "vir": str(_log(rng, 8, 72))}
    if kind in ("ring", "update"):
        o, v = _log(rng, 6, 40), _log(rng, 20, 180)
        case = {"kind": kind, "occ": _parts(rng, o, 3), "vir": _parts(rng, v, 5)}
    else:
        case = {"kind": kind, "occ": " ".join(str(_log(rng, 1, 7)) for _ in range(4))}
        vir = [_log(rng, 6, 24) for _ in range(rng.randint(3, 6))]
        case["vir"] = " ".join(map(str, vir))
        case["irr"] = " ".join(str(i % 4) for i in range(len(vir)))
        if kind == "split":
            case["slices"] = rng.choice([6, 7, 7, 8])
    if kind in ("ring", "ladder"):
        case["async"] = rng.random() < 0.5
    return case


# ---------------------------------------------------------------------------
# block structure and inputs

def _ints(case, key):
    return [int(x) for x in case[key].split()]


def _spaces(case):
    """Occupied and virtual space: per block (start, size, spin, irrep)."""
    both = case["kind"] in ("ladder", "ladder_add", "split", "symm", "quadratic")
    out = []
    for key in ("occ", "vir"):
        sizes = _ints(case, key)
        irr = _ints(case, "irr") if key == "vir" and both else [i % 4 for i in range(len(sizes))]
        rows, at = [], 0
        for spin in (0, 1) if both else (0,):
            for n, x in zip(sizes, irr):
                rows.append((at, n, spin, x))
                at += n
        out.append(rows)
    return {"o": out[0], "v": out[1]}


def _dims(case, kinds):
    sp = _spaces(case)
    return [sum(r[1] for r in sp[k]) for k in kinds]


def _allowed(sp, kinds, idx):
    """Spin conserved between the pairs (0, 1) and (2, 3) and irreps multiplying to the first."""
    b = [sp[k][i] for k, i in zip(kinds, idx)]
    x = 0
    for r in b:
        x = _TABLE[x, r[3]]
    return b[0][2] + b[1][2] == b[2][2] + b[3][2] and x == 0


def _images(sp, kinds, idx, pairs):
    """The blocks that symmetry makes one with block idx: exchanges in each pair, the spin flip, for `vvvv` the exchange of the pairs."""
    half = [len(sp[k]) // 2 for k in kinds]
    out = set()
    for s1, s2, flip, ex in itertools.product((0, 1), (0, 1), (0, 1), (0, 1) if pairs else (0,)):
        p, q = idx[:2], idx[2:]
        if ex:
            p, q = q, p
        p, q = (p[::-1] if s1 else p), (q[::-1] if s2 else q)
        b = p + q
        if flip:
            b = tuple((i + h) % (2 * h) for i, h in zip(b, half))
        out.add(b)
    return out


def _canonical(case, kinds):
    """The stored blocks: of each allowed orbit the block that comes first."""
    sp = _spaces(case)
    every = itertools.product(*[range(len(sp[k])) for k in kinds])
    if "irr" not in case:
        return list(every)
    return [b for b in every if _allowed(sp, kinds, b) and b == min(_images(sp, kinds, b, kinds == "vvvv"))]


def _block(sp, kinds, b):
    return tuple(slice(sp[k][i][0], sp[k][i][0] + sp[k][i][1]) for k, i in zip(kinds, b))


def _normal(dims, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*dims, generator=g, dtype=torch.float64, device="cuda")


def _array(case, kinds, seed):
    """A dense tensor with the symmetry of its kind: amplitudes (`oovv`) decay with |a - i| and are of order 0.01, integrals (`vvvv`) of order 1."""
    x = _normal(_dims(case, kinds), seed)
    if kinds == "oovv":
        o, v = x.shape[0], x.shape[2]
        i, a = torch.arange(o, device="cuda"), torch.arange(v, device="cuda")
        x *= (0.01 / (1.0 + (a[None, :] - i[:, None]).abs().double()))[:, None, :, None]
    if "irr" not in case:
        return x
    x -= x.transpose(0, 1).clone()
    x -= x.transpose(2, 3).clone()
    if kinds == "vvvv":
        x += x.permute(2, 3, 0, 1).clone()
    for d in range(4):                    # the spin flip of all four dimensions at once
        x = x.unflatten(2 * d, (2, x.shape[2 * d] // 2))
    x = (x + x.flip(0, 2, 4, 6)).flatten(0, 1).flatten(1, 2).flatten(2, 3).flatten(3, 4)
    x *= 0.25 if kinds == "oovv" else 0.125
    sp = _spaces(case)
    spin, irr = ([torch.tensor([r[f] for r in sp[k] for _ in range(r[1])], device="cuda") for k in kinds] for f in (2, 3))
    row = (spin[0][:, None] + spin[1][None, :]) * 4 + (irr[0][:, None] ^ irr[1][None, :])
    col = (spin[2][:, None] + spin[3][None, :]) * 4 + (irr[2][:, None] ^ irr[3][None, :])
    for i in range(x.shape[0]):           # blocks that symmetry forbids are zero
        x[i] *= row[i][:, None, None] == col[None]
    return x


def _tensor(ctx, case, kinds, dense):
    """A block tensor with the splits and symmetry of its kind; `dense` fills its stored blocks."""
    sp = _spaces(case)
    bis = lt.block_index_space([sum(r[1] for r in sp[k]) for k in kinds])
    for k in "ov":
        mask = [1 if x == k else 0 for x in kinds]
        if any(mask):
            for r in sp[k][1:]:
                bis.split(mask, r[0])
    bt = lt.block_tensor(ctx, bis)
    if dense is None:
        return bt
    if "irr" in case:
        for p in ((1, 0, 2, 3), (0, 1, 3, 2)):
            bt.insert(lt.se_perm(p, -1.0))
        if kinds == "vvvv":
            bt.insert(lt.se_perm((2, 3, 0, 1), 1.0))
        part = lt.se_part((2, 2, 2, 2))
        spins = list(itertools.product((0, 1), repeat=4))
        good = [s for s in spins if s[0] + s[1] == s[2] + s[3]]
        for s in spins:
            if s not in good:
                part.mark_forbidden(s)
        for s in good:
            f = tuple(1 - x for x in s)
            if s < f:
                part.add_map(s, f, 1.0)
        bt.insert(part)
        label = lt.se_label(workloads.C2V[0])
        for k in "ov":
            mask = [1 if x == k else 0 for x in kinds]
            if any(mask):
                for n, r in enumerate(sp[k]):
                    label.assign(mask, n, r[3])
        label.set_rule([0])
        bt.insert(label)
    for b in _canonical(case, kinds):
        bt.set_block(b, dense[_block(sp, kinds, b)].cpu().numpy())
    return bt


def _contraction(pairs, permc=None):
    c = lt.contraction2(2, 2, 2, permc)
    for p in pairs:
        c.contract(*p)
    return c


def _seeds(seed):
    return [1000003 * (seed + 1) + 7919 * i for i in range(4)]


class _results(dict):
    """Result tensors by name. They stay in HBM, where the program's next step takes them; an entry is unfolded on the host when it is read."""

    def __getitem__(self, key):
        v = dict.__getitem__(self, key)
        return v.to_dense() if isinstance(v, lt.block_tensor) else v.download() if isinstance(v, lt.device_array) else v

    def items(self):
        return [(k, self[k]) for k in self]

    def values(self):
        return [self[k] for k in self]


# ---------------------------------------------------------------------------
# one pass

def prepare(case, seed):
    ctx, kind, s = _context(), case["kind"], _seeds(seed)
    if kind == "permute":
        dims, perm = _ints(case, "dims"), _ints(case, "perm")
        a = lt.device_array(ctx, dims, _normal(dims, s[0]).cpu().numpy())
        return {"kind": kind, "a": a, "b": lt.device_array(ctx, [dims[p] for p in perm]), "perm": perm}
    if kind == "dense":
        o, v = int(case["occ"]), int(case["vir"])
        a, b = (lt.device_array(ctx, (o, o, v, v), _normal((o, o, v, v), x).cpu().numpy()) for x in s[:2])
        return {"kind": kind, "a": a, "b": b, "c": lt.device_array(ctx, (o, o, v, v)),
                "contr": _contraction(_RING, (0, 2, 1, 3))}
    if kind == "update":
        t = [_tensor(ctx, case, "oovv", _array(case, "oovv", x)) for x in s[:3]]
        return {"kind": kind, "t": t[0], "u": t[1], "w": t[2], "r": _tensor(ctx, case, "oovv", None)}
    a = _tensor(ctx, case, "oovv", _array(case, "oovv", s[0]))
    r = _tensor(ctx, case, "oovv", None)
    state = {"kind": kind, "a": a, "r": r}
    if kind == "quadratic":
        state["op"] = lt.btod_contract3(_contraction(_LADDER), _contraction(((2, 0), (3, 1))), a, a, a, kd=0.25)
        return state
    if kind == "ring":
        b = _tensor(ctx, case, "oovv", _array(case, "oovv", s[1]))
        op = lt.btod_contract2(_contraction(_RING, (0, 2, 1, 3)), a, b)
    else:
        b = _tensor(ctx, case, "vvvv", _array(case, "vvvv", s[1]))
        if kind == "split":
            b.set_immutable()
        op = lt.btod_contract2(_contraction(_LADDER), a, b)
    if kind == "ladder_add":
        # the residual before this term: another amplitude-like tensor
        state["r"] = _tensor(ctx, case, "oovv", _array(case, "oovv", s[2]))
    if kind == "split":
        op.set_ozaki(case["slices"])
    if case.get("async"):
        op.set_async(True)
    state.update(b=b, op=lt.btod_symmetrize2(op, _SWAP, True) if kind == "symm" else op)
    return state


def run(s):
    kind = s["kind"]
    if kind == "permute":
        lt.tod_copy(s["a"], s["b"], s["perm"], -0.5)
        return _results(b=s["b"])
    if kind == "dense":
        lt.tod_contract2(s["contr"], s["a"], s["b"], s["c"], 0.5)
        return _results(c=s["c"])
    if kind == "update":
        lt.btod_add([(s["t"], None, 0.75), (s["u"], _SWAP, -0.25)], s["r"])
        return _results(r=s["r"], e=lt.btod_dotprod(s["r"], s["w"]))
    if kind == "ladder_add":
        s["op"].perform_add(s["r"], 0.5)
    elif kind == "split":
        s["op"].perform(s["r"], lt.LT_MODE_OZAKI)
    else:
        s["op"].perform(s["r"])
    return _results(r=s["r"])


def exact(case, seed):
    """The dense contraction in 64 bits, by torch's matrix products."""
    kind, s = case["kind"], _seeds(seed)
    if kind == "permute":
        return {"b": (-0.5 * _normal(_ints(case, "dims"), s[0]).permute(_ints(case, "perm"))).cpu().numpy()}
    if kind == "update":
        t, u, w = (_array(case, "oovv", x) for x in s[:3])
        r = 0.75 * t - 0.25 * u.permute(_SWAP)
        return {"r": r.cpu().numpy(), "e": float((r * w).sum())}
    if kind in ("ring", "dense"):
        if kind == "dense":
            o, v = int(case["occ"]), int(case["vir"])
            a, b = (_normal((o, o, v, v), x) for x in s[:2])
        else:
            a, b = (_array(case, "oovv", x) for x in s[:2])
        o, v = a.shape[0], a.shape[2]
        m = a.permute(0, 2, 1, 3).reshape(o * v, o * v)
        m = m @ b.permute(0, 2, 1, 3).reshape(o * v, o * v)
        c = m.reshape(o, v, o, v).permute(0, 2, 1, 3)
        return {"c": (0.5 * c).cpu().numpy()} if kind == "dense" else {"r": c.cpu().numpy()}
    t = _array(case, "oovv", s[0])
    o, v = t.shape[0], t.shape[2]
    m = t.reshape(o * o, v * v)
    if kind == "quadratic":
        return {"r": (0.25 * (m @ m.T) @ m).reshape(o, o, v, v).cpu().numpy()}
    r = (m @ _array(case, "vvvv", s[1]).reshape(v * v, v * v).T).reshape(o, o, v, v)
    if kind == "symm":
        r = r + r.permute(_SWAP)
    if kind == "ladder_add":
        r = _array(case, "oovv", s[2]) + 0.5 * r
    return {"r": r.cpu().numpy()}


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _elements(case, kinds):
    sp = _spaces(case)
    return sum(int(np.prod([sp[k][i][1] for k, i in zip(kinds, b)])) for b in _canonical(case, kinds))


def _products(case, kinds, inner):
    """2 m n k over the stored result blocks, contracted over the allowed blocks of an antisymmetric pair, each once."""
    sp = _spaces(case)
    total = 0
    pairs = [(p, q) for p in range(len(sp[inner])) for q in range(p, len(sp[inner]))]
    for b in _canonical(case, kinds):
        c = [sp[k][i] for k, i in zip(kinds, b)]
        spin, irr = c[0][2] + c[1][2], _TABLE[c[0][3], c[1][3]]
        k = sum(sp[inner][p][1] * sp[inner][q][1] for p, q in pairs
                if sp[inner][p][2] + sp[inner][q][2] == spin and _TABLE[sp[inner][p][3], sp[inner][q][3]] == irr)
        total += 2 * k * int(np.prod([r[1] for r in c]))
    return total


def work(case):
    kind = case["kind"]
    if kind == "permute":
        return {"bytes": 16 * int(np.prod(_ints(case, "dims"))), "flops": 0}
    if kind in ("dense", "ring"):
        o, v = sum(_ints(case, "occ")), sum(_ints(case, "vir"))
        return {"bytes": 24 * (o * v) ** 2, "flops": 2 * (o * v) ** 3}
    n = _elements(case, "oovv")
    if kind == "update":
        return {"bytes": 40 * n, "flops": 5 * n}       # R is written, and read again by the scalar product
    if kind == "quadratic":
        return {"bytes": 16 * n, "flops": _products(case, "oooo", "v") + _products(case, "oovv", "o")}
    return {"bytes": 8 * (_elements(case, "vvvv") + (3 if kind == "ladder_add" else 2) * n),
            "flops": _products(case, "oovv", "v")}


def tolerance(case):
    """FP64 sums in another order (measured against `exact`: up to 4e-15); the split form drops what its slices do not hold (7 slices: 1e-13)."""
    if case["kind"] == "split":
        return {"rel": {6: 1e-10, 7: 1e-12, 8: 2e-14}[case["slices"]]}
    if case["kind"] == "permute":
        return "exact"
    return {"rel": 2e-14, "max": 1e-12}
