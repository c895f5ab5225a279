"""The workloads whose speed this repository answers for.

Each case is one call that a user's program makes on tensors already on the
GPU: a contraction plan, a permutation plan, an einsum expression or a tree
built node by node, prepared once and run many times.  `listed()` names twelve,
`draw(rng)` gives more of the same kinds and ranges.

A case's "kind" says which entry point it takes:
  pair      einsum_ir_amd.ContractionPlan, one binary contraction
  permute   einsum_ir_amd.PermutePlan
  network   einsum_ir_amd.host.Expression, a tensor network along a path
  mlp       einsum_ir_amd.host.Nodes, linear layers with bias and ReLU
Sizes are written "a=32,b=16"; paths "0-1,0-1".
"""
import math

import torch

import einsum_ir_amd as eir
from einsum_ir_amd import host

# a random network of ten tensors, its intermediates up to 2^20 elements and
# one node with a K of 32768
TEN_TENSORS = "djoA,ritfw,aezqj,niovgx,kcqrsa,cpbetl,gpBhu,mlhd,mybv,wfusnk->xyzAB"
TEN_SIZES = ("A=8,B=16,a=16,b=8,c=4,d=16,e=4,f=4,g=2,h=8,i=4,j=8,k=8,l=16,m=16,n=2,o=16,p=16,q=8,r=8,s=16,t=2,"
             "u=16,v=16,w=16,x=8,y=8,z=8")
TEN_PATH = "1-9,3-8,1-7,0-1,2-3,0-4,0-3,0-2,0-1"
FIVE_TENSORS = "iaje,bf,dcba,cigj,dh->hgfei"
FIVE_PATH = "1-2,2-3,0-1,0-1"
COMPLEX_TREE = "iae,bf,dcba,cg,dh->hgfei"
COMPLEX_PATH = "1-2,1-3,1-2,0-1"


def listed():
    return [
        # a small node in the middle of a network: launch and latency count
        dict(name="small_fp32", kind="pair", dtype="fp32", out="fp32", expr="abkl,cdkl->abcd",
             sizes="a=8,b=16,c=8,d=16,k=16,l=16"),
        # the ordinary multi-mode contraction, both operands K-contiguous
        dict(name="multimode_fp32", kind="pair", dtype="fp32", out="fp32", expr="abkl,cdkl->abcd",
             sizes="a=32,b=16,c=32,d=16,k=32,l=16"),
        # large batched bf16 contraction, fp32 result
        dict(name="batched_bf16", kind="pair", dtype="bf16", out="fp32", expr="zakm,zbkn->zabmn",
             sizes="z=8,a=64,m=64,b=64,n=64,k=1024"),
        # a linear layer over a ragged number of tokens, bf16 in and out
        dict(name="linear_bf16", kind="pair", dtype="bf16", out="bf16", expr="btk,ok->bto",
             sizes="b=8,t=509,k=2048,o=2048"),
        # coupled-cluster contraction at full size: a large fp32 matrix product
        # over two contracted modes, the unit-stride modes of both operands free or contracted
        dict(name="ccsd_fp32", kind="pair", dtype="fp32", out="fp32", expr="aecf,bfde->abcd",
             sizes="a=96,b=96,c=84,d=84,e=84,f=84"),
        # coupled-cluster triples: six free modes, one short contracted mode, the result is the traffic
        dict(name="triples_fp32", kind="pair", dtype="fp32", out="fp32", expr="dega,gfbc->abcdef",
             sizes="a=24,b=20,c=20,d=24,e=20,f=20,g=24"),
        # the same contraction in double precision, as quantum chemistry runs it, at a smaller basis
        dict(name="ccsd_fp64", kind="pair", dtype="fp64", out="fp64", expr="aecf,bfde->abcd",
             sizes="a=48,b=48,c=42,d=42,e=42,f=42"),
        # transposition of a four-mode tensor between two contractions
        dict(name="permute_fp32", kind="permute", dtype="fp32", expr="abcd->dbca", sizes="a=64,b=64,c=64,d=64"),
        # the same in bf16 with mode sizes that are no powers of two
        dict(name="permute_bf16", kind="permute", dtype="bf16", expr="abcd->bdac", sizes="a=36,b=48,c=36,d=512"),
        # five linear layers with bias and ReLU on a batch of 1152, weights locked
        dict(name="mlp_fp32", kind="mlp", batch=1152, widths="784,512,512,512,512,10"),
        # a tensor network along a given path
        dict(name="network_fp32", kind="network", dtype="fp32", complex=False, expr=TEN_TENSORS, sizes=TEN_SIZES,
             path=TEN_PATH),
        # a network of complex tensors (interleaved, as torch.complex64 holds them)
        dict(name="network_complex64", kind="network", dtype="fp32", complex=True, expr=COMPLEX_TREE,
             sizes="a=24,b=32,c=20,d=24,e=28,f=32,g=20,h=24,i=30", path=COMPLEX_PATH),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm, odd ones among them."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _text(sizes):
    return ",".join("%s=%d" % (d, sizes[d]) for d in sorted(sizes))


# layouts of pairs: free modes of the left (M), of the right (N), batch and contracted modes
_FP32 = ["abkl,cdkl->abcd", "aecf,bfde->abcd", "dega,gfbc->abcdef", "acd,dbc->ab", "dca,bd->abc", "ea,ebcd->abcd",
         "eafd,fbec->abcd"]
_BF16 = ["zakm,zbkn->zabmn", "btk,ok->bto", "btk,ko->bto"]


def _roles(expr):
    ins, out = expr.split("->")
    a, b = (set(t) for t in ins.split(","))
    o = set(out)
    return ([d for d in sorted(a & b & o)], [d for d in sorted((a - b) & o)], [d for d in sorted((b - a) & o)],
            [d for d in sorted(a & b - o)])


def _split(rng, dims, total):
    """Sizes of dims whose product is near total."""
    sizes, rest = {}, total
    order = list(dims)
    rng.shuffle(order)
    for i, d in enumerate(order):
        left = len(order) - i
        sizes[d] = max(1, int(round(rest if left == 1 else rest ** (rng.uniform(0.6, 1.4) / left))))
        rest = max(1.0, rest / sizes[d])
    return sizes


def _pair(rng, exprs, dtype, out, free, contracted, most):
    expr = rng.choice(exprs)
    c, m, n, k = _roles(expr)
    while True:
        sizes = _split(rng, c, _log(rng, 2, 12)) if c else {}
        sizes.update(_split(rng, m, _log(rng, *free)))
        sizes.update(_split(rng, n, _log(rng, *free)))
        sizes.update(_split(rng, k, _log(rng, *contracted)))
        if 2 * math.prod(sizes.values()) <= most:
            return dict(kind="pair", dtype=dtype, out=out, expr=expr, sizes=_text(sizes))


def draw(rng):
    what = rng.choice(["small", "fp32", "fp32", "bf16", "bf16", "fp64", "permute", "permute", "mlp", "network",
                       "complex"])
    if what == "small":
        return _pair(rng, _FP32[:1], "fp32", "fp32", (48, 640), (64, 2048), 1e9)
    if what == "fp32":
        return _pair(rng, _FP32, "fp32", "fp32", (300, 12000), (16, 8000), 6e11)
    if what == "bf16":
        return _pair(rng, _BF16, "bf16", rng.choice(["fp32", "bf16"]), (300, 6000), (64, 5000), 4e11)
    if what == "fp64":
        return _pair(rng, _FP32, "fp64", "fp64", (200, 4000), (16, 4000), 5e10)
    if what == "permute":
        expr, lo, hi = rng.choice([("abcd->dbca", (6, 16, 16, 6), (100, 100, 100, 100)),
                                   ("abcd->bdac", (16, 16, 16, 96), (72, 96, 72, 600)),
                                   ("abcd->acdb", (16, 8, 32, 32), (128, 64, 96, 128)),
                                   ("abcd->cabd", (24, 24, 96, 24), (64, 64, 600, 64)),
                                   ("abcd->dcba", (16, 16, 32, 32), (64, 64, 128, 128))])
        sizes = {d: _log(rng, a, b) for d, a, b in zip("abcd", lo, hi)}
        return dict(kind="permute", dtype=rng.choice(["fp32", "fp32", "bf16"]), expr=expr, sizes=_text(sizes))
    if what == "mlp":
        w = [_log(rng, 200, 2000)] + [64 * _log(rng, 2, 32)] * rng.randint(1, 4) + [_log(rng, 8, 128)]
        return dict(kind="mlp", batch=_log(rng, 64, 4000), widths=",".join(map(str, w)))
    cpx = what == "complex"
    case = dict(kind="network", dtype=rng.choice(["fp32", "fp64"]) if cpx else "fp32", complex=cpx)
    while True:
        if not cpx:
            sizes = {d: _log(rng, 4, 12) if d in "ij" else _log(rng, 8, 72) for d in "abcdefghij"}
            case.update(expr=FIVE_TENSORS, sizes=_text(sizes), path=FIVE_PATH)
        elif rng.random() < 0.5:
            sizes = {d: _log(rng, 64, 1500) for d in "kmn"}
            case.update(expr="km,nk->nm", sizes=_text(sizes), path="0-1")
        else:
            sizes = {d: _log(rng, 10, 34) for d in "abcdefghi"}
            case.update(expr=COMPLEX_TREE, sizes=_text(sizes), path=COMPLEX_PATH)
        w = work(case)
        if w["flops"] <= 5e10 and w["bytes"] <= 8e8:
            return case


_TORCH = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp64": torch.float64}
_EIR = {"fp32": eir.FP32, "bf16": eir.BF16, "fp64": eir.FP64}


def _sizes(case):
    return {k: int(v) for k, v in (p.split("=") for p in case["sizes"].split(","))}


def _path(case):
    return [tuple(int(x) for x in p.split("-")) for p in case["path"].split(",")]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(shape, dtype, g):
    """Values of [-1, 1)."""
    return (torch.rand(shape, device="cuda", generator=g, dtype=torch.float64 if dtype == torch.float64
                       else torch.float32) * 2 - 1).to(dtype)


def _mlp_tensors(case, seed):
    g, w = _generator(seed), [int(x) for x in case["widths"].split(",")]
    x = torch.randn((case["batch"], w[0]), device="cuda", generator=g)
    ws = [_uniform((o, i), torch.float32, g) / i ** 0.5 for i, o in zip(w, w[1:])]
    bs = [_uniform((o,), torch.float32, g) / i ** 0.5 for i, o in zip(w, w[1:])]
    return x, ws, bs


def _inputs(case, seed):
    """A case's input tensors, made from the seed alone."""
    g, s = _generator(seed), _sizes(case)
    ins = case["expr"].split("->")[0].split(",")
    dtype = _TORCH[case["dtype"]]
    if case["kind"] != "network":
        return [_uniform([s[d] for d in t], dtype, g) for t in ins]
    # each tensor scaled by the square root of its contracted modes, so that
    # the results of all nodes are of the order of one
    out, tensors = case["expr"].split("->")[1], []
    for t in ins:
        shape = [s[d] for d in t]
        scale = math.prod(s[d] for d in t if d not in out) ** 0.25
        if case["complex"]:
            x = torch.complex(*(torch.randn(shape, device="cuda", generator=g, dtype=dtype) for _ in range(2)))
        else:
            x = torch.randn(shape, device="cuda", generator=g, dtype=dtype)
        tensors.append(x / scale)
    return tensors


def prepare(case, seed):
    stream = torch.cuda.current_stream()
    if case["kind"] == "mlp":
        x, ws, bs = _mlp_tensors(case, seed)
        widths = [x.shape[1]] + [w.shape[0] for w in ws]
        sizes = {i: n for i, n in enumerate([case["batch"]] + widths)}
        out = torch.empty((case["batch"], widths[-1]), device="cuda")
        nodes = host.Nodes(sizes, {0: 1, **{i: n for i, n in sizes.items() if i > 1}}, stream=stream)
        prev = nodes.add_leaf([0, 1], x)
        leaves = [nodes.add_leaf([i + 2, i + 1], w) for i, w in enumerate(ws)]
        for i, leaf in enumerate(leaves):
            last = i == len(leaves) - 1
            prev = nodes.add_binary([0, i + 2], prev, leaf, tensor=out if last else None, aux=bs[i], first=eir.COPY,
                                    main=eir.MADD, last=eir.UNDEFINED_KTYPE if last else eir.RELU)
        nodes.compile(prev)
        for leaf in leaves:
            nodes.store_and_lock_data(leaf)
        return dict(kind="mlp", nodes=nodes, out=out, keep=(x, ws, bs))
    sizes, tensors = _sizes(case), _inputs(case, seed)
    shape = [sizes[d] for d in case["expr"].split("->")[1]]
    if case["kind"] == "permute":
        u = eir.unary_dims(case["expr"], sizes)
        out = torch.empty(shape, device="cuda", dtype=tensors[0].dtype)
        plan = eir.PermutePlan(u["sizes"], u["strides_in"], u["strides_out"], dtype=_EIR[case["dtype"]])
    elif case["kind"] == "pair":
        lp = eir.binary_loops(case["expr"], sizes)
        out = torch.empty(shape, device="cuda", dtype=_TORCH[case["out"]])
        dt = _EIR[case["dtype"]]
        plan = eir.ContractionPlan(lp["dim_types"], lp["sizes"], lp["strides_left"], lp["strides_right"],
                                   lp["strides_out"], dtype_left=dt, dtype_right=dt,
                                   dtype_comp=eir.FP64 if case["dtype"] == "fp64" else eir.FP32,
                                   dtype_out=_EIR[case["out"]])
    else:
        out = torch.empty(shape, device="cuda", dtype=tensors[0].dtype)
        plan = host.Expression(case["expr"], sizes, _path(case), tensors + [out], dtype=_EIR[case["dtype"]],
                               stream=stream, ctype=host.BATCH_INNER if case["complex"] else host.REAL_ONLY)
    return dict(kind=case["kind"], plan=plan, tensors=tensors, out=out, stream=stream)


def run(state):
    if state["kind"] == "mlp":
        state["nodes"].eval_async()
    elif state["kind"] == "network":
        state["plan"].eval_async()
    else:
        state["plan"].execute(*state["tensors"], state["out"], stream=state["stream"])
    return state["out"]


def _steps(case):
    """(left, right, result) modes of each node of a network along its path."""
    ins, out = case["expr"].split("->")
    live, steps = ins.split(","), []
    for i, j in _path(case):
        a, b = live[i], live[j]
        live = [t for k, t in enumerate(live) if k not in (i, j)]
        kept = set("".join(live)) | set(out)
        res = "".join(d for d in dict.fromkeys(a + b) if d in kept) if live else out
        steps.append(((i, j), a, b, res))
        live.append(res)
    return steps


def work(case):
    if case["kind"] == "mlp":
        w, b = [int(x) for x in case["widths"].split(",")], case["batch"]
        pairs = list(zip(w, w[1:]))
        return dict(bytes=4 * (b * (w[0] + w[-1]) + sum(i * o + o for i, o in pairs)),
                    flops=2 * b * sum(i * o for i, o in pairs))
    s = _sizes(case)
    ins, out = case["expr"].split("->")
    numel = lambda t: math.prod(s[d] for d in t)  # noqa: E731
    item = _TORCH[case["dtype"]].itemsize * (2 if case.get("complex") else 1)
    read = item * sum(numel(t) for t in ins.split(","))
    if case["kind"] == "permute":
        return dict(bytes=2 * read, flops=0)
    if case["kind"] == "pair":
        return dict(bytes=read + _TORCH[case["out"]].itemsize * numel(out), flops=2 * math.prod(s.values()))
    flops = sum(numel(set(a) | set(b)) for _, a, b, _ in _steps(case)) * (8 if case["complex"] else 2)
    return dict(bytes=read + item * numel(out), flops=flops)


def tolerance(case):
    # measured against 64 bits: fp32 2e-7 to 1.5e-6 (the largest where 7056 products are summed), fp64 1e-15, bf16
    # results 1.7e-3 (half a unit in the last place of 8 bits)
    if case["kind"] == "permute":
        return "exact"
    if case["kind"] == "mlp":
        return dict(rel=1e-5)
    if case["dtype"] == "fp64":
        return dict(rel=2e-14)
    if case["kind"] == "pair" and case["out"] == "bf16":
        return dict(rel=4e-3, max=1e-2)
    return dict(rel=1e-5)


def exact(case, seed):
    if case["kind"] == "mlp":
        x, ws, bs = _mlp_tensors(case, seed)
        x = x.double()
        for i, (w, b) in enumerate(zip(ws, bs)):
            x = x @ w.double().t().contiguous() + b.double()
            x = x if i == len(ws) - 1 else torch.relu(x)
        return x
    tensors = _inputs(case, seed)
    ins, out = case["expr"].split("->")
    if case["kind"] == "permute":
        return tensors[0].double().permute([ins.index(d) for d in out]).contiguous()
    tensors = [t.to(torch.complex128 if t.is_complex() else torch.float64) for t in tensors]
    if case["kind"] == "pair":
        return torch.einsum(case["expr"], *tensors)
    for (i, j), a, b, res in _steps(case):
        t = torch.einsum("%s,%s->%s" % (a, b, res), tensors[i], tensors[j])
        tensors = [x for k, x in enumerate(tensors) if k not in (i, j)] + [t]
    return tensors[0]
