"""Timed cases of the zeroth-order (ZO) fine-tuning step: what a program that trains with this package
has it do, through the package's public entry points.

A case is a dict of plain values. `kind` names the calls that one pass makes:

  steady    the two parameter passes of every steady ZO step: perturb by -2 eps z, then the fused restore +
            update + next perturbation, over one model's trainable set (ZOTable)
  passes    the same step without cross-step fusion: perturb +1, perturb -2, restore + update, and an update
            of its own (the options zo_fuse_next_perturb = False and zo_fuse_restore = False) (ZOTable)
  spsa      the library's part of half an iteration of the DiZO gamma search: the draw of gamma's noise, the
            projection applied, and reversed with the new norms (normals, ProjTable)
  fo        the library's part of one first-order iteration on gamma: norms, projection with an fp32 ratio,
            the gradient reduction against a snapshot (ProjTable)
  norms     the norms without a table or any allocation, as a captured or memory-tight caller takes them
            (dz_group_sumsq_static)
  normals   z written out: the noise of one tensor for inspection, or a tensor's random initialisation
            (normals)
  train     one whole optimisation step of an OPT model, forwards included (ZOTrainer.training_step)

Parameters live in one flat buffer per model, as programs that flatten their parameters keep them: each
tensor starts at a multiple of 512 bytes (as PyTorch's allocator places separate tensors), or directly behind
the one before it where the case says `packed`.
"""
import ctypes
import math

import numpy as np
import torch

from dizo_amd import _lib as L
from dizo_amd.table import ProjTable, ZOTable, normals

DEV = "cuda"
DT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"fp32": 4, "fp16": 2, "bf16": 2}
EPS, LR = 1e-3, 1e-6  # zo_eps and learning rate of the fine-tuning recipe


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # the test-size model: the smallest calls, where launches and latency count
        dict(name="steady tiny fp16", kind="steady", set="opt", layers=2, d=64, ffn=256, positions=130, dtype="fp16", packed=False),
        # low-rank adapters on the k/v projections of an OPT-2.7B: many short tensors, each below one tile
        dict(name="steady adapters fp16", kind="steady", set="adapters", layers=32, d=2560, rank=8, dtype="fp16", packed=False),
        # the whole trainable set of an OPT-125m in fp32
        dict(name="steady opt-125m fp32", kind="steady", set="opt", layers=12, d=768, ffn=3072, positions=2050, dtype="fp32", packed=False),
        # the whole trainable set of an OPT-2.7B in fp16
        dict(name="steady opt-2.7b fp16", kind="steady", set="opt", layers=32, d=2560, ffn=10240, positions=2050, dtype="fp16", packed=False),
        # the largest: eight layers of an OPT-30B in bf16 (the whole one runs at the same rate)
        dict(name="steady opt-30b-part bf16", kind="steady", set="opt", layers=8, d=7168, ffn=28672, positions=2050, dtype="bf16", packed=False),
        # a flattened, tightly packed parameter buffer of odd sizes: no tensor starts at a vector boundary
        dict(name="passes packed odd bf16", kind="passes", set="opt", layers=6, d=1001, ffn=3003, positions=515, dtype="bf16", packed=True),
        # the gamma search over adapters (the projected set of a run on adapters only)
        dict(name="spsa adapters fp16", kind="spsa", set="adapters", layers=32, d=2560, rank=8, dtype="fp16", packed=False),
        # the gamma search over the k/v projections of an OPT-13B
        dict(name="spsa opt-13b fp16", kind="spsa", set="kv", layers=40, d=5120, dtype="fp16", packed=False),
        # the first-order path over the k/v projections of an OPT-2.7B
        dict(name="fo opt-2.7b fp16", kind="fo", set="kv", layers=32, d=2560, dtype="fp16", packed=False),
        # norms under capture, over the k/v projections of an OPT-125m in fp32
        dict(name="norms opt-125m fp32", kind="norms", set="kv", layers=12, d=768, dtype="fp32", packed=False),
        # z of one feed-forward matrix of an OPT-13B
        dict(name="normals 105M fp16", kind="normals", n=20480 * 5120, offset=13 * 2**20, dtype="fp16"),
        # one optimisation step of an OPT-125m, 16 examples x 2 candidates of 32 to 64 tokens
        dict(name="train opt-125m fp32", kind="train", set="opt", layers=12, d=768, heads=12, ffn=3072, vocab=50272, positions=2050,
             batch=16, dtype="fp32", packed=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: models from the test size to a few OPT-2.7B layers, adapters of
    rank 2 to 64, aligned and packed, odd widths among them, in the three data types."""
    kind = rng.choice(["steady", "steady", "steady", "passes", "passes", "spsa", "spsa", "spsa", "fo", "norms", "normals", "normals", "train"])
    dtype = rng.choice(["fp32", "fp16", "bf16"])
    if kind == "normals":
        return dict(kind=kind, n=_log(rng, 24, 100_000_000), offset=rng.randrange(0, 2**33), dtype=dtype)
    if kind == "train":
        heads = rng.choice([4, 8, 12])
        d = heads * 8 * rng.randint(2, 8)
        return dict(kind=kind, set="opt", layers=rng.randint(2, 8), d=d, heads=heads, ffn=4 * d, vocab=rng.randrange(500, 50272),
                    positions=130, batch=rng.randint(2, 16), dtype=dtype, packed=False)
    packed = rng.random() < 0.25
    d = _log(rng, 64, 2400)
    if rng.random() < 0.6:
        d = max(64, d // 64 * 64)
    if kind in ("steady", "passes") and rng.random() < 0.7:
        return dict(kind=kind, set="opt", layers=rng.randint(1, 16), d=d, ffn=rng.choice([4 * d, 3 * d + 1]),
                    positions=rng.choice([130, 515, 2050]), dtype=dtype, packed=packed)
    if kind not in ("steady", "passes") and rng.random() < 0.5:
        return dict(kind=kind, set="kv", layers=rng.randint(1, 40), d=d, dtype=dtype, packed=packed)
    return dict(kind=kind, set="adapters", layers=rng.randint(1, 48), d=d, rank=_log(rng, 2, 64), dtype=dtype, packed=packed)


def numels(case):
    """Elements of each registered tensor, in named_parameters order."""
    d = case["d"]
    if case["set"] == "kv":
        return [d * d] * (2 * case["layers"])
    if case["set"] == "adapters":  # A (rank x d) and B (d x rank) on k and v
        return [d * case["rank"]] * (4 * case["layers"])
    f = case["ffn"]
    layer = [d * d, d] * 4 + [d, d] + [f * d, f, d * f, d] + [d, d]
    return [case["positions"] * d, d, d] + layer * case["layers"]


def places(case):
    """(first elements, length of the flat buffer)."""
    step = 1 if case["packed"] else 512 // SIZE[case["dtype"]]
    at, out = (3 if case["packed"] else 0), []
    for n in numels(case):
        at = -(-at // step) * step
        out.append(at)
        at += n
    return out, at + 8


# ----------------------------------------------------------------- inputs --
def _flat(case, seed, std):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.empty(places(case)[1], dtype=DT[case["dtype"]], device=DEV).normal_(0.0, std, generator=g)


def _weights(case, seed):
    return _flat(case, seed, 0.02)


def _anchored(case, seed):
    """(anchor, weights a fine-tuning run away from it)"""
    anchor = _weights(case, seed)
    return anchor, anchor + _flat(case, seed + 10**6, 4e-3)


def _views(case, flat):
    return [flat[a:a + n] for a, n in zip(places(case)[0], numels(case))]


def _seeds(seed):
    return 1000 * seed + 17  # the first z seed of a state; later steps count up from it


def _grad(case, seed):
    return float(np.random.RandomState(seed % 2**31).standard_normal())


def _ratios(case, seed):
    """One ratio for each group, near 1 as gamma / norm is in the search."""
    g = torch.Generator().manual_seed(seed)
    return torch.empty(len(numels(case)), dtype=torch.float64).uniform_(0.8, 1.2, generator=g)


def _tokens(case, seed):
    """16 x 2-style batch: each prompt with both verbalizer tokens, left-padded; the label picks one."""
    r = np.random.RandomState(seed % 2**31)
    rows, labels = [], []
    for _ in range(case["batch"]):
        prompt, label = r.randint(2, case["vocab"], r.randint(32, 65)), int(r.randint(2))
        for v in (6587, 372):
            rows.append(np.append(prompt, v % case["vocab"]))
            labels.append(label)
    width = -(-max(len(x) for x in rows) // 8) * 8
    ids, mask = np.ones((len(rows), width), np.int64), np.zeros((len(rows), width), np.int64)
    for i, x in enumerate(rows):
        ids[i, width - len(x):], mask[i, width - len(x):] = x, 1
    return torch.from_numpy(ids).to(DEV), torch.from_numpy(mask).to(DEV), torch.tensor(labels, device=DEV)


def _model(case, seed):
    """(model with its ZO set in a flat buffer, the buffer, the token embedding)"""
    from dizo_amd.synth import OPTShape, build_opt

    shape = OPTShape("case", case["layers"], case["d"], case["heads"], case["ffn"], case["vocab"], case["positions"] - 2)
    model = build_opt(shape, DT[case["dtype"]], DEV)
    flat, emb = _weights(case, seed), _embedding(case, seed)
    params = dict(model.named_parameters())
    params.pop("model.decoder.embed_tokens.weight").data.copy_(emb)
    order = _names(case)
    assert sorted(order) == sorted(params)
    for name, v in zip(order, _views(case, flat)):
        p = params[name]
        if name.endswith("layer_norm.weight"):
            v.add_(1.0)
        p.data = v.view(p.shape)
    return model, flat


def _embedding(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed + 5)
    return torch.empty(case["vocab"], case["d"], dtype=DT[case["dtype"]], device=DEV).normal_(0.0, 0.02, generator=g)


def _names(case):
    """Names of the trainable set, in the order of numels()."""
    out = ["model.decoder.embed_positions.weight", "model.decoder.final_layer_norm.weight", "model.decoder.final_layer_norm.bias"]
    for i in range(case["layers"]):
        at = "model.decoder.layers.%d." % i
        for m in ("self_attn.k_proj", "self_attn.v_proj", "self_attn.q_proj", "self_attn.out_proj", "self_attn_layer_norm", "fc1", "fc2",
                  "final_layer_norm"):
            out += [at + m + ".weight", at + m + ".bias"]
    return out


def prepare(case, seed):
    s = {"case": case, "seed": _seeds(seed), "step": 0}
    kind, dt = case["kind"], DT.get(case["dtype"])
    if kind == "normals":
        return s
    if kind == "train":
        from dizo_amd.trainer import ZOArguments, ZOTrainer

        s["model"], s["flat"] = _model(case, seed)
        ids, mask, labels = _tokens(case, seed)
        s["batch"] = dict(input_ids=ids, attention_mask=mask, labels=labels, option_len=torch.ones_like(labels), num_options=torch.full_like(labels, 2))
        s["trainer"] = ZOTrainer(s["model"], ZOArguments(learning_rate=LR, zo_eps=EPS, max_steps=10**7))
        return s
    if kind in ("steady", "passes"):
        s["flat"] = _weights(case, seed)
        s["table"] = ZOTable(_views(case, s["flat"]))
        s["grad"] = torch.tensor([_grad(case, seed)], device=DEV).to(dt)
        return s
    s["anchor"], s["flat"] = _anchored(case, seed)
    G = len(numels(case))
    s["norms"] = torch.empty(G, dtype=dt, device=DEV)
    if kind == "norms":
        s["outs"] = (torch.empty(G, dtype=torch.float64, device=DEV), torch.empty(G, dtype=torch.float32, device=DEV), s["norms"])
        L.call("dz_init", torch.cuda.current_device())
        return s
    theta0 = _views(case, s["anchor"])
    s["table"] = ProjTable(_views(case, s["flat"]), theta0)
    if kind == "spsa":
        s["ratios"] = _ratios(case, seed).to(dt).to(DEV)
    else:
        s["saved"] = s["flat"].clone()
        s["saved_table"] = ProjTable(_views(case, s["saved"]), theta0)
        s["grads"] = _views(case, _flat(case, seed + 2 * 10**6, 1e-2))
        s["gamma"] = (_ratios(case, seed) * 4e-3 * math.sqrt(numels(case)[0])).float().to(DEV)
        s["dot"] = (torch.empty(G, dtype=torch.float64, device=DEV), torch.empty(G, dtype=torch.float32, device=DEV))
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    seed = s["seed"] + s["step"]  # a step's z seed
    s["step"] += 1
    if kind == "steady":
        s["table"].perturb(seed, -2.0, EPS)
        s["table"].restore_update_perturb(seed, seed + 1, EPS, 0.0, LR, d_grad=s["grad"])
        return s["flat"]
    if kind == "passes":
        t = s["table"]
        t.perturb(seed, 1.0, EPS)
        t.perturb(seed, -2.0, EPS)
        t.restore_update(seed, EPS, 0.0, LR, d_grad=s["grad"])
        t.update(seed + 1, 0.0, LR, d_grad=s["grad"])
        return s["flat"]
    if kind == "spsa":
        G = s["norms"].numel()
        z = normals(seed, L.DZ_STREAM_GAMMA, G, G, s["norms"].dtype, s["norms"].device)
        s["table"].project(s["ratios"], L.DZ_PROJ_APPLY)
        s["table"].project(s["ratios"], L.DZ_PROJ_REVERSE_SUMSQ, norm_T=s["norms"])
        return [s["flat"], s["norms"], z]
    if kind == "fo":
        s["table"].group_sumsq(norm_T=s["norms"])
        s["table"].project(s["gamma"] / (s["norms"] + 1e-8), L.DZ_PROJ_APPLY_F32ALPHA)
        s["saved_table"].group_dot(s["grads"], *s["dot"])
        return [s["flat"], s["norms"], *s["dot"]]
    if kind == "norms":
        ns, outs, size = numels(case), s["outs"], SIZE[case["dtype"]]
        at = [a * size for a in places(case)[0]]
        L.call("dz_group_sumsq_static", L.u64_array([s["flat"].data_ptr() + a for a in at]), L.u64_array([s["anchor"].data_ptr() + a for a in at]),
               L.i64_array(ns), len(ns), {"fp32": L.DZ_DTYPE_F32, "fp16": L.DZ_DTYPE_F16, "bf16": L.DZ_DTYPE_BF16}[case["dtype"]],
               *(ctypes.c_void_p(o.data_ptr()) for o in outs), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        return list(outs)
    if kind == "normals":
        return normals(s["seed"], L.DZ_STREAM_PARAM, case["offset"], case["n"], DT[case["dtype"]], torch.device(DEV, torch.cuda.current_device()))
    np.random.seed(seed % 2**32)  # the trainer draws its z seed from numpy's generator
    loss = s["trainer"].training_step(s["batch"])
    return [loss, s["flat"]]


# ------------------------------------------------------------------- work --
def work(case):
    kind, size = case["kind"], SIZE[case["dtype"]]
    if kind == "normals":
        return {"bytes": case["n"] * size, "flops": 0}
    P = sum(numels(case))
    tensors = P * size
    if kind in ("steady", "passes"):
        return {"bytes": 2 * tensors * (2 if kind == "steady" else 4), "flops": 0}
    if kind == "spsa":  # two passes, each reads theta and theta0 and writes theta
        return {"bytes": 6 * tensors, "flops": 0}
    if kind == "fo":  # norms 2, apply 3, reduction 3
        return {"bytes": 8 * tensors, "flops": 0}
    if kind == "norms":
        return {"bytes": 2 * tensors, "flops": 0}
    # training step: two parameter passes, and two forwards (each matrix once, its products over every token)
    tokens = 2 * case["batch"] * 48
    d, f = case["d"], case["ffn"]
    products = case["layers"] * (4 * d * d + 2 * d * f) + d * case["vocab"]
    return {"bytes": 4 * tensors + 2 * products * size, "flops": 2 * 2 * tokens * products}


def tolerance(case):
    # z and each rounded operation on the parameters are defined bit for bit
    if case["kind"] in ("steady", "passes", "normals"):
        return "exact"
    # sums of squares and products run in 64 bits and come out in 32 or 16: another order of summation moves
    # them by about 1e-15, which all but never changes a rounded value; one that changes is 6e-8 (32 bits) off
    if case["kind"] in ("spsa", "fo", "norms"):
        return {"rel": 1e-6, "max": 1e-5}
    # a whole step: its forwards in the data type
    return {"rel": 1e-5 if case["dtype"] == "fp32" else 1e-2}


# ------------------------------------------------------------------ exact --
def _philox_z(case, seed, stream, first, n):
    """z of elements first .. first + n - 1 as the generator defines it: Philox4x32 with 7 rounds (Salmon et
    al., SC'11) on the counter (stream, q low, 0, q high) for each 8 elements, each 16-bit field a sign and an
    index into the normal quantiles, rounded to the data type."""
    i = torch.arange(32768, dtype=torch.float64, device=DEV)
    quant = torch.special.ndtri(0.5 + (i + 0.5) / 65536).to(DT[case["dtype"]]).double()
    out = torch.empty(n, dtype=torch.float64, device=DEV)
    M = 0xFFFFFFFF
    for at in range(0, n, 1 << 27):
        m = min(n - at, 1 << 27)
        lo = first + at
        q = torch.arange(lo // 8, (lo + m + 7) // 8, dtype=torch.int64, device=DEV)
        x, y, z, w = torch.full_like(q, stream), q & M, torch.zeros_like(q), q >> 32
        k0, k1 = seed & M, seed >> 32
        for _ in range(7):
            p, r = x * 0xD2511F53, z * 0xCD9E8D57
            x, y, z, w = ((r >> 32) & M) ^ y ^ k0, r & M, ((p >> 32) & M) ^ w ^ k1, p & M
            k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
        h = torch.stack([v >> s & 0xFFFF for v in (x, y, z, w) for s in (0, 16)], 1).reshape(-1)[lo % 8:lo % 8 + m]
        v = quant[h & 0x7FFF]
        out[at:at + m] = torch.where(h >= 0x8000, -v, v)
    return out


def _add_z(case, flat, seed, factor):
    at = 0
    for v in _views(case, flat):
        v.add_(_philox_z(case, seed, 0, at, v.numel()), alpha=factor)
        at += -(-v.numel() // 8) * 8


def _norms(case, a, b):
    return torch.stack([(x.double() - y.double()).square().sum() for x, y in zip(_views(case, a), _views(case, b))])


def exact(case, seed):
    kind, first = case["kind"], _seeds(seed)
    if kind == "normals":
        return _philox_z(case, first, 0, case["offset"], case["n"])
    if kind in ("steady", "passes"):
        flat = _weights(case, seed).double()
        g = float(torch.tensor(_grad(case, seed)).to(DT[case["dtype"]]))
        _add_z(case, flat, first, -EPS - LR * g if kind == "steady" else -LR * g)
        _add_z(case, flat, first + 1, EPS if kind == "steady" else -LR * g)
        return flat
    if kind == "train":
        return _exact_train(case, seed)
    anchor, flat = _anchored(case, seed)
    squares = _norms(case, flat, anchor)
    if kind == "norms":
        return [squares, squares.sqrt(), squares.sqrt()]
    if kind == "spsa":
        G = len(numels(case))
        return [flat.double(), squares.sqrt(), _philox_z(case, first, 1, G, G)]
    grads = _flat(case, seed + 2 * 10**6, 1e-2)
    dot = torch.stack([(g.double() * (x.double() - y.double())).sum()
                       for g, x, y in zip(_views(case, grads), _views(case, flat), _views(case, anchor))])
    gamma = (_ratios(case, seed) * 4e-3 * math.sqrt(numels(case)[0])).to(DEV)
    out = flat.double()
    for v, a, ratio in zip(_views(case, out), _views(case, anchor), gamma / squares.sqrt()):
        v.copy_(a.double() + (v - a.double()) * ratio)
    return [out, squares.sqrt(), dot, dot]


def _exact_train(case, seed):
    """The loss at theta + eps z, and theta + eps z - 2 eps z: what one step leaves (its restore and update
    run with the next step's perturbation)."""
    flat = _weights(case, seed)
    names = _names(case)
    for name, v in zip(names, _views(case, flat)):
        if name.endswith("layer_norm.weight"):
            v.add_(1.0)
    flat = flat.double()
    np_state = np.random.get_state()
    np.random.seed(first_seed(seed))
    z_seed = int(np.random.randint(1000000000))
    np.random.set_state(np_state)
    _add_z(case, flat, z_seed, EPS)
    P = dict(zip(names, _views(case, flat)))
    ids, mask, labels = _tokens(case, seed)
    loss = _exact_loss(case, P, _embedding(case, seed).double(), ids, mask, labels)
    _add_z(case, flat, z_seed, -2 * EPS)
    return [loss, flat]


def first_seed(seed):
    return _seeds(seed) % 2**32


def _exact_loss(case, P, emb, ids, mask, labels):
    """OPT in 64 bits: the option-masked classification loss of one batch."""
    F = torch.nn.functional
    d, heads, at = case["d"], case["heads"], "model.decoder."

    def linear(x, name, rows):
        return F.linear(x, P[name + ".weight"].view(rows, -1), P[name + ".bias"])

    def norm(x, name):
        return F.layer_norm(x, (d,), P[name + ".weight"], P[name + ".bias"])

    place = (mask.cumsum(1) * mask - 1) + 2
    x = emb[ids] + P[at + "embed_positions.weight"].view(-1, d)[place]
    B, T = ids.shape
    seen = (torch.ones(T, T, dtype=torch.bool, device=DEV).tril() & mask.bool()[:, None, :])[:, None]
    seen = seen | ~seen.any(-1, keepdim=True)  # rows of padding: any values, which nothing reads
    for i in range(case["layers"]):
        p = at + "layers.%d." % i
        h = norm(x, p + "self_attn_layer_norm")
        q, k, v = (linear(h, p + "self_attn.%s_proj" % m, d).view(B, T, heads, -1).transpose(1, 2).contiguous() for m in "qkv")
        a = (q @ k.transpose(-1, -2).contiguous()) / math.sqrt(d // heads)
        a = a.masked_fill(~seen, -math.inf).softmax(-1)
        x = x + linear((a @ v).transpose(1, 2).reshape(B, T, d), p + "self_attn.out_proj", d)
        h = linear(norm(x, p + "final_layer_norm"), p + "fc1", case["ffn"]).relu()
        x = x + linear(h, p + "fc2", d)
    last = F.linear(norm(x[:, -2], at + "final_layer_norm"), emb).log_softmax(-1)
    chosen = last.gather(1, ids[:, -1:]).view(-1, 2)
    return F.cross_entropy(chosen, labels.view(-1, 2)[:, 0])
