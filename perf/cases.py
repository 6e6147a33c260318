"""The work a user of the MoE layer has it do, as cases that can be timed.

Every case is one MOLEModule driven through its public interface: a forward pass under no_grad (serving), a forward and a
backward pass (training; gradient accumulation over two micro-batches and the load-balancing loss among the options), with
the experts resident on the GPU or in pinned host memory behind the slot pool, on the layer's own ragged layout or on the
reference's padded one, in bf16 or fp32.  Weights are N(0, 0.02), tokens N(0, 1), the output's gradient N(0, 1e-3), as in
bench.py.

A case: kind "forward" | "train", S tokens, M width, E experts, k choices, F hidden width, cf capacity factor (0: nothing is
dropped), dtype "bf16" | "fp32", zipf (per-expert logit bias with Zipf(1.2) loads), padded (reference_layout), offloaded (all
experts in pinned host memory), pool (slots on the GPU), micro (micro-batches of S tokens per pass), aux (weight of l_aux in
the loss, 0: not used).
"""
import math

import torch

from mole_amd import core
from mole_amd.moe.layer import MOLEModule

DEFAULTS = dict(cf=0.0, dtype="bf16", zipf=False, padded=False, offloaded=False, pool=-1, micro=1, aux=0.0)


def _case(name, kind, S, M, E, k, F, **kw):
    return dict(DEFAULTS, name=name, kind=kind, S=S, M=M, E=E, k=k, F=F, **kw)


def listed():
    return [
        # serving: one token of one sequence through the large sparse layer: launches, latency, two experts' weights
        _case("decode 1 token", "forward", 1, 2048, 64, 2, 8192),
        # serving: one token for each of a batch of sequences, a Switch-style layer (every expert gets a few rows)
        _case("decode 61 tokens", "forward", 61, 1024, 16, 1, 4096),
        # serving: a larger decode batch on a fine-grained layer, 256 experts with about eight rows each
        _case("decode 256 fine-grained", "forward", 256, 2048, 256, 8, 1024),
        # serving: the prompt of one request, ragged length
        _case("prefill 3001 tokens", "forward", 3001, 1024, 16, 2, 4096),
        # the reference's own dtype, a short batch forward
        _case("forward fp32 777 tokens", "forward", 777, 512, 8, 2, 2048, cf=1.0, dtype="fp32"),
        # training: small micro-batches of odd length, widths that are no multiple of 64, gradients summed over two of them,
        # load-balancing loss
        _case("train 2 x 513 odd widths", "train", 513, 520, 16, 4, 1416, micro=2, aux=0.01),
        # training: the reference's literal call sequence (extract_critical, encode into [E, C, M], decode)
        _case("train padded layout", "train", 2048, 512, 16, 2, 1024, cf=1.25, padded=True, aux=0.01),
        # training in fp32 at the reference's default capacity factor: the CPU-runnable configuration
        _case("train fp32 4096 tokens", "train", 4096, 512, 8, 2, 2048, cf=1.0, dtype="fp32"),
        # training: Switch-style layer, top-1 with capacity drop (the headline configuration)
        _case("train 16384 top-1", "train", 16384, 1024, 16, 1, 4096, cf=1.25),
        # training: 64 experts under Zipf-distributed loads, 4.3 GB of weights and as much of gradients
        _case("train 8192 skewed", "train", 8192, 2048, 64, 2, 8192, zipf=True),
        # training: the fine-grained layer, 262144 routed rows
        _case("train 32768 fine-grained", "train", 32768, 2048, 256, 8, 1024),
        # training with the experts in pinned host memory and fewer slots on the GPU than experts
        _case("train offloaded experts", "train", 1024, 1024, 8, 2, 4096, offloaded=True, pool=4),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        c = dict(DEFAULTS)
        c["kind"] = rng.choice(["forward", "train"])
        c["dtype"] = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        c["S"] = _log_uniform(rng, 1, 32768)
        grain = rng.choice([64, 64, 64, 8])              # most widths are multiples of 64, some only of 8
        c["M"] = max(grain, _log_uniform(rng, 256, 4096) // grain * grain)
        c["F"] = max(grain, int(c["M"] * rng.choice([0.5, 1, 2, 3, 4])) // grain * grain)
        c["E"] = _log_uniform(rng, 4, 256)
        c["k"] = min(rng.choice([1, 2, 2, 4, 8]), c["E"])
        c["cf"] = rng.choice([0.0, 0.0, 1.0, 1.25, 2.0])
        c["zipf"] = rng.random() < 0.2
        c["padded"] = rng.random() < 0.15
        if c["padded"] and c["cf"] == 0.0:
            c["cf"] = 1.25
        if c["kind"] == "train":
            c["micro"] = rng.choice([1, 1, 1, 2])
            c["aux"] = rng.choice([0.0, 0.01])
            if not c["padded"] and c["micro"] == 1 and rng.random() < 0.15:
                c["E"] = min(c["E"], 16)
                c["k"] = min(c["k"], 2)
                c["offloaded"], c["pool"] = True, max(2, c["E"] // 2)
        weights = 2 * c["E"] * c["M"] * c["F"]
        flops = work(c)["flops"]
        slow = (16 if c["dtype"] == "fp32" else 1) * (4 if grain == 8 else 1)
        if weights > (2.2e9 if c["dtype"] == "bf16" else 1.1e9) or flops * slow > 6.0e12:
            continue
        if c["offloaded"] and weights > 1.0e8:           # host initialisation and pinning take their time
            continue
        if c["padded"] and c["S"] * c["k"] * c["cf"] * (2 * c["M"] + 3 * c["F"]) > 4.0e9:
            continue
        return c


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _layer(case, g):
    E, M, F, off = case["E"], case["M"], case["F"], case["offloaded"]
    pool = case["pool"] if off else -1
    um = core.get_UniMem()
    if off and um is not None and (um.F, um.M, um.dtype, um.pool_size) == (F, M, _dtype(case), pool):
        MOLEModule._instance = []        # the layers of a process share one slot pool; earlier ones may go
    else:
        MOLEModule.reset_instances()
    bias = None
    if case["zipf"]:
        ranks = torch.randperm(E, generator=g, device="cuda").float() + 1.0
        bias = torch.log(ranks ** -1.2)
    m = MOLEModule(E if off else 0, 0 if off else E, M, F, pool, case["k"], 2 if off else 4,
                   {"local_rank": 0, "world_size": 1, "rank": 0}, "gelu", case["micro"], False, off, dtype=_dtype(case),
                   gate_logit_bias=bias, reference_layout=case["padded"])
    with torch.no_grad():
        m.gate[0].linear.weight.normal_(0.0, 1.0 / M ** 0.5, generator=g)
        stores = (m.FC1_W_CPU, m.FC1_B_CPU, m.FC2_W_CPU, m.FC2_B_CPU) if off else (m.FC1_W_GPU, m.FC1_B_GPU, m.FC2_W_GPU, m.FC2_B_GPU)
        for p in stores:
            t = p.all_tensors
            if off:
                t.copy_(torch.empty(t.shape, dtype=t.dtype, device="cuda").normal_(0.0, 0.02, generator=g))
            else:
                t.normal_(0.0, 0.02, generator=g)
    return m


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt, S, M = _dtype(case), case["S"], case["M"]
    st = {"case": case, "layer": _layer(case, g)}
    new = lambda scale: (torch.randn(S, M, device="cuda", generator=g) * scale).to(dt)
    train = case["kind"] == "train"
    st["x"] = [new(1.0).requires_grad_(train) for _ in range(case["micro"])]
    if train:
        st["dy"] = [new(1e-3) for _ in range(case["micro"])]
        st["aux"] = torch.tensor(case["aux"], device="cuda") if case["aux"] else None
    return st


def run(st):
    case, m = st["case"], st["layer"]
    if case["kind"] == "forward":
        with torch.no_grad():
            return {"y": m(st["x"][0], capacity_factor=case["cf"])}
    wg = m.gate[0].linear.weight
    wg.grad = None
    if case["micro"] > 1:                # the optimizer's zero_grad at the start of an accumulation window
        for p in m.s_experts_param():
            p.grad.zero_()
    ys = []
    for x, dy in zip(st["x"], st["dy"]):
        x.grad = None
        y = m(x, capacity_factor=case["cf"])
        if st["aux"] is not None:
            torch.autograd.backward([y, m.l_aux], [dy, st["aux"]])
        else:
            y.backward(dy)
        ys.append(y.detach())
    if case["offloaded"]:
        core.synchronize_tran()          # the optimizer on the host reads the gradients next
        grads = [t.grad_ for t in m.d_experts_param()]
    else:
        grads = [p.grad for p in m.s_experts_param()]
    return {"y": ys, "dx": [x.grad for x in st["x"]], "dwg": wg.grad, "grads": grads}


def _loads(case):
    """Expected rows of every expert and the expected number of experts that get any."""
    S, E, k = case["S"], case["E"], case["k"]
    p = [1.0 / E] * E
    if case["zipf"]:
        w = [(i + 1.0) ** -1.2 for i in range(E)]
        p = [v / sum(w) for v in w]
    cap = k * int(case["cf"] * ((S + E - 1) // E)) if case["cf"] > 0 else S
    hit = [min(1.0, k * v) for v in p]
    total = sum(hit)
    rows = [S * k * h / total for h in hit]
    active = sum(1.0 - (1.0 - h) ** S for h in hit)
    return sum(min(r, cap) for r in rows), min(active, S * k)


def work(case):
    """One pass: tokens, gate, and the weights of the experts that get rows are read once, results (training: the
    gradients of all experts) written once; flops of the gate and of the kept rows' expert products."""
    S, M, E, F, n = case["S"], case["M"], case["E"], case["F"], case["micro"]
    b = 2 if case["dtype"] == "bf16" else 4
    rows, active = _loads(case)
    expert = 2 * F * M + F + M
    nbytes = 2 * S * M * b + 4 * E * M + active * expert * b
    flops = 2.0 * S * M * E + 4.0 * rows * M * F
    if case["kind"] == "train":
        nbytes = n * 4 * S * M * b + 8 * E * M + (active + E) * expert * b
        flops = n * 3.0 * flops
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    """About four times what the outputs differ by from the same layer in fp64 with the same routing decisions (all outputs of
    all listed kinds: bf16 up to 3.4e-3 in the 2-norm and 0.042 for one value, fp32 9.4e-7 and 8.2e-6; wider fp32 layers sum
    longer)."""
    return {"rel": 1.2e-2, "max": 0.16} if case["dtype"] == "bf16" else {"rel": 5e-6, "max": 5e-5}
