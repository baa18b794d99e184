"""The work that a user of this library has it do: MoE layers, from one decode token to a prefill chunk.

Each case is one call (or, for ``stack``, one token's calls) of the public Python entry points:

  experts   ``ExpertStore`` + ``make_experts_forward``: the routed-compute step bound into an engine's
            layer, ``forward(hidden_states, top_k_index, top_k_weights)``; the routing is an input
  block     ``moe_block``: router from its weights, routed experts, shared expert if the shape has one
  layer     ``moe_layer``: RMSNorm, the block and the residual add
  stack     ``moe_layer`` for each of a residency ledger's layers, one token, logits supplied

and the experts are exact bf16, int4 with group-128 bf16 scales, or int4 with one fp16 scale per row.
``prepare`` builds a layer's seeded weights, its pointer table and a workspace, as a program keeps them.
"""
import math

import torch

from tarfa_amd import moe as tm
from tarfa_amd import seeded
from tarfa_amd.experts import ExpertStore, make_experts_forward
from tarfa_amd.moe import MoEShape, Workspace
from tarfa_amd.residency import ResidencyLedger, zipf_logits

EPS = 1e-6


def _case(name, entry, weights, H, E, I, k, Is, T, layers=1):
    return {"name": name, "entry": entry, "weights": weights, "H": H, "E": E, "I": I, "k": k, "Is": Is, "T": T,
            "layers": layers}


def listed():
    return [
        # One decode token through the small layer (the one the CPU reference runs): latency and host calls only.
        _case("decode_small", "experts", "bf16", 1024, 32, 512, 8, 0, 1),
        # The headline: one decode token through the full-size layer, router and shared expert included.
        _case("decode", "block", "bf16", 2560, 256, 1024, 8, 1024, 1),
        # The same token in the int4 fast mode, as a decoder layer calls it (norm in, residual out).
        _case("decode_int4", "layer", "int4", 2560, 256, 1024, 8, 1024, 1),
        # One token through six full-size layers back to back, Zipf-popular routing: the decode loop.
        _case("decode_stack", "stack", "bf16", 2560, 256, 1024, 8, 1024, 1, layers=6),
        # A handful of sequences decoded together (or a short draft verified at once).
        _case("batch_6", "layer", "bf16", 2560, 256, 1024, 8, 1024, 6),
        # The same kind of batch in the int4 fast mode.
        _case("batch_12_int4", "block", "int4", 2560, 256, 1024, 8, 1024, 12),
        # A serving batch of decode tokens: most experts hit by one or two tokens each.
        _case("batch_40", "block", "bf16", 2560, 256, 1024, 8, 1024, 40),
        # A short prompt through a mid-size layer without a shared expert (I no multiple of 512), by way of
        # the engine's experts step.
        _case("prompt_211_mid", "experts", "bf16", 2048, 128, 768, 8, 0, 211),
        # A prompt through the reference's own int4 files' layout.
        _case("prompt_603_int4_rows", "experts", "int4_rows", 2560, 256, 1024, 8, 0, 603),
        # A prefill chunk of ordinary size.
        _case("prefill_1024", "layer", "bf16", 2560, 256, 1024, 8, 1024, 1024),
        # The prefill chunk of the headline configuration, exact and in the int4 fast mode.
        _case("prefill_4096", "block", "bf16", 2560, 256, 1024, 8, 1024, 4096),
        _case("prefill_4096_int4", "block", "int4", 2560, 256, 1024, 8, 1024, 4096),
    ]


def draw(rng):
    while True:
        T = int(math.exp(rng.uniform(0.0, math.log(4096.999))))
        H = rng.choice([1024, 1536, 2048, 2560, 2560, 3072])
        E = rng.choice([32, 64, 128, 160, 256, 256])
        I = rng.choice([512, 640, 768, 1024, 1024])
        k = rng.choice([4, 6, 8, 8, 8])
        weights = rng.choice(["bf16", "bf16", "int4", "int4_rows"])
        entry = rng.choice(["experts", "block", "layer"])
        if T == 1 and rng.random() < 0.3:
            entry = "stack"
        layers = rng.randint(2, 6) if entry == "stack" else 1
        if weights == "int4_rows" and entry in ("layer", "stack"):
            continue                                   # those entry points take bf16 or group-scaled int4
        if weights != "bf16" and T == 1 and (H % 512 or I % 512):
            continue                                   # int4 decode takes multiples of 512
        if E < 2 * k:
            continue
        Is = rng.choice([0, I]) if entry != "experts" else 0
        c = _case("", entry, weights, H, E, I, k, Is, T, layers)
        del c["name"]
        cost, most = work(c), work(listed()[-2])
        if cost["bytes"] > most["bytes"] or cost["flops"] > most["flops"]:
            continue                                   # no more than the headline prefill chunk
        return c


# ---------------------------------------------------------------------------- inputs
def _shape(c):
    return MoEShape(c["H"], c["E"], c["I"], c["k"], c["Is"])


def _quantised(c, layer):
    """The layer's experts in int4: the packed rows and their scales, gate_up then down."""
    parts = []
    for w in (layer.gate_up, layer.down):
        q, s = tm.quantize_int4(w)
        if c["weights"] == "int4_rows":
            s = s.float().amax(-1).to(torch.float16)       # one scale per row
        parts += [q, s.contiguous()]
    return parts


def prepare(case, seed):
    dev = torch.device("cuda")
    shape = _shape(case)
    T, H = case["T"], case["H"]
    st = {"case": case, "shape": shape}
    if case["entry"] == "stack":
        L = case["layers"]
        ledger = ResidencyLedger(shape, L, device=dev, int4=case["weights"] == "int4")
        ledger.fill_seeded(seed)
        st["ledger"], st["ws"] = ledger, Workspace(shape, dev)
        st["shared"] = [seeded.make_block_weights(shape, seed, l, dev)[1] for l in range(L)]
        st["ln_w"] = [tm.fill_bf16(torch.empty(H, dtype=torch.bfloat16, device=dev), seed + 7000 + l, 0.1)
                      for l in range(L)]
        st["h"] = seeded.make_tokens(shape, seed, 1, device=dev)
        st["logits"] = zipf_logits(shape, L, 1, seed, device=dev)[0].reshape(L, 1, -1).contiguous()
        return st
    layer = seeded.make_layer(shape, seed, device=dev)
    st["router_w"], st["shared"] = layer.router_w, layer.shared
    st["x"] = seeded.make_tokens(shape, seed, T, device=dev)
    if case["weights"] == "bf16":
        parts = [layer.gate_up, layer.down]
    else:
        parts = _quantised(case, layer)
    st["parts"] = parts
    del layer
    if case["entry"] == "experts":
        make = {"bf16": ExpertStore.from_slabs, "int4": ExpertStore.from_int4, "int4_rows": ExpertStore.from_int4_rows}
        store = make[case["weights"]](shape, *parts)
        store.workspace.ensure(T)
        st["store"], st["forward"] = store, make_experts_forward(store, jtopk=8)
        st["ids"], st["w"], _ = tm.router_topk(shape, x=st["x"], router_w=st["router_w"])
        return st
    table = {"bf16": tm.expert_table, "int4": tm.expert_table_q4, "int4_rows": tm.expert_table_q4_rows}
    st["table"] = table[case["weights"]](*parts)
    st["ws"] = Workspace(shape, dev, tokens=T)
    if case["entry"] == "layer":
        st["ln_w"] = tm.fill_bf16(torch.empty(H, dtype=torch.bfloat16, device=dev), seed + 7000, 0.1)
    return st


# ---------------------------------------------------------------------------- one pass
def run(st):
    entry, shape = st["case"]["entry"], st["shape"]
    if entry == "experts":
        return st["forward"](None, st["x"], st["ids"], st["w"])
    if entry == "block":
        return tm.moe_block(shape, st["x"], st["table"], st["ws"], router_w=st["router_w"], shared=st["shared"])
    if entry == "layer":
        return tm.moe_layer(shape, st["x"], st["ln_w"], EPS, st["table"], st["ws"], router_w=st["router_w"],
                            shared=st["shared"])
    h, outs = st["h"], []
    for l in range(st["ledger"].L):
        h, ids, w = tm.moe_layer(shape, h, st["ln_w"][l], EPS, st["ledger"].table(l), st["ws"],
                                 logits=st["logits"][l], shared=st["shared"][l])
        outs += [h, ids, w]
    return outs


# ---------------------------------------------------------------------------- what it cannot do without

def work(case):
    H, E, I, k, Is, T, L = (case[n] for n in ("H", "E", "I", "k", "Is", "T", "layers"))
    hit = k if T == 1 else E * (1.0 - (1.0 - k / E) ** T)
    per = {"bf16": 2.0, "int4": 0.5 + 2.0 / 128, "int4_rows": 0.5}[case["weights"]]
    nbytes = hit * 3 * H * I * per + 2 * T * H * 2
    if case["weights"] == "int4_rows":
        nbytes += hit * 2 * (2 * I + H)
    flops = 6.0 * T * k * H * I
    if Is:
        nbytes += 2 * (3 * H * Is + H)
        flops += 6.0 * T * H * Is
    if case["entry"] in ("block", "layer"):
        nbytes += 2 * E * H
        flops += 2.0 * T * E * H
    if case["entry"] == "stack":
        nbytes += 4 * E
    nbytes += T * k * 10
    return {"bytes": nbytes * L, "flops": flops * L}


def tolerance(case):
    # A layer's output is 2e-3 to 6e-3 from the same sums in 64 bits (bf16 roundings after every product and
    # addition; measured for every listed case), and two implementations that round at other places differ by
    # about that much.  A token whose 8th and 9th logits lie within a fp32 sum's rounding may list the other.
    return {"rel": 1e-2, "differ": 2e-4}


# ---------------------------------------------------------------------------- the same in 64 bits
def _dequant(q, s):
    q = q.to(torch.int32)
    n = torch.stack([q & 15, q >> 4], dim=-1).reshape(*q.shape[:-1], -1).double() - 8.0
    if s.dim() == q.dim() - 1:
        s = s.unsqueeze(-1)
    return n * s.double().repeat_interleave(n.shape[-1] // s.shape[-1], dim=-1)


def _expert(parts, e):
    if len(parts) == 2:
        return parts[0][e].double(), parts[1][e].double()
    return _dequant(parts[0][e], parts[1][e]), _dequant(parts[2][e], parts[3][e])


def _mlp(x, gate_up, down):
    g, u = (x @ gate_up.T).chunk(2, dim=-1)
    return (torch.nn.functional.silu(g) * u) @ down.T


def _experts64(x, ids, w, parts):
    out = torch.zeros_like(x)
    for e in torch.unique(ids).tolist():
        t, s = (ids == e).nonzero(as_tuple=True)
        gu, dn = _expert(parts, e)
        out.index_add_(0, t, _mlp(x[t], gu, dn) * w[t, s].unsqueeze(-1))
    return out


def _route64(logits, k):
    p, ids = torch.topk(torch.softmax(logits.double(), dim=-1), k, dim=-1)
    return ids, p / p.sum(-1, keepdim=True)


def _norm64(h, w):
    return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * (1.0 + w.double())


def _block64(x, logits, k, parts, shared):
    ids, w = _route64(logits, k)
    out = _experts64(x, ids, w, parts)
    if shared is not None:
        g, u, d, sg = (t.double() for t in shared)
        out += torch.sigmoid(x @ sg.reshape(-1, 1)) * _mlp(x, torch.cat([g, u]), d)
    return out, ids, w


def exact(case, seed):
    st = prepare(case, seed)
    k = case["k"]
    if case["entry"] == "experts":
        return _experts64(st["x"].double(), st["ids"], st["w"].double(), st["parts"])
    if case["entry"] == "stack":
        h, outs = st["h"].double(), []
        for l in range(case["layers"]):
            y, ids, w = _block64(_norm64(h, st["ln_w"][l]), st["logits"][l], k, st["ledger"].hbm[l], st["shared"][l])
            h = h + y
            outs += [h, ids, w]
        return outs
    h = st["x"].double()
    x = _norm64(h, st["ln_w"]) if case["entry"] == "layer" else h
    out, ids, w = _block64(x, x @ st["router_w"].double().T, k, st["parts"], st["shared"])
    return (h + out if case["entry"] == "layer" else out), ids, w
