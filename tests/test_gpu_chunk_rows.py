"""The prefill GEMMs' chunk sizes: groups at the edges of 16- to 160-row chunks, at widths that take four
or five weight stages per cycle, against the oracle's chain at the bf16 bars; every case asserts the chunk
size that it runs."""
import numpy as np
import pytest
import torch

from oracle import bf16, moe
from tarfa_amd import moe as tm
from tarfa_amd import seeded
from tarfa_amd.moe import MoEShape, Workspace
from tests._util import assert_close_bf16, expert_dicts, f32
from tests.test_chunk_rows import hot, plan, uniform

pytestmark = pytest.mark.gpu

ROWS = [1, 31, 32, 33, 64, 65]


def _ids(rows, seed):
    """One expert per token, expert e taken by rows[e] tokens in a shuffled order."""
    ids = np.repeat(np.arange(len(rows)), rows)
    np.random.default_rng(seed).shuffle(ids)
    return ids[:, None].astype(np.int64)


def _device_rows(shape, T, ws, p):
    """The rows per chunk that the last call's dispatch chose."""
    assert shape.ws_bytes(T) <= ws.buf.numel()
    return int(ws.buf[p[4]:p[4] + 4].cpu().view(torch.int32)[0])


EDGES = [1, 31, 32, 33, 63, 64, 65, 128, 129, 159, 160, 161, 320, 321]


@pytest.mark.parametrize("H,I,rows,chunk", [
    (768, 640, ROWS + [0] * 10, 32), (1280, 512, ROWS, 32), (512, 768, ROWS + [0] * 10, 32),
    (768, 640, EDGES, 64), (1280, 512, EDGES, 64), (512, 768, EDGES, 64),
    (768, 640, EDGES * 4, 160), (1280, 512, EDGES * 3, 160), (512, 768, EDGES * 4, 160)])
def test_bf16_chunk_edges(gpu, H, I, rows, chunk):
    E = len(rows)
    shape = MoEShape(H, E, I, 1, 0)
    layer = seeded.make_layer(shape, H + E, device=gpu)
    ids = _ids(rows, H)
    T = len(ids)
    p = plan(T, H, E, I, 1, counts=rows)
    assert p[0] == chunk
    ws = Workspace(shape, gpu, tokens=T)
    x = seeded.make_tokens(shape, H + E, T, device=gpu)
    w = torch.linspace(0.1, 1.0, T, device=gpu).to(torch.bfloat16)[:, None].contiguous()
    out = tm.experts_forward(shape, x, torch.from_numpy(ids).to(gpu), w, tm.expert_table(layer.gate_up, layer.down),
                             ws)
    assert _device_rows(shape, T, ws, p) == chunk
    gu, dn = expert_dicts(layer.gate_up, layer.down, ids)
    assert_close_bf16(f32(out), moe.experts_prefill(f32(x), ids, f32(w), gu, dn, E), f"H={H} I={I} chunk={chunk}")
    ws.status()


@pytest.mark.parametrize("T,I,routing,chunk", [
    (17, 768, uniform, 32), (90, 768, uniform, 32), (300, 768, uniform, 64), (160, 768, hot, 32),
    (1000, 768, hot, 64), (2000, 768, uniform, 160), (4096, 640, uniform, 160), (4096, 640, hot, 160)])
def test_bf16_chunks_with_shared_expert(gpu, T, I, routing, chunk):
    """The shared expert in the same chunks; a routing that spreads over the experts, and one that sends
    every token to the same four (group sizes that only the dispatch sees).  I = 640: the 160-row down
    GEMM's five-stage cycles."""
    E, k = 16, 4
    shape = MoEShape(768, E, I, k, I)
    layer = seeded.make_layer(shape, T, device=gpu)
    ws = Workspace(shape, gpu, tokens=T)
    x = seeded.make_tokens(shape, T, T, device=gpu)
    logits = seeded.make_logits(shape, T, T, device=gpu)
    if routing is hot:
        logits[:, :k] += 1000.0
    table = tm.expert_table(layer.gate_up, layer.down)
    out, ids, w = tm.moe_block(shape, x, table, ws, logits=logits, shared=layer.shared)
    ids = ids.cpu().numpy()
    assert np.array_equal(ids, moe.router_topk(logits.cpu().numpy(), k)[0])
    p = plan(T, 768, E, I, k, I, counts=np.bincount(ids.ravel(), minlength=E))
    assert p[0] == chunk and _device_rows(shape, T, ws, p) == chunk
    gu, dn = expert_dicts(layer.gate_up, layer.down, ids)
    ref = moe.add_bf16(moe.experts_prefill(f32(x), ids, f32(w), gu, dn, E),
                       moe.shared_expert(f32(x), *[f32(t) for t in layer.shared]))
    assert_close_bf16(f32(out), ref, f"T={T}")
    ws.status()


def _q4(layer, rows, gpu):
    """(table, dequantised gate_up and down per expert) of the layer in int4."""
    parts = []
    for w in (layer.gate_up, layer.down):
        q, s = tm.quantize_int4(w)
        if rows:
            s = s.float().amax(-1).to(torch.float16)           # one scale per row
        parts += [q, s.contiguous()]
    deq = []
    for q, s in (parts[:2], parts[2:]):
        q = q.cpu().numpy()
        n = np.stack([q & 15, q >> 4], axis=-1).reshape(*q.shape[:-1], -1).astype(np.float32) - 8.0
        s = s.float().cpu().numpy()
        s = s[..., None] if rows else np.repeat(s, 128, axis=-1)
        deq.append(bf16.to_f32(bf16.bits(n * s)))
    table = (tm.expert_table_q4_rows if rows else tm.expert_table_q4)(*parts)
    return parts, table, dict(enumerate(deq[0])), dict(enumerate(deq[1]))


@pytest.mark.parametrize("rows", [False, True])
@pytest.mark.parametrize("H,I,E", [(512, 512, 40), (768, 640, 40), (512, 640, 16), (768, 512, 16), (768, 640, 6)])
def test_int4_chunk_edges(gpu, H, I, E, rows):
    """Means of 6, 14 and 38 rows: 16-, 32- and 64-row chunks; K of 4 (the fewest), 5 and 6 stages."""
    shape = MoEShape(H, E, I, 1, 0)
    assert plan(sum(ROWS), H, E, I, 1, q4=1 + rows)[0] == {40: 16, 16: 32, 6: 64}[E]
    layer = seeded.make_layer(shape, H + E, device=gpu)
    parts, table, gu, dn = _q4(layer, rows, gpu)
    ids = _ids(ROWS, H)
    T = len(ids)
    ws = Workspace(shape, gpu, tokens=T)
    x = seeded.make_tokens(shape, H + E, T, device=gpu)
    w = torch.linspace(0.1, 1.0, T, device=gpu).to(torch.bfloat16)[:, None].contiguous()
    out = tm.experts_forward(shape, x, torch.from_numpy(ids).to(gpu), w, table, ws)
    assert_close_bf16(f32(out), moe.experts_prefill(f32(x), ids, f32(w), gu, dn, E), f"H={H} I={I} E={E}")
    ws.status()


@pytest.mark.parametrize("rows", [False, True])
@pytest.mark.parametrize("T,I,chunk,fuse", [(2, 512, 16, 1), (4, 768, 16, 1), (33, 512, 16, 1), (90, 512, 32, 1),
                                            (200, 512, 64, 0), (33, 640, 16, 0), (900, 640, 64, 0)])
def test_int4_chunks_with_shared_expert(gpu, T, I, chunk, fuse, rows):
    """Mean groups of 0.5 to 225 rows; the shared expert's tiles inside the int4 launches (I = 512, up to
    32-row chunks) or in launches of their own."""
    shape = MoEShape(768, 16, I, 4, I)
    assert plan(T, 768, 16, I, 4, I, q4=1 + rows)[:4] == [chunk, 32 if fuse else 64, fuse, 1]
    layer = seeded.make_layer(shape, T, device=gpu)
    parts, table, gu, dn = _q4(layer, rows, gpu)
    ws = Workspace(shape, gpu, tokens=T)
    x = seeded.make_tokens(shape, T, T, device=gpu)
    logits = seeded.make_logits(shape, T, T, device=gpu)
    out, ids, w = tm.moe_block(shape, x, table, ws, logits=logits, shared=layer.shared)
    ids = ids.cpu().numpy()
    assert np.array_equal(ids, moe.router_topk(logits.cpu().numpy(), 4)[0])
    ref = moe.add_bf16(moe.experts_prefill(f32(x), ids, f32(w), gu, dn, 16),
                       moe.shared_expert(f32(x), *[f32(t) for t in layer.shared]))
    assert_close_bf16(f32(out), ref, f"T={T} I={I}")
    ws.status()


@pytest.mark.parametrize("T,E,k", [(1, 8, 8), (64, 256, 16), (128, 495, 8), (128, 497, 8), (129, 256, 8), (33, 1023, 4),
                                   (1024, 3, 1), (1025, 3, 1)])
def test_dispatch_one_launch_bounds(gpu, T, E, k):
    """T k and E around the limits of the one-launch dispatch (1024 entries, 16384 mask words), with sentinels."""
    ids = np.random.default_rng(T * E).integers(0, E + 1, (T, k)).astype(np.int64)     # E: the sentinel
    ws = Workspace(MoEShape(128, E, 64, k if k <= E else E), gpu, tokens=T)
    offsets, perm, inv = tm.dispatch(torch.from_numpy(ids).to(gpu), E, ws)
    o_ref, p_ref = moe.dispatch(ids, E)
    n = int(o_ref[-1])
    assert np.array_equal(offsets.cpu().numpy(), o_ref)
    assert np.array_equal(perm.cpu().numpy()[:n], p_ref)
    inv_ref = np.full(T * k, -1, np.int64)
    inv_ref[p_ref] = np.arange(n)
    assert np.array_equal(inv.cpu().numpy(), inv_ref)
    ws.status()


def test_captured_call_follows_each_replays_routing(gpu):
    """One captured call, replayed on routings that want other chunk sizes (160, 64 and 32 rows), with eager
    calls between: each replay's bits are the eager call's."""
    E, k, T = 16, 4, 2400
    shape = MoEShape(768, E, 768, k, 0)
    layer = seeded.make_layer(shape, T, device=gpu)
    ws = Workspace(shape, gpu, tokens=T)
    x = seeded.make_tokens(shape, T, T, device=gpu)
    table = tm.expert_table(layer.gate_up, layer.down)
    slots = torch.arange(k, device=gpu)
    spread = (torch.arange(T, device=gpu)[:, None] * 5 + slots * 4) % E
    one = slots.repeat(T, 1)
    few = torch.full((T, k), E, dtype=torch.int64, device=gpu)       # 40 tokens routed, the rest skipped
    few[:40] = spread[:40]
    w = torch.full((T, k), 0.25, dtype=torch.bfloat16, device=gpu)
    ids = spread.clone()
    tm.experts_forward(shape, x, ids, w, table, ws)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = tm.experts_forward(shape, x, ids, w, table, ws)
    for routing, rows in ((spread, 160), (one, 64), (few, 32), (spread, 160), (few, 32), (one, 64)):
        want = tm.experts_forward(shape, x, routing, w, table, ws).clone()
        torch.cuda.synchronize()
        ids.copy_(routing)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        p = plan(T, 768, E, 768, k, counts=np.bincount(routing.cpu().numpy().ravel(), minlength=E + 1)[:E])
        assert p[0] == rows and _device_rows(shape, T, ws, p) == rows
    ws.status()
