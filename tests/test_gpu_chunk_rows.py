"""The prefill GEMMs' chunk sizes: groups of 1, 31, 32, 33, 64 and 65 rows through 32- and 64-row chunks
(the rule takes the fewest rows that hold a mean group plus three standard deviations), at widths that
take four or five weight stages per cycle, against the oracle's chain at the bf16 bars."""
import numpy as np
import pytest
import torch

from oracle import moe
from tarfa_amd import moe as tm
from tarfa_amd import seeded
from tarfa_amd.moe import MoEShape, Workspace
from tests._util import assert_close_bf16, expert_dicts, f32

pytestmark = pytest.mark.gpu

ROWS = [1, 31, 32, 33, 64, 65]


def _ids(E, seed):
    """One expert per token, expert e taken by ROWS[e] tokens in a shuffled order."""
    ids = np.repeat(np.arange(len(ROWS)), ROWS)
    np.random.default_rng(seed).shuffle(ids)
    return ids[:, None].astype(np.int64)


@pytest.mark.parametrize("H,I,E", [(768, 640, 16), (768, 640, 6), (1280, 512, 16), (512, 768, 6)])
def test_bf16_chunk_edges(gpu, H, I, E):
    shape = MoEShape(H, E, I, 1, 0)                # mean 14 rows (E = 16) or 38 (E = 6)
    layer = seeded.make_layer(shape, H + E, device=gpu)
    ids = _ids(E, H)
    T = len(ids)
    ws = Workspace(shape, gpu, tokens=T)
    x = seeded.make_tokens(shape, H + E, T, device=gpu)
    w = torch.linspace(0.1, 1.0, T, device=gpu).to(torch.bfloat16)[:, None].contiguous()
    out = tm.experts_forward(shape, x, torch.from_numpy(ids).to(gpu), w, tm.expert_table(layer.gate_up, layer.down),
                             ws)
    gu, dn = expert_dicts(layer.gate_up, layer.down, ids)
    assert_close_bf16(f32(out), moe.experts_prefill(f32(x), ids, f32(w), gu, dn, E), f"H={H} I={I} E={E}")
    ws.status()


@pytest.mark.parametrize("T", [17, 90, 200])
def test_bf16_chunks_with_shared_expert(gpu, T):
    """Mean groups of 4, 22 and 50 rows (32-, 64- and 160-row chunks), the shared expert in the same chunks."""
    shape = MoEShape(768, 16, 768, 4, 768)
    layer = seeded.make_layer(shape, T, device=gpu)
    ws = Workspace(shape, gpu, tokens=T)
    x = seeded.make_tokens(shape, T, T, device=gpu)
    logits = seeded.make_logits(shape, T, T, device=gpu)
    table = tm.expert_table(layer.gate_up, layer.down)
    out, ids, w = tm.moe_block(shape, x, table, ws, logits=logits, shared=layer.shared)
    ids = ids.cpu().numpy()
    assert np.array_equal(ids, moe.router_topk(logits.cpu().numpy(), 4)[0])
    gu, dn = expert_dicts(layer.gate_up, layer.down, ids)
    ref = moe.add_bf16(moe.experts_prefill(f32(x), ids, f32(w), gu, dn, 16),
                       moe.shared_expert(f32(x), *[f32(t) for t in layer.shared]))
    assert_close_bf16(f32(out), ref, f"T={T}")
    ws.status()
