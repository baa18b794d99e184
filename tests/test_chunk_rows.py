"""The prefill path's plan (rows per M-chunk), computed on the host: no GPU."""
import numpy as np
import pytest

from tarfa_amd._lib import lib

CUS = 256


def plan(T, H, E, I, k, Is=0, q4=0, counts=None):
    out = np.zeros(8, np.int64)
    c = None if counts is None else np.ascontiguousarray(counts, np.int32)
    st = lib().tmoe_debug_prefill_plan(T, H, E, I, k, Is, q4, CUS, None if c is None else c.ctypes.data,
                                       out.ctypes.data)
    assert st == 0, st
    return out.tolist()


def uniform(T, E, k, seed=0):
    r = np.random.default_rng(seed)
    return np.bincount(r.random((T, E)).argpartition(k, axis=1)[:, :k].ravel(), minlength=E)


def hot(T, E, k):
    """Every token takes the same k experts."""
    return np.where(np.arange(E) < k, T, 0)


FULL = (2560, 256, 1024, 8, 1024)


@pytest.mark.parametrize("T,routing,rows", [
    (18, uniform, 32), (18, hot, 32), (40, hot, 64), (211, uniform, 32), (603, uniform, 32), (1024, uniform, 64),
    (400, hot, 64), (603, hot, 64), (1024, hot, 160), (1536, hot, 160), (2048, uniform, 160), (4096, uniform, 160)])
def test_bf16_rows_follow_the_group_sizes(T, routing, rows):
    """Measured at the full-size layer with each size forced: a routing that sends every token to the same
    experts took 128 us at T = 400 with 160 rows, 152 with the 32 that a uniform routing wants."""
    H, E, I, k, Is = FULL
    assert plan(T, H, E, I, k, Is, counts=routing(T, E, k))[:2] == [rows, rows]


def test_bf16_rows_few_large_groups():
    """Few groups leave blocks idle at 160 rows (E = 8 of mean 128 rows: 91 us against 73)."""
    assert plan(512, 1280, 8, 1920, 2, counts=uniform(512, 8, 2))[0] == 64
    assert plan(256, 768, 16, 640, 4, 640, counts=uniform(256, 16, 4))[0] in (32, 64)
    assert plan(565, 2048, 14, 1536, 1, 1536, counts=uniform(565, 14, 1))[0] == 160   # one round: 104 us, 64 rows 112


def _cost(s, hit, chunks, H, I):
    first, further, turn = ((305, 91, 100), (308, 107, 114), (325, 197, 241))[s]
    up, dn = I // 128, H // 256
    whole = CUS * (-(-chunks * up // CUS) * H + -(-chunks * dn // CUS) * I)
    unit = up * H + dn * I
    work = (first * hit + further * (chunks - hit)) * unit + 0.63 * turn * (whole - chunks * unit)
    return max(work, turn * whole)


@pytest.mark.parametrize("seed", range(40))
def test_bf16_rows_are_the_cheapest(seed):
    """The choice over random group sizes, up to the most entries a call may have, against the cost in
    Python."""
    r = np.random.default_rng(seed)
    H, I = 256 * int(r.integers(2, 17)), 128 * int(r.integers(4, 33))
    E, k = int(r.integers(1, 1024)), 1
    T = int(np.exp(r.uniform(np.log(20), np.log(524288))))
    p = r.dirichlet(np.full(E, r.choice([0.02, 0.3, 5.0])))
    c = r.multinomial(T, p)
    Is = int(r.choice([0, I]))
    got, shared, _, tiled = plan(T, H, E, I, k, Is, counts=c)[:4]
    smallest = plan(T, H, E, I, k, Is)[0]
    assert got == shared
    if not tiled or smallest == 160:
        assert got == 160
        return
    hit = int((c > 0).sum()) + (Is > 0)
    costs = {rows: _cost(s, hit, int((-(-c // rows)).sum()) + (-(-T // rows) if Is else 0), H, I)
             for s, rows in enumerate((32, 64, 160)) if rows >= smallest}
    assert costs[got] <= min(costs.values()) * (1 + 1e-5)          # the rule is in fp32


@pytest.mark.parametrize("E,k,Is", [(32, 8, 1024), (16, 4, 512), (16, 6, 512), (16, 8, 0), (256, 8, 1024), (8, 2, 512),
                                    (1, 1, 512)])
@pytest.mark.parametrize("q4", [0, 1, 2])
def test_small_calls_take_small_chunks(E, k, Is, q4):
    """Few tokens leave few logits; their descriptors fit the region of their own (int4 E = 32, k = 8,
    T = 2 .. 4 ran 160-row tiles: 151 us against 84 at T = 5, H = 2560, I = 640)."""
    I = Is or 512
    for T in range(2, 6):
        rows, shared, fuse, tiled = plan(T, 1024, E, I, k, Is, q4)[:4]
        assert tiled and (rows == 16 if q4 else rows == 32)
        assert fuse == (q4 > 0 and Is > 0) and shared == (32 if fuse or not q4 else 64)


@pytest.mark.parametrize("seed", range(30))
def test_descriptors_fit_their_region(seed):
    """The most chunks that T k entries can make: every expert one row, the rest on one of them."""
    r = np.random.default_rng(seed)
    E = int(np.exp(r.uniform(0, np.log(1023.9))))
    k = int(r.integers(1, min(E, 16) + 1))
    Is = int(r.choice([0, 768]))
    for T in sorted({2, 3, *np.exp(r.uniform(np.log(2), np.log((1 << 19) / k), 20)).astype(int).tolist()}):
        for q4 in (0, 1):
            rows, shared, _, _, _, room = plan(T, 1024, E, 768, k, Is, q4)[:6]
            hit = min(T * k, E)
            spread = np.full(hit, (T * k) // hit)
            spread[0] += T * k - spread.sum()
            one = np.ones(hit, int)
            one[0] = T * k - hit + 1                   # past T: more than distinct experts per token allow
            for c in (spread, one):
                chunks = int((-(-c // rows)).sum()) + (-(-T // shared) if Is else 0)
                assert chunks <= room, (T, E, k, Is, q4, rows)


@pytest.mark.parametrize("T,E,tile", [
    (4096, 256, [64, 64]), (2048, 256, [64, 32]), (1024, 256, [32, 32]), (16384, 256, [64, 64]),
    (4096, 160, [32, 32]), (16384, 8, [32, 32]), (16384, 16, [32, 32]), (16384, 32, [64, 32]), (128, 1023, [32, 32])])
def test_router_tiles(T, E, tile):
    """Wider tiles only where they fill the chip in fewer or cheaper rounds: E = 160, T = 4096 in 320 blocks and
    E = 8 in 64-wide tiles were slower than the 32 x 32 tiles they replaced (2 % and 11 %)."""
    assert plan(T, 2560, E, 512, min(8, E))[6:8] == tile
