"""GPU: score passes whose keys are split over workgroups.

Short calls, but those whose pass 2 may run in fp6 (16-bit inputs, plain votes), take pass 1 as a
sweep of every score in the screen's four products, each row group's keys split over workgroups and
the row maxima merged; grids of few row groups split pass 2's keys.
The maximum is over the same fp32 values and a key's votes need no other key, so both agree with
the unsplit kernels bit for bit: with the screened pass 1 (STA_SCREEN_PASS1=1), and with the
row-count instances of pass 2, which stay whole.
"""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def say(msg):
    print(f"[case] {msg}", flush=True)


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import _sta_native
    _sta_native.lib()


def _inputs(H, Hkv, N, D, dt, seed):
    from synthetic import base_inv_freq, planted_inputs
    q, k, v = planted_inputs(seed, H, Hkv, N, D, 0.01, dt, DEV)
    return q, k, v, base_inv_freq(D, 10000.0).to(DEV), torch.full((H,), 4.0)


CASES = [
    # (H, Hkv, N, D, dtype, tile, q_pos_base): one short piece; the ends of 64-key chunks and of 256-
    # and 512-row groups; phantom keys; head counts off the XCD map; the last call below the limit of
    # 8192 (row group, chunk) steps and the first above; long rows of few heads (pass 2 split alone)
    (1, 1, 1, 128, torch.bfloat16, 64, 0),
    (2, 1, 65, 128, torch.bfloat16, 64, 0),
    (3, 3, 257, 64, torch.float16, 32, 0),
    (8, 8, 512, 128, torch.float32, 64, 0),
    (5, 5, 513, 64, torch.bfloat16, 64, 0),
    (4, 2, 1000, 128, torch.float16, 32, 37),
    (28, 4, 700, 64, torch.bfloat16, 64, 640),
    (8, 2, 2048, 64, torch.float32, 64, 0),
    (8, 8, 5632, 128, torch.bfloat16, 64, 0),
    (8, 8, 5900, 128, torch.bfloat16, 64, 0),
    (2, 2, 9001, 128, torch.bfloat16, 32, 0),
]


@pytest.mark.parametrize("case", CASES)
def test_row_max_and_votes_match_the_screen(case, monkeypatch):
    import _sta_native as native
    H, Hkv, N, D, dt, tile, qpb = case
    say(f"key split: H={H} Hkv={Hkv} N={N} D={D} {dt} tile={tile} q_pos_base={qpb}")
    q, k, _, invf, tau = _inputs(H, Hkv, N, D, dt, 31)
    sm = 1.0 / math.sqrt(D)
    got = {}
    for screen in (False, True):
        monkeypatch.setenv("STA_SCREEN_PASS1", "1" if screen else "0")
        for score in ("freq", "expmass"):
            r = native.select_vote(q, k, tau, invf, 0.5, 1.0, sm, tile, qpb, want_row_counts=False, select_score=score)
            torch.cuda.synchronize()
            got[screen, score] = [x.cpu().numpy() for x in r if x is not None]
    for score in ("freq", "expmass"):
        for a, b in zip(got[False, score], got[True, score]):
            assert np.array_equal(a, b), f"{score}: {int((a != b).sum())} of {a.size} entries differ"


@pytest.mark.parametrize("H,Hkv,N,D,dt", [(16, 4, 1500, 128, torch.bfloat16), (3, 3, 300, 64, torch.float32),
                                          (8, 8, 4133, 64, torch.float16)])
def test_split_bits_match_the_whole_row_instances(H, Hkv, N, D, dt):
    """PQ pass 2 without row counts (split) against the row-count instance (whole)."""
    import _sta_native as native
    say(f"key split, per-query bits: H={H} N={N} D={D} {dt}")
    q, k, v, invf, tau = _inputs(H, Hkv, N, D, dt, 37)
    whole = native.pq_select_bits(q, k, tau, invf, 0.5, 1.0, 1.0 / math.sqrt(D))
    part = native.PqPlan(q, k, v, tau, invf, invf, 0.5, 1.0, k_max=512, want_votes=True, want_row_max=True).run()
    torch.cuda.synchronize()
    for name in ("row_max", "votes", "bits", "wvotes"):
        a, b = whole[name].cpu().numpy(), part[name].cpu().numpy()
        assert np.array_equal(a, b), f"{name}: {int((a != b).sum())} of {a.size} entries differ"
    rc = whole["row_counts"].cpu().numpy().sum()
    assert int(part["votes"].sum()) == int(rc)


def test_rows_and_keys_that_are_not_finite(monkeypatch):
    """An infinite query row and a NaN key: no bound caps their head's thresholds, and every other
    row keeps what the screen's fallback (three products a score, rounded apart by the lo.lo term:
    1e-4 on the maxima, a vote in 1e4 at the threshold) keeps."""
    import _sta_native as native
    H, N, D = 3, 700, 128
    q, k, _, invf, tau = _inputs(H, H, N, D, torch.bfloat16, 41)
    q[0, 0, 100] = float("inf")
    k[0, 1, 300, 5] = float("nan")
    got = []
    for screen in ("0", "1"):
        monkeypatch.setenv("STA_SCREEN_PASS1", screen)
        votes, _, rm = native.select_vote(q, k, tau, invf, 0.5, 1.0, 1.0 / math.sqrt(D), 64, want_row_counts=False)
        torch.cuda.synchronize()
        got.append((votes.cpu().numpy(), rm.cpu().numpy()))
    (va, ma), (vb, mb) = got
    fine = np.isfinite(mb)
    assert np.array_equal(fine, np.isfinite(ma))
    assert np.abs(ma[fine] - mb[fine]).max() < 1e-4
    assert (va != vb).mean() < 1e-4


@pytest.mark.parametrize("dt,tile", [(torch.bfloat16, 64), (torch.float16, 32)])
def test_concentrated_scores_keep_three_products(dt, tile, monkeypatch):
    """Keys that differ by 2% of their size: the screen cannot single out a row's maximum anywhere, so
    plain votes of 16-bit inputs take three products in both passes, as under STA_EXACT_PASS1=1, bit
    for bit (the fp6 correction moves hundreds of these votes)."""
    import _sta_native as native
    from synthetic import base_inv_freq
    H, N, D = 2, 1500, 128
    say(f"concentrated scores, plain votes: {dt} tile={tile}")
    g = torch.Generator().manual_seed(47)
    q = torch.randn(1, H, N, D, generator=g).to(dt).to(DEV)
    k = (torch.randn(1, H, 1, D, generator=g) + 0.02 * torch.randn(1, H, N, D, generator=g)).to(dt).to(DEV)
    invf = base_inv_freq(D, 10000.0).to(DEV)
    tau = torch.full((H,), 0.03)
    got = []
    for exact in ("0", "1"):
        monkeypatch.setenv("STA_EXACT_PASS1", exact)
        votes, _, rm = native.select_vote(q, k, tau, invf, 0.0, 1.1, 1.0 / math.sqrt(D), tile, want_row_counts=False)
        torch.cuda.synchronize()
        got.append((votes.cpu().numpy(), rm.cpu().numpy()))
    (va, ma), (vb, mb) = got
    assert va.sum() > 10000
    assert np.array_equal(ma, mb) and np.array_equal(va, vb), f"{int((va != vb).sum())} vote entries differ"


@pytest.mark.parametrize("H,Hkv,N,D,dt,scores", [
    (2, 1, 1500, 128, torch.float32, ("freq", "margin", "expmass")), (4, 2, 8300, 64, torch.float32, ("freq", "margin", "expmass")),
    (3, 3, 700, 64, torch.bfloat16, ("margin", "expmass")),           # the row-count instance has no fp6 pass 2
])
@pytest.mark.parametrize("pieces", ["0", "1", "3", "7"])
def test_groups_that_the_screen_gave_up(H, Hkv, N, D, dt, scores, pieces, monkeypatch):
    """The first half of one kv head's keys repeats one key: the screen gives up where rows see little
    else, and the split pass 2 takes the maxima that a sweep of those row groups left.  The row-count
    instance stays whole and sweeps inside.  (Whole plain votes sweep 512 rows where one half of them
    was given up, the row-count instance 256: there all keys of the head are the same.)"""
    import _sta_native as native
    monkeypatch.setenv("STA_SCREEN_PASS1", "1")
    monkeypatch.setenv("STA_SCORE_PIECES", pieces)
    for score in scores:
        say(f"screen gave up: H={H} Hkv={Hkv} N={N} D={D} {dt} {score} pieces={pieces}")
        q, k, _, invf, tau = _inputs(H, Hkv, N, D, dt, 53)
        k[:, 0, : N if score == "freq" and pieces in "01" else N // 2] = k[:, 0, :1]
        got = []
        for counts in (False, True):
            r = native.select_vote(q, k, tau, invf, 0.0, 1.0, 1.0 / math.sqrt(D), 32, want_row_counts=counts, select_score=score)
            torch.cuda.synchronize()
            got.append([r[i].cpu().numpy() for i in range(len(r)) if i != 1])
        for a, b in zip(*got):
            assert np.array_equal(a, b), f"{score}: {int((a != b).sum())} of {a.size} entries differ"


def test_tied_scores_cost_one_sweep():
    """100000 rows of one head, pass 2 in 17 pieces: a call whose scores all tie sweeps the maxima once
    more, 1.4 times a call whose scores do not (3.3 times when every piece swept them)."""
    import time
    import _sta_native as native
    from synthetic import base_inv_freq
    N, D = 100000, 64
    say("tied scores, 1 head x 100000")
    g = torch.Generator(DEV).manual_seed(3)
    q, k = (torch.randn(1, 1, N, D, generator=g, device=DEV) for _ in range(2))
    invf = base_inv_freq(D, 10000.0).to(DEV)
    best = []
    for keys in (k, k[:, :, :1].repeat(1, 1, N, 1)):
        t = []
        for _ in range(4):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            native.select_vote(q, keys, torch.full((1,), 4.0), invf, 0.0, 1.0, 0.125, 64, want_row_counts=False)
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        best.append(min(t[1:]))
    assert best[1] < 2.4 * best[0], f"{best[1] * 1e3:.2f} ms with ties, {best[0] * 1e3:.2f} without"


@pytest.mark.parametrize("H,Hkv,N,D", [(2, 2, 1500, 128), (4, 2, 700, 64)])
@pytest.mark.parametrize("tau", [0.0, 4.0])
@pytest.mark.parametrize("far", [1e6, float("inf")])
def test_one_key_far_out(H, Hkv, N, D, tau, far):
    """The last key a million times as long as the others, or with an infinite element: the rows that
    do not see it keep what the oracle keeps without it, and each of them its best key (the bound on
    the four-product maxima spans all of the head's scores, or is not finite)."""
    import _sta_native as native
    from oracle import sta_oracle as orc
    from parity_helpers import BAND, np_of
    say(f"one key far out: H={H} Hkv={Hkv} N={N} D={D} x{far} tau={tau}")
    q, k, _, invf, _ = _inputs(H, Hkv, N, D, torch.float32, 43)
    taus = torch.full((H,), tau)
    qn, odt = np_of(q[0])
    kn, _ = np_of(k[0])
    sm = 1.0 / math.sqrt(D)
    a = orc.select_vote(qn, kn, odt, taus.numpy(), invf.cpu().numpy(), 0.5, 1.0, sm, 32, 0, band_eps=BAND, want_band=True)
    if far < float("inf"):
        k[:, 0, N - 1] *= far
    else:
        k[:, 0, N - 1, 5] = far
    votes, _, rm = native.select_vote(q, k, taus, invf, 0.5, 1.0, sm, 32, want_row_counts=False)
    torch.cuda.synchronize()
    votes, rm = votes.cpu().numpy().astype(np.int64), rm.cpu().numpy()
    assert np.abs(rm - a["row_max"])[:, : N - 1].max() < 1e-4
    nt = (N - 1) // 32
    assert (np.abs(votes - a["votes"])[:, :nt] <= a["band"][:, :nt]).all()
    assert (votes[:, :nt].sum(-1) >= 32).all()


@pytest.mark.parametrize("H,Hkv,N,D,dt", [(2, 1, 65, 128, torch.float16), (3, 3, 700, 64, torch.float32),
                                          (8, 2, 1601, 128, torch.bfloat16)])
def test_forced_pieces_match_whole_groups(H, Hkv, N, D, dt, monkeypatch):
    """Plain and weighted votes and per-query bits in 2, 5 and more pieces than chunks against one piece:
    the sizes above split or not as the cost rule has it, here they do."""
    import _sta_native as native
    say(f"forced pieces: H={H} Hkv={Hkv} N={N} D={D} {dt}")
    q, k, v, invf, tau = _inputs(H, Hkv, N, D, dt, 71)
    sm = 1.0 / math.sqrt(D)
    got = []
    for pieces in ("1", "2", "5", "64"):
        monkeypatch.setenv("STA_SCORE_PIECES", pieces)
        out = []
        for score in ("freq", "margin", "expmass"):
            r = native.select_vote(q, k, tau, invf, 0.5, 1.0, sm, 32, want_row_counts=False, select_score=score)
            out += [x.clone() for x in r if x is not None]
        p = native.PqPlan(q, k, v, tau, invf, invf, 0.5, 1.0, k_max=512, want_votes=True, want_row_max=True).run()
        out += [p[name].clone() for name in ("row_max", "votes", "bits", "wvotes", "out")]
        torch.cuda.synchronize()
        got.append(out)
    for other in got[1:]:
        for i, (a, b) in enumerate(zip(got[0], other)):
            assert torch.equal(a, b), f"output {i}: {int((a != b).sum())} of {a.numel()} entries differ"


def _oracle(q, k, tau, invf, ps, tile):
    from oracle import sta_oracle as orc
    from parity_helpers import BAND, np_of
    qn, dt = np_of(q[0])
    kn, _ = np_of(k[0])
    return orc.select_vote(qn, kn, dt, tau.numpy(), invf.cpu().numpy(), ps, 1.0, 1.0 / math.sqrt(q.shape[-1]), tile,
                           band_eps=BAND, want_band=True)


def _votes(q, k, tau, invf, ps, tile, counts):
    import _sta_native as native
    votes, rc, rm = native.select_vote(q, k, tau, invf, ps, 1.0, 1.0 / math.sqrt(q.shape[-1]), tile, want_row_counts=counts)
    torch.cuda.synchronize()
    return votes.cpu().numpy().astype(np.int64), rc.cpu().numpy() if counts else None, rm.cpu().numpy()


PATHS = pytest.mark.parametrize("screen,pieces", [("0", "0"), ("0", "4"), ("1", "0"), ("1", "4")])
KINDS = pytest.mark.parametrize("dt,counts", [(torch.bfloat16, False), (torch.bfloat16, True), (torch.float32, False)])


@PATHS
@KINDS
def test_tied_scores(dt, counts, screen, pieces, monkeypatch):
    """One key repeated, and zero query rows, on the short calls' pass 1 and behind the screen, with and
    without row counts: maxima and votes of the oracle."""
    H, N, D = 2, 1500, 128
    say(f"tied scores: {dt} counts={counts} screen={screen} pieces={pieces}")
    g = torch.Generator().manual_seed(5)
    q, k = (torch.randn(1, H, N, D, generator=g) for _ in range(2))
    q[:, :, 300:700] = 0.0
    k[:, 0] = k[:, 0, :1]
    q, k = q.to(dt).to(DEV), k.to(dt).to(DEV)
    invf, tau = _inputs(H, H, 1, D, dt, 1)[3], torch.full((H,), 5.0)
    a = _oracle(q, k, tau, invf, 0.0, 64)
    monkeypatch.setenv("STA_SCREEN_PASS1", screen)
    monkeypatch.setenv("STA_SCORE_PIECES", pieces)
    votes, _, rm = _votes(q, k, tau, invf, 0.0, 64, counts)
    assert np.abs(rm - a["row_max"]).max() < 1e-4
    assert (np.abs(votes - a["votes"]) <= a["band"]).all()


@PATHS
@KINDS
def test_tau_zero_and_below(dt, counts, screen, pieces, monkeypatch):
    """tau = 0: each row keeps its best key and none beyond the band; tau < 0: no key."""
    H, N, D = 2, 2000, 128
    say(f"tau 0 and below: {dt} counts={counts} screen={screen} pieces={pieces}")
    q, k, _, invf, _ = _inputs(H, H, N, D, dt, 12)
    monkeypatch.setenv("STA_SCREEN_PASS1", screen)
    monkeypatch.setenv("STA_SCORE_PIECES", pieces)
    tau = torch.zeros(H)
    a = _oracle(q, k, tau, invf, 0.5, 64)
    votes, rc, _ = _votes(q, k, tau, invf, 0.5, 64, counts)
    assert (np.abs(votes - a["votes"]) <= a["band"]).all()
    rows = np.minimum(64, N - 64 * np.arange(votes.shape[1]))
    assert (votes.sum(-1) >= rows).all()
    if counts:
        assert (rc >= 1).all()
    for low in (-0.5, -3.0):
        votes, rc, _ = _votes(q, k, torch.full((H,), low), invf, 0.5, 64, counts)
        assert votes.sum() == 0 and (not counts or rc.sum() == 0), low


@PATHS
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tau", [0.0, 4.0])
def test_finite_rows_beside_others(dt, tau, screen, pieces, monkeypatch):
    """An infinite and a NaN query row and a NaN key: tiles without such a row, and rows before that
    key, have the votes that the oracle gives them on finite inputs, and a key for every row."""
    H, N, D, tile = 3, 700, 128, 32
    say(f"rows and keys that are not finite: {dt} tau={tau} screen={screen} pieces={pieces}")
    q, k, _, invf, _ = _inputs(H, H, N, D, dt, 41)
    taus = torch.full((H,), tau)
    a = _oracle(q, k, taus, invf, 0.5, tile)
    q[0, 0, 100] = float("inf")
    q[0, 2, 200, 7] = float("nan")
    k[0, 1, 300, 5] = float("nan")
    monkeypatch.setenv("STA_SCREEN_PASS1", screen)
    monkeypatch.setenv("STA_SCORE_PIECES", pieces)
    votes, _, _ = _votes(q, k, taus, invf, 0.5, tile, False)
    ok = np.ones(votes.shape[:2], bool)
    ok[0, 100 // tile] = ok[2, 200 // tile] = ok[1, 300 // tile:] = False
    rows = np.minimum(tile, N - tile * np.arange(votes.shape[1]))
    assert (np.abs(votes - a["votes"])[ok] <= a["band"][ok]).all()
    assert (votes.sum(-1) >= rows)[ok].all()


@PATHS
@KINDS
def test_tau_zero_with_long_rows(dt, counts, screen, pieces, monkeypatch):
    """Rows four times as long: the bound on the four-product maxima exceeds the band, yet no key beyond
    the band of a row's best key passes at tau = 0."""
    H, N, D = 2, 1500, 128
    say(f"tau 0, long rows: {dt} counts={counts} screen={screen} pieces={pieces}")
    q, k, _, invf, _ = _inputs(H, H, N, D, dt, 13)
    q, k = (4 * q.float()).to(dt), (4 * k.float()).to(dt)
    tau = torch.zeros(H)
    a = _oracle(q, k, tau, invf, 0.5, 64)
    monkeypatch.setenv("STA_SCREEN_PASS1", screen)
    monkeypatch.setenv("STA_SCORE_PIECES", pieces)
    votes, _, _ = _votes(q, k, tau, invf, 0.5, 64, counts)
    assert (np.abs(votes - a["votes"]) <= a["band"]).all()
    rows = np.minimum(64, N - 64 * np.arange(votes.shape[1]))
    assert (votes.sum(-1) >= rows).all()


@pytest.mark.parametrize("N", [40, 700])
@pytest.mark.parametrize("screen", ["0", "1"])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_one_key_far_out_of_few(N, screen, dt, monkeypatch):
    """The same with so few keys that the screen scores all of them: every row keeps the oracle's."""
    H, D = 2, 128
    say(f"one key far out of {N}: {dt} screen={screen}")
    q, k, _, invf, tau = _inputs(H, H, N, D, dt, 43)
    a = _oracle(q, k, tau, invf, 0.5, 32)
    k[:, 0, N - 1] *= 1e6
    monkeypatch.setenv("STA_SCREEN_PASS1", screen)
    votes, _, _ = _votes(q, k, tau, invf, 0.5, 32, False)
    nt = (N - 1) // 32
    assert (np.abs(votes - a["votes"])[:, :nt] <= a["band"][:, :nt]).all()


@pytest.mark.parametrize("screen", ["0", "1"])
@pytest.mark.parametrize("score", ["freq", "expmass"])
def test_swept_groups_in_a_graph(screen, score, monkeypatch):
    """A graph over keys that tie and keys that do not, in turn, and a tau that calls for three products
    in between: each replay starts from its own flags and maxima and gives the eager call's outputs."""
    import _sta_native as native
    H, N, D = 3, 1500, 64
    say(f"graph: screen={screen} {score}")
    monkeypatch.setenv("STA_SCREEN_PASS1", screen)
    monkeypatch.setenv("STA_SCORE_PIECES", "3")
    q, k, v, invf, _ = _inputs(H, H, N, D, torch.float32, 79)
    tied = k.clone()
    tied[:, 1] = tied[:, 1, :1]
    kw = dict(pct=30.0, tile=64, k_max=256, want_votes=True, select_score=score)
    kb, tb = k.clone(), torch.full((H,), 5.0, device=DEV)
    plan = native.NoallocPlan(q, kb, v, tb, invf, 0.0, 1.0, invf, 0.5, 1.0, **kw)
    plan.run()
    torch.cuda.synchronize()
    inputs = [(k, 5.0), (tied, 5.0), (k, 0.0), (tied, 0.0), (k, 5.0), (tied, 5.0)]
    refs = [native.shared_attention(q, keys, v, torch.full((H,), t), invf, 0.0, 1.0, invf, 0.5, 1.0, **kw) for keys, t in inputs]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        plan.run()
    torch.cuda.synchronize()
    for i, ((keys, t), ref) in enumerate(zip(inputs, refs)):
        kb.copy_(keys)
        tb.fill_(t)
        g.replay()
        torch.cuda.synchronize()
        for name in ("votes", "idx", "kept_size", "out"):
            assert torch.equal(plan.out[name], ref[name]), f"replay {i}: {name}"
