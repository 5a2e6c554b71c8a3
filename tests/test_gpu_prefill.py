"""GPU parity: prefill / extend attention over the packed paged cache (tq_prefill) vs the float64
oracle (oracle.decode.prefill_dense: each query row is a decode over the tokens it sees; pinned
against a masked score tensor in test_oracle.py).  Bar: rtol 1e-2 / atol 1e-3, as decode.
"""

import math

import numpy as np
import pytest
import torch

from oracle import compress as ocomp
from oracle import decode as odec
from test_gpu_decode import ATOL, RTOL, _cb, build_case

pytestmark = pytest.mark.gpu

H64 = ocomp.wht_closed_form(128, 1.0 / math.sqrt(128.0))


def make_queries(rng, n_new, Hq):
    cu = np.zeros(len(n_new) + 1, np.int32)
    cu[1:] = np.cumsum(n_new)
    q = rng.standard_normal((int(cu[-1]), Hq, 128)).astype(np.float32)
    return q, cu


def oracle_prefill(case, q, cu, Hq, Hkv, kb, kq, vb, sm, cs, causal=True, qp=None):
    G = Hq // Hkv
    kc, vc = _cb(kb).double().numpy(), _cb(vb).double().numpy()
    out = np.zeros(q.shape)
    qpv = q if qp is None else qp
    for s in range(len(case["seq_lens"])):
        L = int(case["seq_lens"][s])
        rows = slice(int(cu[s]), int(cu[s + 1]))
        if L == 0 or cu[s + 1] == cu[s]:
            continue
        for kh in range(Hkv):
            kp = {k: v[:, kh] for k, v in case["k_tok"][s].items()}
            vp = {k: v[:, kh] for k, v in case["v_tok"][s].items()}
            k, sg, rn = odec.dequant_keys(kp, kc, kb, kq)
            v = odec.dequant_values(vp, vc, vb)
            hs = slice(kh * G, (kh + 1) * G)
            out[rows, hs] = odec.prefill_dense(q[rows, hs], qpv[rows, hs], k, sg, rn, v, sm, cs, causal=causal)
    return out


def run_prefill(dev, case, q, cu, kb, kq, vb, bs, sm, cs, causal=True, rotate=False, qp=None,
                dtype=torch.bfloat16, out_dtype=None, max_q_len=None):
    from turboquant.kernels.paged import PagedKVFormat, prefill_paged
    kf = PagedKVFormat(bits=kb, qjl=kq, block_size=bs, layout=case["layouts"][0])
    vf = PagedKVFormat(bits=vb, qjl=False, block_size=bs, layout=case["layouts"][1])
    qt = torch.from_numpy(q).to(dtype).to(dev)
    qpt = torch.from_numpy(qp).to(dtype).to(dev) if qp is not None else None
    out = None
    if out_dtype is not None:
        out = torch.empty(qt.shape, dtype=out_dtype, device=dev)
    out = prefill_paged(qt, torch.from_numpy(cu).to(dev), torch.from_numpy(case["k_cache"]).to(dev), kf,
                        _cb(kb).to(dev), torch.from_numpy(case["v_cache"]).to(dev), vf, _cb(vb).to(dev),
                        torch.from_numpy(case["bt"]).to(dev), torch.from_numpy(case["seq_lens"]).to(dev),
                        sm_scale=sm, corr_scale=cs, q_proj=qpt, causal=causal, rotate=rotate, out=out,
                        max_q_len=max_q_len)
    torch.cuda.synchronize()
    qr = qt.float().cpu().numpy().astype(np.float64)
    qpr = qpt.float().cpu().numpy().astype(np.float64) if qpt is not None else None
    return out.float().cpu().numpy(), qr, qpr


SM, CS = 1 / math.sqrt(128), math.sqrt(math.pi / 2) / 128


@pytest.mark.parametrize("kb,kq,vb,G", [(3, True, 3, 6), (4, False, 4, 4), (2, True, 2, 8), (3, True, 4, 1),
                                        (2, False, 3, 3), (4, True, 2, 12)])
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_bit_widths_and_groups(dev, kb, kq, vb, G, causal):
    Hkv, bs = 2, 16
    Hq = G * Hkv
    lens = [37, 1, 300, 70]
    n_new = [5, 1, 64, 0]
    case = build_case(900 + 5 * kb + vb + G, len(lens), Hq, Hkv, lens, kb, kq, vb, bs)
    rng = np.random.default_rng(G + kb)
    q, cu = make_queries(rng, n_new, Hq)
    got, qr, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, causal=causal)
    want = oracle_prefill(case, qr, cu, Hq, Hkv, kb, kq, vb, SM, CS, causal=causal)
    np.testing.assert_allclose(got, want, rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("kb,kq,vb", [(3, True, 3), (2, False, 4)])
def test_prefill_row_major_paged_tiles(dev, kb, kq, vb):
    """Row-major tiles are read as well as the lane-grouped ones."""
    Hq, Hkv, bs = 8, 2, 32
    lens = [100, 37]
    n_new = [20, 37]
    case = build_case(31 + kb, len(lens), Hq, Hkv, lens, kb, kq, vb, bs, layouts=("rows", "rows"))
    rng = np.random.default_rng(kb)
    q, cu = make_queries(rng, n_new, Hq)
    got, qr, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS)
    want = oracle_prefill(case, qr, cu, Hq, Hkv, kb, kq, vb, SM, CS)
    np.testing.assert_allclose(got, want, rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("bs", [32, 64])
def test_prefill_block_sizes_row_blocks_and_short_sequences(dev, bs):
    """Block sizes above 16, sequences whose rows span several 64-row blocks (130 x 6), more new
    tokens than cache tokens (the first rows see nothing: zero), f16 queries, f32 output."""
    kb, kq, vb, Hq, Hkv = 3, True, 3, 12, 2
    lens = [400, 3, 129]
    n_new = [130, 5, 129]
    case = build_case(1234 + bs, len(lens), Hq, Hkv, lens, kb, kq, vb, bs)
    rng = np.random.default_rng(bs)
    q, cu = make_queries(rng, n_new, Hq)
    got, qr, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, dtype=torch.float16,
                             out_dtype=torch.float32, max_q_len=max(n_new))
    want = oracle_prefill(case, qr, cu, Hq, Hkv, kb, kq, vb, SM, CS)
    np.testing.assert_allclose(got, want, rtol=RTOL, atol=ATOL)
    assert np.all(got[int(cu[1]):int(cu[1]) + 2] == 0.0)


def test_prefill_more_new_tokens_than_max_q_len(dev):
    """A sequence with more new tokens than max_q_len: the ones that are computed keep their positions
    (the causal limit counts all of the sequence's new tokens)."""
    kb, kq, vb, Hq, Hkv, bs = 4, False, 4, 8, 2, 16
    lens, n_new, mq = [300, 250], [70, 30], 64
    case = build_case(61, len(lens), Hq, Hkv, lens, kb, kq, vb, bs)
    rng = np.random.default_rng(5)
    q, cu = make_queries(rng, n_new, Hq)
    got, qr, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, max_q_len=mq)
    want = oracle_prefill(case, qr, cu, Hq, Hkv, kb, kq, vb, SM, CS)
    for s, n in enumerate(n_new):
        rows = slice(int(cu[s]), int(cu[s]) + min(n, mq))
        np.testing.assert_allclose(got[rows], want[rows], rtol=RTOL, atol=ATOL)


def test_prefill_rotated_and_explicit_q_proj(dev):
    kb, kq, vb, Hq, Hkv, bs = 3, True, 3, 8, 2, 16
    lens = [200, 45]
    n_new = [17, 45]
    case = build_case(77, len(lens), Hq, Hkv, lens, kb, kq, vb, bs)
    rng = np.random.default_rng(8)
    q, cu = make_queries(rng, n_new, Hq)
    got, qr, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, rotate=True)
    want = oracle_prefill(case, qr @ H64, cu, Hq, Hkv, kb, kq, vb, SM, CS) @ H64
    np.testing.assert_allclose(got, want, rtol=RTOL, atol=ATOL)
    qp = rng.standard_normal(q.shape).astype(np.float32)
    got, qr, qpr = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, qp=qp)
    want = oracle_prefill(case, qr, cu, Hq, Hkv, kb, kq, vb, SM, CS, qp=qpr)
    np.testing.assert_allclose(got, want, rtol=RTOL, atol=ATOL)


def test_prefill_bad_block_entries_are_masked(dev):
    """A block-table entry outside [0, num_blocks) removes its tokens from every row."""
    kb, kq, vb, Hq, Hkv, bs = 4, False, 4, 4, 1, 16
    lens = [48]
    case = build_case(19, 1, Hq, Hkv, lens, kb, kq, vb, bs)
    case["bt"][0, 1] = case["nb"] + 5        # tokens 16..31 unreadable
    rng = np.random.default_rng(1)
    q, cu = make_queries(rng, [6], Hq)
    got, qr, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, 0.1, 0.0)
    keep = np.r_[0:16, 32:48]
    kc, vc = _cb(kb).double().numpy(), _cb(vb).double().numpy()
    kp = {k: v[keep, 0] for k, v in case["k_tok"][0].items()}
    vp = {k: v[keep, 0] for k, v in case["v_tok"][0].items()}
    k, _, _ = odec.dequant_keys(kp, kc, kb, False)
    v = odec.dequant_values(vp, vc, vb)
    pos_keep = keep
    for i in range(6):
        lim = int(np.searchsorted(pos_keep, 48 - 6 + i, side="right"))
        want = odec.decode_dense(qr[i], None, k[:lim], None, None, v[:lim], 0.1, 0.0)
        np.testing.assert_allclose(got[i], want, rtol=RTOL, atol=ATOL)


def test_prefill_last_row_is_a_decode_step(dev):
    """Full causal prefill of 1000 tokens (G = 6): its last row equals decode_paged of that token on
    the same cache, and sampled rows match the oracle."""
    from turboquant.kernels.paged import PagedKVFormat, decode_paged
    kb, kq, vb, Hq, Hkv, bs = 3, True, 3, 12, 2, 16
    lens = [1000]
    case = build_case(5, 1, Hq, Hkv, lens, kb, kq, vb, bs)
    rng = np.random.default_rng(9)
    q, cu = make_queries(rng, [1000], Hq)
    got, qr, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS)
    kf = PagedKVFormat(bits=kb, qjl=kq, block_size=bs)
    vf = PagedKVFormat(bits=vb, qjl=False, block_size=bs, layout="values")
    qlast = torch.from_numpy(qr[-1:]).to(torch.bfloat16).to(dev)
    dec = decode_paged(qlast, torch.from_numpy(case["k_cache"]).to(dev), kf, _cb(kb).to(dev),
                       torch.from_numpy(case["v_cache"]).to(dev), vf, _cb(vb).to(dev),
                       torch.from_numpy(case["bt"]).to(dev), torch.from_numpy(case["seq_lens"]).to(dev),
                       sm_scale=SM, corr_scale=CS, tokens_per_chunk=256)
    np.testing.assert_allclose(got[-1], dec.float().cpu().numpy()[0], rtol=RTOL, atol=ATOL)
    kc, vc = _cb(kb).double().numpy(), _cb(vb).double().numpy()
    G = Hq // Hkv
    for kh in range(Hkv):
        kp = {k: v[:, kh] for k, v in case["k_tok"][0].items()}
        vp = {k: v[:, kh] for k, v in case["v_tok"][0].items()}
        k, sg, rn = odec.dequant_keys(kp, kc, kb, kq)
        v = odec.dequant_values(vp, vc, vb)
        for i in (0, 1, 15, 16, 17, 511, 998, 999):
            hs = slice(kh * G, (kh + 1) * G)
            want = odec.decode_dense(qr[i, hs], qr[i, hs], k[:i + 1], sg[:i + 1], rn[:i + 1], v[:i + 1], SM, CS)
            np.testing.assert_allclose(got[i, hs], want, rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("kb", [2, 3, 4])
@pytest.mark.parametrize("kq", [False, True])
@pytest.mark.parametrize("vb,G", [(2, 16), (3, 1), (4, 5)])
def test_prefill_stream_formats(dev, kb, kq, vb, G):
    """Every pair of formats of the streaming kernel, on segments that are cut over several waves and
    merged (1000 and 340 tokens, few rows) next to short and empty ones."""
    Hkv, bs = 2, 48
    lens, n_new = [1000, 0, 340, 1, 31], [3, 2, 40, 1, 0]
    case = build_case(40 + 9 * kb + vb + G, len(lens), G * Hkv, Hkv, lens, kb, kq, vb, bs)
    q, cu = make_queries(np.random.default_rng(G), n_new, G * Hkv)
    got, qr, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, max_q_len=40)
    want = oracle_prefill(case, qr, cu, G * Hkv, Hkv, kb, kq, vb, SM, CS)
    np.testing.assert_allclose(got, want, rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("workspace", [True, False])
@pytest.mark.parametrize("name", ["many", "long", "full"])
def test_prefill_stream_shares(dev, monkeypatch, name, workspace, causal):
    """The streaming kernel's ways to share out segments against prefill_kernel (which a separate q_proj
    selects): more sequences than a wave's lanes, each segment whole; one long sequence over all
    waves; more segments than waves; each also without a workspace.  Both are within RTOL / ATOL of the
    oracle, so within twice that of each other."""
    from turboquant import _lib
    kb, kq, vb, Hkv, bs = 3, True, 3, 8, 16
    rng = np.random.default_rng(2)
    if name == "many":
        G, lens = 3, [int(x) for x in rng.integers(0, 200, 70)] + [200]
        n_new = [int(x) for x in rng.integers(0, 40, 71)]
    elif name == "long":
        G, lens, n_new = 4, [6000], [50]
    else:
        G, lens, n_new = 16, [30, 850], [9, 800]
    case = build_case(7, len(lens), G * Hkv, Hkv, lens, kb, kq, vb, bs)
    q, cu = make_queries(rng, n_new, G * Hkv)
    want, _, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, qp=q, causal=causal, out_dtype=torch.float32)
    if not workspace:
        monkeypatch.setattr(_lib.lib(), "tq_prefill_workspace_bytes", lambda *a: 0)
    got, _, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, causal=causal, out_dtype=torch.float32)
    np.testing.assert_allclose(got, want, rtol=2 * RTOL, atol=2 * ATOL)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("lens", [[6000], [250]])
def test_prefill_bad_query_rows_stay_visible(dev, lens, bad):
    """A query row that is not finite gives NaN, also where its keys are cut over several waves (6000
    tokens), and leaves every other row as it was.  The other rows may round anew (their exponent base
    moves with a row of the same tile): both runs are within RTOL / ATOL of the oracle."""
    kb, kq, vb, Hkv, G, bs = 3, True, 3, 2, 4, 16
    case = build_case(11, 1, G * Hkv, Hkv, lens, kb, kq, vb, bs)
    q, cu = make_queries(np.random.default_rng(3), [50], G * Hkv)
    want, _, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, out_dtype=torch.float32)
    q[7, 2] = bad
    got, _, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, out_dtype=torch.float32)
    assert np.isnan(got[7, 2]).all()
    got[7, 2] = want[7, 2]
    np.testing.assert_allclose(got, want, rtol=2 * RTOL, atol=2 * ATOL)


@pytest.mark.parametrize("variant", ["rows", "q_proj", "unaligned_q", "unaligned_out", "zero_scale", "streams"])
def test_prefill_takes_a_workspace_only_where_it_is_used(dev, variant):
    """Calls that prefill_kernel serves allocate nothing beside their output; the streaming kernel's
    allocate what tq_prefill_workspace_bytes says (here more than 32 MB)."""
    from turboquant import _lib
    from turboquant.kernels.paged import PagedKVFormat, allocate_cache, prefill_paged
    S, n, Hq, Hkv, bs = 4, 256, 32, 8, 16
    layouts = ("rows", "rows") if variant == "rows" else ("keys", "values")
    kf = PagedKVFormat(bits=3, qjl=True, block_size=bs, layout=layouts[0])
    vf = PagedKVFormat(bits=3, block_size=bs, layout=layouts[1])
    nb = S * n // bs
    kc, vc = allocate_cache(nb, Hkv, kf, device=dev).zero_(), allocate_cache(nb, Hkv, vf, device=dev).zero_()
    bt = torch.arange(nb, dtype=torch.int32, device=dev).view(S, -1).repeat(1, 2)
    lens = torch.full((S,), n, dtype=torch.int32, device=dev)
    cu = torch.arange(0, (S + 1) * n, n, dtype=torch.int32, device=dev)
    wide = torch.zeros(S * n, Hq, 132, dtype=torch.bfloat16, device=dev)
    plain = torch.zeros(S * n, Hq, 128, dtype=torch.bfloat16, device=dev)
    q = wide[..., 1:129] if variant == "unaligned_q" else plain
    out = wide[..., 2:130] if variant == "unaligned_out" else torch.empty_like(plain)
    cb = _cb(3).to(dev)
    need = _lib.lib().tq_prefill_workspace_bytes(S, n, Hq, Hkv, bt.shape[1], bs)
    assert need > 32 << 20
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated(dev)
    torch.cuda.reset_peak_memory_stats(dev)
    prefill_paged(q, cu, kc, kf, cb, vc, vf, cb, bt, lens, sm_scale=0.0 if variant == "zero_scale" else SM,
                  q_proj=plain if variant == "q_proj" else None, max_q_len=n, out=out)
    peak = torch.cuda.max_memory_allocated(dev) - before
    assert peak >= need if variant == "streams" else peak < 1 << 20


@pytest.mark.parametrize("workspace", [True, False])
@pytest.mark.parametrize("S", [2, 40])
@pytest.mark.parametrize("table", [192, 208, 256, 272, 384, 400, 784])
def test_prefill_dispatch_edges(dev, monkeypatch, table, S, workspace):
    """Both sides of each line of the dispatch on the block table's tokens, with few and with many segments,
    with and without a workspace: short sequences in a table of that width, against prefill_kernel (which
    a separate q_proj selects; both are within RTOL / ATOL of the oracle).  A NaN query row stays NaN."""
    from turboquant import _lib
    kb, kq, vb, G, Hkv, bs = 3, True, 3, 6, 4, 16
    rng = np.random.default_rng(table + S)
    top = min(table, 300)
    lens = [top, 0] + [int(x) for x in rng.integers(1, top + 1, S - 2)]
    n_new = [min(70, n) for n in lens]
    case = build_case(table, S, G * Hkv, Hkv, lens, kb, kq, vb, bs)
    wide = np.full((S, table // bs), -1, np.int32)
    wide[:, :case["bt"].shape[1]] = case["bt"]
    case["bt"] = wide
    q, cu = make_queries(rng, n_new, G * Hkv)
    q[3, 1] = np.nan
    want, _, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, qp=q, out_dtype=torch.float32, max_q_len=70)
    if not workspace:
        monkeypatch.setattr(_lib.lib(), "tq_prefill_workspace_bytes", lambda *a: 0)
    got, _, _ = run_prefill(dev, case, q, cu, kb, kq, vb, bs, SM, CS, out_dtype=torch.float32, max_q_len=70)
    assert np.isnan(got[3, 1]).all() and np.isnan(want[3, 1]).all()
    got[3, 1] = want[3, 1] = 0
    np.testing.assert_allclose(got, want, rtol=2 * RTOL, atol=2 * ATOL)
