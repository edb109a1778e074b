"""Garesun on MI355X against the plain restatement in tests/garesun_oracle.py (float64 on the CPU, token by token).

Small random checkpoints with unequal sizes (tests/garesun_helpers.py) are written to disk and loaded through
`utils.load_model` (registry by config.json, safetensors reader, weight packing).  float32 serving is compared tightly,
bfloat16 within the rounding of a 16-bit projection chain.  Covered: every mechanism alone (operator level and as a one-
layer model); whole prompts against portions of several sizes (down to two tokens) and against token-by-token decoding;
batches of unequal requests against each alone; pages and state slots freed and used again; attention keys far back, at
page and tile borders, in prompts and decoding, with one score made to stand out; the first tokens; long decoding; sizes
that are equal or 1 elsewhere (top = 1, no shared expert, no feed-forward, no token input, partial rotation, shared
latent cache); greedy generation through generate_step and the continuous batch generator."""
import numpy as np
import pytest
import torch

from tests import garesun_helpers as H
from tests import garesun_oracle as O

pytestmark = pytest.mark.gpu
F64 = torch.float64


def _load(tmp_path, cfg, W, dtype, tokens=4096, seqs=6, name="m"):
    from mlx_vlm_amd.utils import load_model

    return load_model(H.write_checkpoint(str(tmp_path / name), cfg, W), dtype=dtype, kv_pool_tokens=tokens, max_seqs=seqs)


def _ids(n, vocab, seed):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed)).numpy().astype(np.int32)


def _whole(lm, ids):
    c = lm.make_cache()
    lg = lm.step([(c[0]._seq, ids)], want="all").cpu()
    c[0]._seq.release()
    return lg


TOL = {"float32": 2e-5, "bfloat16": 4e-2}
Q = {"float32": 1.0, "bfloat16": 0.8}         # bf16: see garesun_helpers.rel_rms


# ------------------------------------------------------------------------------------------------ operators
def test_linear_any_all_formats_and_batched():
    from mlx_vlm_amd import ops

    g = torch.Generator().manual_seed(1)
    for M in (1, 3, 8, 9, 70):
        a, w = torch.randn(M, 37, generator=g), torch.randn(29, 37, generator=g)
        for ta in (torch.float32, torch.bfloat16):
            for tw in (torch.float32, torch.bfloat16):
                for tc in (torch.float32, torch.bfloat16):
                    A, Wt = a.to(ta).cuda(), w.to(tw).cuda()
                    got = ops.linear_any(A, Wt, out_dtype=tc).float().cpu()
                    want = (A.double().cpu() @ Wt.double().cpu().T)
                    tol = 1e-5 if tc == torch.float32 else 1e-2
                    assert (got.double() - want).abs().max() <= tol * want.abs().max(), (M, ta, tw, tc)
    # accumulate onto an fp32 stream; rows do not depend on their neighbours
    a, w = torch.randn(40, 24, generator=g).cuda(), torch.randn(16, 24, generator=g).cuda()
    x = torch.ones(40, 16, device="cuda")
    ops.linear_any(a, w, out=x, accumulate=True)
    assert torch.allclose(x.cpu(), 1 + a.cpu() @ w.cpu().T, atol=1e-5)
    assert torch.equal(ops.linear_any(a[:20], w), ops.linear_any(a, w)[:20])
    # per-head maps inside wider rows
    Hh, D, R, X = 3, 5, 7, 2
    q = torch.randn(11, Hh * (D + X), generator=g).cuda()
    wk = torch.randn(Hh, R, D, generator=g).cuda()
    out = torch.zeros(11, Hh * (R + X), device="cuda")
    ops.linear_any(q, wk.view(Hh * R, D), out=out, M=11, N=R, K=D, batch=Hh, stride_a=D + X, stride_w=R * D, stride_c=R + X)
    want = torch.einsum("thd,hrd->thr", q.view(11, Hh, D + X)[..., :D], wk)
    assert torch.allclose(out.view(11, Hh, R + X)[..., :R], want, atol=1e-5)
    assert out.view(11, Hh, R + X)[..., R:].abs().max() == 0


@pytest.mark.parametrize("M, N, K", [(300, 1600, 96), (333, 1030, 1000), (70, 7000, 52), (17, 260, 2080), (16, 16, 32), (5, 40, 37), (65, 96, 33), (1, 24, 8)])
def test_linear_any_f32_tiles(M, N, K):
    """every tile shape and both ways the ranges of k are run (rows 1, 16, 17, ... of the same operands take other tiles): the same bits per row;
    against float64 within K roundings of the sum of magnitudes"""
    from mlx_vlm_amd import ops

    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g).cuda()
    for tw in (torch.float32, torch.bfloat16):
        w = torch.randn(N, K, generator=g).to(tw).cuda()
        out = ops.linear_any(a, w)
        bound = a.double().abs() @ w.double().abs().T * (K * 2.0 ** -24)
        assert ((out.double() - a.double() @ w.double().T).abs() <= bound).all()
        if tw == torch.float32:
            for n in {1, min(9, M), min(16, M), min(40, M)}:
                assert torch.equal(ops.linear_any(a[M - n:], w), out[M - n:]), n
    # rows that are not whole 16-byte pieces
    b = torch.randn(M, K + 1, generator=g).cuda()[:, :K]
    w = torch.randn(N, K, generator=g).cuda()
    assert torch.equal(ops.linear_any(b, w), ops.linear_any(b.contiguous(), w) if K % 4 == 0 else ops.linear_any(b.clone(), w))


@pytest.mark.parametrize("M, N, K, batch", [(1, 40, 33, 1), (17, 260, 40, 1), (33, 1030, 97, 1), (100, 7000, 37, 1), (300, 600, 1031, 1), (70, 520, 129, 12), (257, 64, 515, 3), (65, 4100, 8, 1)])
@pytest.mark.parametrize("ta,tw", [("float32", "float32"), ("float32", "bfloat16"), ("bfloat16", "float32"), ("bfloat16", "bfloat16")])
def test_rows_that_are_not_whole_pieces_have_the_bits_of_those_that_are(M, N, K, batch, ta, tw):
    """every tile shape over rows at odd pitches and odd addresses, against the same rows padded to whole 16-byte pieces (zeros past K: the same chains).  (bf16 times
    bf16 rows take other kernels when they are aligned: against float64 there)"""
    from mlx_vlm_amd import ops

    g = torch.Generator().manual_seed(M + N + K)
    ta, tw = getattr(torch, ta), getattr(torch, tw)
    a, w = torch.randn(M, batch, K, generator=g).to(ta), torch.randn(batch, N, K, generator=g).to(tw)
    K8 = (K + 7) & ~7
    out, got = [], None
    for odd in (True, False):
        pad = K + 1 - K % 2 if odd else K8                   # (an odd number)
        abuf, wbuf = torch.zeros(M * batch * pad + 1, dtype=ta), torch.zeros(batch * N * pad + 1, dtype=tw)
        av, wv = (b[int(odd):][: b.numel() - 1].view(-1, pad) for b in (abuf, wbuf))
        av[:, :K], wv[:, :K] = a.reshape(-1, K), w.reshape(-1, K)
        ad, wd = abuf.cuda()[int(odd):][: M * batch * pad].view(M, batch * pad), wbuf.cuda()[int(odd):][: batch * N * pad].view(batch * N, pad)
        o = torch.empty(M, batch * N, device="cuda")
        ops.linear_any(ad, wd, out=o, M=M, N=N, K=K, batch=batch, stride_a=pad, stride_w=N * pad, stride_c=N)
        out.append(o)
    if M > 1 and tw == torch.bfloat16:
        ref = (a.double().transpose(0, 1) @ w.double().transpose(1, 2)).transpose(0, 1).reshape(M, batch * N).cuda()
        room = (a.double().abs().transpose(0, 1) @ w.double().abs().transpose(1, 2)).transpose(0, 1).reshape(M, batch * N).cuda() * (K * 2.0 ** -24)
        assert ((out[0].double() - ref).abs() <= room).all()
    elif not (M <= 8 and (ta, tw) != (torch.float32, torch.float32)):
        assert torch.equal(*out)


def test_stream_row_operators():
    from mlx_vlm_amd import ops

    g = torch.Generator().manual_seed(2)
    x = (torch.randn(9, 50, generator=g) * 3 + 1.5)
    w = torch.randn(50, generator=g)
    got = ops.layernorm_nobias(x.cuda(), w.cuda(), 1e-5).cpu()
    assert torch.allclose(got.double(), O.layer_norm_nobias(x.double(), w.double(), 1e-5), atol=1e-5)
    y = torch.randn(9, 50, generator=g)
    xs = x.clone().cuda()
    ops.unit_rms_add_(xs, y.cuda(), w.cuda(), 1e-5)
    assert torch.allclose(xs.cpu().double(), x.double() + O.unit_rms(y.double(), 1e-5) * w.double(), atol=1e-5)
    ids = torch.tensor([3, 0, 6, 6, 1, 2, 5, 4, 3], dtype=torch.int32)
    table = torch.randn(7, 12, generator=g)
    gate = torch.randn(9, 4, generator=g)
    got = ops.gelu_tanh_gate_rows(gate.cuda(), table.cuda(), ids.cuda(), 8).cpu()
    assert torch.allclose(got.double(), O.gelu_tanh(gate.double()) * table.double()[ids.long()][:, 8:12], atol=1e-6)
    emb = ops.embed_scale_f32(ids.cuda(), table.to(torch.bfloat16).cuda(), 2.5).cpu()
    assert torch.equal(emb, table.to(torch.bfloat16).float()[ids.long()] * 2.5)


@pytest.mark.parametrize("E,top", [(5, 2), (8, 8), (70, 1), (130, 6)])
def test_moe_route_top_k_and_softmax_over_chosen(E, top):
    from mlx_vlm_amd import ops

    z = torch.randn(33, E, generator=torch.Generator().manual_seed(E))
    z[0, :] = 0.25                                    # all equal: the lowest indices win
    gate, idx, wgt = (t.cpu() for t in ops.moe_route(z.cuda(), top))
    val, ref_idx = torch.topk(z[1:], top, dim=-1)
    assert torch.equal(idx[1:].long(), ref_idx)
    assert torch.allclose(wgt[1:], torch.softmax(val, -1), atol=1e-6)
    assert sorted(idx[0].tolist()) == list(range(top))
    dense = torch.zeros(33, E).scatter_(1, idx.long(), wgt)
    assert torch.equal(gate, dense)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("kind", ["retention", "mlstm", "latent_attention"])
def test_each_mixer_alone_and_each_feed_forward_shape(tmp_path, kind, dtype):
    for j, kw in enumerate((dict(mlp=None), dict(), dict(top=1, shared_ff=0), dict(experts=3, top=3))):
        cfg = H.config([H.layer(kind, **kw)], side=(0 if j == 0 else 8))
        W = H.weights(cfg, seed=10 + j)
        lm = _load(tmp_path, cfg, W, dtype, name=f"{kind}{j}").language_model
        ids = _ids(50, cfg["vocab"], j)
        want = O.Oracle(cfg, W, F64).forward(ids)
        assert H.rel_rms(_whole(lm, ids), want, Q[dtype]) < TOL[dtype], (kind, kw)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_layers_match_layer_by_layer(tmp_path, dtype):
    cfg = H.config(H.MIXED)
    W = H.weights(cfg, seed=3)
    lm = _load(tmp_path, cfg, W, dtype).language_model
    ids = _ids(70, cfg["vocab"], 5)
    orc = O.Oracle(cfg, W, F64)
    orc.forward(ids)
    lm._trace = []
    try:
        _whole(lm, ids)
        for i, (got, want) in enumerate(zip(lm._trace, orc.trace)):
            err = H.rel_rms(got.cpu(), want, Q[dtype])
            assert err < (1e-5 if dtype == "float32" else 2e-2), (i, cfg["layers"][i]["type"], float(err))
    finally:
        lm._trace = None


@pytest.mark.parametrize("gated,rot,D,Dv,Hh", [(1, 0, 128, 128, 3), (1, 0, 40, 130, 2), (1, 0, 13, 7, 1), (1, 0, 13, 8, 3), (0, 32, 32, 48, 3), (0, 20, 70, 16, 2), (0, 128, 128, 128, 2)])
def test_chunk_parallel_recurrences_against_the_token_by_token_kernel(gated, rot, D, Dv, Hh):
    """segments around the borders of a chunk next to short ones, fresh and carried states, workspaces of one chunk and of all: read-outs, states
    and maxima against float64, no further off than 1.5 times the token-by-token kernel (or 2^-20 of the largest value: sums of another order)"""
    from mlx_vlm_amd import _lib, ops

    g = torch.Generator().manual_seed(D + Dv)
    lens, pos0 = [1, 16, 17, 63, 64, 65, 200, 5], [0, 3, 0, 9, 0, 700, 130, 0]
    T, n, C, slots = sum(lens), len(lens), Dv + gated, len(lens) + 1
    cu = [sum(lens[:i]) for i in range(n + 1)]
    q, k = (torch.randn(T, Hh * D, generator=g).bfloat16() for _ in range(2))
    v, gate = (torch.randn(T, Hh * Dv, generator=g).bfloat16() for _ in range(2))
    ip, fp = torch.randn(T, Hh, generator=g).bfloat16() * 3, (torch.randn(T, Hh, generator=g) * 6).bfloat16()          # forget gates from 0 to 1
    ib, fb, cap = torch.zeros(Hh).bfloat16(), torch.full((Hh,), 2.0).bfloat16(), 12.0
    decay = torch.tensor([0.999, 0.9, 0.3][:Hh])
    inv = torch.tensor([1e4 ** (-2 * i / max(rot, 1)) for i in range(rot // 2)])
    state0 = torch.randn(slots, Hh, D, C, generator=g)
    m0 = torch.randn(slots, Hh, generator=g)
    # float64, token by token
    want, ends, mends = torch.zeros(T, Hh, C, dtype=F64), state0.double().clone(), m0.double().clone()
    for i in range(n):
        S = state0[i + 1].double().clone() if pos0[i] else torch.zeros(Hh, D, C, dtype=F64)
        m = m0[i + 1].double().clone() if pos0[i] else torch.zeros(Hh, dtype=F64)
        for t in range(cu[i], cu[i + 1]):
            qt, kt, vt = (x[t].double().view(Hh, -1) for x in (q, k, v))
            if rot:
                a = (pos0[i] + t - cu[i]) * inv.double()
                turn = lambda x: torch.cat([x[:, : rot // 2] * a.cos() - x[:, rot // 2: rot] * a.sin(), x[:, rot // 2: rot] * a.cos() + x[:, : rot // 2] * a.sin(), x[:, rot:]], 1)      # noqa: E731
                qt, kt = turn(qt), turn(kt)
            qt, kt = qt * 0.5, kt * 0.25
            if gated:
                it = cap * torch.tanh((ip[t].double() + ib.double()) / cap)
                ft = torch.nn.functional.logsigmoid(cap * torch.tanh((fp[t].double() + fb.double()) / cap))
                mn = torch.maximum(ft + m, it)
                da, db, m = torch.exp(ft + m - mn), torch.exp(it - mn), mn
                vt = torch.cat([vt, torch.ones(Hh, 1, dtype=F64)], 1)
            else:
                da, db = decay.double(), torch.ones(Hh, dtype=F64)
            S = da.view(Hh, 1, 1) * S + db.view(Hh, 1, 1) * kt.unsqueeze(2) * vt.unsqueeze(1)
            want[t] = torch.einsum("hdc,hd->hc", S, qt)
        ends[i + 1], mends[i + 1] = S, m
    dev = {x: y.cuda() for x, y in dict(q=q, k=k, v=v, gate=gate, ip=ip, fp=fp, ib=ib, fb=fb, decay=decay, inv=inv).items()}
    tab = torch.tensor(cu + list(range(1, n + 1)) + pos0, dtype=torch.int32).cuda()
    prep = (4 * Hh if gated else 2 * Hh * D) * T + 4

    def run(ws_floats):
        st, ms = state0.cuda(), m0.cuda()
        raw, out = torch.empty(T, Hh, C, device="cuda"), torch.empty(T, Hh * Dv, dtype=torch.bfloat16, device="cuda")
        mtok, mprev = torch.empty(T, Hh, device="cuda"), torch.empty(n, Hh, device="cuda")
        ws = torch.full((ws_floats,), float("nan"), device="cuda") if ws_floats else None
        a = _lib.RecurrenceArgs()
        a.q, a.k, a.v, a.g = (dev[x].data_ptr() for x in ("q", "k", "v", "gate"))
        a.ldq = a.ldk = Hh * D
        a.ldv = a.ldg = a.ldo = Hh * Dv
        a.qscale, a.kscale, a.eps, a.gate_act, a.gated, a.rot_dims = 0.5, 0.25, 1e-5, 1, gated, rot
        if gated:
            a.ipre, a.fpre, a.ldi, a.ldf, a.ib, a.fb, a.cap = dev["ip"].data_ptr(), dev["fp"].data_ptr(), Hh, Hh, dev["ib"].data_ptr(), dev["fb"].data_ptr(), cap
            a.mstate, a.mtok, a.mprev = ms.data_ptr(), mtok.data_ptr(), mprev.data_ptr()
        else:
            a.decay, a.inv_freq = dev["decay"].data_ptr(), dev["inv"].data_ptr()
        a.seg_start, a.seg_slot, a.seg_pos0 = tab.data_ptr(), tab[n + 1:].data_ptr(), tab[2 * n + 1:].data_ptr()
        a.state, a.raw, a.out, a.H, a.D, a.Dv = st.data_ptr(), raw.data_ptr(), out.data_ptr(), Hh, D, Dv
        if ws is not None:
            a.ws, a.ws_floats = ws.data_ptr(), ws.numel()
        ops.linear_recurrence(a, n, T, False)
        torch.cuda.synchronize()
        return raw.cpu().double(), st.cpu().double(), ms.cpu().double()

    serial = run(0)
    for chunks in (1, 3, T // 64 + n):
        for got, ref, old in zip(run(prep + chunks * Hh * D * C), (want, ends, mends), serial):
            err, lim = (got - ref).abs().max(), ref.abs().max()
            assert err <= max(1.5 * (old - ref).abs().max(), lim * 2.0 ** -20), (chunks, float(err), float((old - ref).abs().max()), float(lim))
    assert all(torch.equal(x, y) for x, y in zip(run(Hh * D * Dv), serial))         # no room behind the prepared rows: token by token


@pytest.mark.parametrize("gated,rot,q_act,decays", [(1, 20, 0, None), (1, 0, 1, None), (1, 20, 1, None), (0, 0, 1, [0.9, 0.5]), (0, 20, 0, [0.9, 0.5]),
                                                    (0, 20, 0, [-0.9, 0.0]), (0, 0, 0, [-0.97, 1.0])])
def test_a_workspace_changes_no_recurrence(gated, rot, q_act, decays):
    """every form of the call that is accepted, with a workspace and without: gated heads with rotated keys, and with the flag of an activation that gated heads
    do not have; decays of either sign, zero and one.  Sums of another order: 2^-18 of the largest value"""
    from mlx_vlm_amd import _lib, ops

    g, T, Hh, D, Dv = torch.Generator().manual_seed(rot + q_act), 150, 2, 32, 24
    C = Dv + gated
    q, k = (torch.randn(T, Hh * D, generator=g).bfloat16().cuda() for _ in range(2))
    v, gate = (torch.randn(T, Hh * Dv, generator=g).bfloat16().cuda() for _ in range(2))
    pre = torch.randn(2, T, Hh, generator=g).bfloat16().cuda()
    bias, decay = torch.ones(Hh).bfloat16().cuda(), torch.tensor(decays or [0.5] * Hh).cuda()
    inv = torch.tensor([1e4 ** (-2 * i / 20) for i in range(10)]).cuda()
    state0, m0 = torch.randn(2, Hh, D, C, generator=g), torch.randn(2, Hh, generator=g)
    tab = torch.tensor([0, T, 1, 7], dtype=torch.int32).cuda()

    def run(ws):
        state, ms, mtok, mprev = state0.cuda(), m0.cuda(), torch.empty(T, Hh, device="cuda"), torch.empty(1, Hh, device="cuda")
        raw, out = torch.empty(T, Hh, C, device="cuda"), torch.empty(T, Hh * Dv, dtype=torch.bfloat16, device="cuda")
        a = _lib.RecurrenceArgs()
        a.q, a.k, a.v, a.g, a.ldq, a.ldk, a.ldv, a.ldg, a.ldo = q.data_ptr(), k.data_ptr(), v.data_ptr(), gate.data_ptr(), Hh * D, Hh * D, Hh * Dv, Hh * Dv, Hh * Dv
        a.qscale, a.kscale, a.eps, a.gate_act, a.gated, a.rot_dims, a.q_act, a.decay, a.inv_freq = 0.5, 0.25, 1e-5, 1, gated, rot, q_act, decay.data_ptr(), inv.data_ptr()
        a.ipre, a.fpre, a.ldi, a.ldf, a.ib, a.fb, a.cap = pre[0].data_ptr(), pre[1].data_ptr(), Hh, Hh, bias.data_ptr(), bias.data_ptr(), 12.0
        a.mstate, a.mtok, a.mprev = ms.data_ptr(), mtok.data_ptr(), mprev.data_ptr()
        a.seg_start, a.seg_slot, a.seg_pos0 = tab.data_ptr(), tab[2:].data_ptr(), tab[3:].data_ptr()
        a.state, a.raw, a.out, a.H, a.D, a.Dv = state.data_ptr(), raw.data_ptr(), out.data_ptr(), Hh, D, Dv
        if ws is not None:
            a.ws, a.ws_floats = ws.data_ptr(), ws.numel()
        ops.linear_recurrence(a, 1, T, False)
        torch.cuda.synchronize()
        return raw.cpu().double(), state.cpu().double(), ms.cpu().double()

    for got, want in zip(run(torch.empty(1 << 20, device="cuda")), run(None)):
        assert (got - want).abs().max() <= want.abs().max() * 2.0 ** -18


@pytest.mark.parametrize("gated,rot", [(0, 0), (0, 8), (1, 0)])
def test_a_workspace_and_more_segments_than_a_grid_dimension_has(gated, rot):
    """65536 segments of one token and one of 40: served with a workspace as without, and to the same bits"""
    from mlx_vlm_amd import _lib, ops

    g, n, D = torch.Generator().manual_seed(5), 65537, 8
    T, C = n + 39, D + gated
    q, k, v, gate = (torch.randn(T, D, generator=g).bfloat16().cuda() for _ in range(4))
    pre, bias, decay = torch.randn(2, T, 1, generator=g).bfloat16().cuda(), torch.ones(1).bfloat16().cuda(), torch.tensor([0.9]).cuda()
    inv = torch.tensor([1.0, 0.1, 0.01, 0.001]).cuda()
    cu = torch.cat([torch.arange(n, dtype=torch.int32), torch.tensor([T], dtype=torch.int32)]).cuda()
    slots, pos0 = torch.arange(n, dtype=torch.int32).cuda(), torch.zeros(n, dtype=torch.int32).cuda()

    def run(ws):
        state, ms, mtok, mprev = torch.zeros(n, 1, D, C, device="cuda"), torch.zeros(n, 1, device="cuda"), torch.zeros(T, 1, device="cuda"), torch.zeros(n, 1, device="cuda")
        raw, out = torch.empty(T, 1, C, device="cuda"), torch.empty(T, D, dtype=torch.bfloat16, device="cuda")
        a = _lib.RecurrenceArgs()
        a.q, a.k, a.v, a.g, a.ldq, a.ldk, a.ldv, a.ldg, a.ldo = q.data_ptr(), k.data_ptr(), v.data_ptr(), gate.data_ptr(), D, D, D, D, D
        a.qscale, a.kscale, a.eps, a.gate_act, a.gated, a.rot_dims, a.decay, a.inv_freq = 0.5, 0.25, 1e-5, 1, gated, rot, decay.data_ptr(), inv.data_ptr()
        a.ipre, a.fpre, a.ldi, a.ldf, a.ib, a.fb, a.cap = pre[0].data_ptr(), pre[1].data_ptr(), 1, 1, bias.data_ptr(), bias.data_ptr(), 12.0
        a.mstate, a.mtok, a.mprev = ms.data_ptr(), mtok.data_ptr(), mprev.data_ptr()
        a.seg_start, a.seg_slot, a.seg_pos0 = cu.data_ptr(), slots.data_ptr(), pos0.data_ptr()
        a.state, a.raw, a.out, a.H, a.D, a.Dv = state.data_ptr(), raw.data_ptr(), out.data_ptr(), 1, D, D
        if ws is not None:
            a.ws, a.ws_floats = ws.data_ptr(), ws.numel()
        ops.linear_recurrence(a, n, T, False)
        torch.cuda.synchronize()
        return raw, state, ms

    assert all(torch.equal(x, y) for x, y in zip(run(torch.empty(1 << 22, device="cuda")), run(None)))


@pytest.mark.parametrize("gated,rot", [(0, 0), (0, 20), (1, 0)])
def test_values_that_are_not_finite_stay_with_later_tokens(gated, rot):
    """an infinity and a NaN among the values of a prompt: the read-outs of the tokens before them, and of the columns beside them, are what they are without
    them (sums of another order within 16 tokens: 2^-20 of the largest); what follows is not finite in those columns"""
    from mlx_vlm_amd import _lib, ops

    g, T, Hh, D, Dv = torch.Generator().manual_seed(rot), 200, 2, 32, 40
    C = Dv + gated
    q, k = (torch.randn(T, Hh * D, generator=g).bfloat16().cuda() for _ in range(2))
    v, gate = (torch.randn(T, Hh * Dv, generator=g).bfloat16().cuda() for _ in range(2))
    pre, bias, decay = torch.randn(2, T, Hh, generator=g).bfloat16().cuda(), torch.ones(Hh).bfloat16().cuda(), torch.tensor([0.9, 0.99]).cuda()
    inv, tab, ws = torch.tensor([1e4 ** (-2 * i / 20) for i in range(10)]).cuda(), torch.tensor([0, T, 0, 0], dtype=torch.int32).cuda(), torch.empty(1 << 20, device="cuda")

    def run(v):
        state, ms, mtok, mprev = torch.zeros(1, Hh, D, C, device="cuda"), torch.zeros(1, Hh, device="cuda"), torch.empty(T, Hh, device="cuda"), torch.empty(1, Hh, device="cuda")
        raw, out = torch.empty(T, Hh, C, device="cuda"), torch.empty(T, Hh * Dv, dtype=torch.bfloat16, device="cuda")
        a = _lib.RecurrenceArgs()
        a.q, a.k, a.v, a.g, a.ldq, a.ldk, a.ldv, a.ldg, a.ldo = q.data_ptr(), k.data_ptr(), v.data_ptr(), gate.data_ptr(), Hh * D, Hh * D, Hh * Dv, Hh * Dv, Hh * Dv
        a.qscale, a.kscale, a.eps, a.gate_act, a.gated, a.rot_dims, a.decay, a.inv_freq = 0.5, 0.25, 1e-5, 1, gated, rot, decay.data_ptr(), inv.data_ptr()
        a.ipre, a.fpre, a.ldi, a.ldf, a.ib, a.fb, a.cap = pre[0].data_ptr(), pre[1].data_ptr(), Hh, Hh, bias.data_ptr(), bias.data_ptr(), 12.0
        a.mstate, a.mtok, a.mprev = ms.data_ptr(), mtok.data_ptr(), mprev.data_ptr()
        a.seg_start, a.seg_slot, a.seg_pos0 = tab.data_ptr(), tab[2:].data_ptr(), tab[3:].data_ptr()
        a.state, a.raw, a.out, a.H, a.D, a.Dv, a.ws, a.ws_floats = state.data_ptr(), raw.data_ptr(), out.data_ptr(), Hh, D, Dv, ws.data_ptr(), ws.numel()
        ops.linear_recurrence(a, 1, T, False)
        torch.cuda.synchronize()
        return raw.cpu()

    want, bad = run(v), v.clone()
    bad[75, 3], bad[75, 39], bad[137, 7] = float("inf"), float("nan"), float("-inf")          # head 0, columns 3 and 39, then 7
    got = run(bad)
    close = lambda x, y: bool(((x - y).abs() <= want.abs().max() * 2.0 ** -20).all())          # noqa: E731
    for col, first in ((3, 75), (39, 75), (7, 137)):
        assert close(got[:first, 0, col], want[:first, 0, col]) and not torch.isfinite(got[first:, 0, col]).any()
    rest = [c for c in range(C) if c not in (3, 39, 7)]
    assert close(got[:, 0, rest], want[:, 0, rest]) and close(got[:, 1], want[:, 1])


def test_one_workspace_serves_all_recurrent_layers(tmp_path):
    """a prompt over four recurrent layers of two kinds: what the step holds on to has one workspace, as large as the neediest layer's"""
    cfg = H.config([H.layer("retention"), H.layer("mlstm"), H.layer("retention", heads=2, dim=40), H.layer("mlstm")])
    lm = _load(tmp_path, cfg, H.weights(cfg), "bfloat16")
    lm = getattr(lm, "language_model", lm)
    T = 200
    _whole(lm, _ids(T, cfg["vocab"], 1))
    flat = [x.numel() for x in lm._keep if isinstance(x, torch.Tensor) and x.dtype == torch.float32 and x.dim() == 1]
    need = [(4 * ns.H if ns.type == "mlstm" else 2 * ns.H * ns.D) * T + 4 + (T // 64 + 1) * ns.H * ns.D * (ns.Dv + (ns.type == "mlstm")) for ns in lm._L]
    assert flat == [max(need)]


# ------------------------------------------------------------------------------------------------ schedules
@pytest.fixture(scope="module")
def mixed32(tmp_path_factory):
    cfg = H.config(H.MIXED)
    W = H.weights(cfg, seed=7)
    lm = _load(tmp_path_factory.mktemp("g32"), cfg, W, "float32", tokens=1024, seqs=4).language_model
    return cfg, W, lm


def _portions(lm, ids, sizes):
    """feed ids in portions of the given sizes (cycled), every row's logits"""
    c = lm.make_cache()
    out, o, j = [], 0, 0
    while o < len(ids):
        n = min(sizes[j % len(sizes)], len(ids) - o)
        out.append(lm.step([(c[0]._seq, ids[o:o + n])], want="all").cpu())
        o, j = o + n, j + 1
    c[0]._seq.release()
    return torch.cat(out)


def test_portions_and_token_by_token_equal_the_whole_prompt(mixed32):
    cfg, W, lm = mixed32
    ids = _ids(150, cfg["vocab"], 11)          # crosses two page borders and the recurrence's 16-token staging blocks
    whole = _whole(lm, ids)
    assert H.rel_rms(whole, O.Oracle(cfg, W, F64).forward(ids)) < TOL["float32"]
    for sizes in ([2], [3, 61, 2, 64], [37, 2, 3], [64], [63, 1, 1, 65], [1]):
        got = _portions(lm, ids, sizes)
        assert torch.equal(got, whole), sizes               # float32 serving: the same bits however the prompt is cut


def test_bf16_portions_and_decode(tmp_path):
    cfg = H.config(H.MIXED)
    W = H.weights(cfg, seed=8)
    lm = _load(tmp_path, cfg, W, "bfloat16", tokens=1024, seqs=4).language_model
    ids = _ids(140, cfg["vocab"], 12)
    want = O.Oracle(cfg, W, F64).forward(ids)
    for sizes in ([140], [2, 30, 64, 5], [100] + [1] * 40):
        assert H.rel_rms(_portions(lm, ids, sizes), want, Q["bfloat16"]) < TOL["bfloat16"], sizes


def test_unequal_batch_equals_each_alone_and_slots_are_reused(mixed32):
    cfg, W, lm = mixed32
    V = cfg["vocab"]
    reqs = [_ids(n, V, 20 + n) for n in (130, 1, 23, 70, 66, 5, 90)]
    alone = [_whole(lm, r) for r in reqs]
    free0, slots0 = lm.pool.free_pages, len(lm.pool._free_seqs)
    # four live requests at a time (the pool has four slots); the others queue and take over freed pages / slots
    live, done, queue, got = {}, {}, list(range(len(reqs))), {i: [] for i in range(len(reqs))}
    rng = np.random.default_rng(0)
    seen_slots = []
    while queue or live:
        while queue and len(live) < 4:
            i = queue.pop(0)
            live[i] = [lm.make_cache(), 0]
            seen_slots.append(live[i][0][0]._seq.seq)
        entries, who = [], []
        for i, (c, o) in live.items():
            if rng.random() < 0.25 and len(live) > 1:
                continue                                   # left out of this step
            n = int(min(len(reqs[i]) - o, rng.choice([1, 1, 2, 3, 17, 64])))
            entries.append((c[0]._seq, reqs[i][o:o + n]))
            who.append((i, n))
        if not entries:
            continue
        lg = lm.step(entries, want="all").cpu()
        r = 0
        for i, n in who:
            got[i].append(lg[r:r + n])
            r += n
            live[i][1] += n
            if live[i][1] == len(reqs[i]):
                live.pop(i)[0][0]._seq.release()
    assert len(set(seen_slots)) <= 4 and len(seen_slots) == len(reqs)          # slots were used again
    assert lm.pool.free_pages == free0 and len(lm.pool._free_seqs) == slots0   # everything was given back
    for i in range(len(reqs)):
        assert torch.equal(torch.cat(got[i]), alone[i]), i     # ... and whatever else is in the batch, whichever slot and pages


def test_pool_exhaustion_is_an_error_not_a_fault(tmp_path):
    cfg = H.config([H.layer("latent_attention")])
    lm = _load(tmp_path, cfg, H.weights(cfg), "float32", tokens=128, seqs=2).language_model
    a, b = lm.make_cache(), lm.make_cache()
    lm.step([(a[0]._seq, _ids(100, 97, 0))])
    with pytest.raises(RuntimeError):
        lm.step([(b[0]._seq, _ids(10, 97, 1))])               # both pages are taken
    with pytest.raises(RuntimeError):
        lm.make_cache()                                          # both slots are taken
    a[0]._seq.release()
    lm.step([(b[0]._seq, _ids(100, 97, 1))])
    b[0]._seq.release()


# ------------------------------------------------------------------------------------------------ far keys, borders
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_latent_attention_finds_one_key_anywhere(dtype):
    """operator level: one cached row is made to score far above the rest; the output must be that row's latent, wherever
    it sits (first token, page borders 63 / 64, tile borders 255 / 256, far back, the query's own position)"""
    from mlx_vlm_amd import ops
    from mlx_vlm_amd.models.cache import PAGE

    R, Dr, Hh, n = 24, 8, 3, 700
    g = torch.Generator().manual_seed(4)
    rows = torch.randn(n, R + Dr, generator=g) * 0.1
    pages = torch.randperm(16, generator=g)[: (n + PAGE - 1) // PAGE].to(torch.int32)         # scattered pages
    pool = torch.zeros(16, PAGE, R + Dr)
    for j in range(n):
        pool[pages[j // PAGE], j % PAGE] = rows[j]
    pool_d = pool.to(dtype).cuda()
    bt = torch.zeros(2, 16, dtype=torch.int32)
    bt[1, : len(pages)] = pages
    qdir = torch.randn(R + Dr, generator=g)
    qdir /= qdir.norm()
    for key in (0, 1, 63, 64, 65, 255, 256, 257, 511, 512, 640, 699):
        for qpos in (key, key + 1, 699):
            if qpos >= n:
                continue
            p2 = pool_d.clone()
            p2[pages[key // PAGE], key % PAGE] = (rows[key] + 6.0 * qdir).to(dtype)
            q = (qdir * 8.0).repeat(Hh, 1).reshape(1, Hh, R + Dr).cuda()
            out = ops.latent_attn(q, p2, torch.tensor([1], dtype=torch.int32).cuda(), torch.tensor([qpos], dtype=torch.int32).cuda(),
                                  bt.cuda(), Hh, R, Dr, 1.0).cpu()
            want = p2[pages[key // PAGE], key % PAGE, :R].float().cpu()
            assert (out[0] - want).abs().max() < 1e-3, (key, qpos)
        if key + 1 < n:                                        # ... and one position BEFORE the key it must not be seen
            out = ops.latent_attn(q, p2, torch.tensor([1], dtype=torch.int32).cuda(), torch.tensor([key - 1 if key else 0], dtype=torch.int32).cuda(),
                                  bt.cuda(), Hh, R, Dr, 1.0).cpu()
            if key:
                assert (out[0] - want).abs().max() > 0.05, key


def test_far_key_through_the_model_in_prompt_and_decoding(tmp_path):
    """model level: a latent-attention layer whose query and key projections are scaled up, so that softmax weight sits on
    few keys; a token 600 back is then visible in the logits - compared in a prompt, in portions and decoded one by one"""
    cfg = H.config([H.layer("latent_attention", heads=2, kv_rank=16, dim=16), H.layer("retention")], side=0)
    W = H.weights(cfg, seed=21)
    W["l0.mix.q"] = (W["l0.mix.q"].float() * 4).to(torch.bfloat16)
    W["l0.mix.uk"] = (W["l0.mix.uk"].float() * 4).to(torch.bfloat16)
    lm = _load(tmp_path, cfg, W, "float32", tokens=2048, seqs=2).language_model
    ids = _ids(700, cfg["vocab"], 3)
    ids[650:] = ids[40:90]                       # the tail repeats tokens seen 610 back
    want = O.Oracle(cfg, W, F64).forward(ids)
    whole = _whole(lm, ids)
    assert H.rel_rms(whole[600:], want[600:]) < TOL["float32"]
    assert H.rel_rms(_portions(lm, ids, [640] + [1] * 60)[600:], want[600:]) < TOL["float32"]
    assert H.rel_rms(_portions(lm, ids, [255, 2, 63])[600:], want[600:]) < TOL["float32"]


def test_first_tokens_and_a_one_token_request(mixed32):
    cfg, W, lm = mixed32
    for n in (1, 2, 3):
        ids = _ids(n, cfg["vocab"], 40 + n)
        assert H.rel_rms(_whole(lm, ids), O.Oracle(cfg, W, F64).forward(ids)) < TOL["float32"], n


def test_long_decoding_keeps_the_recurrent_state(tmp_path):
    cfg = H.config([H.layer("mlstm"), H.layer("retention", decay=[0.999, 0.9, 0.5])], side=4)
    W = H.weights(cfg, seed=31)
    lm = _load(tmp_path, cfg, W, "float32", tokens=1024, seqs=2).language_model
    ids = _ids(400, cfg["vocab"], 9)
    want = O.Oracle(cfg, W, F64).forward(ids)
    got = _portions(lm, ids, [20] + [1] * 380)
    assert H.rel_rms(got[-50:], want[-50:]) < TOL["float32"]


def test_other_sizes_wide_heads_and_many_experts(tmp_path):
    layers = [H.layer("mlstm", heads=1, dim=72, vdim=130, experts=20, top=4, ff=8), H.layer("latent_attention", heads=1, kv_rank=264, dim=8, rot_dim=2, vdim=40),
              H.layer("retention", heads=7, dim=8, vdim=8, rot_dims=2, decay=[0.9] * 7), H.layer("latent_attention", heads=2, kv_rank=264, rot_dim=2, kv_from=1)]
    cfg = H.config(layers, vocab=301, width=100, side=3, scale=0.7, eps=1e-3)
    W = H.weights(cfg, seed=41)
    ids = _ids(90, 301, 2)
    want = O.Oracle(cfg, W, F64).forward(ids)
    for dtype in ("float32", "bfloat16"):
        lm = _load(tmp_path, cfg, W, dtype, name=dtype).language_model
        assert H.rel_rms(_portions(lm, ids, [70, 2, 1]), want, Q[dtype]) < TOL[dtype], dtype


# ------------------------------------------------------------------------------------------------ generation paths
def _greedy_oracle(cfg, W, prompt, n):
    """teacher: float64 greedy continuation, and the margin of every choice"""
    orc = O.Oracle(cfg, W, F64)
    lg = orc.forward(prompt)[-1]
    out, margins = [], []
    for _ in range(n):
        top2 = torch.topk(lg, 2).values
        margins.append(float(top2[0] - top2[1]))
        out.append(int(lg.argmax()))
        lg = orc.forward([out[-1]])[-1]
    return out, margins


def test_greedy_generation_through_generate_step_and_the_batch_generator(tmp_path):
    from mlx_vlm_amd.batch import BatchGenerator
    from mlx_vlm_amd.generate import generate_step

    cfg = H.config(H.MIXED[:4])
    W = H.weights(cfg, seed=51)
    W["head"] = (W["head"].float() * 6).to(torch.bfloat16)          # wide margins: greedy choices survive bf16 logits
    model = _load(tmp_path, cfg, W, "float32", tokens=2048, seqs=8)
    prompts = [_ids(n, cfg["vocab"], 60 + n) for n in (9, 70, 33)]
    refs = [_greedy_oracle(cfg, W, p, 12) for p in prompts]

    def agree(got, ref):
        toks, margins = ref
        for a, b, m in zip(got, toks, margins):
            if a != b:
                assert m < 0.05, (got, toks, margins)            # a tie within the bf16 rounding of the sampler's logits
                return
    for p, ref in zip(prompts, refs):
        got = [t for t, _ in generate_step(p[None], model, None, None, max_tokens=12, temperature=0.0)]
        assert len(got) == 12
        agree(got, ref)
    gen = BatchGenerator(model, None, max_tokens=12, completion_batch_size=2, prefill_batch_size=2, compute_logprobs=True)
    uids = gen.insert([p for p in prompts])
    out = {u: [] for u in uids}
    while gen.has_work:
        _, rs = gen.next()
        for r in rs:
            out[r.uid].append(r.token)
    gen.close()
    for u, ref in zip(uids, refs):
        assert len(out[u]) == 12
        agree(out[u], ref)
    assert len(model.language_model.pool._free_seqs) >= 7         # rows gave their slots back (the scratch row keeps one)


def test_trace_session_replays_mixed_steps(tmp_path):
    from mlx_vlm_amd.batch import TraceSession

    cfg = H.config(H.MIXED[:3])
    W = H.weights(cfg, seed=61)
    model = _load(tmp_path, cfg, W, "float32", tokens=256, seqs=4)
    a, b = _ids(100, cfg["vocab"], 1), _ids(30, cfg["vocab"], 2)
    wa, wb = O.Oracle(cfg, W, F64).forward(a), O.Oracle(cfg, W, F64).forward(b)
    s = TraceSession(model)
    assert s.step([("a", a[:64].tolist(), [])]) is None
    lg = s.step([("a", a[64:99].tolist(), [0, 34]), ("b", b[:29].tolist(), [28])])
    assert H.rel_rms(lg, torch.stack([wa[64], wa[98], wb[28]])) < TOL["float32"]
    lg = s.step([("b", b[29:].tolist(), [0]), ("a", a[99:].tolist(), [0])], end=["a", "b"])
    assert H.rel_rms(lg, torch.stack([wb[29], wa[99]])) < TOL["float32"]
    assert model.language_model.pool.free_pages == 4


def test_captured_decode_steps_equal_eager_ones(tmp_path):
    """a captured decode step is replayed many times, with eager work (another request's prompt, a release, synchronisations)
    between the replays; every replay's logits and token must equal the eager step's"""
    from mlx_vlm_amd.sample_utils import make_sampler

    cfg = H.config(H.MIXED)
    W = H.weights(cfg, seed=71)
    lm = _load(tmp_path, cfg, W, "bfloat16", tokens=2048, seqs=6).language_model
    sargs = make_sampler().engine_args()
    prompts = [_ids(n, cfg["vocab"], 80 + n) for n in (40, 7, 66)]

    def run(use_graph):
        caches = lm.make_cache_batch(3)
        lg = lm.prefill(torch.cat([torch.as_tensor(p) for p in prompts]).cuda().reshape(-1, 1), None, caches, [len(p) for p in prompts])
        st = lm.decode_begin(caches, lg.argmax(-1), np.zeros((3, 1)), max_new_tokens=80)
        out = []
        for i in range(70):                                          # crosses a page border in every row
            lm.decode_run(st, 1, sargs, use_graph=use_graph)
            out.append((st.tok.cpu().clone(), st.logits.float().cpu().clone()))
            if i % 9 == 4:                                           # eager work between replays
                other = lm.make_cache()
                lm.step([(other[0]._seq, _ids(30 + i, cfg["vocab"], i))])
                torch.cuda.synchronize()
                other[0]._seq.release()
        for c in caches:
            c[0]._seq.release()
        return out
    eager, graph = run(False), run(True)
    assert any(isinstance(v, tuple) for v in lm._graphs.values())            # a graph was captured and used
    for i, ((t0, l0), (t1, l1)) in enumerate(zip(eager, graph)):
        assert torch.equal(t0, t1) and torch.equal(l0, l1), i


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_latent_attention_prompt_form_equals_row_form(dtype):
    """the two attention kernels (query blocks through LDS / one row per workgroup) against a dense softmax, ragged batch:
    two sequences at different offsets on scattered pages, blocks that end inside a tile"""
    from mlx_vlm_amd import ops
    from mlx_vlm_amd.models.cache import PAGE

    R, Dr, Hh = 40, 8, 3
    g = torch.Generator().manual_seed(9)
    lens, offs = [37, 5], [150, 0]                   # sequence 0: 37 new tokens after 150 cached ones; sequence 1: 5 from the start
    bt = torch.zeros(3, 8, dtype=torch.int32)
    bt[1, :3] = torch.tensor([5, 2, 7])
    bt[2, :1] = torch.tensor([4])
    pool = (torch.randn(8, PAGE, R + Dr, generator=g) * 0.5).to(dtype)
    tok_seq = torch.tensor([1] * 37 + [2] * 5, dtype=torch.int32)
    tok_pos = torch.tensor(list(range(150, 187)) + list(range(5)), dtype=torch.int32)
    q = torch.randn(42, Hh, R + Dr, generator=g)
    gate = torch.randn(42, Hh, generator=g).to(dtype)
    qb_start = torch.tensor([0, 16, 32, 37], dtype=torch.int32)
    qb_count = torch.tensor([16, 16, 5, 5], dtype=torch.int32)
    a = ops.latent_attn(q.cuda(), pool.cuda(), tok_seq.cuda(), tok_pos.cuda(), bt.cuda(), Hh, R, Dr, 0.3, gate=gate.cuda()).cpu()
    b = ops.latent_attn_blocks(q.cuda(), pool.cuda(), qb_start.cuda(), qb_count.cuda(), tok_seq.cuda(), tok_pos.cuda(), bt.cuda(), Hh, R, Dr,
                               0.3, gate=gate.cuda()).cpu()
    want = torch.zeros(42, Hh, R, dtype=torch.float64)
    for t in range(42):
        sq, pos = int(tok_seq[t]), int(tok_pos[t])
        rows = torch.stack([pool[bt[sq, j // PAGE], j % PAGE] for j in range(pos + 1)]).double()
        w = torch.softmax(torch.einsum("hd,jd->hj", q[t].double(), rows) * 0.3, -1)
        want[t] = torch.einsum("hj,jr->hr", w, rows[:, :R]) * torch.sigmoid(gate[t].double())[:, None]
    assert (a.double() - want).abs().max() < 2e-5 and (b.double() - want).abs().max() < 2e-5


def test_sampled_generation_uses_the_device_sampler_and_refuses_what_is_not_built(tmp_path):
    from mlx_vlm_amd.generate import generate_step

    cfg = H.config(H.MIXED[:3])
    model = _load(tmp_path, cfg, H.weights(cfg, seed=91), "bfloat16", tokens=1024, seqs=4)
    p = _ids(20, cfg["vocab"], 5)
    runs = [[t for t, _ in generate_step(p[None], model, None, None, max_tokens=16, temperature=0.8, top_p=0.9, seed=7)] for _ in range(2)]
    assert runs[0] == runs[1] and len(runs[0]) == 16 and all(0 <= t < cfg["vocab"] for t in runs[0])
    other = [t for t, _ in generate_step(p[None], model, None, None, max_tokens=16, temperature=0.8, top_p=0.9, seed=8)]
    greedy = [t for t, _ in generate_step(p[None], model, None, None, max_tokens=16, temperature=0.0)]
    assert other != runs[0] or greedy != runs[0]                    # the draw depends on the seed / temperature
    with pytest.raises(NotImplementedError):
        list(generate_step(p[None], model, None, None, max_tokens=4, repetition_penalty=1.3))
    assert len(model.language_model.pool._free_seqs) == 4           # every generation gave its slot back


# ------------------------------------------------------------------------------------------------ steps of few rows
@pytest.mark.parametrize("M", [2, 3, 8, 16, 17, 32, 33, 300])
@pytest.mark.parametrize("N,K,batch", [(1, 8, 1), (8, 1536, 1), (100, 200, 3), (257, 72, 1), (1544, 136, 1), (4104, 64, 1), (8192, 264, 1), (16, 4096, 1), (16, 4104, 1),
                                       (512, 128, 28), (128, 512, 12), (64, 1536, 1), (65, 1536, 1),
                                       (512, 128, 12), (256, 192, 28), (100, 64, 130), (130, 72, 60), (20, 40, 300)])          # (maps: pieces of columns that do not come out even)
def test_linear_any_few_rows_over_bf16_weights(M, N, K, batch):
    """tiles of R columns (R = 1 to 16, one or two a wave), pieces of 64 of K cut short, both sides of the lines in rows, columns and K, a pitch, bf16 and
    fp32 rows and results, accumulation.  Every sum is at most K / 256 + 12 roundings of 2^-24 of partial sums below sum |a w|: 2^-19 of it"""
    from mlx_vlm_amd import ops

    g = torch.Generator().manual_seed(N + K + M)
    a, w = torch.randn(M, batch * K + 16, generator=g), (torch.randn(batch * N, K + 8, generator=g)).bfloat16().cuda()[:, :K]
    for ta in (torch.bfloat16, torch.float32):
        at = a.to(ta).cuda()[:, : batch * K]
        ad, wd = at.double().reshape(M, batch, K).transpose(0, 1), w.double().view(batch, N, K).transpose(1, 2)
        want, room = (ad @ wd).transpose(0, 1).reshape(M, batch * N), (ad.abs() @ wd.abs()).transpose(0, 1).reshape(M, batch * N) * 2.0 ** -19
        for tc in (torch.bfloat16, torch.float32):
            out = torch.full((M, batch * N), 3.0, dtype=tc, device="cuda")
            for add in ([False, True] if tc == torch.float32 else [False]):
                ops.linear_any(at, w, out=out, M=M, N=N, K=K, batch=batch, stride_a=K, stride_w=N * w.stride(0), stride_c=N, accumulate=add)
                ref = want * (2 if add else 1)
                over = (out.double() - ref).abs() - room * (2 if add else 1) - ref.abs() * (2.0 ** -8 if tc == torch.bfloat16 else 2.0 ** -24)
                assert over.max() <= 0, (ta, tc, add)


@pytest.mark.parametrize("N,K,add", [(64, 3584, False), (1536, 4096, True), (6144, 3000, True), (1536, 17920, True)])
def test_fp32_results_of_few_rows_are_as_close_as_the_streaming_form_s(N, K, add):
    """distance to float64 over 2, 4 and 8 rows of several draws (some 10^4 sums: the mean square is known to a few parts in a hundred): no larger than that of the
    kernel that takes such rows otherwise"""
    from mlx_vlm_amd import ops

    g, e = torch.Generator(device="cuda").manual_seed(K), [0.0, 0.0]
    for M in (2, 4, 8) * (8 if N < 1000 else 1):
        a, w = (torch.randn(n, K, generator=g, device="cuda").bfloat16() for n in (M, N))
        ref = a.double() @ w.double().T
        for i, f in enumerate((ops.linear_any, ops.linear_rows_bf16w)):
            x = torch.zeros(M, N, device="cuda")
            f(a, w, out=x, accumulate=add)
            e[i] += (x.double() - ref).pow(2).sum().item()
    assert e[0] <= 1.05 * e[1], e


@pytest.mark.parametrize("experts", [6, 36])
@pytest.mark.parametrize("rows", [1, 2, 3, 4])
def test_steps_of_few_rows_sum_onto_the_stream_in_fp32(tmp_path, rows, experts):
    """output projection of 1 to 4 decode rows over [mixer | experts] wider than 4096 and wider than 20480: the stream after a layer is the stream before it plus the
    float64 product of the layer's bf16 rows, within the roundings of fp32 sums (a bf16 row on the way would be off by 2^-9)"""
    cfg = H.config([H.layer("retention", ff=600, shared_ff=600, experts=experts) for _ in range(2)], side=0)
    lm = _load(tmp_path, cfg, H.weights(cfg), "bfloat16")
    lm = getattr(lm, "language_model", lm)
    ns, seen, linear = lm._L[1], [], lm._linear
    lm._linear = lambda a, w, **kw: (seen.append(a.double()) if w is ns.wout else None, linear(a, w, **kw))[1]
    lm._trace = []
    caches = [lm.make_cache() for _ in range(rows)]
    lm.step([(c[0]._seq, _ids(1, cfg["vocab"], 5 + i)) for i, c in enumerate(caches)], want="all")
    before, after = (x.double() for x in lm._trace)
    assert len(seen) == 1 and seen[0].shape == (rows, ns.wout.shape[1])
    added = seen[0] @ ns.wout.double().T
    # at most K / 256 + 12 roundings of partial sums below sum |a w|, and one of the stream
    bound = seen[0].abs() @ ns.wout.double().abs().T * ((ns.wout.shape[1] / 256 + 12) * 2.0 ** -24) + after.abs() * 2.0 ** -24
    assert ((after - before - added).abs() <= bound).all()
    assert (after - before - added).norm() < 2.0 ** -20 * added.norm()


@pytest.mark.parametrize("M,N,K", [(2, 1536, 8960), (8, 1536, 17920), (33, 264, 4160), (64, 3584, 4352)])
def test_gemm_rows_splits_a_long_k_in_a_capture_too(M, N, K):
    from mlx_vlm_amd import ops

    g = torch.Generator().manual_seed(M)
    a, w = torch.randn(M, K, generator=g).bfloat16().cuda(), torch.randn(N, K, generator=g).bfloat16().cuda()
    want = ops.gemm(a, w)
    assert torch.equal(ops.gemm_rows(a, w), want)
    out = torch.empty_like(want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.gemm_rows(a, w, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("M,N,K", [(2, 16384, 16384), (64, 16448, 16384), (3, 16320, 16384), (2, 41024, 16384)])
def test_gemm_rows_of_many_columns_in_a_capture(M, N, K):
    """both sides of the lines in columns up to which a very long K is split: the captured product has the bits of the eager one"""
    from mlx_vlm_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M)
    a, w = (torch.randn(n, K, generator=g, device="cuda").bfloat16() for n in (M, N))
    want, out = ops.gemm_rows(a, w), torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    ref = a.double() @ w[:512].double().T
    assert (want[:, :512].double() - ref).norm() <= 2.0 ** -8 * ref.norm()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.gemm_rows(a, w, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


# ------------------------------------------------------------------------------------------------ experts of prompts, pair by pair
@pytest.mark.parametrize("T,K,E,top,ff,N,shared", [(300, 128, 5, 2, 64, 72, 1), (70, 64, 3, 3, 128, 64, 0), (65, 192, 40, 4, 192, 264, 1), (513, 64, 0, 0, 64, 8, 1)])
@pytest.mark.parametrize("act", [1, 5])
def test_pairs_with_a_shared_expert_and_fp32_rows(T, K, E, top, ff, N, shared, act):
    """squared-relu and gated experts, one more that every token takes, fp32 rows summed in the residual step.  The activations are rounded to bf16 once
    as in the oracle: what is left is the order of fp32 sums, which moves one activation in some thousands to the neighbouring bf16 value:
    2^-13 (rms) bounds both"""
    from mlx_vlm_amd import ops

    g = torch.Generator().manual_seed(T + E)
    bf, per, n = torch.bfloat16, 1 if act == 5 else 2, E + shared
    h, wup = torch.randn(T, K, generator=g).to(bf), (torch.randn(n * per * ff + 8, K, generator=g) / K ** 0.5).to(bf)
    wdown = (torch.randn(N, n * ff + 8, generator=g) / ff ** 0.5).to(bf)
    gate = torch.zeros(T, E)
    for t in range(T):
        pick = torch.randperm(max(E, 1), generator=g)[: top - (t % 4 == 0)] if top else []
        gate[t, pick] = torch.rand(len(pick), generator=g) + 0.1
    rows, slots = ops.moe_grouped_rows(h.cuda(), wup.cuda(), wdown.cuda(), gate.cuda(), top, act, ff=ff, shared=shared, out_dtype=torch.float32)
    assert rows.dtype == torch.float32 and slots.shape == (T, top + shared)
    want = torch.zeros(T, N, dtype=F64)
    full = torch.cat([gate, torch.ones(T, shared)], 1).double()
    for e in range(n):
        z = h.double() @ wup.double()[e * per * ff: (e + 1) * per * ff].T
        m = torch.relu(z) ** 2 if act == 5 else torch.nn.functional.silu(z[:, :ff]) * z[:, ff:]
        want += (full[:, e:e + 1] * m).to(bf).double() @ wdown.double()[:, e * ff: (e + 1) * ff].T
    x0, y, w = torch.randn(T, N, generator=g), torch.randn(T, N + 4, generator=g).to(bf), torch.randn(N, generator=g).to(bf)
    for yy in (None, y.cuda()[:, :N]):
        for ww in (None, w.cuda()):
            x = x0.clone().cuda()
            hh = ops.add_slots_rms_(x, rows, slots, 0.7, y=yy, w=ww, w_offset=1.0, eps=1e-5)
            ref = x0.double() + 0.7 * (want + (0 if yy is None else y.double()[:, :N]))
            assert (x.cpu().double() - ref).norm() < 2.0 ** -13 * ref.norm()
            assert (hh is None) == (ww is None)
            if ww is not None:
                nr = ref / torch.sqrt(ref.pow(2).mean(-1, keepdim=True) + 1e-5) * (1 + w.double())
                assert (hh.cpu().double() - nr).norm() < 2.0 ** -8 * nr.norm()


@pytest.mark.parametrize("D", [16384, 16392, 70])
def test_slots_step_of_any_width(D):
    """rows wider than a workgroup's registers hold, and rows that do not come in pieces of four; three fp32 additions and the norm's rounding"""
    from mlx_vlm_amd import ops

    g = torch.Generator().manual_seed(D)
    x, rows, y, w = (torch.randn(n, D, generator=g) for n in (3, 5, 3, 1))
    y, w, slots = y.bfloat16().cuda(), w[0].bfloat16().cuda(), torch.tensor([[0, 4], [-1, 2], [-1, -1]], dtype=torch.int32)
    got = x.clone().cuda()
    h = ops.add_slots_rms_(got, rows.cuda(), slots.cuda(), 0.5, y=y, w=w, w_offset=1.0, eps=1e-6)
    want = x.double() + 0.5 * (y.cpu().double() + torch.stack([sum((rows[s].double() for s in t if s >= 0), torch.zeros(D, dtype=F64)) for t in slots.tolist()]))
    assert (got.cpu().double() - want).abs().max() <= 2.0 ** -21
    nr = want / torch.sqrt(want.pow(2).mean(-1, keepdim=True) + 1e-6) * (1 + w.cpu().double())
    assert ((h.cpu().double() - nr).abs() <= nr.abs() * 2.0 ** -8 + 1e-6).all()


@pytest.mark.parametrize("family", ["garesun", "tilalorn"])
@pytest.mark.parametrize("lens", [[64], [131, 5, 70], [300, 1]])
def test_experts_pair_by_pair_against_all_of_them(tmp_path, family, lens):
    """a bf16 step whose experts are evaluated pair by pair against the general form of the same model (every expert for every token): both differ from
    float64 by the rounding of 16-bit projections, and a token whose choice is a near tie may take another expert: nine rows in ten"""
    from tests import tilalorn_helpers as TH

    if family == "garesun":
        cfgs = [H.config([H.layer("retention", ff=64, shared_ff=sff, experts=6), H.layer("latent_attention", ff=64, shared_ff=sff)], width=128) for sff in (64, 0)]
        make = H.weights
    else:
        cfgs = [TH.config([TH.latent(mlp=TH.moe(ff=64)), TH.attention(mlp=TH.moe(experts=8, groups=2, keep=1, ff=128))], width=64)]
        make = TH.weights
    for j, cfg in enumerate(cfgs):
        lm = _load(tmp_path, cfg, make(cfg), "bfloat16", name=f"m{j}")
        lm = getattr(lm, "language_model", lm)
        got = []
        for size in (1, 1 << 30):
            lm.GROUPED_SIZE = size
            caches = [lm.make_cache() for _ in lens]
            got.append(lm.step([(c[0]._seq, _ids(n, cfg["vocab"], n)) for c, n in zip(caches, lens)], want="all").cpu())
            for c in caches:
                c[0]._seq.release()
        assert not torch.equal(got[0], got[1])                 # (two routes)
        assert H.rel_rms(got[0], got[1].double(), 0.9) < 2 * TOL["bfloat16"]


@pytest.mark.parametrize("family,experts", [("garesun", 256), ("tilalorn", 272)])
def test_more_experts_than_the_plan_takes(tmp_path, family, experts):
    """a prompt above the size from which pairs are evaluated, with more experts (shared ones counted) than a plan holds: every expert for every token, as for a
    shorter prompt"""
    from tests import tilalorn_helpers as TH

    if family == "garesun":
        cfg = H.config([H.layer("retention", ff=64, shared_ff=64, experts=experts)], width=64)
        W = H.weights(cfg)
    else:
        cfg = TH.config([TH.attention(mlp=TH.moe(experts=experts, groups=2, keep=1, ff=64))], width=64)
        W = TH.weights(cfg)
    lm = _load(tmp_path, cfg, W, "bfloat16")
    lm = getattr(lm, "language_model", lm)
    got = []
    for size in (1, 1 << 30):
        lm.GROUPED_SIZE = size
        got.append(_whole(lm, _ids(40, cfg["vocab"], 3)))
    assert torch.equal(*got)


@pytest.mark.parametrize("rows", [1, 2, 3, 8])
def test_decode_rows_at_a_checkpoint_s_width_row_by_row(tmp_path, rows):
    """steps of 1 to 8 rows over projections as wide as a real model's (what the kernels of few rows, the split K and the matrix-core attention are chosen by),
    every row of logits against float64: four in five within the rounding of a 16-bit chain (a router's near tie moves a row by itself, not its neighbours)"""
    moe = dict(experts=8, top=2, ff=512, shared_ff=512)
    cfg = H.config([H.layer("mlstm", heads=12, dim=128, vdim=128, **moe), H.layer("latent_attention", heads=12, dim=128, rot_dim=64, vdim=128, kv_rank=512, **moe),
                    H.layer("retention", heads=12, dim=128, vdim=128, rot_dims=128, **moe)], vocab=512, width=1536)
    W = H.weights(cfg)
    lm = _load(tmp_path, cfg, W, "bfloat16", seqs=rows + 1)
    lm = getattr(lm, "language_model", lm)
    steps, texts = 4, [_ids(20 + 9 * r + 4, cfg["vocab"], r) for r in range(rows)]
    want = torch.stack([O.Oracle(cfg, W, F64).forward(t)[-steps:] for t in texts], 1)
    caches = [lm.make_cache() for _ in texts]
    lm.step([(c[0]._seq, t[:-steps]) for c, t in zip(caches, texts)])
    got = torch.stack([lm.step([(c[0]._seq, t[len(t) - steps + i: len(t) - steps + i + 1]) for c, t in zip(caches, texts)]).cpu() for i in range(steps)])
    assert H.rel_rms(got.view(-1, cfg["vocab"]), want.reshape(-1, cfg["vocab"]), 0.8) < TOL["bfloat16"]
