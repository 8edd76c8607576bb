"""The decode step's projections over packed operands against fp64 (needs an MI355X).

Bounds. The inputs are fp16, so every product is exact in fp32, and a sum of k
fp32 terms in any order is within k * 2^-24 of the sum of the terms' absolute
values; the result is rounded to fp16 once (2^-11 relative). With a norm the
operand x * scale * weight is itself rounded to fp16 once (2^-11 of each term)
and the scale is an fp32 rsqrt. SwiGLU's silu adds a few fp32 roundings and its
derivative (at most 1.1) carries the gate's error.
"""
from __future__ import annotations

import pytest
import torch

from engine.kernels.paged_attention_integration import decode_linear, pack_rows, pack_weight

pytestmark = pytest.mark.gpu

EPS = 1e-6


def _data(rows, n, k, device, seed):
    g = torch.Generator(device=device).manual_seed(seed)
    x = torch.randn(rows, k, generator=g, device=device).half()
    w = (torch.randn(n, k, generator=g, device=device) * k ** -0.5).half()
    return x, w, g


def _within(got, want, terms, rel_terms):
    """|got - want| <= one fp16 rounding + rel_terms of the summed absolute terms."""
    bound = want.abs() * 2.0 ** -11 + terms * rel_terms + 2.0 ** -24
    worst = ((got.double() - want).abs() / bound).max().item()
    print(f"[decode-linear] worst error / bound {worst:.3f}", flush=True)
    assert worst <= 1.0


# Row counts at the edges of the 16-row tiles, K from one step (most wavefronts idle) through both
# wavefront counts; tiles past the end of N or M: test_tiles_past_the_end.
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 33, 100, 128, 256])
@pytest.mark.parametrize("n,k", [(32, 32), (1152, 896), (80, 2336), (896, 4864)])
def test_linear_with_bias_residual_and_sums(cuda_device, rows, n, k):
    x, w, g = _data(rows, n, k, cuda_device, rows * 31 + n + k)
    bias = torch.randn(n, generator=g, device=cuda_device).half()
    want = x.double() @ w.double().t() + bias.double()
    terms = x.double().abs() @ w.double().abs().t() + bias.double().abs()
    wp = pack_weight(w)
    got = decode_linear(x, wp, bias=bias, packed=False)
    _within(got, want, terms, k * 2.0 ** -24)
    assert torch.equal(got, decode_linear(pack_rows(x), wp, bias=bias, packed=False))
    if n % 32:
        return
    res = torch.randn(rows, n, generator=g, device=cuda_device).half()
    out = decode_linear(x, wp, bias=bias, residual=pack_rows(res), sums=True)
    _within(out.unpack(), want + res.double(), terms + res.double().abs(), (k + 1) * 2.0 ** -24)
    squares = out.unpack().double().square()
    assert torch.allclose(out.sums.double().sum(0), squares.sum(1), rtol=n * 2.0 ** -24, atol=0)
    assert out.sums.shape == (n // 16, rows)


# Row-major weights, loaded two K steps at a time: K of fewer steps than wavefronts, ranges that end
# inside a pair, both wavefront counts; rows of a wider buffer.
@pytest.mark.parametrize("rows", [1, 17, 50, 100, 128, 241, 256])
@pytest.mark.parametrize("n,k", [(32, 32), (1136, 96), (1152, 896), (1136, 2336), (896, 4864)])
def test_row_major_weights(cuda_device, rows, n, k):
    x, w, g = _data(rows, n, k, cuda_device, rows * 13 + n + k)
    wide = torch.full((n, k + 24), float("nan"), device=cuda_device).half()
    wide[:, :k] = w
    bias = torch.randn(n, generator=g, device=cuda_device).half()
    want = x.double() @ w.double().t() + bias.double()
    terms = x.double().abs() @ w.double().abs().t() + bias.double().abs()
    got = decode_linear(x, w, bias=bias, packed=False)
    _within(got, want, terms, k * 2.0 ** -24)
    for again in (decode_linear(pack_rows(x), w, bias=bias, packed=False),
                  decode_linear(x, wide[:, :k], bias=bias, packed=False)):
        assert torch.equal(got, again)
    if n % 32:
        return
    res = torch.randn(rows, n, generator=g, device=cuda_device).half()
    out = decode_linear(x, w, bias=bias, residual=pack_rows(res), sums=True)
    _within(out.unpack(), want + res.double(), terms + res.double().abs(), (k + 1) * 2.0 ** -24)
    squares = out.unpack().double().square()
    assert torch.allclose(out.sums.double().sum(0), squares.sum(1), rtol=n * 2.0 ** -24, atol=0)


def _tile(kind, rows, n, k, cus=256):
    """The dispatch of launch_decode_linear: (wavefronts, column tiles, row tiles) of a workgroup."""
    mt, nt, up = -(-rows // 16), n // 16, lambda a, b: -(-a // b)  # noqa: E731
    if kind == "silu":
        if mt == 1 or mt * up(nt, 2) <= cus:
            return 4, 2, 1
        if mt == 2 or up(mt, 2) * up(nt, 2) <= cus:
            return 4, 2, 2
        return (4, 3, 2) if mt == 3 or up(mt, 2) * up(nt, 3) <= cus else (4, 3, 4)
    nw = 8 if k > 32 * 4 * 14 else 4
    if mt * nt <= cus:
        return nw, 1, 1
    if kind == "row" and nw == 8:
        if mt > 1 and up(mt, 2) * nt <= cus:
            return nw, 1, 2
        return (nw, 2, 1) if mt == 1 else (nw, 2, 2)
    return (nw, 2, 1) if mt == 1 or mt * up(nt, 2) <= cus else (nw, 2, 2)


# (kind, rows, n, k): every kernel of the dispatch, with columns and rows of tiles past the end of N
# and M wherever its tile has more than one.
_PAST_THE_END = [
    *(("plain", rows, 1136, k) for rows in (3, 100, 200) for k in (96, 2336)),
    *(("norm", rows, 1136, k) for rows in (3, 100, 200) for k in (96, 2304)),
    *(("row", rows, 1136, k) for rows in (3, 100, 200) for k in (96, 2336)),
    ("row", 70, 1136, 2336), ("row", 5, 4112, 2336),
    ("silu", 100, 1136, 96), ("silu", 140, 1136, 96), ("silu", 200, 1184, 96),
    ("silu", 200, 4864, 896),
]


def test_every_kernel_runs_past_the_end():
    """_PAST_THE_END against the dispatch: each kernel once with a remainder in N and in M."""
    tiles = {(1, 1), (2, 1), (2, 2)}
    want = {(kind, nw, *t) for kind in ("plain", "norm", "row") for nw in (4, 8) for t in tiles}
    want |= {("row", 8, 1, 2), ("silu", 4, 2, 1), ("silu", 4, 2, 2), ("silu", 4, 3, 2),
             ("silu", 4, 3, 4)}
    columns, rows_ = set(), set()
    for kind, rows, n, k in _PAST_THE_END:
        tile = _tile(kind, rows, n, k)
        if tile[1] == 1 or n // 16 % tile[1]:
            columns.add((kind, *tile))
        if rows % 16 and (tile[2] == 1 or -(-rows // 16) % tile[2]):
            rows_.add((kind, *tile))
    assert columns == want and rows_ == want


@pytest.mark.parametrize("kind,rows,n,k", _PAST_THE_END)
def test_tiles_past_the_end(cuda_device, kind, rows, n, k):
    """Row-major outputs: packed ones have whole pairs of column tiles."""
    assert torch.cuda.get_device_properties(cuda_device).multi_processor_count == 256
    x, w, g = _data(rows, 2 * n if kind == "silu" else n, k, cuda_device, rows + n + k)
    gain = torch.randn(k, generator=g, device=cuda_device).half()
    xd = x.double()
    rel = k * 2.0 ** -24
    if kind in ("norm", "silu"):
        xd = xd * torch.rsqrt(xd.square().mean(1, keepdim=True) + EPS) * gain.double()
        rel = 2.0 ** -11 + (k + 8) * 2.0 ** -24
    want, terms = xd @ w.double().t(), xd.abs() @ w.double().abs().t()
    packed = pack_rows(x)
    norm = (gain, EPS) if kind in ("norm", "silu") else None
    got = decode_linear(packed, w if kind == "row" else pack_weight(w), norm=norm,
                        silu=kind == "silu", packed=False)
    # Operands below fp16's normal range are rounded to a multiple of 2^-24 of the scaled row.
    small = w.double().abs().sum(1)[None, :] * 2.0 ** -24 if norm else torch.zeros_like(want)
    if kind != "silu":
        _within(got, want, terms + small / rel, rel)
        if kind != "norm":
            assert torch.equal(got, decode_linear(x, w if kind == "row" else pack_weight(w),
                                                  packed=False))
        return
    gate, up = want[:, :n], want[:, n:]
    err = rel * terms + small
    want = torch.nn.functional.silu(gate) * up
    bound = 1.1 * err[:, :n] * (up.abs() + err[:, n:]) + gate.abs() * err[:, n:]
    _within(got, want, bound + want.abs() * 2.0 ** -21, 1.0)
    if n % 32 == 0:
        out = decode_linear(packed, pack_weight(w), norm=norm, silu=True)
        assert torch.equal(out.unpack(), got)


@pytest.mark.parametrize("rows", [1, 16, 31, 48, 64, 100, 128, 256])
@pytest.mark.parametrize("n,k", [(32, 64), (1152, 896), (224, 2304)])
def test_norm_and_swiglu(cuda_device, rows, n, k):
    x, w, g = _data(rows, 2 * n, k, cuda_device, rows * 17 + n + k)
    # Rows of very different sizes: the scale's power of two differs from row to row.
    x = (x * torch.logspace(-3, 3, rows, device=cuda_device)[:, None]).half()
    gain = torch.randn(k, generator=g, device=cuda_device).half()
    xd = x.double()
    normed = xd * torch.rsqrt(xd.square().mean(1, keepdim=True) + EPS) * gain.double()
    y = normed @ w.double().t()
    terms = normed.abs() @ w.double().abs().t()
    # One rounding of each operand (2^-11), the fp32 scale (a few 2^-24), the sum; operands below
    # fp16's normal range are rounded to a multiple of 2^-24 of the power-of-two scaled row.
    rel = 2.0 ** -11 + (k + 8) * 2.0 ** -24
    small = w.double().abs().sum(1)[None, :] * 2.0 ** -24
    packed = pack_rows(x)
    got = decode_linear(packed, pack_weight(w[:n]), norm=(gain, EPS), packed=False)
    _within(got, y[:, :n], terms[:, :n] + small[:, :n] / rel, rel)
    act = decode_linear(packed, pack_weight(w), norm=(gain, EPS), silu=True).unpack()
    gate, up = y[:, :n], y[:, n:]
    want = torch.nn.functional.silu(gate) * up
    err = rel * terms + small
    bound = 1.1 * err[:, :n] * (up.abs() + err[:, n:]) + gate.abs() * err[:, n:]
    _within(act, want, bound + want.abs() * 2.0 ** -21, 1.0)


def test_normed_values_up_to_the_largest_fp16(cuda_device):
    """A normed value that fp16 holds is not an infinity on the way, whatever the row's scale."""
    rows, n, k = 33, 32, 96
    x = torch.zeros(rows, k, device=cuda_device, dtype=torch.float16)
    x[:, 0] = torch.logspace(-1, 1, rows, base=2.0, device=cuda_device).half()
    gain = torch.full((k,), 6600.0, device=cuda_device).half()  # times sqrt(96): 64666
    w = (torch.rand(n, k, device=cuda_device) * 2.0 ** -8).half()
    got = decode_linear(pack_rows(x), pack_weight(w), norm=(gain, EPS), packed=False)
    xd = x.double()
    normed = xd * torch.rsqrt(xd.square().mean(1, keepdim=True) + EPS) * gain.double()
    assert normed.max() < 65504
    want = normed @ w.double().t()
    _within(got, want, want.abs(), 2.0 ** -11 + (k + 8) * 2.0 ** -24)


def test_sums_of_the_previous_launch_feed_the_norm(cuda_device):
    """A residual row written by one launch is normalised by the next from its partial sums."""
    x, w, g = _data(37, 896, 896, cuda_device, 3)
    h = decode_linear(x, pack_weight(w), sums=True)
    again = pack_rows(h.unpack())
    assert torch.equal(again.unpack(), h.unpack())
    gain = torch.rand(896, generator=g, device=cuda_device).half()
    w2 = pack_weight(_data(1, 1152, 896, cuda_device, 4)[1])
    a = decode_linear(h, w2, norm=(gain, EPS), packed=False)
    b = decode_linear(again, w2, norm=(gain, EPS), packed=False)
    # The row sums differ in order only: the scale by a few 2^-24, the result by an fp16 step.
    assert ((a.float() - b.float()).abs() <= b.float().abs() * 2.0 ** -10 + 2.0 ** -24).all()


def test_rows_with_infinities_and_nans_stay_in_their_rows(cuda_device):
    x, w, _ = _data(20, 64, 96, cuda_device, 5)
    x[3, 7], x[18, 0] = float("inf"), float("nan")
    gain = torch.ones(96, device=cuda_device).half()
    got = decode_linear(pack_rows(x), pack_weight(w), norm=(gain, EPS), packed=False)
    bad = torch.zeros(20, dtype=torch.bool, device=cuda_device)
    bad[[3, 18]] = True
    assert torch.isnan(got[bad]).all() and torch.isfinite(got[~bad]).all()


def test_stack_and_layer_paths_agree(cuda_device):
    """A decode step through the fused stack, and one that takes the layers one by one (a layer
    with a forward hook), give the same logits up to fp16 roundings; the hook fires."""
    from engine import workloads
    from engine.kernels.paged_attention_integration import KernelPagedManualDecode
    from engine.memory.block_allocator import BlockTable

    config = dict(vocab_size=512, hidden_size=128, intermediate_size=256, num_hidden_layers=3,
                  num_attention_heads=4, num_key_value_heads=2, max_position_embeddings=4096,
                  rope_theta=1e6, tie_word_embeddings=False)
    with torch.inference_mode():
        model = workloads.decode_model(cuda_device, 11, config)
        logits, fired = [], []
        for hook in (False, True):
            runner = KernelPagedManualDecode(model, num_blocks=64, device=str(cuda_device),
                                             use_graphs=False)
            gen = torch.Generator(device=cuda_device).manual_seed(2)
            for c in runner.pool.k_cache + runner.pool.v_cache:
                c.normal_(0, 0.6, generator=gen)
            seqs = [{"seq_id": i, "block_table": BlockTable(i, 16, [2 * i, 2 * i + 1], 9 + i),
                     "last_token_id": 5 * i} for i in range(5)]
            handle = model.model.layers[1].register_forward_hook(
                lambda *a: fired.append(1)) if hook else None
            runner.decode_step(seqs)
            if handle:
                handle.remove()
            logits.append(torch.stack([s["last_logits"] for s in seqs]).float())
    assert fired == [1]
    # Three layers of fp16 activations: the layer path rounds more often (normed rows, projections
    # before the residual add); 2^-11 per rounding over some twenty roundings.
    diff = (logits[0] - logits[1]).norm() / logits[1].norm()
    print(f"[decode-linear] stack against layers: {diff.item():.2e}", flush=True)
    assert diff <= 20 * 2.0 ** -11


@pytest.mark.parametrize("use_graphs", [False, True])
def test_o_and_down_follow_their_parameters(cuda_device, use_graphs):
    """In-place changes of the two weights that are not merged with others reach the next step, also
    through a graph captured before, as in the layer path."""
    from engine import workloads
    from engine.kernels.paged_attention_integration import KernelPagedManualDecode
    from engine.memory.block_allocator import BlockTable

    config = dict(vocab_size=512, hidden_size=128, intermediate_size=256, num_hidden_layers=2,
                  num_attention_heads=4, num_key_value_heads=2, max_position_embeddings=4096,
                  rope_theta=1e6, tie_word_embeddings=False)
    with torch.inference_mode():
        model = workloads.decode_model(cuda_device, 13, config)

        def logits(runner):
            gen = torch.Generator(device=cuda_device).manual_seed(2)
            for c in runner.pool.k_cache + runner.pool.v_cache:
                c.normal_(0, 0.6, generator=gen)
            seqs = [{"seq_id": i, "block_table": BlockTable(i, 16, [i], 5 + i),
                     "last_token_id": 7 * i} for i in range(5)]
            runner.decode_step(seqs)
            return torch.stack([s["last_logits"] for s in seqs]).float()

        runner = KernelPagedManualDecode(model, num_blocks=8, device=str(cuda_device),
                                         use_graphs=use_graphs)
        old = logits(runner)
        model.model.layers[0].self_attn.o_proj.weight.mul_(-3)
        model.model.layers[1].mlp.down_proj.weight.data.copy_(
            model.model.layers[1].mlp.down_proj.weight * 2)
        new = logits(runner)
        handle = model.model.layers[0].register_forward_hook(lambda *a: None)  # the layer path
        want = logits(KernelPagedManualDecode(model, num_blocks=8, device=str(cuda_device),
                                              use_graphs=False))
        handle.remove()
    # Two layers of fp16 activations: some fourteen roundings of 2^-11.
    assert (new - want).norm() <= 14 * 2.0 ** -11 * want.norm()
    assert (new - old).norm() >= 0.1 * want.norm()


def test_packed_copies_only_where_memory_is_left(cuda_device, monkeypatch):
    """All layers' packed copies within a quarter of the free memory, or none: the step then runs
    layer by layer. A later runner packs them if it finds the room."""
    from engine import workloads
    from engine.kernels import paged_attention_integration as integration
    from engine.memory.block_allocator import BlockTable

    config = dict(vocab_size=512, hidden_size=128, intermediate_size=256, num_hidden_layers=2,
                  num_attention_heads=4, num_key_value_heads=2, max_position_embeddings=4096,
                  rope_theta=1e6, tie_word_embeddings=False)
    copies = 2 * 2 * (256 * 128 + 512 * 128)  # two layers' q/k/v and gate/up, two bytes each
    free = integration._free_bytes(cuda_device)
    held = torch.empty(64 << 20, dtype=torch.uint8, device=cuda_device)
    assert 0 <= free - integration._free_bytes(cuda_device) - held.numel() <= 16 << 20
    with torch.inference_mode():
        model = workloads.decode_model(cuda_device, 14, config)
        logits = []
        for room, packed in ((4 * copies - 1, False), (4 * copies, True)):
            monkeypatch.setattr(integration, "_free_bytes", lambda device: room)
            runner = integration.KernelPagedManualDecode(model, num_blocks=4,
                                                         device=str(cuda_device))
            assert all(hasattr(m, "_pa_fused") and hasattr(m, "_pa_packed") == packed
                       for m in model.model.layers)
            for c in runner.pool.k_cache + runner.pool.v_cache:
                c.zero_()
            seq = {"seq_id": 0, "block_table": BlockTable(0, 16, [3], 5), "last_token_id": 9}
            runner.decode_step([seq])
            logits.append(seq["last_logits"].float())
    # Two layers of fp16 activations: some fourteen roundings of 2^-11.
    assert (logits[0] - logits[1]).norm() <= 14 * 2.0 ** -11 * logits[0].norm()


@pytest.mark.parametrize("use_graphs", [False, True])
def test_ids_nobody_checked_go_through_the_embedding_module(cuda_device, monkeypatch, use_graphs):
    """decode_step refuses ids outside the table and embeds the others in the step's first launch; a
    model call with ids of its own asks the module, which refuses them as it always does."""
    from engine import workloads
    from engine.kernels import paged_attention_integration as integration
    from engine.memory.block_allocator import BlockTable

    launches = []
    embed = integration.decode_embed
    monkeypatch.setattr(integration, "decode_embed", lambda *a: launches.append(1) or embed(*a))
    config = dict(vocab_size=512, hidden_size=128, intermediate_size=256, num_hidden_layers=1,
                  num_attention_heads=4, num_key_value_heads=2, max_position_embeddings=4096,
                  rope_theta=1e6, tie_word_embeddings=False)
    with torch.inference_mode():
        model = workloads.decode_model(cuda_device, 12, config)
        runner = integration.KernelPagedManualDecode(model, num_blocks=8, device=str(cuda_device),
                                                     use_graphs=use_graphs)
        seq = {"seq_id": 0, "block_table": BlockTable(0, 16, [3], 5), "last_token_id": 511}
        runner.pool.k_cache[0].zero_(), runner.pool.v_cache[0].zero_()
        runner.decode_step([seq])
        assert launches
        with pytest.raises(IndexError):
            runner.decode_step([dict(seq, last_token_id=512)])
        launches.clear()
        ctx = integration.PagedAttentionContext(runner.pool, [seq["block_table"]], [6])
        with integration.patch_paged_attention(model, ctx):
            out = model(input_ids=torch.full((1, 1), 511, device=cuda_device),
                        position_ids=torch.full((1, 1), 5, device=cuda_device), use_cache=False)
        assert not launches
    # The same embedding row; rotary rows an fp16 rounding apart at most (2^-11 of a row's key).
    diff = (out.logits[0, -1].float() - seq["last_logits"].float()).norm()
    assert diff <= 2.0 ** -10 * seq["last_logits"].float().norm()


@pytest.mark.parametrize("rows,hidden,dim,freq", [
    (1, 32, 64, torch.float32), (17, 896, 64, torch.float16), (130, 2336, 128, torch.float32)])
def test_embed_matches_the_modules(cuda_device, rows, hidden, dim, freq):
    """Embedding rows bit for bit; cos and sin as torch computes them in fp32 (an fp16 rounding
    boundary apart at most); an id outside the table gives NaNs in its row only."""
    from engine.kernels.paged_attention_integration import decode_embed

    g = torch.Generator(device=cuda_device).manual_seed(rows)
    table = torch.randn(1000, hidden, generator=g, device=cuda_device).half()
    ids = torch.randint(0, 1000, (rows,), generator=g, device=cuda_device)
    pos = torch.randint(0, 32768, (rows,), generator=g, device=cuda_device)
    inv = 1e6 ** (-torch.arange(0, dim, 2, device=cuda_device).float() / dim)
    inv = inv.to(freq)
    packed, cos, sin = decode_embed(ids, pos, table, inv, 0.5)
    assert torch.equal(packed.unpack(), table[ids])
    assert torch.allclose(packed.sums[0].double(), table[ids].double().square().sum(1),
                          rtol=hidden * 2.0 ** -24, atol=0)
    angle = (pos.float()[:, None] * inv.float()[None, :]).repeat(1, 2)
    for got, want in ((cos, angle.cos() * 0.5), (sin, angle.sin() * 0.5)):
        assert ((got.float() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -22).all()
    if rows > 1:
        ids[1], ids[-1] = -1, 1000
        out = decode_embed(ids, pos, table, inv)[0].unpack()
        bad = torch.zeros(rows, dtype=torch.bool, device=cuda_device)
        bad[[1, rows - 1]] = True
        assert torch.isnan(out[bad]).all() and torch.equal(out[~bad], table[ids[~bad]])


# Ranges of one load, ragged parts, an empty one, more than the L2 share; batches that leave CUs
# free and that take the two-launch form (where nothing is fetched).
@pytest.mark.parametrize("seqs,longest", [(1, 40), (9, 700), (128, 300), (1, 5000)])
@pytest.mark.parametrize("sizes", [[16], [8, 1000, 0, 77777], [1 << 20, 40 << 20, 8]])
def test_prefetch_changes_nothing(cuda_device, seqs, longest, sizes):
    from engine.kernels.paged_attention_integration import paged_rope_decode_attention

    g = torch.Generator(device=cuda_device).manual_seed(seqs)
    width = -(-longest // 16)
    blocks = seqs * width + 3
    lens = torch.randint(1, longest + 1, (seqs,), generator=g, device=cuda_device).int()
    lens[-1] = longest
    tables = torch.randperm(blocks, generator=g, device=cuda_device)[:seqs * width]
    tables = tables.view(seqs, width).int()
    rows = [torch.randn(seqs, h, 64, generator=g, device=cuda_device).half() for h in (14, 2, 2)]
    cos, sin = torch.randn(2, seqs, 64, generator=g, device=cuda_device).half()
    pools = [torch.randn(blocks, 16, 2, 64, generator=g, device=cuda_device).half()
             for _ in range(2)]
    ranges = [torch.zeros(n // 2, dtype=torch.float16, device=cuda_device) for n in sizes]
    results = []
    for prefetch in ((), ranges):
        own = [p.clone() for p in pools]
        out = paged_rope_decode_attention(*rows, cos, sin, *own, tables, lens, 0.125,
                                          prefetch=prefetch)
        results.append((out, *own))
    assert all(torch.equal(a, b) for a, b in zip(*results))
