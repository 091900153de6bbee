"""GPU parity of the OneTrans block kernels against the CPU oracle
(oracle/onetrans.py, autocast mode, whose rounding points are pinned against
torch's CPU autocast) on the same seeded inputs.

Tolerance (bf16 path), per element: every bf16 intermediate (Q, K, V,
attention output, GELU activations) and the block's update y - x_tail
satisfy |got - want| <= 2e-2 * (|want| + terms), where ``terms`` is the sum
of the absolute terms of the dot products that produce the value
(``oracle.onetrans.term_magnitudes``: |h| . |W|^T for a GEMM output, P . |V|
for attention).  That is the bf16 relative tolerance of 2e-2, measured
against the magnitude a rounding difference scales with.  Beyond it, fewer
than 1 % of the elements may differ by more than 2^-7 of that scale (one
bf16 ulp): GEMM and softmax summation orders differ from the oracle's, so a
bf16 value may round to its neighbour, and nothing larger."""
import pytest
import torch

from oracle import onetrans as ot

pytestmark = pytest.mark.gpu

ELEM_TOL = 2e-2
ULP = 2.0 ** -7


def _close(name, got, want, terms=None, tight_frac=0.01):
    got, want = got.double().cpu(), want.double().cpu()
    assert got.shape == want.shape, (name, got.shape, want.shape)
    assert torch.isfinite(got).all(), f"{name}: non-finite values"
    scale = want.abs() if terms is None else want.abs() + terms.double().reshape(want.shape)
    err = (got - want).abs()
    worst = (err / scale.clamp_min(1e-30)).max().item()
    beyond = (err > ULP * scale).double().mean().item()
    print(f"{name}: worst err / (|want| + terms) {worst:.2e}, beyond one ulp {beyond:.2e}", flush=True)
    assert bool((err <= ELEM_TOL * scale).all()), f"{name}: worst err / (|want| + terms) {worst:.3e}"
    assert beyond < tight_frac, f"{name}: {beyond:.3%} of the elements beyond one bf16 ulp"


def _gpu_weights(w, dev):
    bf = lambda t: t.to(torch.bfloat16).contiguous().to(dev)  # noqa: E731
    return dict(norm1_w=w["norm1"].float().contiguous().to(dev), s_qkv_w=bf(w["s_qkv"]),
                ns_qkv_w=bf(w["ns_qkv"]), out_w=bf(w["out"]), norm2_w=w["norm2"].float().contiguous().to(dev),
                s_w1=bf(w["s_w1"]), s_w2=bf(w["s_w2"]), ns_w1=bf(w["ns_w1"]), ns_w2=bf(w["ns_w2"]))


def _ws_view(ws, layout, name, shape, dtype=torch.bfloat16):
    off, size = layout[name]
    n = 1
    for s in shape:
        n *= s
    return ws[off:off + size].view(dtype)[:n].view(*shape)


def _check_layer(pdm, dev, x, w, q_len, label="", v_sums=False):
    """Runs one block on the GPU and checks its intermediates and output against the oracle on the same x.  With
    v_sums the attention output is also allowed what its V may differ by: D * 2^-24 * |h| . |W| (fp32 sums of D
    products in another order) and two columns of h on the other side of a bf16 rounding (the row's fp32 norm differs in
    its last bit: one column in about 60,000).  A query that sees one key copies that key's V, whatever cancelled in it,
    and among many samples some V is far smaller than its terms (1.0e-7 against 1.5e-7 out of terms of 5.0; 3e-5 against
    3e-4 with one column of h rounded the other way)."""
    B, kv, D = x.shape
    H = D // 64
    F = w["s_w1"].shape[0]
    print(f"block {label} B={B} kv={kv} q_len={q_len} D={D} n_ns={w['ns_qkv'].shape[0]}", flush=True)
    want, parts = ot.block_forward(x, w, q_len, H, mode="autocast", return_parts=True)
    terms = ot.term_magnitudes(x, w, q_len, H, parts)
    layout = pdm.ops.onetrans_workspace_layout(B, kv, q_len, D, F)
    ws = torch.empty(layout["total"][0], dtype=torch.uint8, device=dev)
    got = pdm.ops.onetrans_block_raw(x.to(dev), _gpu_weights(w, dev), H, q_len, workspace=ws)
    torch.cuda.synchronize()
    # intermediates still held by the workspace: K, V^T, the attention output, GELU activations
    k = _ws_view(ws, layout, "k", (B, kv, D))
    kv_ld = (kv + 63) // 64 * 64  # V^T row stride: rows start on 128-byte lines
    vt = _ws_view(ws, layout, "vt", (B, H, 64, kv_ld))[..., :kv]
    v = vt.permute(0, 3, 1, 2).reshape(B, kv, D)
    o = _ws_view(ws, layout, "q", (B, q_len, D))
    _close("k", k, parts["k"], terms["k"])
    _close("v", v, parts["v"], terms["v"])
    o_terms = terms["o"].double().reshape(B, q_len, D)
    if v_sums:  # the scale is multiplied by ELEM_TOL in _close
        w_max = max(w["s_qkv"].abs().max().item(), w["ns_qkv"].abs().max().item() if w["ns_qkv"].numel() else 0.0)
        h_max = (x * x.square().mean(-1, keepdim=True).rsqrt() * w["norm1"]).abs().max().item()
        o_terms = o_terms + (terms["v"].max().item() * D * 2.0 ** -24 + 2 * 2.0 ** -8 * h_max * w_max) / ELEM_TOL
    _close("attention out", o, parts["o"], o_terms)
    if "g" in layout:  # the separate FFN kernels keep RMSNorm2 rows and GELU activations in the workspace
        g = _ws_view(ws, layout, "g", (B, q_len, F))
        h2 = _ws_view(ws, layout, "h", (B, q_len, D))
        _close("rmsnorm2", h2, parts["h2"].to(torch.bfloat16), terms["h2"])
        _close("gelu(ffn up)", g, parts["g"], terms["g"])
    x_tail = x[:, kv - q_len:]
    got = got.cpu()
    _close("block update y - x_tail", got - x_tail, want - x_tail, terms["y"])
    return got


def _run_case(pdm, dev, B, kv, q_len, n_ns, D=256, F=1024, seed=0, x_std=1.0, w_std=0.02, norm_std=0.0, v_sums=False):
    w = ot.random_weights(D, F, n_ns, std=w_std, seed=seed, norm_std=norm_std)
    x = torch.randn(B, kv, D, generator=torch.Generator().manual_seed(seed + 1)) * x_std
    return _check_layer(pdm, dev, x, w, q_len, v_sums=v_sums)


@pytest.mark.parametrize("B,kv,q_len,n_ns", [
    (3, 40, 40, 4),      # full layer, ragged sizes
    (5, 70, 37, 16),     # pyramid layer: keep a tail
    (2, 33, 16, 16),     # q_len == n_ns: no S-token query
    (130, 48, 48, 2),    # B > one GEMM row tile of NS tokens
    (4, 64, 20, 0),      # no NS tokens
    (6, 240, 100, 16),   # 4 query tiles over 240 keys: the 4-wave attention with 8 copy rounds
    (2, 600, 600, 16),   # 19 query tiles over 608 padded keys: 8 waves, Q read from memory, <10,8>
    (3, 500, 300, 16),   # 10 query tiles over 512 padded keys: Q does not fit beside K/V^T in LDS, <10,8>
    (4, 250, 200, 16),   # 7 query tiles over 256 padded keys: the <4,8> instance
])
def test_block_matches_oracle(pdm, dev, B, kv, q_len, n_ns):
    _run_case(pdm, dev, B, kv, q_len, n_ns, seed=B + kv)


def test_block_d128_ffn384_and_norm_weights(pdm, dev):
    _run_case(pdm, dev, 6, 50, 30, 5, D=128, F=384, seed=7, norm_std=0.3, w_std=0.05)


def test_block_d384_tiled_path(pdm, dev):
    """d_model 384 (the reference's OneTransL width) runs the FFN as separate kernels."""
    _run_case(pdm, dev, 5, 45, 21, 3, D=384, F=1536, seed=8, norm_std=0.2)


def test_block_d512_tiled_path(pdm, dev):
    """d_model 512 (8 heads), the FFN as separate kernels."""
    _run_case(pdm, dev, 3, 40, 20, 3, D=512, F=2048, seed=9, norm_std=0.2)


@pytest.mark.parametrize("B,kv,q_len,n_ns,D", [
    (1, 608, 608, 5, 128),   # 19 query tiles on four workgroups per head, the longest keys held in LDS
    (2, 300, 20, 4, 256),    # one query tile: one workgroup
    (3, 290, 65, 4, 128),    # three tiles, the last of one row: three workgroups
    (64, 290, 70, 2, 128),   # 128 heads: two workgroups each
    (65, 290, 70, 2, 128),   # 130 heads: one each
])
def test_block_attention_workgroups_per_head(pdm, dev, B, kv, q_len, n_ns, D):
    """The split of a head's query tiles over workgroups at its edges, with the tolerance of every block test."""
    _run_case(pdm, dev, B, kv, q_len, n_ns, D=D, F=2 * D, seed=B + kv, norm_std=0.1)


@pytest.mark.parametrize("B,kv,q_len,n_ns,D", [
    (1, 5, 5, 4, 384),      # one S token: a block of 31 padding rows, every column split of the small grid
    (2, 47, 20, 7, 128),    # 40 S tokens: the last block stores one run of 8 V^T tokens
    (3, 71, 40, 6, 512),    # 65 S tokens: the last block holds one token, no multiple of 8
    (2, 30, 30, 0, 384),    # no NS tokens
    (3, 16, 16, 16, 384),   # no S tokens
    (140, 37, 24, 3, 384),  # NS tokens over two row tiles of 128 samples, the second partial
    (300, 61, 45, 3, 384),  # 13,500 kept rows: 128 x 128 tiles of the residual projections, the last one partial
    (330, 61, 43, 5, 256),  # 14,190 kept rows: just above the fused FFN's limit
    (325, 61, 43, 5, 256),  # 13,975 kept rows: just below it
    (700, 101, 50, 2, 128),  # enough row tiles that no column split is made; 99 S tokens, Q of the tail only
])
def test_block_row_projection_edges(pdm, dev, B, kv, q_len, n_ns, D):
    """The Q/K/V and FFN-up projections (32-token blocks of a sample, 32-sample blocks of an NS token, column
    splits) and the residual projections at the edges of their blocks, with the tolerance of every block test."""
    _run_case(pdm, dev, B, kv, q_len, n_ns, D=D, F=2 * D, seed=B + kv, norm_std=0.1)


@pytest.mark.parametrize("B,kv,q_len,n_ns,D", [
    (513, 21, 21, 5, 384),  # NS tokens over five row tiles of 128 samples, the last of one sample
    (130, 35, 2, 2, 128),   # one S token behind a whole block, run token by token and not kept as a query
    (130, 36, 3, 2, 256),   # two of them, one kept; the FFN-up's only S token
    (512, 1, 1, 0, 512),    # one S token and no whole block, no NS tokens
    (512, 40, 8, 2, 128),   # 38 S tokens: the six behind a whole block token by token, all kept
    (512, 9, 9, 2, 256),    # seven S tokens: a block for Q/K/V, token by token for the FFN-up
    (256, 18, 18, 2, 384),  # 16 S tokens: token by token for the FFN-up, a block for Q/K/V
    (260, 52, 50, 3, 512),  # 49 and 47 S tokens: a whole block and 17 or 15 behind it
])
def test_block_row_projection_tokens_of_many_samples(pdm, dev, B, kv, q_len, n_ns, D):
    """Row tiles that hold one token of 128 samples: the NS tokens, and the few S tokens behind a sample's last whole
    block of 32."""
    _run_case(pdm, dev, B, kv, q_len, n_ns, D=D, F=2 * D, seed=B + kv, norm_std=0.1, v_sums=True)


@pytest.mark.parametrize("D", [256, 384])
def test_block_stores_norm2_rows_only_on_request(pdm, dev, D):
    """Nothing in the library reads RMSNorm2's rows: a call without PDM_BLOCK_KEEP_NORM2 leaves their region of the
    workspace as it was, and the result is the same bit for bit."""
    import ctypes

    B, kv, q_len, n_ns, F = 6, 45, 40, 3, 2 * D
    L = pdm._lib
    w = _gpu_weights(ot.random_weights(D, F, n_ns, std=0.02, seed=23, norm_std=0.1), dev)
    x = torch.randn(B, kv, D, generator=torch.Generator().manual_seed(23)).to(dev)
    layout = pdm.ops.onetrans_workspace_layout(B, kv, q_len, D, F)
    names = ("norm1_w", "s_qkv_w", "ns_qkv_w", "out_w", "norm2_w", "s_w1", "s_w2", "ns_w1", "ns_w2")
    outs, kept = [], []
    for flags in (0, L.PDM_BLOCK_KEEP_NORM2):
        ws = torch.full((layout["total"][0],), 0xAB, dtype=torch.uint8, device=dev)
        out = torch.empty(B, q_len, D, device=dev)
        desc = L.BlockDesc(B, D, D // 64, n_ns, F, kv, q_len, flags)
        status = L.lib().pdm_onetrans_block_fwd(ctypes.byref(desc), x.data_ptr(),
                                                ctypes.byref(L.BlockWeights(*[w[k].data_ptr() for k in names])),
                                                out.data_ptr(), ws.data_ptr(), ws.numel(), L.stream_ptr(dev))
        L.check(status, "pdm_onetrans_block_fwd")
        torch.cuda.synchronize()
        outs.append(out)
        off, size = layout["h"]
        kept.append(bool((ws[off:off + size] == 0xAB).all()))
    assert kept == [True, False]
    assert torch.equal(outs[0], outs[1])


def test_block_and_stack_workspace_without_room_for_the_split_ffn(pdm, dev):
    """d_model 256: a workspace of Q, K and V^T alone runs the fused FFN on a small batch (checked against the oracle),
    one byte less is refused, and so for a stack, whose guard bytes behind the workspace stay untouched."""
    B, kv, q_len, n_ns, D, F = 5, 70, 37, 4, 256, 512
    w = ot.random_weights(D, F, n_ns, std=0.02, seed=24, norm_std=0.1)
    wd = _gpu_weights(w, dev)
    x = torch.randn(B, kv, D, generator=torch.Generator().manual_seed(24))
    least = pdm.ops.onetrans_workspace_layout(B, kv, q_len, D, F)["h"][0]
    full = torch.full((least + 4096,), 0xAB, dtype=torch.uint8, device=dev)
    got = pdm.ops.onetrans_block_raw(x.to(dev), wd, D // 64, q_len, workspace=full[:least]).cpu()
    assert bool((full[least:] == 0xAB).all())
    want, parts = ot.block_forward(x, w, q_len, D // 64, mode="autocast", return_parts=True)
    tail = x[:, kv - q_len:]
    _close("block update y - x_tail", got - tail, want - tail,
           ot.term_magnitudes(x, w, q_len, D // 64, parts)["y"])
    with pytest.raises(ValueError, match="workspace"):
        pdm.ops.onetrans_block_raw(x.to(dev), wd, D // 64, q_len, workspace=full[:least - 1])
    # a stack: the largest layer's Q, K, V^T, then two buffers of the largest inner output
    q_s = [60, 33, 20]
    least = pdm.ops.onetrans_workspace_layout(B, kv, 64, D, F)["h"][0] + 2 * ((B * 64 * D * 4 + 255) // 256 * 256)
    full = torch.full((least + 4096,), 0xAB, dtype=torch.uint8, device=dev)
    got = pdm.ops.onetrans_stack_raw(x.to(dev), [wd] * 3, D // 64, q_s, workspace=full[:least]).cpu()
    assert bool((full[least:] == 0xAB).all())
    want = ot.stack_forward(x, [w] * 3, q_s, D // 64)
    tail = x[:, kv - 24:].double()
    assert ((got.double() - want.double()).norm() / (want.double() - tail).norm()).item() <= 1e-2
    with pytest.raises(ValueError, match="workspace"):
        pdm.ops.onetrans_stack_raw(x.to(dev), [wd] * 3, D // 64, q_s, workspace=full[:least - 1])


def test_block_wide_ffn(pdm, dev):
    """d_model 256 with an FFN of 65,536: one sample's hidden activations are 68 MB, so 32 samples' would lie more than
    2^31 bytes apart."""
    _run_case(pdm, dev, 2, 520, 520, 2, D=256, F=65536, seed=21, w_std=0.01)


def test_block_samples_far_apart(pdm, dev):
    """33 samples of 262,150 tokens at d_model 128: the same token of 32 samples lies more than 2^31 bytes apart in K,
    and K of all samples fills 2.2 GB.  The first, the 32nd and the last sample are compared with the oracle."""
    B, kv, q_len, n_ns, D, F = 33, 262150, 20, 3, 128, 128
    w = ot.random_weights(D, F, n_ns, std=0.02, seed=22, norm_std=0.1)
    x = torch.empty(B, kv, D, device=dev)
    for b in range(B):
        x[b] = torch.randn(kv, D, generator=torch.Generator(device=dev).manual_seed(b), device=dev)
    print(f"block B={B} kv={kv} q_len={q_len} D={D}", flush=True)
    got = pdm.ops.onetrans_block_raw(x, _gpu_weights(w, dev), D // 64, q_len).cpu()
    for b in (0, 31, 32):
        xs = x[b:b + 1].cpu()
        want, parts = ot.block_forward(xs, w, q_len, D // 64, mode="autocast", return_parts=True)
        terms = ot.term_magnitudes(xs, w, q_len, D // 64, parts)
        tail = xs[:, kv - q_len:]
        _close(f"sample {b} update", got[b:b + 1] - tail, want - tail, terms["y"])


def test_block_baseline_shape_reduced_batch(pdm, dev):
    """The 4-layer benchmark's first layer (400 tokens, 16 NS, d 256, FFN 1024) at batch 8."""
    _run_case(pdm, dev, 8, 400, 400, 16, seed=11)


def test_block_batch1024_short_sequence(pdm, dev):
    """Batch 1024 (the benchmark's batch: 48 k rows of the streaming Q/K/V projection, hundreds of fused-FFN row tiles
    and 4096 attention (sample, head) pairs over the persistent grids) at a short sequence of 48 tokens keeping 32."""
    _run_case(pdm, dev, 1024, 48, 32, 16, seed=12, norm_std=0.1)


def test_block_vt_paired_tiles(pdm, dev):
    """Batch 160 with 128 S tokens: four 32-token blocks per sample, of which the streaming Q/K/V projection writes the
    32 tokens of every V^T row, and a tail of which half a block is kept."""
    _run_case(pdm, dev, 160, 144, 32, 16, seed=14, norm_std=0.1)


def test_block_ffn_ns_last_round(pdm, dev):
    """Batch 1024 keeping 80 of 96 tokens: 640 FFN row tiles of 128 rows, one whole round of 512 resident
    workgroups (256 CUs x 2) on the S tiles and a last round holding the 128 NS tiles (per-token weights)."""
    _run_case(pdm, dev, 1024, 96, 80, 16, seed=15, norm_std=0.1)


def test_block_ns_tiles_cross_tokens(pdm, dev):
    """Batch 1100 with 16 NS tokens on the streaming Q/K/V projection: nine tiles of 128 samples per NS token (the last
    partial); 33 S tokens (one whole block and one token run by itself) with the kept tail starting inside the block."""
    _run_case(pdm, dev, 1100, 49, 20, 16, seed=13, norm_std=0.1)


@pytest.mark.parametrize("B,kv,q_len,n_ns", [
    # 128 S tokens, 3,600 S tiles of 32 over 256 workgroups: shares of 14 or 15 consecutive tiles, so some write two
    # tiles' V^T as whole lines together and others a tile alone (a share starting at token 64 pairs it with token 96, a
    # share's last tile at token 0 goes alone)
    (900, 144, 32, 16),
    # 16 NS tokens: 82 tiles of 32 samples each (the last of 8), shares that cross from one NS token's weight to the
    # next; 33 S tokens (a whole and a single-row tile per sample), the kept tail starting inside the whole one
    (2600, 49, 20, 16),
    (2599, 48, 48, 16),   # 32 S tokens: unpaired tiles only; every token kept; the last NS tile of 7 samples
    (1277, 95, 17, 0),    # no NS tokens; two whole tiles and one of 31 rows; a tail inside the last tile
    (3001, 41, 3, 3),     # kept tail of the NS tokens alone
    (120, 1001, 520, 5),  # 32 tiles per sample, an odd number of keys, streaming attention
    (2450, 49, 20, 16),   # 120,050 rows: just above the line between the two projections
    (2448, 49, 20, 16),   # 119,952 rows: just below it
])
def test_block_stationary_projection(pdm, dev, B, kv, q_len, n_ns):
    """d_model 256 with more than 120,000 rows: the weight-stationary Q/K/V projection at ragged sizes, every sample
    compared."""
    assert (B * kv > 120_000) == ((B, kv) != (2448, 49))
    _run_case(pdm, dev, B, kv, q_len, n_ns, D=256, F=256, seed=B, norm_std=0.1, v_sums=True)


@pytest.mark.parametrize("B,kv,q_len,n_ns,D,F", [
    (1010, 100, 100, 2, 512, 512),  # 526 and 528 row tiles x 4 column tiles
    (1301, 110, 104, 5, 384, 384),  # 705 and 706 x 3
])
def test_block_residual_192_row_tiles(pdm, dev, B, kv, q_len, n_ns, D, F):
    """Enough rows for the 192 x 128 tiles of the residual projections (2,048 of them), the last S tile and every NS
    token's last tile partial.  The first and last samples and those at the edges of the NS tiles are compared."""
    tiles = lambda n_s, n_ns_: (-(-B * n_s // 192) + n_ns_ * -(-B // 192)) * D // 128  # noqa: E731
    assert tiles(q_len, 0) >= 2048 and tiles(q_len - n_ns, n_ns) >= 2048
    assert B * q_len % 192 and B * (q_len - n_ns) % 192 and B % 192
    print(f"block B={B} kv={kv} q_len={q_len} D={D} n_ns={n_ns}, sampled", flush=True)
    w = ot.random_weights(D, F, n_ns, std=0.02, seed=B, norm_std=0.1)
    x = torch.randn(B, kv, D, generator=torch.Generator().manual_seed(B + 1))
    got = pdm.ops.onetrans_block_raw(x.to(dev), _gpu_weights(w, dev), D // 64, q_len).cpu()
    edge = B // 192 * 192
    pick = torch.tensor([0, 1, 2, 95, 190, 191, 192, 193, 383, 384, edge - 1, edge, edge + 1, B - 3, B - 2, B - 1])
    xs = x[pick]
    want, parts = ot.block_forward(xs, w, q_len, D // 64, mode="autocast", return_parts=True)
    terms = ot.term_magnitudes(xs, w, q_len, D // 64, parts)
    tail = xs[:, kv - q_len:]
    _close("block update y - x_tail", got[pick] - tail, want - tail, terms["y"])


@pytest.mark.parametrize("B,kv,q_len,D", [
    (2, 720, 300, 256),    # above the LDS-resident attention's 608 keys: the streaming attention kernel
    (1, 1516, 1516, 256),  # the reference OneTransL's first layer (L_S = 1500 + 16 NS, full causal)
    (3, 1000, 700, 384),   # 6 heads: 18 (sample, head) pairs x 3 query blocks of 256, the last partial
    (2, 650, 650, 384),    # just above 608 keys, full causal, d_model 384
])
def test_block_long_sequence_streaming_attention(pdm, dev, B, kv, q_len, D):
    _run_case(pdm, dev, B, kv, q_len, 16, D=D, F=4 * D, seed=kv, norm_std=0.1)


def _load_block(blk, w):
    with torch.no_grad():
        blk.norm1.weight.copy_(w["norm1"])
        blk.attn.s_qkv.weight.copy_(w["s_qkv"])
        blk.attn.ns_qkv_weight.copy_(w["ns_qkv"])
        blk.attn.out_proj.weight.copy_(w["out"])
        blk.norm2.weight.copy_(w["norm2"])
        blk.ffn.s_w1.weight.copy_(w["s_w1"])
        blk.ffn.s_w2.weight.copy_(w["s_w2"])
        blk.ffn.ns_w1.copy_(w["ns_w1"])
        blk.ffn.ns_w2.copy_(w["ns_w2"])


@pytest.mark.parametrize("B,L_S,schedule,D", [
    (16, 384, [384, 256, 128, 64], 256),  # the benchmark's 4-layer pyramid: (kv, q) = (400,400),(400,272),(272,144),(144,80)
    (4, 96, [96, 64, 32, 0], 256),        # down to the NS tokens only
    (2, 984, [984, 656, 328, 0], 384),    # d_model 384, 6 heads: streaming attention at kv 1000 and 672, then LDS
])
def test_stack_pyramid_matches_oracle(pdm, dev, B, L_S, schedule, D):
    """OneTransStack (the block loop of onetrans.py:568-582) with an explicit schedule.  Each layer is
    checked element-wise against the oracle on the GPU's own input to that layer; the stack's output
    equals the chained layers bit for bit, and stays within 1e-2 (relative L2) of the oracle's stack."""
    F, n_ns, H = 4 * D, 16, D // 64
    stack = pdm.OneTransStack(D, H, n_ns, len(schedule), schedule=schedule).to(dev).eval()
    layers = []
    for i, blk in enumerate(stack.blocks):
        w = ot.random_weights(D, F, n_ns, std=0.02, seed=100 + i, norm_std=0.1)
        _load_block(blk, w)
        layers.append(w)
    x = torch.randn(B, L_S + n_ns, D, generator=torch.Generator().manual_seed(5))
    got = stack(x.to(dev)).cpu()
    assert got.shape == (B, schedule[-1] + n_ns, D)
    h = x
    for i, (w, q_s) in enumerate(zip(layers, schedule)):
        h = _check_layer(pdm, dev, h, w, q_s + n_ns, label=f"layer {i}")
    assert torch.equal(got, h)
    want = ot.stack_forward(x, layers, schedule, H)
    drift = ((got.double() - want.double()).norm() / (want.double() - x[:, -got.shape[1]:].double()).norm()).item()
    print(f"stack drift (relative L2 of the update) {drift:.2e}", flush=True)
    assert drift <= 1e-2


def test_stack_default_schedule_is_reference_pyramid(pdm, dev):
    """Without an explicit schedule the stack keeps pyramid_schedule(L_S, n_ns, n_layers) queries."""
    D, n_ns, H = 128, 4, 2
    stack = pdm.OneTransStack(D, H, n_ns, 3).to(dev).eval()
    x = torch.randn(2, 40 + n_ns, D, device=dev)
    assert stack(x).shape == (2, pdm.pyramid_schedule(40, n_ns, 3)[-1] + n_ns, D)


def test_block_rejects_bad_shapes(pdm, dev):
    w = _gpu_weights(ot.random_weights(256, 1024, 2), dev)
    x = torch.zeros(2, 10, 256, device=dev)
    with pytest.raises(ValueError):
        pdm.ops.onetrans_block_raw(x, w, 4, 1)  # q_len < n_ns
    with pytest.raises(pdm._lib.PdmError, match="head dim"):
        pdm.ops.onetrans_block_raw(x, w, 2, 10)  # head dim 128
