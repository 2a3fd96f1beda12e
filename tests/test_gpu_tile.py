"""GPU: the expert stages above the token crossover on the register-fed tiles
(64 rows x 256 weight rows, ftm_tile.hip) against the oracle, at the sizes
where a tile can go wrong: partly filled row blocks, a second M tile of one
row, channels and columns that end inside a tile, one and several K steps,
scale groups wider than a step, a shared expert beside the routed ones."""
from dataclasses import replace

import numpy as np
import pytest
import torch

import ftm_oracle as O
from ftm_helpers import np_, oracle_spec, rel_rms, to_f32

from ftmoe import _native as nat
from ftmoe import synthetic as S

pytestmark = pytest.mark.gpu

# The oracle rounds h and the router weights to bf16 as the layer does; what
# is left is the output's rounding (2^-9 / sqrt(3) = 1.1e-3 relative RMS) and
# h values that fall on the other side of a rounding boundary in another
# summation order.
REL_RMS = 4e-3


def _check(syn, gpu, ids=None, w=None, cast=lambda n, t: t):
    T = syn.x.shape[0]
    ref = O.layer_reference(oracle_spec(syn), np_(syn.x), ids=ids, w=w)
    dsyn = syn.to(gpu)
    layer = S.build_layer(dsyn, bank={n: cast(n, t) for n, t in dsyn.bank.items()})
    if ids is None:
        run = lambda: layer.forward(dsyn.x)  # noqa: E731
    else:
        i, v = torch.from_numpy(ids).to(gpu), torch.from_numpy(w).to(gpu)
        run = lambda: layer.forward_routed(dsyn.x, i, v)  # noqa: E731
    out = run()
    torch.cuda.synchronize()
    err = rel_rms(to_f32(out), ref["out"])
    assert err < REL_RMS, err
    assert torch.equal(run(), out)
    return layer


def _skewed(T, E, k, counts, seed):
    """Caller routing that gives expert e counts[e] tokens (the rest spread over the others)."""
    rng = np.random.RandomState(seed)
    ids = np.full((T, k), -1, np.int32)
    for e, c in enumerate(counts):
        rows = rng.choice(np.flatnonzero((ids >= 0).sum(1) < k), c, replace=False)
        for t in rows:
            ids[t, (ids[t] >= 0).sum()] = e
    return ids, O.round_bf16(rng.rand(T, k).astype(np.float32))


@pytest.mark.parametrize("T,H,I,shared,group", [(64, 256, 384, 0, 128), (129, 384, 128, 0, 128), (200, 256, 256, 192, 128),
                                                (90, 512, 256, 128, 256)])
def test_gptq_tiles_match_oracle(gpu, T, H, I, shared, group):
    """GPTQ with zero points of every value and groups of one or two K steps."""
    cfg = replace(S.SMALL["c2_gptq"], H=H, I=I, shared_inter=shared, group=group)
    syn = S.generate(cfg, T=T, seed=T + H)
    g = torch.Generator().manual_seed(T)
    for n in ("qzeros_gate_up", "qzeros_down"):
        z = syn.bank[n]
        syn.bank[n] = torch.randint(-2**31, 2**31 - 1, z.shape, generator=g, dtype=torch.int64).to(torch.int32)
    layer = _check(syn, gpu)
    assert layer.stage_kernel(T, nat.STAGE_W13) == "k_tile"
    assert layer.stage_kernel(T, nat.STAGE_W2) == "k_tile"


@pytest.mark.parametrize("T,H,I,shared,groups", [(64, 256, 128, 0, 1), (130, 320, 192, 0, 1), (100, 512, 256, 128, 2),
                                                 (75, 384, 256, 0, 1)])
def test_int8_tiles_match_oracle(gpu, T, H, I, shared, groups):
    """INT8 per channel and with K groups of 256 / 128, K ending in a half
    step (H = 320, I = 192), channels and columns that end inside a tile."""
    cfg = replace(S.SMALL["c1_int8"], H=H, I=I, shared_inter=shared, int8_num_groups=groups)
    layer = _check(S.generate(cfg, T=T, seed=T + H), gpu)
    assert layer.stage_kernel(T, nat.STAGE_W13) == "k_tile"
    assert layer.stage_kernel(T, nat.STAGE_W2) == "k_tile"


@pytest.mark.parametrize("name", ["c1_int8", "c2_gptq", "c3_fp8", "c3_fp8_wide", "c4_mxfp4", "bf16", "bf16_wide"])
def test_tiles_with_uneven_experts(gpu, name):
    """Experts of 1, 15, 16, 17, 32, 33, 64, 65 and 129 rows, some of none.
    bf16 layers with fewer stage-A tiles than CUs keep the LDS-ring tiles
    (bf16), with more they take the register-fed ones (bf16_wide).  FP8 with
    fewer than 16 tokens per expert: the bf16 tiles (c3_fp8_wide)."""
    T, E, k = 144, 16, 4
    cfg = S.SMALL["c1_int8"] if name.startswith("bf16") else S.SMALL[name.removesuffix("_wide")]
    if name == "bf16":
        cfg = replace(cfg, fmt="bf16")
    elif name == "bf16_wide":  # 144 x 4 / 64 + 16 row tiles x 11 of 128 channels
        cfg = replace(cfg, fmt="bf16", I=1408)
    elif name == "c3_fp8_wide":
        E, cfg = 64, replace(cfg, I=512)
    syn = S.generate(replace(cfg, E=E, k=k), T=T, seed=9)
    ids, w = _skewed(T, E, k, [1, 15, 16, 17, 0, 32, 33, 64, 65, 129, 0, 48], 3)
    layer = _check(syn, gpu, ids, w)
    if name.startswith("bf16"):
        assert layer.stage_kernel(T, nat.STAGE_W13) == ("k_tile" if name == "bf16_wide" else "k_gemm_a_ring")
    if name.startswith("c3_fp8"):
        assert layer.stage_kernel(T, nat.STAGE_W13) == ("k_tile" if name == "c3_fp8_wide" else "k_gemm_mx")


@pytest.mark.parametrize("fmt", ["c1_int8", "c2_gptq", "c3_fp8", "bf16"])
@pytest.mark.parametrize("T", [47, 48])
def test_tiles_of_few_rows(gpu, fmt, T):
    """64 experts of 512 channels cover the chip: tiles from 3 tokens per
    expert (48 tokens, top-4) on, most of a row block empty; the GEMV stages
    below."""
    cfg = replace(S.SMALL["c1_int8"], fmt="bf16") if fmt == "bf16" else S.SMALL[fmt]
    layer = _check(S.generate(replace(cfg, E=64, k=4, H=256, I=512, shared_inter=0), T=T, seed=T), gpu)
    assert (layer.stage_kernel(T, nat.STAGE_W13) == "k_tile") == (T >= 48)
    assert (layer.stage_kernel(T, nat.STAGE_W2) == "k_tile") == (T >= 48)


@pytest.mark.parametrize("E,shared,H,T", [
    (256, True, 2048, 481),   # the shared gate's row beside whole tiles, a token block of one
    (60, False, 2880, 1480),  # rows padded to a tile, a last stage of 320 elements
    (62, True, 1024, 3890),   # the shared gate's row inside a padded tile
    (290, True, 320, 2720),   # one partial stage, 291 rows: three past the tiles
])
def test_router_mm_bit_exact(gpu, E, shared, H, T):
    """The prefill router on the fp32 matrix cores keeps the fma chains and
    the butterfly that the oracle replays."""
    from ftmoe.banks import Proj
    from ftmoe.layer import MoeLayer

    I, k = 16, 4
    rng = np.random.RandomState(E + T)
    bits = lambda v: O.f32_to_bf16_bits(v.astype(np.float32))  # noqa: E731
    dev = lambda b: torch.from_numpy(b.view(np.int16)).view(torch.bfloat16).to(gpu)  # noqa: E731
    gate, x = bits(rng.randn(E, H) * 0.05), bits(rng.randn(T, H))
    sgate, s13, s2 = bits(rng.randn(1, H) * 0.05), bits(rng.randn(2 * I, H) * 0.05), bits(rng.randn(H, I))
    shd = {"w13": dev(s13), "w2": dev(s2), "gate": dev(sgate)} if shared else None
    w13 = Proj("bf16", torch.zeros(E, 2 * I, H, dtype=torch.bfloat16, device=gpu), 2 * I, H)
    w2 = Proj("bf16", torch.zeros(E, H, I, dtype=torch.bfloat16, device=gpu), H, I)
    layer = MoeLayer(w13=w13, w2=w2, num_experts=E, hidden=H, inter=I, topk=k, gate_w=dev(gate), shared=shd,
                     act_dtype=torch.bfloat16)
    assert layer.stage_kernel(T, nat.STAGE_ROUTER) == "k_router_mm"
    out, ids, w, logits = layer.forward(dev(x), return_routing=True)
    torch.cuda.synchronize()
    ref = O.router_logits(x, gate)
    rid, rw = O.route(ref, k, "softmax_topk", True)
    np.testing.assert_array_equal(to_f32(logits), ref)
    np.testing.assert_array_equal(ids.cpu().numpy(), rid)
    np.testing.assert_array_equal(w.cpu().numpy(), rw)
    if shared:  # zero banks: the output is the shared expert's, times its gate
        f = lambda b: torch.from_numpy(b.view(np.int16)).view(torch.bfloat16).double()  # noqa: E731
        gu = f(x) @ f(s13).t()
        h = (torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]).bfloat16().double()
        want = (h @ f(s2).t()) * torch.sigmoid((f(x) @ f(sgate).t()).bfloat16().double())
        assert rel_rms(to_f32(out), want.numpy()) < 2 * REL_RMS  # the gate's own rounding as well
    else:
        assert torch.count_nonzero(out) == 0


def test_gptq_tiles_take_outlier_channels(gpu):
    """Activations enter the GPTQ tiles as the bf16 values they are: one channel
    of each 128 at 1e4 that no weight reads (every code at its zero point) does
    not cost the others a bit.  What it does cost is the fp32 rounding of
    sum q x before the zero point leaves: H / 128 = 4 groups of 15 x 1e4 at
    2^-24 each, at most 0.04 of a step of s, against a sum of 512 products of
    about 4 s."""
    T, k = 80, 4
    syn = S.generate(replace(S.SMALL["c2_gptq"], H=512, I=256, shared_inter=0), T=T, seed=4)
    qw, z = syn.bank["qweight_gate_up"], syn.bank["qzeros_gate_up"]
    zero = torch.stack([(z >> (4 * i)) & 15 for i in range(8)], -1).reshape(z.shape[0], z.shape[1], -1) + 1
    assert int(zero.max()) <= 15
    for g in range(4):
        word, sh = (128 * g + 5) // 8, 4 * 5
        qw[:, word] = (qw[:, word] & ~(15 << sh)) | (zero[:, g].to(torch.int32) << sh)
    syn.x[:, 5::128] = 1e4
    rng = np.random.RandomState(2)
    ids = np.stack([rng.choice(16, k, replace=False) for _ in range(T)]).astype(np.int32)
    layer = _check(syn, gpu, ids, O.round_bf16(rng.rand(T, k).astype(np.float32)))
    assert layer.stage_kernel(T, nat.STAGE_W13) == "k_tile"


@pytest.mark.parametrize("T,H,kernel", [(100, 384, "k_tile"), (200, 2048, "k_stage_a_lean"), (300, 2048, "k_tile")])
def test_fp8_below_16_tokens_takes_outlier_channels(gpu, T, H, kernel):
    """Below 16 tokens per expert FP8 layers read bf16 activations, on the GEMV
    stages and on the tiles: a channel of each 128 at 1e6 that no weight reads
    leaves the others exact."""
    E, k = (64, 4) if H == 384 else (256, 8)
    syn = S.generate(replace(S.SMALL["c3_fp8"], E=E, k=k, H=H, I=512, shared_inter=0), T=T, seed=6)
    syn.bank["weight_gate_up"].view(torch.uint8)[:, :, 5::128] = 0
    syn.x[:, 5::128] = 1e6
    rng = np.random.RandomState(3)
    ids = np.stack([rng.choice(E, k, replace=False) for _ in range(T)]).astype(np.int32)
    layer = _check(syn, gpu, ids, O.round_bf16(rng.rand(T, k).astype(np.float32)))
    assert layer.stage_kernel(T, nat.STAGE_W13) == kernel


@pytest.mark.parametrize("H", [256, 320])
def test_bf16_output_does_not_depend_on_the_tile_kind(gpu, H):
    """The register-fed tiles (144 tokens: 275 stage-A tiles) and the LDS-ring
    ones (their first 80 tokens: 231) sum in the same order: the same bits."""
    cfg = replace(S.SMALL["c1_int8"], fmt="bf16", E=16, k=4, H=H, I=1408)
    syn = S.generate(cfg, T=144, seed=H).to(gpu)
    layer = S.build_layer(syn)
    assert layer.stage_kernel(144, nat.STAGE_W13) == "k_tile" and layer.stage_kernel(80, nat.STAGE_W13) == "k_gemm_a_ring"
    out, part = layer.forward(syn.x), layer.forward(syn.x[:80].contiguous())
    torch.cuda.synchronize()
    assert torch.equal(out[:80], part)


@pytest.mark.parametrize("fmt,kernel", [("c3_fp8", "k_gemm_mx"), ("c1_int8", "k_tile"), ("c2_gptq", "k_tile"),
                                        ("c4_mxfp4", "k_gemm_mx")])
def test_shared_expert_bits_beside_any_experts(gpu, fmt, kernel):
    """Routed banks of zeros leave the shared expert's output: beside every
    format's tiles the same bits as beside bf16 experts on the LDS-ring tiles."""
    T, H, Is = 200, 384, 192
    outs = []
    for f, I, want in ((fmt, 128, kernel), ("bf16", 64, "k_gemm_a_ring")):
        cfg = S.SMALL["c1_int8"] if f == "bf16" else S.SMALL[f]
        cfg = replace(cfg, fmt=f if f == "bf16" else cfg.fmt, E=8, k=2, H=H, I=I, shared_inter=Is, act="silu",
                      route_mode="softmax_topk", gate_bias=False, expert_bias=False)
        syn = S.generate(cfg, T=T, seed=1)
        for n, t in syn.bank.items():
            if f == "bf16" or n.startswith(("scale", "weight_scale", "blocks")):
                t.zero_()
        if outs:
            syn.x, syn.gate_w, syn.shared = first.x, first.gate_w, first.shared
        first = syn
        dsyn = syn.to(gpu)
        layer = S.build_layer(dsyn)
        assert layer.stage_kernel(T, nat.STAGE_W13) == want
        outs.append(layer.forward(dsyn.x))
    torch.cuda.synchronize()
    assert torch.count_nonzero(outs[0]) > 0
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("name,T,H,I,shared,group,kernel", [
    ("int8", 64, 256, 256, 0, 64, "k_gemm_a_ring"),     # four groups of 64
    ("int8", 130, 384, 384, 192, 192, "k_gemm_a_ring"),  # two of 192: one and a half K steps of the bf16 tiles
    ("int8", 70, 2112, 128, 0, 64, "k_gemm_a"),          # 33 groups: their scales do not fit beside the ring
    ("fp8", 64, 320, 384, 0, 128, "k_gemm_a_ring"),      # H and its scale blocks end in a half block
    ("fp8", 130, 256, 192, 192, 64, "k_gemm_a_ring"),    # 64 x 64 blocks
    ("fp8_bf16_scales", 90, 256, 256, 128, 128, "k_gemm_a_ring"),
])
def test_lds_tiles_match_oracle(gpu, name, T, H, I, shared, group, kernel):
    """Quantised layers above the crossover that the register-fed tiles do not
    take stay on the LDS tiles."""
    cast = lambda n, t: t  # noqa: E731
    if name == "int8":
        cfg = replace(S.SMALL["c1_int8"], H=H, I=I, shared_inter=shared, int8_num_groups=H // group)
        if I % (64 * (H // group)) and I != H:  # w2 per channel
            syn = S.generate(replace(cfg, int8_num_groups=1), T=T, seed=T)
            w = torch.randn(cfg.E, 2 * I, H, generator=torch.Generator().manual_seed(T)) * 0.02
            syn.bank.update(S.quantize_bank(cfg.fmt, w, "gate_up", int8_num_groups=H // group))
        else:
            syn = S.generate(cfg, T=T, seed=T)
    else:
        syn = S.generate(replace(S.SMALL["c3_fp8"], E=8, k=2, H=H, I=I, shared_inter=shared, group=group), T=T, seed=T)
    if name == "fp8_bf16_scales":
        for n in ("scale_gate_up", "scale_down"):
            syn.bank[n] = syn.bank[n].bfloat16().float()
        cast = lambda n, t: t.bfloat16() if n.startswith("scale") else t  # noqa: E731
    layer = _check(syn, gpu, cast=cast)
    assert layer.stage_kernel(T, nat.STAGE_W13) == kernel
    assert layer.stage_kernel(T, nat.STAGE_W2) == "k_gemm_b"


@pytest.mark.parametrize("name", ["c4_mxfp4", "c3_fp8", "c2_gptq", "c1_int8", "c1_int8_groups", "bf16"])
def test_tiles_of_rows_past_32_bit_offsets(gpu, name):
    """Activation rows that span more than 4 GiB go by 64-bit addresses: the
    first and last tokens of 270000 have the bits that they have by
    themselves."""
    from ftmoe import layer as L

    k, E, I = 8, 16, 1024
    T = 270_000  # h: T x k rows of 2048 bytes and more
    cfg = S.SMALL["c1_int8" if name in ("bf16", "c1_int8_groups") else name]
    cfg = replace(cfg, E=E, k=k, H=256, I=I, shared_inter=0, expert_bias=False,
                  int8_num_groups=2 if name == "c1_int8_groups" else 1, fmt="bf16" if name == "bf16" else cfg.fmt)
    syn = S.generate(cfg, T=64, seed=11, device=gpu)
    layer = S.build_layer(syn)
    x = torch.randn(T, 256, device=gpu, generator=torch.Generator(device=gpu).manual_seed(1)).bfloat16()
    with torch.cuda.stream(torch.cuda.Stream()):
        torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
        out = layer.forward(x)
        parts = [(sl, layer.forward(x[sl].contiguous())) for sl in (slice(0, 4096), slice(T - 4096, T))]
        torch.cuda.synchronize()
        L._WS.pop(L._ws_key(x.device))  # the stream's workspace of 7 GB and more
    for sl, part in parts:
        assert layer.stage_kernel(4096, nat.STAGE_W2) == layer.stage_kernel(T, nat.STAGE_W2)
        assert torch.equal(out[sl], part)
