"""GPU tests of the decode-step kernels around the quantized linears:
pe_decode_attention, pe_add_rms_norm and pe_silu_mul against float64 torch
statements on the CPU of the same bf16 inputs.

Tolerances: outputs are rounded to bf16 once (relative 2^-9 of the value); the
fp32 sums before it are off by far less, so 2^-8 of the value, plus 2^-9 of the
output's largest value for sums that cancel, bounds every element."""

import math

import pytest
import torch

from gpu_helpers import DEV, say

pytestmark = pytest.mark.gpu


def _close(got, want, what):
    got, want = got.double().cpu(), want.double()
    bound = want.abs() * 2.0 ** -8 + want.abs().max() * 2.0 ** -9
    bad = (got - want).abs() > bound
    assert not bool(bad.any()), f"{what}: off by {float((got - want).abs().max()):.3e}"


@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 520), (16, 4096), (2, 8192), (2, 8200),
                                       (1, 32768)])
@pytest.mark.parametrize("residual", [False, True])
def test_add_rms_norm(rows, cols, residual):
    from polarengine_vllm.decode_runner import _add_norm
    say(f"add_rms_norm {rows}x{cols} residual={residual}")
    g = torch.Generator().manual_seed(rows * 31 + cols)
    x, r = (torch.randn(rows, cols, generator=g).to(torch.bfloat16) for _ in range(2))
    w = (1 + 0.1 * torch.randn(cols, generator=g)).to(torch.bfloat16)
    got_x, got_h = _add_norm(x.to(DEV), r.to(DEV) if residual else None, w.to(DEV), 1e-6)
    want_x = (x.float() + r.float()).to(torch.bfloat16) if residual else x
    assert torch.equal(got_x.cpu(), want_x)
    v = want_x.double()
    _close(got_h, v / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-6) * w.double(), "norm")


@pytest.mark.parametrize("rows,inter", [(1, 8), (7, 1000), (16, 12288)])
def test_silu_mul(rows, inter):
    from polarengine_vllm.decode_runner import _silu_mul
    say(f"silu_mul {rows}x{inter}")
    gu = 4 * torch.randn(rows, 2 * inter, generator=torch.Generator().manual_seed(inter))
    gu[0, :4] = torch.tensor([200.0, -200.0, 0.0, -1e30])
    gu = gu.to(torch.bfloat16)
    gate, up = gu[:, :inter].double(), gu[:, inter:].double()
    got = _silu_mul(gu.to(DEV)).double().cpu()
    want = gate / (1 + torch.exp(-gate)) * up
    assert bool(((got - want).abs() <= want.abs() * 2.0 ** -8 + 1e-30).all())


# fewer tiles than workgroups, several rounds, a ragged last tile; each K form;
# the last two shapes do not fit and take the library product
@pytest.mark.parametrize("rows,vocab,k", [(1, 8, 1024), (16, 300, 1024), (3, 16384 + 5, 2048),
                                          (16, 9000, 4096), (1, 5000, 8192), (7, 777, 3072),
                                          (17, 64, 1024), (2, 64, 640)])
def test_lm_head(rows, vocab, k):
    """fp32 sums of bf16 products: an error of K 2^-24 of the sum of magnitudes
    bounds any order (the library form rounds to bf16 as well: 2^-8)."""
    from polarengine_vllm.decode_runner import _lm_head
    from polarengine_vllm import _lib
    say(f"lm_head {rows}x{vocab}x{k}")
    g = torch.Generator().manual_seed(vocab)
    h = torch.randn(rows, k, generator=g).to(torch.bfloat16)
    w = (torch.randn(vocab, k, generator=g) / math.sqrt(k)).to(torch.bfloat16)
    got = _lm_head(h.to(DEV), w.to(DEV)).double().cpu()
    want, mag = h.double() @ w.double().T, h.double().abs() @ w.double().abs().T
    bound = mag * (k * 2.0 ** -24)
    if not _lib.lib().pe_lm_head_fits(rows, vocab, k):
        bound = bound + want.abs() * 2.0 ** -8
    assert got.shape == want.shape and bool(((got - want).abs() <= bound).all())


# one step, a step's edges, several steps per split, several splits, odd lengths
@pytest.mark.parametrize("d,group,kvh,batch,max_len,positions", [
    (64, 1, 3, 2, 65, (0, 1, 63, 64)),
    (128, 4, 8, 1, 1088, (0, 64, 1023, 1024, 1087)),
    (128, 8, 2, 3, 515, (127, 128, 514)),
    (64, 2, 8, 16, 1001, (5, 640, 1000)),
    (256, 2, 2, 2, 190, (63, 128, 189)),
    (64, 1, 8, 129, 130, (100, 129)),      # more rows than counters: one split each
    (128, 2, 1, 1, 9000, (8191, 8999)),    # the most splits, several steps in each
    # the other instances, each with one split and with several
    (256, 8, 2, 1, 700, (3, 64, 699)),     # two output passes in the last sum
    (256, 4, 1, 2, 300, (63, 299)),
    (256, 1, 2, 1, 300, (5, 299)),
    (64, 4, 2, 1, 300, (5, 299)),
    (64, 8, 1, 3, 300, (64, 299)),
    (128, 1, 2, 1, 300, (5, 299)),
])
def test_decode_attention(d, group, kvh, batch, max_len, positions):
    from polarengine_vllm.decode_runner import DecodeRunner, DecoderConfig
    cfg = DecoderConfig(hidden=256, layers=1, heads=kvh * group, kv_heads=kvh, head_dim=d,
                        intermediate=256, vocab=64)
    run = DecodeRunner(cfg, batch, max_len, DEV, seed=3)
    g = torch.Generator().manual_seed(d + group + max_len)
    kc = torch.randn(run.k_cache.shape, generator=g).to(torch.bfloat16)
    vc = torch.randn(run.v_cache.shape, generator=g).to(torch.bfloat16)
    # positions that are not written yet hold NaN: they must not be read into a result
    H = kvh * group
    for pos in positions:
        say(f"decode attention d={d} group={group} kvh={kvh} batch={batch} L={max_len} pos={pos}")
        run.k_cache.copy_(kc)
        run.v_cache.copy_(vc)
        run.k_cache[..., pos:] = float("nan")
        run.v_cache[..., pos:, :] = float("nan")
        qkv = torch.randn(batch, (H + 2 * kvh) * d, generator=g).to(torch.bfloat16)
        got = run._attention(torch.tensor([pos], device=DEV))(0, qkv.to(DEV))
        cos, sin = run.cos[pos].double().cpu(), run.sin[pos].double().cpu()
        qk = qkv[:, :(H + kvh) * d].double().view(batch, H + kvh, d)
        a, b = qk[..., :d // 2], qk[..., d // 2:]
        qk = torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
        k_new, v_new = run.k_cache[0, ..., pos].cpu(), run.v_cache[0, :, :, pos].cpu()
        _close(k_new, qk[:, H:], "new key")
        assert torch.equal(v_new, qkv[:, (H + kvh) * d:].view(batch, kvh, d))
        k, v = kc[0, ..., :pos + 1].double(), vc[0, :, :, :pos + 1].double()
        k[..., pos], v[:, :, pos] = k_new.double(), v_new.double()
        q = qk[:, :H].view(batch, kvh, group, d)
        p = torch.softmax(q @ k / math.sqrt(d), -1)
        _close(got, (p @ v).reshape(batch, H * d), "attention")
        after_k, after_v = run.k_cache[0].cpu(), run.v_cache[0].cpu()  # nothing else is written
        assert torch.equal(after_k[..., :pos], kc[0, ..., :pos])
        assert torch.equal(after_v[:, :, :pos], vc[0, :, :, :pos])
        assert bool(after_k[..., pos + 1:].isnan().all()) and bool(after_v[:, :, pos + 1:].isnan().all())
        # the counters are left zero: the same call again gives the same bits
        assert torch.equal(run._attention(torch.tensor([pos], device=DEV))(0, qkv.to(DEV)), got)


@pytest.mark.parametrize("d,group", [(64, 1), (128, 4), (256, 8)])
def test_decode_attention_infinite_scores(d, group):
    """Scores of -inf weigh nothing, in whole splits and next to finite ones."""
    from polarengine_vllm.decode_runner import DecodeRunner, DecoderConfig
    say(f"decode attention: infinite scores d={d} group={group}")
    cfg = DecoderConfig(hidden=256, layers=1, heads=2 * group, kv_heads=2, head_dim=d,
                        intermediate=256, vocab=64)
    L, pos, H = 400, 390, 2 * group
    run = DecodeRunner(cfg, 1, L, DEV, seed=3)
    g = torch.Generator().manual_seed(d + group)
    kc = torch.randn(run.k_cache.shape, generator=g).to(torch.bfloat16)
    run.v_cache.copy_(torch.randn(run.v_cache.shape, generator=g))
    # positive queries, no rotation: a key of -inf in one dimension scores -inf
    run.cos, run.sin = torch.ones_like(run.cos), torch.zeros_like(run.sin)
    qkv = torch.randn(1, (H + 4) * d, generator=g).abs().to(torch.bfloat16)
    for name, dead in (("a whole split and more", range(0, 200)), ("all but a few", range(3, pos))):
        k = kc.clone()
        k[0, 0, 0, 5, list(dead)] = float("-inf")
        run.k_cache.copy_(k)
        got = run._attention(torch.tensor([pos], device=DEV))(0, qkv.to(DEV)).double().cpu()
        q = qkv[:, :H * d].double().view(1, 2, group, d)
        k, v = run.k_cache[0, ..., :pos + 1].double().cpu(), run.v_cache[0, :, :, :pos + 1].double().cpu()
        want = torch.softmax(q @ k / math.sqrt(d), -1) @ v
        _close(got, want.reshape(1, H * d), name)


def test_decode_attention_refuses():
    from polarengine_vllm.decode_runner import DecodeRunner, DecoderConfig
    cfg = DecoderConfig(hidden=256, layers=1, heads=4, kv_heads=2, head_dim=64, intermediate=256,
                        vocab=64)
    run = DecodeRunner(cfg, 2, 32, DEV, seed=3)
    say("decode attention: wrong batch and wrong pos are refused on the host")
    attend = run._attention(torch.tensor([1], device=DEV))
    with pytest.raises(RuntimeError):
        attend(0, torch.zeros(3, 8 * 64, device=DEV, dtype=torch.bfloat16))
    with pytest.raises(RuntimeError):
        run._attention(torch.tensor([1], device=DEV, dtype=torch.int32))
    with pytest.raises(RuntimeError):
        run._attention(torch.tensor([1, 2], device=DEV))


def test_decode_step_refuses_operands_that_do_not_fit():
    from polarengine_vllm.decode_runner import DecodeRunner, DecoderConfig
    cfg = DecoderConfig(hidden=256, layers=1, heads=4, kv_heads=2, head_dim=64, intermediate=256,
                        vocab=64)
    tokens, pos = torch.tensor([1, 2], device=DEV), torch.tensor([3], device=DEV)
    say("decode step: norm weights, stream and cache that do not fit are refused on the host")
    ones = torch.ones(256, device=DEV)
    for change in (lambda r: r.layers[0].update(in_norm=ones.cpu()),
                   lambda r: r.layers[0].update(post_norm=ones[:128]),
                   lambda r: setattr(r, "final_norm", torch.ones(512, device=DEV)),
                   lambda r: setattr(r, "embed", r.embed.half()),
                   lambda r: setattr(r, "k_cache", r.k_cache[..., :24].contiguous()),
                   lambda r: setattr(r, "v_cache", r.v_cache.half())):
        run = DecodeRunner(cfg, 2, 32, DEV, seed=3)
        change(run)
        with pytest.raises(RuntimeError):
            run.step(tokens, pos)
    run.final_norm, run.v_cache = 2 * ones, run.v_cache.to(torch.bfloat16)  # fp32 weights are taken
    assert run.step(tokens, pos).shape == (2, 64)


def test_decode_step_follows_its_rotary_tables():
    """Tables replaced or changed in place are the ones that attention uses, in
    the kernel as in the torch form."""
    from polarengine_vllm.decode_runner import DecodeRunner, DecoderConfig
    cfg = DecoderConfig(hidden=256, layers=1, heads=4, kv_heads=2, head_dim=64, intermediate=256,
                        vocab=64)
    say("decode attention: replaced rotary tables")
    g = torch.Generator().manual_seed(8)
    qkv = torch.randn(2, 8 * 64, generator=g).to(DEV, torch.bfloat16)
    ang = torch.rand(32, 32, generator=g).to(DEV) * 6
    pos = torch.tensor([0], device=DEV)
    keys = []
    for form in ("replaced", "in place"):
        run = DecodeRunner(cfg, 2, 32, DEV, seed=3)
        if form == "replaced":
            run.cos, run.sin = ang.cos(), ang.sin()
        else:
            run.cos.copy_(ang.cos())
            run.sin.copy_(ang.sin())
        assert torch.equal(run.cos, ang.cos()) and torch.equal(run.sin, ang.sin())
        for attend in (run._attention(pos), run._attention_torch(pos)):
            attend(0, qkv)
            k = run.k_cache[0, ..., 0].double().cpu()
            a, b = qkv[:, 256:384].double().cpu().view(2, 2, 64).chunk(2, -1)
            c, s = ang[0].cos().double().cpu(), ang[0].sin().double().cpu()
            _close(k, torch.cat([a * c - b * s, b * c + a * s], -1), f"key, tables {form}")
            keys.append(k)
    assert torch.equal(keys[0], keys[2])
