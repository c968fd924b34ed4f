"""GPU parity for the feed-forward block's tail fused into the combine
(ksl_moe_combine_post, ksl_moe_block_forward) and the layer drop-in
(moe_block_forward / patch_moe_blocks), against the oracle's block_tail
(TF modeling_diffusion_gemma.py:733-743 on the fused RMSNorm).

Bar (TAIL_* in tests/_helpers.py): the combine part is bit-exact (same fma
chain as the oracle); the two row sums of squares are taken in another fp32
order than the oracle's exact sums, which moves a bf16 rounding of the
normalised values by one ulp now and then. So: >= 99.9% of the outputs
bit-exact, and every output within 2 bf16 ulps or within an absolute
2^-4 * |layer_scalar| (one ulp of an intermediate of magnitude < 8 carried
through the second norm and the residual add, where the final value is
small). The measured figures are printed.
"""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as mo
from tests._helpers import Fixed, assert_tail_close, bf16_bits
from tests.conftest import load_mod, load_pkg

pytestmark = pytest.mark.gpu


def _np(t):
    return t.detach().cpu().numpy()


def _f32(t):
    return t.detach().float().cpu().numpy()


def _tail_inputs(T, tk, H, seed, wdt):
    g = torch.Generator().manual_seed(seed)
    out3 = (4 * torch.randn(T * tk, H, generator=g)).to(torch.float16)
    inv = torch.randperm(T * tk, generator=g).to(torch.int32)
    w = torch.rand(T, tk, generator=g) + 0.1
    w = (w / w.sum(-1, keepdim=True)).to(wdt)
    h1 = torch.randn(T, H, generator=g).to(torch.bfloat16)
    res = (2 * torch.randn(T, H, generator=g)).to(torch.bfloat16)
    w2 = (1 + 0.2 * torch.randn(H, generator=g)).to(torch.bfloat16)
    wp = (1 + 0.2 * torch.randn(H, generator=g)).to(torch.bfloat16)
    return out3, inv, w, h1, res, w2, wp


def _oracle_tail(out3, inv, w, h1, res, w2, wp, ls, eps2, eps):
    m = mo.f32_to_bf16(mo.combine_fma(_np(out3), _np(inv).astype(np.int64), _f32(w)))
    return mo.block_tail(m, _f32(h1), _f32(res), _f32(w2), _f32(wp), ls, eps2, eps)


def _combine_post(lib, out3, inv, w, h1, res, w2, wp, ls_t, y, eps2=1e-6, eps=1e-6):
    T, H = h1.shape
    tk = w.shape[1]
    rc = lib.load().ksl_moe_combine_post(
        lib.ptr(out3), lib.ptr(inv), lib.ptr(w), lib.dtype_code(w.dtype), T, tk, H,
        lib.ptr(h1), h1.stride(0), lib.ptr(res), res.stride(0), lib.ptr(w2), eps2, lib.ptr(wp), eps,
        lib.ptr(ls_t), lib.DTYPE_BF16 if ls_t is None else lib.dtype_code(ls_t.dtype),
        lib.ptr(y), y.stride(0), lib.stream_of(y))
    lib.check(rc, "ksl_moe_combine_post")


POST_CASES = [
    # (T, topk, H, weight dtype, layer scalar (value, dtype) or None, seed)
    (256, 8, 2816, torch.float32, (0.75, torch.bfloat16), 51),
    (37, 5, 256, torch.bfloat16, None, 52),
    (3, 12, 8192, torch.float16, (0.7071, torch.float32), 53),
    (64, 1, 128, torch.float32, (1.0, torch.float32), 54),
    (5, 8, 4096, torch.float32, (-1.5, torch.bfloat16), 55),
]


@pytest.mark.parametrize("T,tk,H,wdt,ls,seed", POST_CASES)
def test_combine_post_vs_oracle(gpu, T, tk, H, wdt, ls, seed):
    lib = load_mod("_lib")
    out3, inv, w, h1, res, w2, wp = _tail_inputs(T, tk, H, seed, wdt)
    ls_t = None if ls is None else torch.tensor([ls[0]], dtype=ls[1])
    lsv = 1.0 if ls is None else float(ls_t.float()[0])
    ref = _oracle_tail(out3, inv, w, h1, res, w2, wp, lsv, 1e-6, 1e-6)
    dev = [t.to(gpu) for t in (out3, inv, w, h1, res, w2, wp)]
    ls_d = None if ls_t is None else ls_t.to(gpu)
    y = torch.empty(T, H, dtype=torch.bfloat16, device=gpu)
    print(f"combine_post T={T} topk={tk} H={H} w={wdt} ls={ls}", flush=True)
    _combine_post(lib, *dev, ls_d, y)
    torch.cuda.synchronize()
    got = bf16_bits(y)
    assert_tail_close(got, ref, lsv, f"combine_post T={T} H={H}")
    # the same bits again, and with the output written over the residual
    y2 = torch.empty_like(y)
    _combine_post(lib, *dev, ls_d, y2)
    res_io = dev[4].clone()
    _combine_post(lib, *dev[:4], res_io, dev[5], dev[6], ls_d, res_io)
    torch.cuda.synchronize()
    assert np.array_equal(bf16_bits(y2), got)
    assert np.array_equal(bf16_bits(res_io), got)


def test_combine_post_separate_eps(gpu):
    lib = load_mod("_lib")
    T, tk, H = 16, 4, 512
    out3, inv, w, h1, res, w2, wp = _tail_inputs(T, tk, H, 56, torch.float32)
    out3 = (out3.float() * 1e-3).to(torch.float16)   # small rows: eps2 matters
    ref = _oracle_tail(out3, inv, w, h1, res, w2, wp, 1.0, 1e-2, 1e-6)
    dev = [t.to(gpu) for t in (out3, inv, w, h1, res, w2, wp)]
    y = torch.empty(T, H, dtype=torch.bfloat16, device=gpu)
    _combine_post(lib, *dev, None, y, eps2=1e-2, eps=1e-6)
    torch.cuda.synchronize()
    assert_tail_close(bf16_bits(y), ref, 1.0, "combine_post eps2=1e-2")
    same_eps = _oracle_tail(out3, inv, w, h1, res, w2, wp, 1.0, 1e-6, 1e-6)
    assert not np.array_equal(same_eps, ref)   # the case does exercise eps2


def test_block_forward_canvas_256(gpu):
    """ksl_moe_block_forward on the 256-token canvas (H 2816, I 704, 128 experts,
    top-8): the tail against the oracle applied to the MoE output of
    ksl_moe_layer_forward (the MoE itself has its own parity tests)."""
    lib = load_mod("_lib")
    wl = load_mod("workloads")
    T, H, I, E, tk = 256, wl.H_DG, wl.I_DG, wl.E_DG, wl.TOPK_DG
    x, pre_w, ids, wts = wl.layer_inputs(T, 61)
    exp = wl.make_experts(E, H, I, 62, device=gpu)
    g = torch.Generator().manual_seed(63)
    h1 = torch.randn(T, H, generator=g).to(torch.bfloat16)
    w2 = (1 + 0.2 * torch.randn(H, generator=g)).to(torch.bfloat16)
    wp = (1 + 0.2 * torch.randn(H, generator=g)).to(torch.bfloat16)
    ls = torch.tensor([0.625], dtype=torch.bfloat16)
    xd, pre_d, ids_d, w_d, h1_d, w2_d, wp_d, ls_d = (t.to(gpu) for t in (x, pre_w, ids, wts, h1, w2, wp, ls))
    L = lib.load()
    nbytes = L.ksl_moe_workspace_bytes(T, tk, E, H, I)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=gpu)
    m = torch.empty(T, H, dtype=torch.bfloat16, device=gpu)
    y = torch.empty(T, H, dtype=torch.bfloat16, device=gpu)
    st = lib.stream_of(xd)
    bufs = [lib.ptr(getattr(exp, k)) for k in ("gu_q", "gu_s", "gu_z", "dn_q", "dn_s", "dn_z")]
    v2 = load_mod("fused_moe_w4_v2")
    dn_t = v2.tiled_down(exp.dn_q, exp.dn_s, exp.dn_z)  # the block runs on the load-time repacked down weights
    bufs_t = bufs[:3] + [lib.ptr(dn_t)] + bufs[4:]
    print("block_forward T=256 H=2816 I=704 E=128 top-8", flush=True)
    rc = L.ksl_moe_layer_forward(lib.ptr(xd), lib.DTYPE_BF16, H, lib.ptr(pre_d), lib.DTYPE_BF16, 1e-6,
                                 lib.ptr(ids_d), lib.ptr(w_d), lib.DTYPE_F32, *bufs, lib.DN_LAYOUT_REF, None, None,
                                 T, tk, E, H, I,
                                 lib.ACT_SILU, lib.ptr(m), lib.DTYPE_BF16, H, lib.ptr(ws), nbytes, st)
    lib.check(rc, "ksl_moe_layer_forward")
    rc = L.ksl_moe_block_forward(lib.ptr(xd), H, lib.ptr(pre_d), 1e-6, lib.ptr(ids_d), lib.ptr(w_d), lib.DTYPE_F32,
                                 *bufs_t, lib.DN_LAYOUT_TILED, None, None, T, tk, E, H, I, lib.ACT_SILU, lib.ptr(h1_d), H,
                                 lib.ptr(w2_d), 1e-6,
                                 lib.ptr(wp_d), 1e-6, lib.ptr(ls_d), lib.DTYPE_BF16, lib.ptr(y), H,
                                 lib.ptr(ws), nbytes, st)
    lib.check(rc, "ksl_moe_block_forward")
    torch.cuda.synchronize()
    ref = mo.block_tail(bf16_bits(m), _f32(h1), _f32(x), _f32(w2), _f32(wp), 0.625, 1e-6, 1e-6)
    assert_tail_close(bf16_bits(y), ref, 0.625, "block_forward canvas 256")


def _packed_layer(gpu, T, seed):
    """A transformers DiffusionGemmaDecoderTextLayer (H 256, 16 experts of I 128,
    top-4, bf16) carrying packed W4 experts bound as the reference's loader binds
    them (kernels/load_w4_checkpoint.py:76-83), its norms and router patched;
    attention and the MLP return fixed tensors."""
    from transformers.models.diffusion_gemma.configuration_diffusion_gemma import DiffusionGemmaTextConfig
    from transformers.models.diffusion_gemma import modeling_diffusion_gemma as tfm
    pkg = load_pkg()
    wl = load_mod("workloads")
    H, I, E = 256, 128, 16
    cfg = DiffusionGemmaTextConfig(num_experts=E, hidden_size=H, moe_intermediate_size=I, top_k_experts=4,
                                   intermediate_size=384, num_attention_heads=2, num_key_value_heads=1,
                                   head_dim=128, rms_norm_eps=1e-6, num_hidden_layers=2,
                                   hidden_activation="gelu_pytorch_tanh")
    lay = tfm.DiffusionGemmaDecoderTextLayer(cfg, 1).to(torch.bfloat16)
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for mod in lay.modules():
            if isinstance(mod, tfm.DiffusionGemmaRMSNorm) and mod.with_scale:
                mod.weight.copy_(1 + 0.2 * torch.randn(mod.weight.shape, generator=g))
        lay.router.proj.weight.copy_(0.05 * torch.randn(E, H, generator=g))
        lay.layer_scalar.fill_(0.75)
    lay.self_attn = Fixed(torch.randn(2, T, H, generator=g).to(torch.bfloat16), as_tuple=True)
    lay.mlp = Fixed((3 * torch.randn(2, T, H, generator=g)).to(torch.bfloat16))
    lay = lay.to(gpu)
    lay.self_attn.out = lay.self_attn.out.to(gpu)
    lay.mlp.out = lay.mlp.out.to(gpu)
    ex = wl.make_experts(E, H, I, seed + 1, act="gelu", device=gpu)
    for k in ("gu_q", "gu_s", "gu_z", "dn_q", "dn_s", "dn_z"):
        setattr(lay.experts, k, getattr(ex, k))
    lay.experts.forward = pkg.fused_experts_forward.__get__(lay.experts, lay.experts.__class__)
    pkg.patch_rmsnorms(lay, verbose=False)
    pkg.patch_routers(lay, verbose=False)
    hidden = torch.randn(2, T, H, generator=g).to(torch.bfloat16).to(gpu)
    return lay, hidden, pkg


def test_patched_layer_matches_stock_forward(gpu):
    """TF DiffusionGemmaDecoderTextLayer.forward with the reference's bindings
    (fused experts, fused RMSNorm) vs the same layer after patch_moe_blocks."""
    lay, hidden, pkg = _packed_layer(gpu, 40, 71)
    with torch.no_grad():
        stock = type(lay).forward(lay, hidden)
    assert pkg.patch_moe_blocks(lay, verbose=False) == 1
    with torch.no_grad():
        ours = lay(hidden)
    torch.cuda.synchronize()
    assert ours.shape == stock.shape and ours.dtype == torch.bfloat16
    assert_tail_close(bf16_bits(ours.reshape(-1, 256)), bf16_bits(stock.reshape(-1, 256)), 0.75,
                      "patched layer vs stock forward")


def test_block_checks_the_zero_points_of_an_unseen_module(gpu):
    """A packed module that no load-time helper saw is checked on its first
    block forward, as the other forwards do: a zero-point outside the contract
    (an integer in [0, 15]) is refused, not truncated."""
    lay, hidden, pkg = _packed_layer(gpu, 40, 73)
    mod = load_mod("moe_block")
    lay.experts.gu_z[3, 5, 0] = 16.0
    with torch.no_grad(), pytest.raises(ValueError, match="zero-points"):
        mod.moe_block_forward(lay, hidden, hidden.clone())
    lay.experts.gu_z[3, 5, 0] = 15.0
    with torch.no_grad():
        assert mod.moe_block_forward(lay, hidden, hidden.clone()).shape == hidden.shape
