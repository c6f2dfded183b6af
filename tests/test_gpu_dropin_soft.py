"""GPU parity of the reference's two soft samplers and its batched soft build, through the
C ABI and the drop-in module.

* plz_gumbel_lcg / plz_gumbel_lcg_triton against the reference's own Triton sampler outputs
  (tests/golden/lcg_triton_golden.npz, written from triton_soft_forward.py:51-66 by
  tests/golden/make_lcg_golden.py): every draw of the Triton variant, and the draws of the
  CUDA variant where the two reference samplers agree by construction. The GPU's logf and the
  golden's numpy log may differ by an ulp, so floats are compared at 2e-6; the discrete check
  below is bit-exact.
* A wrong bit anywhere in a hash changes its noise, and with it the argmax of the noisy
  softmax: the hard-noisy build from the GPU noise of each variant must equal the oracle's
  build from the oracle's noise bit for bit, except at near ties of (logit + noise) / tau.
* fused_lut_linear_soft(semantics="triton") against the oracle (forward: palette of the plain
  logits' argmax; backward from the Triton-variant noise of the module's own step counter).
* fused_compute_P_W_batched (fused_lut_linear_cuda.py:1016-1077): the reference's test pattern
  (test_batched_compute_pw.py:199-246: batched layer i == the single-layer build at seed
  step_seed ^ (i * 0x9E3779B9), group size 16) and the oracle (P within one fp16 ulp, W_soft
  within one bf16 ulp).
"""
import os

import numpy as np
import pytest
import torch

import oracle as O
from helpers import assert_close, f32

pytestmark = pytest.mark.gpu
ops = pytest.importorskip("palettize_hip.ops")
from palettize_hip import PLZ_W_HARD_NOISY  # noqa: E402
from palettize_hip import fused_lut_linear_cuda as FL  # noqa: E402
from palettize_hip.qwen_model import PalettizedLinear  # noqa: E402

GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden",
                    "lcg_triton_golden.npz")


@pytest.fixture(scope="module")
def gold():
    return np.load(GOLD)


def test_gumbel_lcg_variants_against_reference_golden(dev, gold):
    # a 32 x 32 grid draws idx (k*32 + n)*4 + c = 0..4095, the golden's first 4096 entries
    N = K = 32
    nk = O.lcg_index(N, K).ravel()
    for s in gold["seeds"]:
        s = int(s)
        want = gold[f"noise_{s}"][:4096]
        tri = f32(ops.gumbel_lcg(N, K, s, device=dev, variant="triton")).ravel()
        assert np.allclose(tri, want[nk], rtol=2e-6, atol=2e-6), f"triton variant, seed {s}"
        cud = f32(ops.gumbel_lcg(N, K, s, device=dev)).ravel()
        agree = O.lcg_variants_agree(s, nk)
        assert np.allclose(cud[agree], want[nk][agree], rtol=2e-6, atol=2e-6), f"cuda, seed {s}"
        assert np.allclose(cud, O.c_gumbel_lcg(s, N, K).ravel(), rtol=2e-6, atol=2e-6)


@pytest.mark.parametrize("variant", ["cuda", "triton"])
def test_gumbel_lcg_hard_build_is_bit_exact(dev, variant):
    N, K, seed, tau = 256, 1024, 0x5EED1234, 0.5
    g = torch.Generator().manual_seed(9)
    logits = torch.randn(N, K, 4, generator=g).to(torch.bfloat16)
    pal = torch.sort(torch.randn(N, K // 256, 4, generator=g) * 0.02, dim=-1).values
    noise = ops.gumbel_lcg(N, K, seed, device=dev, variant=variant)
    w, _ = ops.soft_build_w(logits.to(dev), noise, pal.to(dev), tau, PLZ_W_HARD_NOISY)
    want_noise = O.lcg_gumbel(seed, N, K, variant).astype(np.float64)
    _, _, w_fwd = O.soft_weights(f32(logits), want_noise, pal.numpy(), tau, O.W_HARD_NOISY)
    got = w.view(torch.int16).cpu().numpy().view(np.uint16)
    want = O.bf16_bits(w_fwd.astype(np.float32))
    z = (f32(logits).astype(np.float64) + want_noise) / tau
    top2 = np.sort(z, axis=-1)[..., -2:]
    tie = top2[..., 1] - top2[..., 0] <= 1e-5 * (1.0 + np.abs(top2[..., 1]))
    bad = got != want
    assert not np.any(bad & ~tie), f"{int(np.sum(bad & ~tie))} hard weights differ"
    # the noise decides the pick on a large share of weights (a wrong hash would show)
    am_plain = np.argmax(f32(logits), axis=-1)
    am_noisy = np.argmax(z, axis=-1)
    assert np.mean(am_plain != am_noisy) > 0.3


def test_dropin_soft_triton_semantics(dev):
    M, K, N, GS, tau = 64, 512, 512, 256, 1.0
    g = torch.Generator().manual_seed(21)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    logits = (torch.randn(4, K, N, generator=g) * 1.5).to(torch.float16)
    pal = torch.sort(torch.randn(N // GS, 4, generator=g) * 0.02, dim=-1).values.to(torch.bfloat16)
    gy = torch.randn(M, N, generator=g).to(torch.bfloat16)
    xd = x.to(dev).requires_grad_(True)
    ld = logits.to(dev).requires_grad_(True)
    pd = pal.to(dev).requires_grad_(True)
    FL._TRITON_STEP_SEED = 40
    cuda_seed = FL._SOFT_STEP_SEED
    y = FL.fused_lut_linear_soft(xd, pd, ld, None, GS, tau, semantics="triton")
    assert FL._TRITON_STEP_SEED == 41 and FL._SOFT_STEP_SEED == cuda_seed
    y.backward(gy.to(dev))
    nat_l = f32(logits).transpose(2, 1, 0)                       # [N, K, 4]
    nat_p = np.repeat(f32(pal), GS, axis=0)[:, None, :].repeat(K // 256, axis=1)
    noise = O.lcg_gumbel(41, N, K, "triton").astype(np.float64)
    _, _, w_ste = O.soft_weights(nat_l, noise, nat_p, tau, O.W_HARD_PLAIN)
    w_ste = O.bf16_round(w_ste.astype(np.float32))
    assert_close(f32(y), f32(x).astype(np.float64) @ w_ste.T, what="triton-semantics y")
    gl, gp = O.soft_backward(f32(x), f32(gy), nat_l, noise, nat_p, tau)
    assert_close(f32(ld.grad).transpose(2, 1, 0), gl, what="triton-semantics grad_logits")
    gp_ref = gp.sum(axis=1).reshape(N // GS, GS, 4).sum(axis=1)
    assert_close(f32(pd.grad), gp_ref, what="triton-semantics grad_palette")
    assert_close(f32(xd.grad), f32(gy).astype(np.float64) @ w_ste, what="triton-semantics grad_x")


def test_palettized_linear_soft_semantics_flags(dev):
    lin = torch.nn.Linear(256, 256, bias=False)
    idx = torch.randint(0, 4, (256, 256), generator=torch.Generator().manual_seed(3)).to(dev)
    a = PalettizedLinear(lin, idx, 1, 4, 256, False, use_soft_indices=True)
    b = PalettizedLinear(lin, idx, 1, 4, 256, False, use_soft_indices=True,
                         soft_semantics="triton")
    assert (a._use_cuda, a._use_triton) == (True, False)
    assert (b._use_cuda, b._use_triton) == (False, True)
    with pytest.raises(ValueError):
        PalettizedLinear(lin, idx, 1, 4, 256, False, soft_semantics="cutlass")


def _pw_oracle(logits, pal_bits, gs, tau, seed):
    """(P [K, N, 4], W_soft [K, N]) of the reference's batched kernel from the oracle."""
    lg = logits.astype(np.float32)                                # (4, K, N)
    _, K, N = lg.shape
    nat_l = lg.transpose(2, 1, 0)                                 # [N, K, 4]
    per_row = np.repeat(O.bf16_to_f32(pal_bits), gs, axis=0)[:N]  # [N, 4]
    nat_p = np.repeat(per_row[:, None, :], max(1, -(-K // 256)), axis=1)
    noise = O.lcg_gumbel(seed, N, K, "cuda").astype(np.float64)
    P, w_soft, _ = O.soft_weights(nat_l, noise, nat_p, tau, O.W_SOFT)
    return P.transpose(1, 0, 2), w_soft.T


def test_fused_compute_P_W_batched_reference_pattern(dev):
    """test_batched_compute_pw.py:199-246 on this build: shapes (K, N) (32, 64), (16, 32),
    (48, 64), group size 16, tau 0.5, step seed 12345."""
    mod = FL._get_module()
    torch.manual_seed(0)
    shapes, GS, tau, seed = [(32, 64), (16, 32), (48, 64)], 16, 0.5, 12345
    logits_list = [torch.randn(4, K, N, dtype=torch.float16, device=dev) for K, N in shapes]
    palette_list = [torch.randn(N // GS, 4, dtype=torch.bfloat16, device=dev) for _, N in shapes]
    flat = mod.fused_compute_P_W_batched(logits_list, palette_list, GS, tau, seed)
    assert len(flat) == 6
    for i, ((K, N), lg, pl) in enumerate(zip(shapes, logits_list, palette_list)):
        layer_seed = (seed ^ (i * 0x9E3779B9)) & 0xFFFFFFFF
        x_dummy = torch.zeros(1, K, dtype=torch.bfloat16, device=dev)
        P1, W1 = mod.fused_lut_linear_soft_fwd_aos(x_dummy, pl, lg, GS, tau, layer_seed)
        P, W = flat[2 * i], flat[2 * i + 1]
        assert P.shape == (K, N, 4) and W.shape == (K, N)
        assert torch.equal(P, P1) and torch.equal(W, W1), f"layer {i}"
        Pr, Wr = _pw_oracle(lg.cpu().numpy(), pl.view(torch.int16).cpu().numpy().view(np.uint16),
                            GS, tau, layer_seed)
        Pg = P.float().cpu().numpy().astype(np.float64)
        assert np.all(np.abs(Pg - Pr) <= np.maximum(np.abs(Pr) * 2.0 ** -10, 2.0 ** -24)), i
        Wg = W.float().cpu().numpy().astype(np.float64)
        assert np.all(np.abs(Wg - Wr) <= np.abs(Wr) * 2.0 ** -7 + 1e-6 * np.abs(Wr).max()), i
    with pytest.raises(ValueError, match="G mismatch"):
        mod.fused_compute_P_W_batched(logits_list[:1], [palette_list[1]], GS, tau, seed)


def test_fused_compute_P_W_batched_on_student(dev):
    """Walks a module for soft PalettizedLinears (skipping hard ones and non-palettized
    modules), at Qwen-like shapes, odd group sizes rejected."""
    g = torch.Generator().manual_seed(5)

    def pl(K, N, soft=True):
        lin = torch.nn.Linear(K, N, bias=False)
        idx = torch.randint(0, 4, (K, N), generator=g)
        pal = torch.sort(torch.randn(N // 256, 4, generator=g) * 0.02, -1).values
        m = PalettizedLinear(lin, idx, N // 256, 4, 256, False, initial_palette=pal,
                             use_soft_indices=soft).to(dev)
        if soft:  # logits off the one-hot init, so the noise matters
            with torch.no_grad():
                m.index_logits.copy_((torch.randn(4, K, N, generator=g) * 1.5).half())
        return m

    student = torch.nn.Module()
    student.q = pl(2560, 1024)
    student.frozen = pl(256, 512, soft=False)
    student.other = torch.nn.Linear(8, 8)
    student.down = pl(1024, 2560)
    out = FL.fused_compute_P_W_batched(student, 0.5, 777)
    assert len(out) == 2
    for i, m in enumerate((student.q, student.down)):
        P, W = out[i]
        K, N = m.index_logits.shape[1:]
        assert P.shape == (K, N, 4) and P.dtype == torch.float16 and W.dtype == torch.bfloat16
        seed = (777 ^ (i * 0x9E3779B9)) & 0xFFFFFFFF
        # the oracle on the first 64 input rows k (all N): a cut of whole rows keeps every
        # element's draw index (k*N + n)*4 + c
        rows = slice(0, 64)
        Pr, Wr = _pw_oracle(m.index_logits.detach()[:, rows].cpu().numpy(),
                            m.palette.detach().view(torch.int16).cpu().numpy().view(np.uint16),
                            256, 0.5, seed)
        Pg = P[rows].float().cpu().numpy().astype(np.float64)
        assert np.all(np.abs(Pg - Pr) <= np.maximum(np.abs(Pr) * 2.0 ** -10, 2.0 ** -24)), i
        Wg = W[rows].float().cpu().numpy().astype(np.float64)
        assert np.all(np.abs(Wg - Wr) <= np.abs(Wr) * 2.0 ** -7 + 1e-6 * np.abs(Wr).max()), i
    assert FL.fused_compute_P_W_batched(torch.nn.Linear(4, 4), 1.0, 1) == []
    student.down.group_size = 128
    with pytest.raises(ValueError, match="must share group_size"):
        FL.fused_compute_P_W_batched(student, 0.5, 777)


@pytest.mark.parametrize("semantics", ["cuda", "triton"])
@pytest.mark.parametrize("M,K,N,GS,dt,pdt,ste,strided", [
    (1, 8, 8, 256, torch.float16, torch.bfloat16, True, False),
    (70, 264, 520, 100, torch.bfloat16, torch.float32, True, True),
    (300, 512, 1032, 256, torch.float16, torch.bfloat16, False, False),
    (2000, 1048, 264, 3, torch.float16, torch.float16, True, False),
    (33, 256, 256, 256, torch.float16, torch.bfloat16, True, True)])
def test_soft_reference_layout_route_against_the_native_one(dev, semantics, M, K, N, GS, dt, pdt,
                                                            ste, strided, monkeypatch):
    """The soft linear in (K, N) order (noise drawn in its kernels) against the same call through
    the native layout (noise tensor, K padded): group sizes that split a lane's four columns,
    partial groups and unused ones, strided logits, both samplers, a reduction in one and in
    several splits. The forward weight is the same, so y differs by summation order only."""
    g = torch.Generator().manual_seed(M + K + N)
    logits = (torch.randn(4, K, N, generator=g) * 2).to(dt).to(dev)
    pal = (torch.randn(-(-N // GS) + 1, 4, generator=g) * 0.02).to(pdt).to(dev)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(dev)
    gy = torch.randn(M, N, generator=g).to(torch.bfloat16).to(dev)
    bias = torch.randn(N, generator=g).to(torch.bfloat16).to(dev)
    if strided:
        logits = logits.transpose(1, 2).contiguous().transpose(1, 2)
    outs = []
    for native in (False, True):
        FL._SOFT_STEP_SEED = FL._TRITON_STEP_SEED = 77
        if native:
            monkeypatch.setattr(FL, "_soft_in_reference_layout", lambda *a: False)
        leaves = [t.detach().clone().requires_grad_(True) for t in (x, pal, bias)]
        lg = logits.detach().requires_grad_(True)
        y = FL.fused_lut_linear_soft(leaves[0], leaves[1], lg, leaves[2], GS, 0.7, ste=ste,
                                     semantics=semantics)
        y.backward(gy)
        outs.append([y] + [t.grad for t in leaves] + [lg.grad])
    for a, b, what in zip(*outs, ("y", "grad_x", "grad_palette", "grad_bias", "grad_logits")):
        assert a.dtype == b.dtype and a.shape == b.shape, what
        assert_close(f32(a), f32(b).astype(np.float64), what=f"{what} (routes)")
    # the weights themselves: the hard picks bit for bit; W_soft within one bf16 ulp (2^-7
    # relative), since the compiler may fuse the two kernels' fp32 sums differently
    hard = ops._lib.PLZ_W_HARD_PLAIN if semantics == "triton" else PLZ_W_HARD_NOISY
    mode = hard if ste else ops._lib.PLZ_W_SOFT
    w = ops.soft_ref_build_w(logits.contiguous(), pal, GS, 78, 0.7, mode, semantics)
    Kp = FL._pad_k(K)
    noise = ops.gumbel_lcg(N, Kp, 78, device=dev, variant=semantics)
    wn, _ = ops.soft_build_w(FL.logits_from_reference(logits, K), noise,
                             FL.palette_from_reference(pal, N, K, GS), 0.7, mode)
    wn = wn[:, :K].t()
    assert torch.equal(w, wn) if ste else torch.allclose(w.float(), wn.float(), rtol=2 ** -7,
                                                         atol=1e-8)


@pytest.mark.parametrize("N,kg,GS,G", [(8, 1, 256, 1), (1032, 3, 100, 11), (4096, 10, 256, 16),
                                       (264, 38, 3, 90)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_palette_expand_and_fold(dev, N, kg, GS, G, dt):
    """Reference palettes to the native layout and the gradient back: partial, many and unused
    groups. The expansion is exact; a group's sum is fp32 in another order (n terms of random
    sign: error below n 2^-24 of the sum of magnitudes), rounded to the palette's type."""
    g = torch.Generator().manual_seed(N + kg)
    pal = torch.randn(G, 4, generator=g).to(dt).to(dev)
    want = pal.float().repeat_interleave(GS, 0)[:N][:, None].expand(N, kg, 4)
    assert torch.equal(FL.palette_from_reference(pal, N, 256 * kg, GS), want)
    assert torch.equal(FL._expand_palette(pal, N, 256 * kg, GS), want)
    grad = torch.randn(N, kg, 4, generator=g).to(dev)
    ref, mag = (torch.zeros(G, 4, dtype=torch.float64, device=dev) for _ in range(2))
    rows = torch.arange(N, device=dev) // GS
    ref.index_add_(0, rows, grad.double().sum(1))
    mag.index_add_(0, rows, grad.double().abs().sum(1))
    eps = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}[dt]
    for fold in (FL._fold_palette_grad, FL.palette_grad_to_reference):
        got = fold(grad, GS, G, dt)
        assert got.dtype == dt and bool(((got.double() - ref).abs() <=
                                         eps * ref.abs() + GS * kg * 2.0 ** -24 * mag + 1e-7).all())


@pytest.mark.parametrize("semantics", ["cuda", "triton"])
def test_soft_palette_of_other_strides(dev, semantics):
    """A palette whose (G, 4) is the transpose of a dense (4, G), or every other row of one: the
    same outputs, noise and gradients as the dense (G, 4)."""
    M, K, N, GS = 33, 256, 1032, 256
    g = torch.Generator().manual_seed(5)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).to(dev)
    logits = torch.randn(4, K, N, generator=g).to(torch.float16).to(dev)
    dense = (torch.randn(-(-N // GS), 4, generator=g) * 0.02).to(torch.bfloat16).to(dev)
    gy = torch.randn(M, N, generator=g).to(torch.bfloat16).to(dev)
    spaced = torch.zeros(2 * dense.shape[0], 4, dtype=dense.dtype, device=dev)
    spaced[::2] = dense
    outs = []
    for pal in (dense, dense.t().contiguous().t(), spaced[::2]):
        FL._SOFT_STEP_SEED = FL._TRITON_STEP_SEED = 11
        leaves = [x.clone().requires_grad_(True), pal.detach().requires_grad_(True),
                  logits.clone().requires_grad_(True)]
        y = FL.fused_lut_linear_soft(leaves[0], leaves[1], leaves[2], None, GS, 0.7,
                                     semantics=semantics)
        assert (FL._SOFT_STEP_SEED, FL._TRITON_STEP_SEED) == \
            ((12, 11) if semantics == "cuda" else (11, 12))
        outs.append([y, *torch.autograd.grad(y, leaves, gy)])
    for other in outs[1:]:
        for a, b, what in zip(outs[0], other, ("y", "grad_x", "grad_palette", "grad_logits")):
            assert torch.equal(a, b), what


@pytest.mark.parametrize("K", [512, 264])
@pytest.mark.parametrize("write", ["in place", "data"])
@pytest.mark.parametrize("train", [(0, 1, 2), (1,), (0,)], ids=["all", "palette", "x"])
def test_inputs_written_between_the_soft_forward_and_its_backward(dev, K, write, train):
    """The backward belongs to the forward's values: logits, palette and (at a K that is not a
    multiple of 256) x written after the forward, with or without torch's version counter seeing
    it, change none of its gradients."""
    M, N, GS = 40, 520, 256
    g = torch.Generator().manual_seed(K)
    vals = [torch.randn(M, K, generator=g).to(torch.bfloat16),
            (torch.randn(-(-N // GS), 4, generator=g) * 0.02).to(torch.bfloat16),
            torch.randn(4, K, N, generator=g).to(torch.float16)]
    gy = torch.randn(M, N, generator=g).to(torch.bfloat16).to(dev)
    grads = []
    for touch in (False, True):
        FL._SOFT_STEP_SEED = 30
        leaves = [v.to(dev).requires_grad_(i in train) for i, v in enumerate(vals)]
        y = FL.fused_lut_linear_soft(leaves[0], leaves[1], leaves[2], None, GS, 0.7)
        if touch:
            for t in leaves if K % 256 else leaves[1:]:
                if write == "data":
                    t.data.mul_(-3.0)
                else:
                    with torch.no_grad():
                        t.mul_(-3.0)
        grads.append(torch.autograd.grad(y, [leaves[i] for i in train], gy))
    for a, b, i in zip(*grads, train):
        assert torch.equal(a, b), ("grad_x", "grad_palette", "grad_logits")[i]


def test_palette_helpers_keep_type_and_gradient_on_the_gpu(dev):
    """The same calls as on the CPU (test_abi.py), with the same types and gradients."""
    from test_abi import _palette_helpers
    _palette_helpers(FL, dev)


@pytest.mark.parametrize("N,kg,GS,folds", [(9728, 38, 9728, 2), (9728, 13, 9728, 1),
                                           (9728, 14, 9728, 2), (1024, 38, 1 << 20, 1),
                                           (4096, 38, 1 << 20, 2), (9728, 38, 4864, 2),
                                           (9000, 38, 4001, 2), (9728, 38, 2432, 1)])
def test_large_palette_groups_are_folded_in_two_steps(dev, N, kg, GS, folds, monkeypatch):
    """A group of more than 2^17 entries is folded in parts first (a lone group of any size, groups
    with a last partial one, a prime number of rows): the fp64 sum up to n terms' rounding."""
    calls = []
    fold = ops.palette_fold
    monkeypatch.setattr(ops, "palette_fold", lambda *a: calls.append(1) or fold(*a))
    grad = torch.randn(N, kg, 4, generator=torch.Generator().manual_seed(kg)).to(dev)
    G = -(-N // GS) + 1
    got = FL._fold_palette_grad(grad, GS, G, torch.float32)
    assert len(calls) == folds and got.shape == (G, 4)
    ref, mag = (torch.zeros(G, 4, dtype=torch.float64, device=dev) for _ in range(2))
    rows = torch.arange(N, device=dev) // GS
    ref.index_add_(0, rows, grad.double().sum(1))
    mag.index_add_(0, rows, grad.double().abs().sum(1))
    n = min(GS, N) * kg
    assert bool(((got.double() - ref).abs() <= n * 2.0 ** -24 * mag).all())
