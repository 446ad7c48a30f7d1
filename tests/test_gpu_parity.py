"""Parity of the HIP path (through the C ABI) against the CPU oracle on identical seeded inputs.

Tolerance, one rule for every comparison in this file (`_close`): rtol = 2e-2 element-wise against the
reference evaluated in fp32 on the same (already rounded) inputs, atol = 2e-2 * max(1, mean|ref|), and a
relative Frobenius error below 1e-2.  The absolute term follows the magnitude of the tensor because
an element's rounding error is set by the size of the terms that were summed (which is what
mean|ref| measures), not by the element's own value: an element of a weight gradient that happens
to come out near zero from 8192 products of size 1 cannot be held to 2e-2 of itself.  For outputs
of typical size below one (Y, dX, G, U, H, dG, dU with the stated input distributions) the rule is
the plain rtol = atol = 2e-2.  `test_cfg3_fp16_forward_backward_llama3_8b` holds the rule against a
yardstick: torch's own fp16 module on the same inputs against the same oracle.
"""

import contextlib
import warnings

import numpy as np
import pytest
import torch

from cases import CFG2, CFG3, CFG4, CFG5, Case, make_inputs
from oracle import eager as oracle
from oracle import philox

pytestmark = pytest.mark.gpu

RTOL = ATOL = 2e-2


def _dev():
    assert torch.cuda.is_available(), "GPU tests need a visible AMD GPU"
    return torch.device("cuda", 0)


def _close(name, got, ref):
    got = got.detach().float().cpu()
    ref = ref.detach().float().cpu()
    assert got.shape == ref.shape, f"{name}: shape {tuple(got.shape)} vs {tuple(ref.shape)}"
    assert torch.isfinite(got).all(), f"{name}: non-finite values"
    err = (got - ref).abs()
    atol = ATOL * max(1.0, ref.abs().mean().item() if ref.numel() else 0.0)
    bad = err > atol + RTOL * ref.abs()
    rel_fro = ((got - ref).norm() / ref.norm().clamp_min(1e-30)).item()
    # elements outside the plain band, whatever the magnitude of the tensor scaled the absolute term to
    plain = int((err > ATOL + RTOL * ref.abs()).sum()) if err.numel() else 0
    print(
        f"  {name}: max_abs_err={err.max().item() if err.numel() else 0.0:.3e} rel_fro={rel_fro:.3e} "
        f"atol={atol:.3g} outside_plain_{RTOL:g}_{ATOL:g}_band={plain}/{err.numel()}",
        flush=True,
    )
    assert not bad.any(), (
        f"{name}: {int(bad.sum())} of {bad.numel()} elements outside rtol={RTOL}, atol={atol:.3g}; "
        f"max_abs_err={err.max().item():.4e}, rel_fro={rel_fro:.3e}"
    )
    assert rel_fro < 1e-2, f"{name}: relative Frobenius error {rel_fro:.3e}"


def _oracle_inputs(t):
    return {k: (None if v is None else v.float()) for k, v in t.items()}


def _run_module_case(c: Case, lean: bool = False, yardstick: bool = False):
    from triton_gated_mlp import FusedGatedMLP
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    print(f"case {c.name}: M={c.M} K={c.K} N={c.N} dtype={c.dtype} bias={c.bias} p={c.p} act={c.act}", flush=True)
    t = make_inputs(c)
    mlp = FusedGatedMLP(hidden_size=c.K, intermediate_size=c.N, bias=c.bias, dropout_p=c.p, hidden_act=c.act)
    mlp = mlp.to(dev).to(c.dtype)
    with torch.no_grad():
        mlp.gate_proj.weight.copy_(t["W_gate"])
        mlp.up_proj.weight.copy_(t["W_up"])
        mlp.down_proj.weight.copy_(t["W_down"])
        if c.bias:
            mlp.gate_proj.bias.copy_(t["b_gate"])
            mlp.up_proj.bias.copy_(t["b_up"])
            mlp.down_proj.bias.copy_(t["b_down"])
    mlp.train(c.p > 0.0)
    mlp.dropout_seed = c.dropout_seed
    mlp.recompute_activations = lean
    x = t["x"].to(dev).requires_grad_(c.backward)

    with contextlib.nullcontext() if c.backward else torch.no_grad():
        y = mlp(x)
    keep = None
    if c.p > 0.0:
        # one mask per row chunk the module ran (a single one unless the batch was split)
        states = mlp.last_dropout_states
        assert states and states[0][0] == 0 and sum(s[1] for s in states) == c.M
        assert mlp.last_dropout_state == states[-1][2:]
        parts = []
        for row0, rows, seed, offset in states:
            keep_dev = ops_fwd.dropout_mask(rows, c.N, c.p, seed, offset, device=dev)
            keep_np = philox.keep_mask(rows, c.N, c.p, seed, offset)
            assert np.array_equal(keep_dev.cpu().numpy(), keep_np), "device keep mask differs from the NumPy Philox oracle"
            parts.append(keep_np)
        keep = torch.from_numpy(np.concatenate(parts, axis=0))

    o = _oracle_inputs(t)
    if not c.backward:
        ref = oracle.forward(
            o["x"], o["W_gate"], o["b_gate"], o["W_up"], o["b_up"], o["W_down"], o["b_down"], keep, c.p, c.act
        )
        _close("Y", y, ref["Y"])
        return
    grads_in = [x, mlp.gate_proj.weight, mlp.up_proj.weight, mlp.down_proj.weight]
    names = ["dX", "dW_gate", "dW_up", "dW_down"]
    if c.bias:
        grads_in += [mlp.gate_proj.bias, mlp.up_proj.bias, mlp.down_proj.bias]
        names += ["db_gate", "db_up", "db_down"]
    grads = torch.autograd.grad(y, grads_in, grad_outputs=t["dY"].to(dev))
    ref = oracle.backward(
        o["x"], o["W_gate"], o["b_gate"], o["W_up"], o["b_up"], o["W_down"], o["b_down"], o["dY"], keep, c.p, c.act
    )
    _close("Y", y, ref["Y"])
    for n, g in zip(names, grads):
        _close(n, g, ref[n])
    if yardstick:
        from triton_gated_mlp import EagerGatedMLP, copy_weights

        eager = EagerGatedMLP(hidden_size=c.K, intermediate_size=c.N, bias=c.bias, dropout_p=0.0, hidden_act=c.act)
        eager = eager.to(dev).to(c.dtype)
        copy_weights(mlp, eager)
        xe = t["x"].to(dev).requires_grad_(True)
        ge = torch.autograd.grad(eager(xe), [xe, eager.gate_proj.weight, eager.up_proj.weight, eager.down_proj.weight],
                                 grad_outputs=t["dY"].to(dev))
        for n, g_fused, g_eager in zip(names[:4], grads[:4], ge):
            r = ref[n]
            band = ATOL + RTOL * r.abs()
            e_f, e_e = (g_fused.float().cpu() - r).abs(), (g_eager.float().cpu() - r).abs()
            out_f, out_e = int((e_f > band).sum()), int((e_e > band).sum())
            print(f"  yardstick {n}: outside plain band fused {out_f}, torch fp16 {out_e} of {r.numel()}; "
                  f"max_abs_err fused {e_f.max().item():.3e}, torch fp16 {e_e.max().item():.3e}", flush=True)
            assert out_f <= 1.5 * out_e + 1000, f"{n}: the fused path leaves the plain band far more often than torch's fp16 path"
            assert e_f.max().item() <= 2.0 * e_e.max().item() + ATOL


def test_cfg2_fp16_forward_llama7b():
    _run_module_case(CFG2)


def test_cfg3_fp16_forward_backward_llama3_8b():
    """The headline configuration at full size.  Also the yardstick for the weight-gradient tolerance
    (atol = 2e-2 * max(1, mean|ref|)): an element of dW sums M = 8192 products of operands that were
    themselves rounded to fp16 on the way (dG, dU, H), so its error has an absolute size set by the
    typical magnitude of dW (tens), whatever the element's own value, and elements far below typical
    cannot meet a bound relative to themselves.  torch's own fp16 module (EagerGatedMLP on the GPU,
    hipBLASLt GEMMs) is run on the same inputs: against the same fp32 oracle it leaves the plain
    2e-2/2e-2 band for about as many elements, and the fused gradients are as close as torch's."""
    _run_module_case(CFG3, yardstick=True)


def test_cfg4_bf16_bias_dropout_forward_backward():
    _run_module_case(CFG4)


def test_cfg5_fp16_decode_forward():
    _run_module_case(CFG5)


def test_cfg1_fp32_forward_against_golden_fixture():
    """Baseline configuration 1 (fp32, M=128, K=512, N=256, bias=False, x ~ U[0,1) from torch.rand,
    nn.Linear default init, seed 0; EagerGatedMLP.forward, src/triton_gated_mlp/gated_mlp.py:92-98)
    through FusedGatedMLP on the float32 HIP path, against the committed fixture and the oracle.
    Inputs are built exactly as tests/golden/make_cfg1.py builds them."""
    from golden import make_cfg1
    from triton_gated_mlp import FusedGatedMLP, copy_weights

    dev = _dev()
    torch.manual_seed(0)
    ref_mod = oracle.OracleGatedMLP(hidden_size=512, intermediate_size=256, bias=False, dropout_p=0.0).float()
    torch.manual_seed(0)
    x = torch.rand(128, 512)
    fix = np.load(make_cfg1.FIXTURE)
    assert np.array_equal(fix["x_head"], x[0, :8].numpy()), "torch's generator changed: regenerate the fixture"
    assert np.array_equal(fix["w_gate_head"], ref_mod.gate_proj.weight[0, :8].detach().numpy())
    fused = FusedGatedMLP(hidden_size=512, intermediate_size=256, bias=False, dropout_p=0.0).float()
    copy_weights(ref_mod, fused)
    fused = fused.to(dev)
    with torch.no_grad():
        y = fused(x.to(dev)).cpu()
        y_ref = ref_mod(x)
    assert y.dtype == torch.float32 and y.shape == (128, 512)
    # fp32 operands, fp32 accumulation on both sides: only the summation order differs
    assert torch.allclose(y, y_ref, rtol=1e-4, atol=1e-5), f"max abs err {(y - y_ref).abs().max().item():.3e}"
    np.testing.assert_allclose(y[::16, ::64].numpy(), fix["y_strided"], rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(y.double().sum().item(), float(fix["y_sum"]), rtol=1e-5)
    print(f"  cfg1: max_abs_err={(y - y_ref).abs().max().item():.3e}", flush=True)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize(
    "M,K,N,bias,p",
    [
        (128, 256, 512, True, 0.0),  # the reference's module test shape (tests/test_gated_mlp_fwd.py:23-38)
        (512, 256, 512, False, 0.0),  # 3-D input case B=16, M=32 (tests/test_gated_mlp_bwd.py:27-45)
        (64, 256, 512, False, 0.0),  # B,M,N,K = 2,32,512,256 (tests/test_gated_mlp_bwd.py:97)
        (200, 136, 264, True, 0.25),  # ragged: nothing a multiple of the tile
        (1, 64, 128, True, 0.0),
        (256, 512, 1024, True, 0.5),
        (768, 1024, 2048, False, 0.0),
    ],
)
def test_small_shapes_forward_backward(M, K, N, bias, p, dtype):
    _run_module_case(Case(f"small_{M}x{K}x{N}", M, K, N, dtype, bias=bias, p=p, backward=True, seed=M + K + N))


@pytest.mark.parametrize(
    "M,K,N,dtype,bias,p",
    [
        (3001, 2048, 4096, torch.float16, False, 0.0),  # odd token count on the 256-tile and 128-tile kernels
        (1000, 1024, 4104, torch.bfloat16, True, 0.1),  # ragged tokens and ragged intermediate size
        (50, 512, 1024, torch.float16, True, 0.0),  # fewer rows than one tile
        (4099, 1024, 2048, torch.float16, False, 0.0),  # three rows into the last tile-row
    ],
)
def test_ragged_token_counts_on_the_pipelined_kernels(M, K, N, dtype, bias, p):
    """Token counts (and intermediate sizes) that are not multiples of the tile run on the same
    kernels as whole tiles: the part of a tile beyond the end of an operand reads as zero.  The
    weight gradients reduce over the ragged dimension."""
    _run_module_case(Case(f"ragged_{M}x{K}x{N}", M, K, N, dtype, bias=bias, p=p, backward=True, seed=M))


@pytest.mark.parametrize(
    "M,K,N,dtype,bias",
    [
        (17, 2048, 8192, torch.float16, True),  # one more row than the skinny-M kernels take
        (64, 1024, 4096, torch.float16, False),
        (300, 1024, 4096, torch.bfloat16, True),
        (130, 4096, 14336, torch.float16, False),  # Llama-3-8B widths, short batch
        (40, 1024, 4160, torch.float16, False),  # 130 reduction tiles for dX do not divide by 16 splits
        (100, 5120, 13824, torch.float16, True),  # Llama-2-13B widths: the gate/up GEMM splits as well
    ],
)
def test_short_batches_split_the_long_reductions(M, K, N, dtype, bias):
    """Down projection and input gradient of a short batch have a few output tiles and a long
    reduction; the library asks for a workspace and splits the reduction over several workgroups
    per tile.  Same results as ever, to the usual tolerance."""
    from triton_gated_mlp import _cabi

    code = _cabi.dtype_code(dtype)
    assert _cabi.lib().gmlp_workspace_bytes(_cabi.GMLP_OP_LINEAR_FWD, M, N, K, code) > 0
    assert _cabi.lib().gmlp_workspace_bytes(_cabi.GMLP_OP_DX_BWD, M, K, N, code) > 0
    if N == 13824:
        assert _cabi.lib().gmlp_workspace_bytes(_cabi.GMLP_OP_GATEUP_FWD, M, K, N, code) > 0
    _run_module_case(Case(f"short_{M}x{K}x{N}", M, K, N, dtype, bias=bias, p=0.0, backward=True, seed=M + 1))


def test_split_reduction_without_workspace_gives_the_unsplit_result():
    """NULL workspace is always accepted: one workgroup per tile, same numbers up to summation order."""
    from triton_gated_mlp import _cabi
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(5)
    a = torch.randn(48, 8192, generator=g).to(torch.float16).to(dev)
    W = (0.02 * torch.randn(1024, 8192, generator=g)).to(torch.float16).to(dev)
    split = ops_fwd.linear_fwd(a, W)
    plain = torch.empty_like(split)
    _cabi.check(_cabi.lib().gmlp_linear_fwd(a.data_ptr(), W.data_ptr(), None, plain.data_ptr(), 48, 8192, 1024, 0,
                                            None, 0, _cabi.stream_ptr(dev)))
    ref = a.float().cpu() @ W.float().cpu().T
    _close("split", split, ref)
    _close("plain", plain, ref)
    assert (split.float() - plain.float()).abs().max().item() < 1e-2


OTHER_ACTS = ["gelu", "relu", "leaky_relu", "sigmoid", "tanh", "no_act"]


@pytest.mark.parametrize("act", OTHER_ACTS)
def test_other_activations_forward_backward(act):
    """hidden_act beyond silu (the reference's ACT_FWD table, src/triton_gated_mlp/gated_mlp.py:28-37):
    full-tile kernels, bias, dropout; fp16."""
    _run_module_case(Case(f"act_{act}", 384, 256, 640, torch.float16, bias=True, p=0.1, backward=True, seed=21, act=act))


@pytest.mark.parametrize("act,dtype", [("gelu", torch.bfloat16), ("relu", torch.bfloat16), ("tanh", torch.float32)])
def test_other_activations_ragged_shapes_and_dtypes(act, dtype):
    _run_module_case(Case(f"act_{act}_ragged", 200, 136, 264, dtype, bias=True, p=0.25, backward=True, seed=22, act=act))


@pytest.mark.parametrize("act", OTHER_ACTS)
def test_other_activations_decode_path(act):
    """The weight-streaming kernels for M <= 16 (both variants: K % 256 == 0 and not), called directly:
    the module only routes to them for widths that fill the chip."""
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    for c in (
        Case(f"act_{act}_decode", 8, 1024, 1536, torch.float16, bias=True, seed=23, act=act),
        Case(f"act_{act}_decode_generic", 16, 96, 512, torch.float16, bias=False, seed=24, act=act),
    ):
        t = make_inputs(c)
        d = {k: (None if v is None else v.to(dev)) for k, v in t.items()}
        y = ops_fwd.decode_fwd(d["x"], d["W_gate"], d["b_gate"], d["W_up"], d["b_up"], d["W_down"], d["b_down"], act)
        o = _oracle_inputs(t)
        ref = oracle.forward(o["x"], o["W_gate"], o["b_gate"], o["W_up"], o["b_up"], o["W_down"], o["b_down"], act=act)
        _close(f"{c.name} Y", y, ref["Y"])


@pytest.mark.parametrize("act", ["gelu", "no_act"])
def test_other_activations_operator_level(act):
    """mlp_hidden_states_fwd / _bwd with act_fn, the reference operator signatures
    (src/triton_gated_mlp/ops/fwd.py:198-206, ops/bwd.py:466-468).  The reference's no_act backward
    multiplies by G instead of 1 (_act_bwd, ops/act.py:15-18); the true derivative is checked here."""
    from triton_gated_mlp import mlp_hidden_states_bwd, mlp_hidden_states_fwd

    dev = _dev()
    c = Case(f"op_{act}", 256, 128, 384, torch.float16, backward=True, seed=25, act=act)
    t = make_inputs(c)
    g = torch.Generator().manual_seed(26)
    dH = torch.randn(c.M, c.N, generator=g).to(c.dtype)
    x, Wu, Wg = t["x"].to(dev), t["W_up"].to(dev), t["W_gate"].to(dev)
    h = mlp_hidden_states_fwd(x, Wu, None, Wg, None, act, 0.0)
    dx, dWu, dWg = mlp_hidden_states_bwd(x, Wu, Wg, dH.to(dev), act_fn=act)
    o = _oracle_inputs(t)
    f = oracle.hidden_forward(o["x"], o["W_gate"], None, o["W_up"], None, act=act)
    hb = oracle.hidden_backward(dH.float(), f["G"], f["U"], act=act)
    _close("H", h, f["H"])
    _close("dX", dx, hb["dU"] @ o["W_up"] + hb["dG"] @ o["W_gate"])
    _close("dW_up", dWu, hb["dU"].T @ o["x"])
    _close("dW_gate", dWg, hb["dG"].T @ o["x"])


def test_device_activation_functions_against_float64_closed_forms():
    """The kernels evaluate erf and tanh through short fp32 approximations; this pins them far below
    the storage tolerance.  gating_bwd in float32 with dH = U = 1 returns act(G) as dU and act'(G) as
    dG, compared with scipy / numpy in float64 on a dense grid that includes both tails and 0."""
    from scipy.special import erf, expit

    from triton_gated_mlp.ops import bwd as ops_bwd

    dev = _dev()
    x32 = torch.linspace(-12.0, 12.0, 64 * 4096, dtype=torch.float32).reshape(64, 4096).clone()
    x32[0, :2] = torch.tensor([0.0, -0.0])
    x = x32.double().numpy()
    cdf, pdf = 0.5 * (1.0 + erf(x / np.sqrt(2.0))), np.exp(-0.5 * x * x) / np.sqrt(2.0 * np.pi)
    closed = {
        "silu": (x * expit(x), expit(x) * (1.0 + x * (1.0 - expit(x)))),
        "gelu": (x * cdf, cdf + x * pdf),
        "sigmoid": (expit(x), expit(x) * (1.0 - expit(x))),
        "tanh": (np.tanh(x), 1.0 - np.tanh(x) ** 2),
    }
    one = torch.ones_like(x32).to(dev)
    for act, (f, df) in closed.items():
        dg, du = ops_bwd.gating_bwd(one, x32.to(dev), one, 0.0, 0, 0, act)
        err_f = np.abs(du.cpu().double().numpy() - f).max()
        err_d = np.abs(dg.cpu().double().numpy() - df).max()
        assert err_f < 2e-6 and err_d < 2e-6, (act, err_f, err_d)  # |x| <= 12: a few fp32 ulps of the value
    # tanh keeps its relative accuracy through 0 (no 1 - e^{-2x} cancellation)
    tiny = torch.logspace(-6, -1, 4096, dtype=torch.float32).reshape(1, -1)
    _, du = ops_bwd.gating_bwd(torch.ones_like(tiny).to(dev), tiny.to(dev), torch.ones_like(tiny).to(dev), 0.0, 0, 0, "tanh")
    rel = np.abs(du.cpu().double().numpy() / np.tanh(tiny.double().numpy()) - 1.0).max()
    assert rel < 1e-6, rel


def test_three_dimensional_input_matches_flattened():
    """[B, S, K] input gives the 2-D result on x.view(-1, K) (tests/test_gated_mlp_bwd.py:37-45)."""
    from triton_gated_mlp import FusedGatedMLP

    dev = _dev()
    torch.manual_seed(0)
    mlp = FusedGatedMLP(256, 512, bias=False).to(dev).to(torch.float16)
    x = torch.rand(16, 32, 256, device=dev, dtype=torch.float16)
    y3 = mlp(x)
    y2 = mlp(x.view(-1, 256))
    assert y3.shape == x.shape
    assert torch.equal(y3.view(-1, 256), y2)


def test_operator_level_fwd_bwd_match_closed_form():
    """mlp_hidden_states_fwd/bwd against the closed form (pattern of tests/test_gated_mlp_bwd.py:89-129)."""
    from triton_gated_mlp import mlp_hidden_states_bwd, mlp_hidden_states_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(7)
    BM, N, K = 64, 512, 256
    x = torch.rand(BM, K, generator=g).half()
    W_up = (torch.rand(N, K, generator=g) / 8).half()
    W_gp = (torch.rand(N, K, generator=g) / 8).half()
    dH = torch.rand(BM, N, generator=g).half()
    h = mlp_hidden_states_fwd(x.to(dev), W_up.to(dev), None, W_gp.to(dev), None, "silu", 0.0)
    ref = oracle.hidden_forward(x.float(), W_gp.float(), None, W_up.float(), None)
    _close("hidden", h, ref["H"])
    dx, dW_up, dW_gp = mlp_hidden_states_bwd(x.to(dev), W_up.to(dev), W_gp.to(dev), dH.to(dev))
    hb = oracle.hidden_backward(dH.float(), ref["G"], ref["U"])
    _close("dx", dx, hb["dU"] @ W_up.float() + hb["dG"] @ W_gp.float())
    _close("dW_up", dW_up, hb["dU"].T @ x.float())
    _close("dW_gp", dW_gp, hb["dG"].T @ x.float())


def test_autograd_function_reference_signature():
    """FusedGatedMLPFunction.apply(x, W_up, b_up, W_gp, b_gp) with biases and bias gradients."""
    from triton_gated_mlp import FusedGatedMLPFunction

    dev = _dev()
    g = torch.Generator().manual_seed(11)
    M, K, N = 96, 128, 256
    mk = lambda *s: torch.randn(*s, generator=g).mul(0.1).half()
    x, W_up, b_up, W_gp, b_gp, dH = mk(M, K), mk(N, K), mk(N), mk(N, K), mk(N), mk(M, N)
    args = [a.to(dev).requires_grad_(True) for a in (x, W_up, b_up, W_gp, b_gp)]
    h = FusedGatedMLPFunction.apply(*args)
    grads = torch.autograd.grad(h, args, grad_outputs=dH.to(dev))
    ref_in = [a.float().requires_grad_(True) for a in (x, W_up, b_up, W_gp, b_gp)]
    ref = oracle.hidden_forward(ref_in[0], ref_in[3], ref_in[4], ref_in[1], ref_in[2])["H"]
    ref_grads = torch.autograd.grad(ref, ref_in, grad_outputs=dH.float())
    _close("hidden", h, ref)
    for n, a, b in zip(("dx", "dW_up", "db_up", "dW_gp", "db_gp"), grads, ref_grads):
        _close(n, a, b)


def test_eval_mode_ignores_dropout_and_is_deterministic():
    from triton_gated_mlp import FusedGatedMLP

    dev = _dev()
    torch.manual_seed(3)
    mlp = FusedGatedMLP(256, 512, bias=True, dropout_p=0.5).to(dev).to(torch.bfloat16)
    x = torch.randn(64, 256, device=dev, dtype=torch.bfloat16)
    mlp.eval()
    y0, y1 = mlp(x), mlp(x)
    assert torch.equal(y0, y1)
    mlp.train()
    mlp.dropout_seed = 5
    a = mlp(x)
    mlp._dropout_calls = 0
    b = mlp(x)
    assert torch.equal(a, b), "same seed and offset must give the same mask"
    assert not torch.equal(a, y0)


def test_dropout_mask_matches_numpy_philox_and_rate():
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    for (M, N, p, seed, off) in [(64, 128, 0.1, 1234, 0), (33, 72, 0.5, 2**40 + 17, 3), (1024, 2048, 0.25, 99, 2**33)]:
        got = ops_fwd.dropout_mask(M, N, p, seed, off, device=dev).cpu().numpy()
        ref = philox.keep_mask(M, N, p, seed, off)
        assert np.array_equal(got, ref)
        rate = got.mean()
        sigma = (p * (1 - p) / (M * N)) ** 0.5
        assert abs(rate - (1 - p)) < 5 * sigma + 1e-9


def test_forward_mask_output_equals_standalone_mask():
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(5)
    M, K, N = 300, 128, 520
    x = torch.randn(M, K, generator=g).half().to(dev)
    Wg = (0.05 * torch.randn(N, K, generator=g)).half().to(dev)
    Wu = (0.05 * torch.randn(N, K, generator=g)).half().to(dev)
    hs = ops_fwd.gateup_fwd(x, Wg, None, Wu, None, 0.3, seed=77, offset=1, save_activations=True, return_mask=True)
    ref = philox.keep_mask(M, N, 0.3, 77, 1)
    assert np.array_equal(hs.mask.cpu().numpy(), ref)
    o = oracle.hidden_forward(x.float().cpu(), Wg.float().cpu(), None, Wu.float().cpu(), None, torch.from_numpy(ref), 0.3)
    _close("H", hs.hidden, o["H"])
    _close("G", hs.gate, o["G"])
    _close("U", hs.up, o["U"])


@pytest.mark.parametrize("with_mask", [False, True])
def test_gateup_as_whole_rounds_plus_remaining_columns(with_mask):
    """A grid of large tiles that ends in a thinly filled round of workgroups is launched as two
    column ranges (here 352 tiles on 256 compute units: 32 tile columns, then 12 on small tiles).
    Biases, kept G and U, and the dropout mask must line up across the seam: the mask of an element
    depends on its index in the whole tensor.  With and without the keep-mask output (the two
    epilogue implementations)."""
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(6)
    M, K, N, p = 2048, 64, 5632, 0.3
    x = torch.randn(M, K, generator=g).half().to(dev)
    Wg = (0.1 * torch.randn(N, K, generator=g)).half().to(dev)
    Wu = (0.1 * torch.randn(N, K, generator=g)).half().to(dev)
    bg = (0.1 * torch.randn(N, generator=g)).half().to(dev)
    bu = (0.1 * torch.randn(N, generator=g)).half().to(dev)
    hs = ops_fwd.gateup_fwd(x, Wg, bg, Wu, bu, p, seed=123, offset=2, save_activations=True, return_mask=with_mask)
    ref = philox.keep_mask(M, N, p, 123, 2)
    if with_mask:
        assert np.array_equal(hs.mask.cpu().numpy(), ref)
    f = lambda t: t.float().cpu()
    o = oracle.hidden_forward(f(x), f(Wg), f(bg), f(Wu), f(bu), torch.from_numpy(ref), p)
    _close("H", hs.hidden, o["H"])
    _close("G", hs.gate, o["G"])
    _close("U", hs.up, o["U"])
    # dropped elements are exact zeros, kept ones are not (up to the odd underflow): the mask
    # itself, read off H on both sides of the seam at column 4096
    zero = (hs.hidden == 0).cpu().numpy()
    assert (zero[:, :4096] == (ref[:, :4096] == 0)).mean() > 0.999
    assert (zero[:, 4096:] == (ref[:, 4096:] == 0)).mean() > 0.999


def test_linear_as_whole_rounds_plus_remaining_columns():
    """The same two-launch form for the plain projection: 352 large tiles on 256 compute units,
    bias included; also a shape with exactly one round, which must stay a single launch's result."""
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(8)
    for M, R, C in [(2048, 64, 11264), (2048, 64, 8192)]:
        a = torch.randn(M, R, generator=g).half().to(dev)
        W = (0.1 * torch.randn(C, R, generator=g)).half().to(dev)
        b = (0.1 * torch.randn(C, generator=g)).half().to(dev)
        y = ops_fwd.linear_fwd(a, W, b)
        ref = a.float().cpu() @ W.float().cpu().T + b.float().cpu()
        _close(f"linear {M}x{R}->{C}", y, ref)


def test_backward_gemms_as_whole_rounds_plus_remaining_rows():
    """dH (with the gating-backward epilogue and dropout) and dX with 352 large tiles on 256 compute
    units: launched as 11 tile rows that make a whole round plus the remaining 5 as a problem of
    their own.  G, U, dG, dU and the dropout counters must line up across the seam at row 2816."""
    from triton_gated_mlp.ops import bwd as ops_bwd

    dev = _dev()
    g = torch.Generator().manual_seed(9)
    M, K, N, p = 4096, 64, 5632, 0.25
    dy = torch.randn(M, K, generator=g).half().to(dev)
    Wd = (0.1 * torch.randn(K, N, generator=g)).half().to(dev)
    G = torch.randn(M, N, generator=g).half().to(dev)
    U = torch.randn(M, N, generator=g).half().to(dev)
    dg, du = ops_bwd.dh_bwd(dy, Wd, G, U, p, 321, 4)
    keep = torch.from_numpy(philox.keep_mask(M, N, p, 321, 4))
    f = lambda t: t.float().cpu()
    ref = oracle.hidden_backward(f(dy) @ f(Wd), f(G), f(U), keep, p)
    _close("dG", dg, ref["dG"])
    _close("dU", du, ref["dU"])
    zero = (du == 0).cpu().numpy()
    for rows in (slice(0, 2816), slice(2816, M)):
        assert (zero[rows] == (keep[rows].numpy() == 0)).mean() > 0.999

    M, K, N = 4096, 5632, 64
    dG = torch.randn(M, N, generator=g).half().to(dev)
    dU = torch.randn(M, N, generator=g).half().to(dev)
    Wg = (0.1 * torch.randn(N, K, generator=g)).half().to(dev)
    Wu = (0.1 * torch.randn(N, K, generator=g)).half().to(dev)
    dx = ops_bwd.dx_bwd(dG, dU, Wg, Wu)
    _close("dX", dx, f(dG) @ f(Wg) + f(dU) @ f(Wu))


@pytest.mark.parametrize("band", ["columns", "rows"])
def test_grouped_weight_gradients_with_a_band_of_the_last_problem_on_its_own(band):
    """528 large tiles on 256 compute units: the last problem of the group gives up a band of 16
    tiles (two tile columns, or two tile rows when it is the tall one), which runs as a launch of
    its own through a moved pointer and a trimmed buffer size.  A reduction length that is not a
    multiple of 64 makes the trimmed size matter: reduction rows past the end must read as zero."""
    from triton_gated_mlp.ops import bwd as ops_bwd

    dev = _dev()
    g = torch.Generator().manual_seed(10)
    Mred = 200
    shapes = [(5632, 2048), (5632, 2048), (2048, 5632)] if band == "columns" else [(2048, 5632), (2048, 5632), (5632, 2048)]
    pairs = []
    for R, C in shapes:
        pairs.append((torch.randn(Mred, R, generator=g).half().to(dev), torch.randn(Mred, C, generator=g).half().to(dev)))
    outs = ops_bwd.dw_bwd_grouped(pairs)
    for (lhs, rhs), out in zip(pairs, outs):
        ref = lhs.float().cpu().T @ rhs.float().cpu()
        _close(f"dW {tuple(out.shape)}", out, ref)


def test_full_size_properties_cfg3_linearity_and_zero():
    """Size-independent checks at the headline shape: x = 0 gives Y = 0 (no bias), and the down
    projection is linear in H (Y(2H) = 2Y(H))."""
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    c = CFG3
    g = torch.Generator(device="cpu").manual_seed(1)
    Wd = (0.02 * torch.randn(c.K, c.N, generator=g)).half().to(dev)
    H = torch.randn(c.M, c.N, generator=g).half().to(dev)
    y1 = ops_fwd.linear_fwd(H, Wd)
    y2 = ops_fwd.linear_fwd(H * 2, Wd)
    assert torch.allclose(y2.float(), 2 * y1.float(), rtol=2e-3, atol=2e-3)
    Wg = (0.02 * torch.randn(c.N, c.K, generator=g)).half().to(dev)
    z = ops_fwd.gateup_fwd(torch.zeros(c.M, c.K, dtype=torch.float16, device=dev), Wg, None, Wg, None)
    assert not z.hidden.any()


# ---- float32: the reference's own four tests run in float32 (tests/test_gated_mlp_fwd.py:23-82,
# tests/test_gated_mlp_bwd.py:27-129); same shapes, inputs and tolerances here.


def test_reference_fp32_module_forward():
    from triton_gated_mlp import EagerGatedMLP, FusedGatedMLP, copy_weights

    dev = _dev()
    torch.manual_seed(0)
    eager = EagerGatedMLP(dropout_p=0.0).to(dev).float()  # defaults: K=256, N=512, bias=True
    fused = FusedGatedMLP(dropout_p=0.0).to(dev).float()
    copy_weights(eager, fused)
    x = torch.rand((128, eager.hidden_size), device=dev, dtype=torch.float32)
    y_e, y_f = eager(x), fused(x)
    assert torch.allclose(y_f, y_e, rtol=1e-6, atol=1e-2)  # the reference's effective tolerance
    assert torch.allclose(y_f, y_e, rtol=1e-4, atol=1e-5)  # what fp32 accumulation actually gives
    ref = oracle.forward(x.cpu().double(), *[t.detach().cpu().double() for t in (
        eager.gate_proj.weight, eager.gate_proj.bias, eager.up_proj.weight, eager.up_proj.bias,
        eager.down_proj.weight, eager.down_proj.bias)])["Y"]
    assert torch.allclose(y_f.cpu().double(), ref, rtol=1e-4, atol=1e-5)


def test_reference_fp32_operator_forward():
    from triton_gated_mlp import EagerGatedMLP, eager_fwd, mlp_hidden_states_fwd

    dev = _dev()
    torch.manual_seed(1)
    m = EagerGatedMLP(dropout_p=0.0, bias=False).to(dev).float()
    x = torch.rand((128, m.hidden_size), device=dev)
    ref = eager_fwd(x, m.up_proj.weight, None, m.gate_proj.weight, None)
    out = mlp_hidden_states_fwd(x, m.up_proj.weight, None, m.gate_proj.weight, None, m.act_fn, m.dropout.p)
    assert torch.allclose(out, ref, rtol=1e-4, atol=1e-5)
    # the reference builds this test's module with hidden_act="no_act" (tests/test_gated_mlp_fwd.py:41-82)
    up = torch.nn.functional.linear(x, m.up_proj.weight)
    gate = torch.nn.functional.linear(x, m.gate_proj.weight)
    out = mlp_hidden_states_fwd(x, m.up_proj.weight, None, m.gate_proj.weight, None, "no_act", 0.0)
    assert torch.allclose(out, gate * up, rtol=1e-4, atol=1e-5)


def test_reference_fp32_module_backward_3d_input():
    from triton_gated_mlp import EagerGatedMLP, FusedGatedMLP, copy_weights

    dev = _dev()
    torch.manual_seed(2)
    eager = EagerGatedMLP(dropout_p=0.0, bias=False).to(dev).float()
    fused = FusedGatedMLP(dropout_p=0.0, bias=False).to(dev).float()
    copy_weights(eager, fused)
    x = torch.rand((16, 32, eager.hidden_size), device=dev, requires_grad=True)
    y_e, y_f = eager(x), fused(x)
    assert y_f.shape == x.shape
    assert torch.allclose(y_f, y_e, atol=1e-3)
    go = torch.rand_like(x)
    g_e = torch.autograd.grad(y_e, (x, eager.up_proj.weight, eager.gate_proj.weight, eager.down_proj.weight), grad_outputs=go)
    g_f = torch.autograd.grad(y_f, (x, fused.up_proj.weight, fused.gate_proj.weight, fused.down_proj.weight), grad_outputs=go)
    for a, b in zip(g_f, g_e):
        rel = ((a - b).norm() / b.norm()).item()
        assert rel < 1e-5, rel


def test_reference_fp32_operator_backward():
    from triton_gated_mlp import mlp_hidden_states_bwd

    dev = _dev()
    torch.manual_seed(3)
    B, M, N, K = 2, 32, 512, 256
    kw = dict(device=dev, dtype=torch.float32)
    x = torch.rand((B * M, K), **kw) / K
    W_up, W_gp = torch.rand((N, K), **kw) / K, torch.rand((N, K), **kw) / K
    go = torch.rand((B * M, N), **kw) / K
    a, b = x @ W_up.T, x @ W_gp.T
    sig = torch.sigmoid(b)
    goap = go * a * (sig * (1 + b * (1 - sig)))
    goc = go * torch.nn.functional.silu(b)
    dx, dW_up, dW_gp = mlp_hidden_states_bwd(x, W_up, W_gp, go)
    for got, ref in ((dx, goc @ W_up + goap @ W_gp), (dW_up, goc.T @ x), (dW_gp, goap.T @ x)):
        rel = ((got - ref).norm() / ref.norm()).item()
        assert rel < 1e-5, rel  # the reference asks 1e-7 of its own kernels; fp32 MFMA order differs from BLAS


def test_fp32_bias_dropout_forward_backward_against_oracle():
    _run_module_case(Case("fp32_200x136x264", 200, 136, 264, torch.float32, bias=True, p=0.25, backward=True, seed=5))


def test_empty_and_degenerate_inputs():
    from triton_gated_mlp import FusedGatedMLP

    dev = _dev()
    torch.manual_seed(6)
    mlp = FusedGatedMLP(256, 512, bias=True).to(dev).half()
    # no tokens
    x0 = torch.zeros(0, 256, device=dev, dtype=torch.float16, requires_grad=True)
    y0 = mlp(x0)
    assert y0.shape == (0, 256)
    g = torch.autograd.grad(y0, [x0, mlp.gate_proj.weight, mlp.down_proj.bias], grad_outputs=torch.zeros_like(y0))
    assert g[0].shape == (0, 256) and not g[1].any() and not g[2].any()
    assert mlp(torch.zeros(4, 0, 256, device=dev, dtype=torch.float16)).shape == (4, 0, 256)
    # leading dimensions of one and a single token, with gradients
    x1 = torch.randn(1, 1, 256, device=dev, dtype=torch.float16, requires_grad=True)
    y1 = mlp(x1)
    (gx,) = torch.autograd.grad(y1, [x1], grad_outputs=torch.ones_like(y1))
    f = lambda t: t.detach().float().cpu()
    ref = oracle.backward(f(x1).view(1, 256), f(mlp.gate_proj.weight), f(mlp.gate_proj.bias), f(mlp.up_proj.weight),
                          f(mlp.up_proj.bias), f(mlp.down_proj.weight), f(mlp.down_proj.bias), torch.ones(1, 256))
    _close("Y single token", y1.view(1, 256), ref["Y"])
    _close("dX single token", gx.view(1, 256), ref["dX"])


def test_non_contiguous_inputs_and_partial_gradients():
    from triton_gated_mlp import FusedGatedMLP

    dev = _dev()
    torch.manual_seed(7)
    mlp = FusedGatedMLP(256, 768, bias=False).to(dev).to(torch.bfloat16)
    base = torch.randn(96, 512, device=dev, dtype=torch.bfloat16)
    x_nc = base[:, ::2]  # stride 2 along the feature dimension
    assert not x_nc.is_contiguous()
    y_nc = mlp(x_nc)
    assert torch.equal(y_nc, mlp(x_nc.contiguous()))
    # only the input needs a gradient (weights frozen): no weight-gradient launches, same dX
    x = x_nc.contiguous().requires_grad_(True)
    y = mlp(x)
    dy = torch.randn_like(y)
    (dx_full,) = torch.autograd.grad(y, [x], grad_outputs=dy, retain_graph=True)
    for q in mlp.parameters():
        q.requires_grad_(False)
    (dx_frozen,) = torch.autograd.grad(mlp(x), [x], grad_outputs=dy)
    assert torch.equal(dx_full, dx_frozen)
    # only the weights need a gradient
    for q in mlp.parameters():
        q.requires_grad_(True)
    xw = x.detach()
    gw = torch.autograd.grad(mlp(xw), list(mlp.parameters()), grad_outputs=dy)
    f = lambda t: t.detach().float().cpu()
    ref = oracle.backward(f(xw), f(mlp.gate_proj.weight), None, f(mlp.up_proj.weight), None, f(mlp.down_proj.weight),
                          None, f(dy))
    for n, got in zip(("dW_gate", "dW_up", "dW_down"), gw):
        _close(n, got, ref[n])


def test_many_tokens_tall_shape():
    """M much larger than K and N (65536 tokens): 32-bit index paths and the tile scheduler."""
    _run_module_case(Case("tall_65536x256x512", 65536, 256, 512, torch.float16, bias=False, backward=True, seed=8))


def test_batches_beyond_32bit_offsets_run_as_row_chunks(monkeypatch):
    """A batch whose [M, N] activations exceed the pipelined kernels' 32-bit byte offsets is split
    into row chunks by the module (here the limit is lowered to 512 rows: three chunks, the last one
    ragged); outputs and all gradients, weight gradients summed over the chunks, match the oracle."""
    from triton_gated_mlp.ops import fwd as ops_fwd

    assert ops_fwd.max_rows_32bit(8192, 28672, torch.float16) * 28672 * 2 < 2**31
    monkeypatch.setattr(ops_fwd, "max_rows_32bit", lambda K, N, dtype: 512)
    _run_module_case(Case("chunked_1300x256x640", 1300, 256, 640, torch.float16, bias=True, backward=True, seed=31))
    _run_module_case(Case("chunked_1024x256x640", 1024, 256, 640, torch.bfloat16, bias=False, backward=True, seed=32))
    # with dropout every chunk draws a mask of its own; the oracle rebuilds them from last_dropout_states
    _run_module_case(Case("chunked_1300x256x640_p", 1300, 256, 640, torch.float16, bias=True, p=0.2, backward=True, seed=33))


def test_memory_lean_backward_is_bit_identical():
    """recompute_activations=True (keep x only, as the reference does) gives the same gradients."""
    from triton_gated_mlp import FusedGatedMLP

    dev = _dev()
    torch.manual_seed(4)
    mlp = FusedGatedMLP(512, 1024, bias=True, dropout_p=0.2).to(dev).to(torch.bfloat16).train()
    x = torch.randn(384, 512, device=dev, dtype=torch.bfloat16, requires_grad=True)
    dy = torch.randn(384, 512, device=dev, dtype=torch.bfloat16)
    grads = []
    for lean in (False, True):
        mlp.recompute_activations = lean
        mlp.dropout_seed, mlp._dropout_calls = 77, 0
        y = mlp(x)
        grads.append((y, *torch.autograd.grad(y, [x, *mlp.parameters()], grad_outputs=dy)))
    for a, b in zip(*grads):
        assert torch.equal(a, b)


@pytest.mark.parametrize(
    "case",
    [
        Case("lean_384x512x1024", 384, 512, 1024, torch.bfloat16, bias=True, p=0.2, backward=True, seed=4, dropout_seed=77),
        Case("lean_1000x1024x4104", 1000, 1024, 4104, torch.float16, bias=False, p=0.0, backward=True, seed=5),
        # the size of the bf16 baseline configuration (biases, dropout)
        Case("lean_cfg4", CFG4.M, CFG4.K, CFG4.N, CFG4.dtype, bias=True, p=CFG4.p, backward=True, seed=6),
    ],
    ids=lambda c: c.name,
)
def test_memory_lean_backward_against_oracle(case):
    """recompute_activations=True keeps x only and recomputes G, U, H in backward (what the
    reference does, src/triton_gated_mlp/gated_mlp.py:182, ops/bwd.py:184-193): Y and all seven
    gradients against the oracle, with the Philox mask rebuilt from the recorded seed and offset."""
    _run_module_case(case, lean=True)


def test_benchmark_sweep_reports_both_providers_and_step_memory():
    """The sweep harness (reference: src/triton_gated_mlp/benchmark.py:27-45, 69-123) on two small
    cubes: finite TFLOPS for torch eager and the fused module, and a peak-memory column that is
    the step's own (at least the three [M, N] activations the fused backward keeps, and far from
    the hundreds of MB the process holds besides)."""
    from triton_gated_mlp import benchmark

    dev = _dev()
    perf, mem = benchmark.sweep([256, 512], dev)
    assert [r["N"] for r in perf] == [256, 512] and [r["N"] for r in mem] == [256, 512]
    for rp, rm in zip(perf, mem):
        s = rp["N"]
        for prov in ("torch", "fused"):
            assert np.isfinite(rp[prov]) and rp[prov] > 0.0
            assert rp[prov + "_min"] <= rp[prov] <= rp[prov + "_max"]
            assert rm[prov + "_total"] >= rm[prov] > 0.0
        kept_mb = 3 * s * s * 2 / 1024 / 1024  # G, U, H in fp16
        assert kept_mb <= rm["fused"] < 40 * kept_mb, f"fused step peak {rm['fused']:.2f} MB at {s}"


def _streamk_expected(op, M, K, N, code=0):
    from triton_gated_mlp import _cabi

    return _cabi.lib().gmlp_workspace_bytes(op, M, K, N, code)


def test_streamk_seams_every_gemm_kind_against_fp32_matmul():
    """Grids of large tiles that end in a thinly filled round with a long reduction run their last
    round's tiles as stream-K pieces (several workgroups per tile, fp32 partial sums through the
    workspace, a second launch adds them up in a fixed order).  Every kind of GEMM of the MLP on a
    shape that takes that path (the workspace query says so), against fp32 products of the same
    rounded operands; twice, bit-identical (no dependence on timing)."""
    from triton_gated_mlp import _cabi
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(17)
    rnd = lambda *shape, s=1.0: (s * torch.randn(*shape, generator=g)).half()
    f = lambda t: t.float()

    # down projection: out [2048, 11264] = 352 tiles (1.375 rounds), reduction 5184 = 81 tiles; 96 tiles
    # over 256 workgroups: ranges that straddle tiles (the other cases below cut every tile into a
    # whole number of pieces)
    M, R, C = 2048, 5184, 11264
    assert _streamk_expected(_cabi.GMLP_OP_LINEAR_FWD, M, R, C) == (96 + 256) * 65536 * 4
    a, w, b = rnd(M, R), rnd(C, R, s=0.02), rnd(C, s=0.1)
    y = ops_fwd.linear_fwd(a.to(dev), w.to(dev), b.to(dev))
    assert torch.equal(y, ops_fwd.linear_fwd(a.to(dev), w.to(dev), b.to(dev)))
    _close("linear stream-K", y, f(a) @ f(w).T + f(b))
    # the same call without a workspace (one workgroup per tile throughout): same values up to the
    # order of the fp32 additions in the shared-out tiles
    y0 = torch.empty_like(y)
    ad, wd, bd = a.to(dev), w.to(dev), b.to(dev)
    _cabi.check(_cabi.lib().gmlp_linear_fwd(ad.data_ptr(), wd.data_ptr(), bd.data_ptr(), y0.data_ptr(), M, R, C, 0, None, 0,
                                            _cabi.stream_ptr(dev)))
    torch.cuda.synchronize()
    assert (y.float() - y0.float()).abs().max().item() <= 2e-3 * y0.float().abs().max().item()
    assert not torch.equal(y, torch.zeros_like(y))

    # the same with ragged edges (2000 rows, 11256 columns) in bf16: pieces of edge tiles, predicated sums
    M, R, C = 2000, 5184, 11256
    assert _streamk_expected(_cabi.GMLP_OP_LINEAR_FWD, M, R, C, 1) == (96 + 256) * 65536 * 4
    a, w, b = [v.bfloat16() for v in (rnd(M, R), rnd(C, R, s=0.02), rnd(C, s=0.1))]
    y = ops_fwd.linear_fwd(a.to(dev), w.to(dev), b.to(dev))
    assert torch.equal(y, ops_fwd.linear_fwd(a.to(dev), w.to(dev), b.to(dev)))
    _close("linear stream-K ragged bf16", y, f(a) @ f(w).T + f(b))

    # gate/up: [2048, 5120] hidden = 8 x 40 tiles of 256 x 128, reduction 4352; biases, dropout, G and U kept
    M, K, N = 2048, 4352, 5120
    assert _streamk_expected(_cabi.GMLP_OP_GATEUP_FWD, M, K, N) > 0
    x, wg, wu, bg, bu = rnd(M, K), rnd(N, K, s=0.02), rnd(N, K, s=0.02), rnd(N, s=0.1), rnd(N, s=0.1)
    p, seed = 0.25, 4242
    hs = ops_fwd.gateup_fwd(x.to(dev), wg.to(dev), bg.to(dev), wu.to(dev), bu.to(dev), p, seed, 3, save_activations=True)
    hs2 = ops_fwd.gateup_fwd(x.to(dev), wg.to(dev), bg.to(dev), wu.to(dev), bu.to(dev), p, seed, 3, save_activations=True)
    assert torch.equal(hs.hidden, hs2.hidden) and torch.equal(hs.gate, hs2.gate) and torch.equal(hs.up, hs2.up)
    keep = torch.from_numpy(philox.keep_mask(M, N, p, seed, 3))
    ref = oracle.hidden_forward(f(x), f(wg), f(bg), f(wu), f(bu), keep, p)
    _close("gate/up stream-K H", hs.hidden, ref["H"])
    _close("gate/up stream-K G", hs.gate, ref["G"])
    _close("gate/up stream-K U", hs.up, ref["U"])

    # dH with the gating epilogue: [2048, 10240] = 320 tiles, reduction 4352
    M, K, N = 2048, 4352, 10240
    assert _streamk_expected(_cabi.GMLP_OP_DH_BWD, M, K, N) > 0
    dy, wdn, G, U = rnd(M, K), rnd(K, N, s=0.02), rnd(M, N), rnd(M, N)
    dg, du = ops_bwd.dh_bwd(dy.to(dev), wdn.to(dev), G.to(dev), U.to(dev), p, seed, 5)
    dg2, du2 = ops_bwd.dh_bwd(dy.to(dev), wdn.to(dev), G.to(dev), U.to(dev), p, seed, 5)
    assert torch.equal(dg, dg2) and torch.equal(du, du2)
    keep = torch.from_numpy(philox.keep_mask(M, N, p, seed, 5))
    hb = oracle.hidden_backward(f(dy) @ f(wdn), f(G), f(U), keep, p)
    _close("dH stream-K dG", dg, hb["dG"])
    _close("dH stream-K dU", du, hb["dU"])

    # dX: [2048, 10240] = 320 tiles, two reduction segments of 2176 = 68 tiles together
    M, K, N = 2048, 10240, 2176
    assert _streamk_expected(_cabi.GMLP_OP_DX_BWD, M, K, N) > 0
    dgv, duv, wg, wu = rnd(M, N), rnd(M, N), rnd(N, K, s=0.02), rnd(N, K, s=0.02)
    dx = ops_bwd.dx_bwd(dgv.to(dev), duv.to(dev), wg.to(dev), wu.to(dev))
    assert torch.equal(dx, ops_bwd.dx_bwd(dgv.to(dev), duv.to(dev), wg.to(dev), wu.to(dev)))
    _close("dX stream-K", dx, f(dgv) @ f(wg) + f(duv) @ f(wu))

    # dW, one problem: [10240, 2048] = 320 tiles, reduction over 4360 token rows (not a multiple of 64)
    Mred, R, C = 4360, 10240, 2048
    assert _streamk_expected(_cabi.GMLP_OP_DW_BWD, Mred, R, C) > 0
    lhs, rhs = rnd(Mred, R), rnd(Mred, C)
    dw = ops_bwd.dw_bwd(lhs.to(dev), rhs.to(dev))
    assert torch.equal(dw, ops_bwd.dw_bwd(lhs.to(dev), rhs.to(dev)))
    _close("dW stream-K", dw, f(lhs).T @ f(rhs))

    # dW, grouped: 64 + 64 + 256 = 384 tiles (1.5 rounds); the shared-out tiles are the last 128 of
    # the last problem (reduction of 102 tiles: half a round saved is worth the second launch)
    Mred = 6528
    pairs = [(rnd(Mred, 2048), rnd(Mred, 2048)), (rnd(Mred, 2048), rnd(Mred, 2048)), (rnd(Mred, 4096), rnd(Mred, 4096))]
    dev_pairs = [(a_.to(dev), b_.to(dev)) for a_, b_ in pairs]
    outs = ops_bwd.dw_bwd_grouped(dev_pairs)
    outs2 = ops_bwd.dw_bwd_grouped(dev_pairs)
    for (a_, b_), got, again in zip(pairs, outs, outs2):
        assert torch.equal(got, again)
        _close("dW grouped stream-K", got, f(a_).T @ f(b_))


def test_streamk_pieces_that_straddle_tiles_every_gemm_kind():
    """352 large tiles = one whole round and 96 tiles: 96 does not divide 256, so the shared-out
    tiles go to 256 workgroups as even ranges of (tile, reduction tile) pairs that begin and end
    inside tiles (the multi-piece loop, slot = workgroup + tile, the search for a tile's first
    workgroup in the second stage).  Every kind of GEMM: two accumulator sets (gate/up), the dH
    epilogue with its prefetch, a piece crossing the seam between dX's two reduction segments, both
    operands reduction-strided with a ragged reduction (dW); against fp32 products on the host."""
    from triton_gated_mlp import _cabi
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(23)
    rnd = lambda *shape, s=1.0: (s * torch.randn(*shape, generator=g)).half()
    f = lambda t: t.float()
    straddling = (96 + 256) * 65536 * 4  # slots of a plan without whole pieces per tile

    M, K, N = 2048, 5184, 5632  # gate/up: 8 x 44 tiles of 256 x 128, 81 reduction tiles
    assert _streamk_expected(_cabi.GMLP_OP_GATEUP_FWD, M, K, N) == straddling
    x, wg, wu, bg = rnd(M, K), rnd(N, K, s=0.02), rnd(N, K, s=0.02), rnd(N, s=0.1)
    hs = ops_fwd.gateup_fwd(x.to(dev), wg.to(dev), bg.to(dev), wu.to(dev), None, save_activations=True)
    hs2 = ops_fwd.gateup_fwd(x.to(dev), wg.to(dev), bg.to(dev), wu.to(dev), None, save_activations=True)
    assert torch.equal(hs.hidden, hs2.hidden) and torch.equal(hs.gate, hs2.gate) and torch.equal(hs.up, hs2.up)
    ref = oracle.hidden_forward(f(x), f(wg), f(bg), f(wu), None, None, 0.0)
    _close("gate/up straddling H", hs.hidden, ref["H"])
    _close("gate/up straddling G", hs.gate, ref["G"])
    _close("gate/up straddling U", hs.up, ref["U"])

    M, K, N = 2048, 5184, 11264  # dH: 8 x 44 tiles of 256 x 256
    assert _streamk_expected(_cabi.GMLP_OP_DH_BWD, M, K, N) == straddling
    dy, wdn, G, U = rnd(M, K), rnd(K, N, s=0.02), rnd(M, N), rnd(M, N)
    dg, du = ops_bwd.dh_bwd(dy.to(dev), wdn.to(dev), G.to(dev), U.to(dev))
    dg2, du2 = ops_bwd.dh_bwd(dy.to(dev), wdn.to(dev), G.to(dev), U.to(dev))
    assert torch.equal(dg, dg2) and torch.equal(du, du2)
    hb = oracle.hidden_backward(f(dy) @ f(wdn), f(G), f(U), None, 0.0)
    _close("dH straddling dG", dg, hb["dG"])
    _close("dH straddling dU", du, hb["dU"])

    M, K, N = 2048, 11264, 2624  # dX: two segments of 41 reduction tiles; pieces of 30-31 cross the seam
    assert _streamk_expected(_cabi.GMLP_OP_DX_BWD, M, K, N) == straddling
    dgv, duv, wg, wu = rnd(M, N), rnd(M, N), rnd(N, K, s=0.02), rnd(N, K, s=0.02)
    dx = ops_bwd.dx_bwd(dgv.to(dev), duv.to(dev), wg.to(dev), wu.to(dev))
    assert torch.equal(dx, ops_bwd.dx_bwd(dgv.to(dev), duv.to(dev), wg.to(dev), wu.to(dev)))
    _close("dX straddling", dx, f(dgv) @ f(wg) + f(duv) @ f(wu))

    Mred, R, C = 5192, 2048, 11264  # dW: 82 reduction tiles, the last one of 8 rows
    assert _streamk_expected(_cabi.GMLP_OP_DW_BWD, Mred, R, C) == straddling
    lhs, rhs = rnd(Mred, R), rnd(Mred, C)
    dw = ops_bwd.dw_bwd(lhs.to(dev), rhs.to(dev))
    assert torch.equal(dw, ops_bwd.dw_bwd(lhs.to(dev), rhs.to(dev)))
    _close("dW straddling", dw, f(lhs).T @ f(rhs))


def test_grouped_launch_of_one_problem_whose_tiles_all_go_to_streamk():
    """A single weight gradient of 200 large tiles with a long reduction: fewer tiles than compute
    units, so the plan shares out every tile and the grouped launch has no whole-tile grid left to
    run (which must not be launched empty).  Against the fp32 product and gmlp_dw_bwd."""
    import ctypes

    from triton_gated_mlp import _cabi
    from triton_gated_mlp.ops import bwd as ops_bwd

    dev = _dev()
    Mred, R, C = 16384, 2560, 5120
    RC = (ctypes.c_int64 * 1)
    nbytes = _cabi.lib().gmlp_dw_bwd_grouped_workspace_bytes(
        1, Mred, ctypes.cast(RC(R), ctypes.c_void_p), ctypes.cast(RC(C), ctypes.c_void_p), 0)
    assert nbytes == (200 + 256) * 65536 * 4  # all 200 tiles shared out over 256 workgroups
    g = torch.Generator().manual_seed(29)
    lhs = torch.randn(Mred, R, generator=g).half()
    rhs = torch.randn(Mred, C, generator=g).half()
    (grouped,) = ops_bwd.dw_bwd_grouped([(lhs.to(dev), rhs.to(dev))])
    single = ops_bwd.dw_bwd(lhs.to(dev), rhs.to(dev))
    torch.cuda.synchronize()
    assert torch.equal(grouped, single)
    _close("dW, one problem, all tiles as pieces", grouped, lhs.float().T @ rhs.float())


@pytest.mark.parametrize(
    "M,K,N,dtype,bias,p",
    [
        (2048, 2048, 5632, torch.bfloat16, True, 0.1),   # mid-size grids, biases, dropout
        (300, 1024, 4096, torch.float16, True, 0.0),     # short batch: split reductions, ragged rows
        (2048, 4352, 5120, torch.float16, False, 0.25),  # stream-K in the forward GEMMs
        (1000, 520, 1048, torch.bfloat16, True, 0.0),    # widths that are multiples of 8 only (predicated kernels)
        (192, 512, 768, torch.float32, True, 0.1),       # float32 path
    ],
)
def test_whole_pass_entry_points_equal_the_separate_launches(M, K, N, dtype, bias, p):
    """gmlp_mlp_fwd and gmlp_mlp_bwd (one library call per pass; what the module uses) give, bit for
    bit, what the per-GEMM entry points give when called one after the other, call after call, and
    leave out exactly the gradients that were not asked for.  (The separate entry
    points are the ones held against the oracle throughout this file; the module-level cases go
    through the one-call entries and are held against the oracle as well.)"""
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(31)
    rnd = lambda *shape, s=1.0: (s * torch.randn(*shape, generator=g)).to(dtype).to(dev)
    x, wg, wu, wd, dy = rnd(M, K), rnd(N, K, s=0.03), rnd(N, K, s=0.03), rnd(K, N, s=0.03), rnd(M, K)
    bg, bu, bd = (rnd(N, s=0.1), rnd(N, s=0.1), rnd(K, s=0.1)) if bias else (None, None, None)
    seed, off = 77, 2
    hs = ops_fwd.gateup_fwd(x, wg, bg, wu, bu, p, seed, off, save_activations=True)
    y_ref = ops_fwd.linear_fwd(hs.hidden, wd, bd)
    y, hs1 = ops_fwd.mlp_fwd(x, wg, bg, wu, bu, wd, bd, p, seed, off, save_activations=True)
    assert torch.equal(y, y_ref) and torch.equal(hs1.hidden, hs.hidden)
    assert torch.equal(hs1.gate, hs.gate) and torch.equal(hs1.up, hs.up)
    y2, hs2 = ops_fwd.mlp_fwd(x, wg, bg, wu, bu, wd, bd, p, seed, off, save_activations=False)
    assert torch.equal(y2, y_ref) and hs2.gate is None and hs2.up is None

    dg, du = ops_bwd.dh_bwd(dy, wd, hs.gate, hs.up, p, seed, off)
    ref = {
        "dx": ops_bwd.dx_bwd(dg, du, wg, wu),
        "dW_gate": None, "db_gate": None, "dW_up": None, "db_up": None, "dW_down": None, "db_down": None,
    }
    ref["dW_gate"], ref["dW_up"], ref["dW_down"] = ops_bwd.dw_bwd_grouped([(dg, x), (du, x), (dy, hs.hidden)])
    if bias:
        ref["db_gate"], ref["db_up"], ref["db_down"] = ops_bwd.colsum_grouped([dg, du, dy])
    names = list(ref)
    all_of = tuple(ref[n] is not None for n in names)
    for call in range(2):
        got = ops_bwd.mlp_bwd(dy, x, wg, wu, wd, hs.gate, hs.up, hs.hidden, all_of, p, seed, off)
        torch.cuda.synchronize()
        for n, a, b in zip(names, got, (ref[n] for n in names)):
            assert (a is None) == (b is None), n
            assert a is None or torch.equal(a, b), f"{n} differs (call {call})"
    # subsets: only the input gradient; only the down projection's gradients; everything but dX
    for want in ((True,) + (False,) * 6, (False,) * 5 + (True, bias), (False,) + all_of[1:]):
        got = ops_bwd.mlp_bwd(dy, x, wg, wu, wd, hs.gate, hs.up, hs.hidden, want, p, seed, off)
        torch.cuda.synchronize()
        for n, w, a in zip(names, want, got):
            assert (a is not None) == bool(w), n
            assert a is None or torch.equal(a, ref[n]), f"{n} differs for subset {want}"


def _launched(run):
    """Names of the kernels that run() launches, and its result."""
    from torch.profiler import ProfilerActivity, profile

    run()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as prof:
        result = run()
        torch.cuda.synchronize()
    return [e.name for e in prof.events() if "gmlp" in e.name], result


# dX beside the weight gradients in one grid: rows of a dX tile and of a weight gradient's, whether dX and whether the
# weight gradients are split, or None for a dX of its own (shared-out tiles, or one grid takes longer by
# estimate); then the weight gradients' tile where they are a grid with the bias gradients when dX is not in it.  16-bit types,
# then float32; on a whole MI355X.  Single tiles, remainders in every direction, few rows, many.  Lengths that are not a
# multiple of the 64 of a reduction tile have instances of their own (N, the reduction of dX).
_GRADIENT_GRIDS = [
    # M, K, N, 16-bit, without dX, float32, without dX
    (1, 8, 8, (128, 128, 0, 0), 128, (64, 64, 0, 0), 64),
    (129, 136, 264, (128, 128, 0, 0), 128, (64, 64, 1, 0), 64),
    (33, 512, 1528, (128, 128, 1, 0), 128, (64, 64, 1, 0), 64),
    (512, 512, 1536, (128, 128, 1, 0), 128, (64, 64, 1, 0), 64),
    (1024, 1024, 2816, (256, 256, 1, 0), 256, None, 128),
    (1000, 1024, 2824, (128, 256, 1, 0), 256, None, 128),
    (3000, 1536, 4096, (192, 256, 0, 0), None, None, None),
    (2999, 1528, 4104, (192, 256, 0, 0), None, (128, 128, 1, 0), 128),
    (384, 1984, 5440, (128, 256, 1, 0), 128, (128, 128, 1, 0), 128),
    (271, 2456, 6600, (128, 256, 1, 0), 128, (128, 128, 1, 0), 128),
    (6656, 1472, 1472, (192, 256, 0, 0), 128, (128, 128, 1, 1), None),
    (3456, 384, 1536, (128, 128, 1, 1), None, (128, 128, 1, 1), None),
    (842, 5032, 13520, None, 256, (128, 128, 1, 0), 128),
    (884, 3376, 448, (256, 256, 0, 0), 128, None, 64),
    (896, 3496, 392, (256, 256, 0, 0), 128, None, 64),
    (1022, 136, 6768, (256, 256, 1, 0), 128, None, 64),
    (387, 3968, 576, (128, 256, 0, 0), 128, (128, 128, 1, 0), 128),
    (513, 2240, 856, (128, 256, 0, 0), 128, (128, 128, 1, 0), 128),
    (710, 72, 488, (128, 128, 1, 1), None, (64, 64, 1, 1), None),
    (2381, 240, 128, (128, 128, 0, 1), None, (64, 64, 0, 1), None),
    (1281, 136, 72, (128, 128, 0, 1), None, (64, 64, 0, 1), None),
    (565, 48, 64, (128, 128, 0, 0), 128, (64, 64, 0, 1), None),
    (1632, 720, 72, (128, 128, 0, 1), None, (128, 128, 0, 1), None),
    (442, 3080, 136, (128, 128, 0, 0), 128, (128, 128, 0, 0), 64),
    (590, 352, 544, (128, 128, 1, 0), 128, (64, 64, 1, 0), 64),
    (2902, 2816, 3584, (256, 256, 0, 0), 256, None, 128),
]


def _gradient_grid(names):
    """(dX rows, weight gradient rows, dX split, weight gradients split) of the grid among launched kernels, or None."""
    import re

    # (names come mangled, where a repeated type is a back reference, or, float32's, demangled)
    found = [re.search(r"dx_dw_kernel(.*?)DxDwGroup", n) for n in names if "dx_dw_kernel" in n]
    assert len(found) <= 1 and all(found), names
    if not found:
        return None
    tiles = [int(t) for t in re.findall(r"(?:Li|<|, )(\d+)(?=E|,)", found[0][1])]
    stored = re.findall("EpiStore|EpiPartial", found[0][1])
    return tiles[0], tiles[-1], int(stored[0] == "EpiPartial"), int(stored[-1] == "EpiPartial")


def test_gradient_grid_cases_cover_every_instance():
    both = [(False, False), (True, False), (False, True), (True, True)]
    large = [(t, 256, x, False) for t in (128, 192, 256) for x in (False, True) if not (t == 192 and x)]
    half = large + [(128, 128, *splits) for splits in both]
    assert {(grid, N % 64 != 0) for _, _, N, grid, *_ in _GRADIENT_GRIDS if grid} == {(g, t) for g in half for t in (False, True)}
    assert {grid for *_, grid, _ in _GRADIENT_GRIDS if grid} == {(t, t, *splits) for t in (64, 128) for splits in both}
    assert {(w, full) for _, _, _, _, w, _, full in _GRADIENT_GRIDS} >= {(128, 64), (256, 128), (None, None)}


@pytest.mark.parametrize("M,K,N,half,half_w,full,full_w", _GRADIENT_GRIDS, ids=lambda v: str(v) if isinstance(v, int) else "")
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_input_and_weight_gradients_in_one_grid(M, K, N, half, half_w, full, full_w, dtype):
    """gmlp_mlp_bwd may run dX, whichever weight gradients are wanted and the bias gradients as one grid: the same sums in
    the same order as the entry points of their own (held against the oracle elsewhere), hence equal bit for bit.  Which
    grid ran, with every gradient and without dX, by the launched kernels' names."""
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    g = torch.Generator(device=_dev()).manual_seed(M + N)
    rnd = lambda *shape, s=1.0: (s * torch.randn(*shape, generator=g, device=_dev())).to(dtype)
    x, wg, wu, wd, dy = rnd(M, K), rnd(N, K, s=0.03), rnd(N, K, s=0.03), rnd(K, N, s=0.03), rnd(M, K)
    gate, up, hidden = rnd(M, N), rnd(M, N), rnd(M, N)
    dg, du = ops_bwd.dh_bwd(dy, wd, gate, up)
    dx = ops_bwd.dx_bwd(dg, du, wg, wu)
    pairs = [(dg, x), (du, x), (dy, hidden)]
    for want_dx, wanted, biases in ((1, (1, 1, 1), 1), (1, (1, 0, 0), 0), (1, (0, 1, 1), 1), (1, (0, 0, 1), 0), (0, (1, 1, 1), 1)):
        dws = iter(ops_bwd.dw_bwd_grouped([p for p, w in zip(pairs, wanted) if w]))
        dbs = iter(ops_bwd.colsum_grouped([p[0] for p, w in zip(pairs, wanted) if w]) if biases else ())
        need = (bool(want_dx), *(bool(w and (i == 0 or biases)) for w in wanted for i in (0, 1)))
        if all(wanted) and biases and torch.cuda.get_device_properties(dy.device).multi_processor_count == 256:
            names, got = _launched(lambda: ops_bwd.mlp_bwd(dy, x, wg, wu, wd, gate, up, hidden, need))
            alone = full_w if dtype == torch.float32 else half_w
            grid = (full if dtype == torch.float32 else half) if want_dx else None
            expected = grid or (alone and (alone, alone, 0, 0))  # (dX by itself: the bias gradients join the weights')
            assert _gradient_grid(names) == expected, names
        else:
            got = ops_bwd.mlp_bwd(dy, x, wg, wu, wd, gate, up, hidden, need)
        assert torch.equal(got[0], dx) if want_dx else got[0] is None, f"dX differs beside {wanted}"
        for w, a, b in zip(wanted, got[1::2], got[2::2]):
            assert torch.equal(a, next(dws)) if w else a is None, f"a weight gradient differs for {wanted}"
            assert torch.equal(b, next(dbs)) if w and biases else b is None, f"a bias gradient differs for {wanted}"
    # ... and the hidden-state operator's backward, whose grid has no down projection
    from triton_gated_mlp import FusedGatedMLPFunction

    leaves = [t.detach().clone().requires_grad_(True) for t in (x, wu, rnd(N), wg, rnd(N))]
    grad = rnd(M, N)
    FusedGatedMLPFunction.apply(*leaves).backward(grad)
    hs = ops_fwd.gateup_fwd(x, wg, leaves[4].detach(), wu, leaves[2].detach(), save_activations=True)
    dg, du = ops_bwd.gating_bwd(grad, hs.gate, hs.up)
    dwu, dwg = ops_bwd.dw_bwd_grouped([(du, x), (dg, x)])
    dbu, dbg = ops_bwd.colsum_grouped([du, dg])
    for t, want in zip(leaves, (ops_bwd.dx_bwd(dg, du, wg, wu), dwu, dbu, dwg, dbg)):
        assert torch.equal(t.grad, want)
    torch.cuda.synchronize()


@pytest.mark.parametrize("M,K,N,dtype", [(710, 72, 488, torch.float16), (33, 512, 1528, torch.bfloat16), (590, 352, 544, torch.float32)])
def test_hidden_backward_entry_with_any_outputs_and_workspace(M, K, N, dtype):
    """gmlp_hidden_bwd for every set of gradients with all of its workspace, part of it and (without bias gradients)
    none: the values of the separate calls with the same workspace, nothing written beyond it."""
    import ctypes

    from triton_gated_mlp import _cabi

    dev, lib, code = _dev(), _cabi.lib(), _cabi.dtype_code(dtype)
    g = torch.Generator(device=dev).manual_seed(31)
    rnd = lambda *shape: torch.empty(shape, device=dev).normal_(generator=g).to(dtype)
    dh, x, wg, wu, gate, up = rnd(M, N), rnd(M, K), rnd(N, K), rnd(N, K), rnd(M, N), rnd(M, N)
    dg, du, dg_ref, du_ref = (torch.empty_like(dh) for _ in range(4))
    stream, p, act = _cabi.stream_ptr(dev), _cabi.ptr, _cabi.act_code("gelu")
    flags = (_cabi.GMLP_GRAD_X, _cabi.GMLP_GRAD_W_GATE, _cabi.GMLP_GRAD_W_UP, _cabi.GMLP_GRAD_B_GATE, _cabi.GMLP_GRAD_B_UP)
    sizes = ((M, K), (N, K), (N, K), (N,), (N,))
    new = lambda size: torch.full(size, float("nan"), device=dev, dtype=dtype)
    _cabi.check(lib.gmlp_gating_bwd(p(dh), p(gate), p(up), p(dg_ref), p(du_ref), M, N, code, act, 0.1, 5, 7, stream))

    def apart(want, ws, nbytes):
        """The same by the entry points of their own."""
        outs = [new(size) if w else None for size, w in zip(sizes, want)]
        if want[0]:
            _cabi.check(lib.gmlp_dx_bwd(p(dg_ref), p(du_ref), p(wg), p(wu), p(outs[0]), M, K, N, code, ws, nbytes, stream))
        chosen = [(d, o) for d, o in ((dg_ref, outs[1]), (du_ref, outs[2])) if o is not None]
        if chosen:
            array = lambda kind, values: ctypes.cast((kind * len(values))(*values), ctypes.c_void_p)
            lhs, rhs, dws = (array(ctypes.c_void_p, v) for v in zip(*[(p(d), p(x), p(o)) for d, o in chosen]))
            R, C = array(ctypes.c_int64, [N] * len(chosen)), array(ctypes.c_int64, [K] * len(chosen))
            _cabi.check(lib.gmlp_dw_bwd_grouped(len(chosen), lhs, rhs, dws, M, R, C, code, ws, nbytes, stream))
        for d, o in ((dg_ref, outs[3]), (du_ref, outs[4])):
            if o is not None:
                _cabi.check(lib.gmlp_colsum(p(d), p(o), ws, M, N, code, stream))
        return outs

    for subset in range(32):
        want = [subset >> i & 1 for i in range(5)]
        grads = sum(f for f, w in zip(flags, want) if w)
        need = lib.gmlp_grads_workspace_bytes(_cabi.GMLP_PASS_HIDDEN_BWD, grads, M, K, N, code)
        least = (want[3] + want[4]) * lib.gmlp_workspace_bytes(_cabi.GMLP_OP_COLSUM, M, 0, N, code)
        for nbytes in sorted({need, max(need // 2 // 16 * 16, least), least}):
            buffer = torch.full((need + 4096,), 0xA5, device=dev, dtype=torch.uint8)
            scratch = torch.empty(need + 16, device=dev, dtype=torch.uint8)
            outs = [new(size) if w else None for size, w in zip(sizes, want)]
            _cabi.check(lib.gmlp_hidden_bwd(
                p(dh), p(x) if want[1] or want[2] else None, *((p(wg), p(wu)) if want[0] else (None, None)), p(gate), p(up), p(dg), p(du),
                *(p(o) for o in outs), M, K, N, code, act, 0.1, 5, 7, p(buffer) if nbytes else None, nbytes, stream))
            ref = apart(want, p(scratch) if nbytes else None, nbytes)
            assert torch.equal(dg, dg_ref) and torch.equal(du, du_ref)
            for i, (a, b) in enumerate(zip(outs, ref)):
                assert a is None or torch.equal(a, b), (want, nbytes, i)
            assert (buffer[nbytes:] == 0xA5).all(), (want, nbytes)


@pytest.mark.parametrize(
    "M,K,N,dtype,apart",  # rows on both sides of the line; few tiles that all start at once, many, and float32
    [(8192, 200, 600, torch.bfloat16, False), (65536, 200, 600, torch.bfloat16, True), (16384, 40, 56, torch.float16, False),
     (43686, 264, 296, torch.float16, True), (8192, 64, 128, torch.float32, False), (82604, 176, 184, torch.float32, True)],
)
def test_bias_gradients_of_long_batches_leave_the_gradients_grid(M, K, N, dtype, apart):
    """A workgroup of the gradients' grid sums all rows of its columns: behind tiles that take less time, launches of their
    own are faster.  Same sums either way, which path by the launched kernels (on a whole MI355X)."""
    from triton_gated_mlp.ops import bwd as ops_bwd

    dev = _dev()
    g = torch.Generator(device=dev).manual_seed(M + N)
    rnd = lambda *shape: torch.empty(shape, device=dev).normal_(generator=g).mul_(0.1).to(dtype)
    dy, x, wg, wu, wd, gate, up, hidden = (rnd(M, K), rnd(M, K), rnd(N, K), rnd(N, K), rnd(K, N), rnd(M, N), rnd(M, N), rnd(M, N))
    names, got = _launched(lambda: ops_bwd.mlp_bwd(dy, x, wg, wu, wd, gate, up, hidden))
    dg, du = ops_bwd.dh_bwd(dy, wd, gate, up)
    for i, db in zip((2, 4, 6), ops_bwd.colsum_grouped([dg, du, dy])):
        assert torch.equal(got[i], db)
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert any("dx_dw_kernel" in n for n in names), names
        assert any("colsum" in n for n in names) == apart, names


def test_random_shapes_every_operator_against_fp32_products():
    """Two dozen seeded random shapes through the five GEMM operators: token counts from 1 to a few
    thousand, widths that are multiples of 64 (tuned kernels: large, medium, two-launch, split and
    stream-K grids as the dispatcher picks them) or only of 8 (predicated kernel), both 16-bit
    dtypes; each result against the fp32 product of the same rounded operands, computed on the host,
    and the gate/up and dH epilogues against the oracle's closed forms."""
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    rng = np.random.default_rng(20240611)
    g = torch.Generator(device="cpu").manual_seed(99)
    f = lambda t: t.float().cpu()
    for case in range(24):
        dtype = torch.float16 if case % 2 == 0 else torch.bfloat16
        unit = 8 if case % 6 == 5 else 64
        M = int(rng.choice([1, 7, 33, 100, 255, 256, 257, 700, 1500, 2304, 3000]))
        K = int(rng.integers(1, 3072 // unit + 1)) * unit
        N = int(rng.integers(1, 4096 // unit + 1)) * unit
        print(f"random case {case}: M={M} K={K} N={N} {dtype}", flush=True)
        rnd = lambda *shape, s=1.0: (s * torch.randn(*shape, generator=g)).to(dtype).to(dev)
        x, wg, wu, wd = rnd(M, K), rnd(N, K, s=0.03), rnd(N, K, s=0.03), rnd(K, N, s=0.03)
        dy = rnd(M, K)
        # forward
        hs = ops_fwd.gateup_fwd(x, wg, None, wu, None, save_activations=True)
        G, U = f(x) @ f(wg).T, f(x) @ f(wu).T
        _close("G", hs.gate, G)
        _close("U", hs.up, U)
        _close("H", hs.hidden, torch.nn.functional.silu(G) * U)
        y = ops_fwd.linear_fwd(hs.hidden, wd)
        _close("Y", y, f(hs.hidden) @ f(wd).T)
        # backward, from the device's own (rounded) G, U and H so that every operator is checked alone
        dg, du = ops_bwd.dh_bwd(dy, wd, hs.gate, hs.up)
        hb = oracle.hidden_backward(f(dy) @ f(wd), f(hs.gate), f(hs.up), None, 0.0)
        _close("dG", dg, hb["dG"])
        _close("dU", du, hb["dU"])
        dx = ops_bwd.dx_bwd(dg, du, wg, wu)
        ref_dx = f(dg) @ f(wg) + f(du) @ f(wu)
        _close("dX", dx, ref_dx)
        pairs = [(dg, x), (du, x), (dy, hs.hidden)]
        for name, got, (a_, b_) in zip(("dW_gate", "dW_up", "dW_down"), ops_bwd.dw_bwd_grouped(pairs), pairs):
            ref = f(a_).T @ f(b_)
            _close(name, got, ref)
        _close("dW_gate alone", ops_bwd.dw_bwd(dg, x), f(dg).T @ f(x))


@pytest.mark.parametrize(
    "M,K,N",
    [
        (32, 32, 32),        # one partial reduction tile in every GEMM
        (1, 8, 8),           # a single chunk of it
        (257, 120, 136),     # one whole tile and all but one chunk of the next; one chunk of a third
        (130, 1096, 2056),   # split reductions (several workgroups per tile), rotated start
        (4500, 3272, 3400),  # large tiles, thin last round: stream-K or two launches
    ],
)
def test_reduction_tails_every_operator_against_fp32_products(M, K, N):
    """Reduction lengths that end inside a 64-wide reduction tile.  What the tail of a row would alias
    if it were not cut off is the start of the next row, so every row of the left operand starts with
    8 elements 64 times the usual size: one aliased chunk is far outside the tolerance, whatever the
    other operand holds there."""
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    print(f"reduction tails: M={M} K={K} N={N}", flush=True)
    g = torch.Generator().manual_seed(5)
    rnd = lambda *shape, s=1.0: s * torch.randn(*shape, generator=g)

    def heavy(t):
        t[:, :8] *= 64.0
        return t.half().to(dev)

    f = lambda t: t.float().cpu()
    x, dy, h = heavy(rnd(M, K, s=0.1)), heavy(rnd(M, K, s=0.1)), heavy(rnd(M, N, s=0.1))
    dg, du = heavy(rnd(M, N, s=0.1)), heavy(rnd(M, N, s=0.1))
    wg, wu, wd = (rnd(*s, s=0.03).half().to(dev) for s in ((N, K), (N, K), (K, N)))
    hs = ops_fwd.gateup_fwd(x, wg, None, wu, None, save_activations=True)
    _close("G", hs.gate, f(x) @ f(wg).T)
    _close("U", hs.up, f(x) @ f(wu).T)
    _close("Y", ops_fwd.linear_fwd(h, wd), f(h) @ f(wd).T)
    ones = torch.ones_like(hs.up)
    du_got = ops_bwd.dh_bwd(dy, wd, ones, ones, act_fn="no_act")[1]  # dU = dH
    _close("dH", du_got, f(dy) @ f(wd))
    _close("dX", ops_bwd.dx_bwd(dg, du, wg, wu), f(dg) @ f(wg) + f(du) @ f(wu))


@pytest.mark.parametrize(
    "M,K,N",
    [
        (129, 4096, 14344),  # 128x256 tiles: one row beyond a tile, ragged columns; 8 to 16 splits
        (200, 4104, 8200),   # the same with reduction tails
        (1030, 2056, 5640),  # several rows of them, splits that end inside a tile
        (3000, 256, 520),    # weight gradients with a split reduction (few tiles, many tokens)
        (2500, 136, 72),     # the same, single tiles, ragged last split
        (1345, 2264, 8120),  # 192-row tiles: gate/up and dH, one row beyond a tile, reduction tails
        (2048, 2048, 5640),  # the same without tails, 10.7 tile rows, ragged columns
        (5717, 1640, 6432),  # down and dX
    ],
)
def test_wide_tiles_and_split_gradients_against_fp32_products(M, K, N):
    """Grids that the planner gives to the 128x256 tiles (three ring entries of both operands), and split
    reductions of dH and of the grouped weight gradients; twice, bit-identical."""
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    print(f"wide tiles, split gradients: M={M} K={K} N={N}", flush=True)
    g = torch.Generator().manual_seed(8)
    rnd = lambda *shape, s=1.0: (s * torch.randn(*shape, generator=g)).bfloat16().to(dev)
    f = lambda t: t.float()  # products in fp32 on the device: plain 2-D torch matmuls
    x, dy, h, G, U = rnd(M, K), rnd(M, K), rnd(M, N), rnd(M, N), rnd(M, N)
    wg, wu, wd = rnd(N, K, s=0.03), rnd(N, K, s=0.03), rnd(K, N, s=0.03)

    def run():
        hs = ops_fwd.gateup_fwd(x, wg, None, wu, None, save_activations=True)
        dg, du = ops_bwd.dh_bwd(dy, wd, G, U)
        return [hs.gate, hs.up, ops_fwd.linear_fwd(h, wd), dg, du, ops_bwd.dx_bwd(G, U, wg, wu),
                *ops_bwd.dw_bwd_grouped([(G, x), (U, x), (dy, h)])]

    got = run()
    hb = oracle.hidden_backward(f(dy) @ f(wd), f(G), f(U), None, 0.0)
    refs = [f(x) @ f(wg).T, f(x) @ f(wu).T, f(h) @ f(wd).T, hb["dG"], hb["dU"], f(G) @ f(wg) + f(U) @ f(wu),
            f(G).T @ f(x), f(U).T @ f(x), f(dy).T @ f(h)]
    for name, a, b in zip(("G", "U", "Y", "dG", "dU", "dX", "dW_gate", "dW_up", "dW_down"), got, refs):
        _close(name, a, b)
    assert all(torch.equal(a, b) for a, b in zip(got, run()))


# The GEMMs with long epilogues: output tile (gate/up: of each accumulator set) and wavefronts of gate/up with SiLU, with
# another activation, and of dH; on a whole MI355X.
_LONG_EPILOGUES = [
    # M, K, N, gate/up SiLU, gate/up GELU, dH
    (200, 3080, 14344, (128, 128, 8), (128, 128, 8), (128, 128, 4)),  # reduction tails, a row tile of 72, ragged columns
    (200, 3072, 14344, (128, 128, 8), (128, 128, 8), (128, 128, 4)),
    (1000, 3080, 8192, (256, 128, 4), (256, 128, 4), (128, 256, 8)),  # dH: a row tile of 104, reduction tails
    (1000, 3072, 8192, (256, 128, 4), (256, 128, 4), (128, 256, 8)),
    (893, 712, 5112, (192, 128, 8), (192, 128, 8), (128, 128, 4)),    # 12 reduction tiles; three loads of A a wavefront
    (900, 960, 4104, (192, 128, 8), (192, 128, 8), (128, 128, 4)),    # 15
    (900, 968, 4104, (192, 128, 4), (192, 128, 8), (128, 128, 4)),    # 16: SiLU's epilogue no longer outweighs the loop
    (900, 1536, 4104, (192, 128, 4), (192, 128, 8), (128, 128, 4)),   # 24
    (900, 1984, 4104, (192, 128, 4), (192, 128, 8), (128, 128, 4)),   # 31
    (900, 1992, 4104, (192, 128, 4), (192, 128, 4), (128, 128, 4)),   # 32: nor does GELU's
    (900, 2048, 4104, (192, 128, 4), (192, 128, 4), (128, 128, 4)),
    (1289, 464, 6344, (128, 64, 4), (128, 64, 4), (192, 256, 4)),     # dH: three ring entries of A
    (391, 64, 136, (128, 64, 4), (128, 64, 4), (128, 128, 4)),        # one reduction tile: the loop in place does not run
]


@pytest.mark.parametrize("M,K,N,silu,gelu,dh", _LONG_EPILOGUES, ids=lambda v: str(v) if isinstance(v, int) else "")
@pytest.mark.parametrize("act", ["silu", "gelu"])  # epilogue in the accumulators' layout and behind the transpose
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gate_up_and_dh_tiles_and_wavefronts_against_fp32_products(M, K, N, silu, gelu, dh, act, dtype):
    """Every output of the two GEMMs with long epilogues, biases and dropout on; twice, bit-identical; with the launched
    kernels' tiles and wavefronts."""
    import re

    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    print(f"long epilogues: M={M} K={K} N={N} {act} {dtype}", flush=True)
    g = torch.Generator().manual_seed(21)
    rnd = lambda *shape, s=1.0: (s * torch.randn(*shape, generator=g)).to(dtype).to(dev)
    f = lambda t: t.float()
    x, dy, G, U = rnd(M, K), rnd(M, K), rnd(M, N), rnd(M, N)
    wg, wu, wd, bg, bu = rnd(N, K, s=0.03), rnd(N, K, s=0.03), rnd(K, N, s=0.03), rnd(N, s=0.1), rnd(N, s=0.1)

    def run():
        hs = ops_fwd.gateup_fwd(x, wg, bg, wu, bu, dropout_p=0.1, seed=5, save_activations=True, act_fn=act)
        return [hs.hidden, hs.gate, hs.up, *ops_bwd.dh_bwd(dy, wd, G, U, dropout_p=0.1, seed=5, act_fn=act)]

    names, got = _launched(run)
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        # tile rows, tile columns, (MFMA shape), wavefronts below and beside each other
        numbers = r"gemm_kernel_pipelined.*?" + r"(?:Li|, )(\d+)E?" * 5
        found = [tuple(map(int, m.groups())) for m in (re.search(numbers, n) for n in names) if m]
        launched = [(rows, cols, down * beside) for rows, cols, _, down, beside in found]
        assert launched == [silu if act == "silu" else gelu, dh], names
    keep = torch.from_numpy(philox.keep_mask(M, N, 0.1, 5, 0)).to(dev)
    gate, up = f(x) @ f(wg).T + f(bg), f(x) @ f(wu).T + f(bu)
    hb = oracle.hidden_backward(f(dy) @ f(wd), f(G), f(U), keep, 0.1, act)
    refs = [oracle.ACTS[act][0](gate) * up * keep.float() / 0.9, gate, up, hb["dG"], hb["dU"]]
    for name, a, b in zip(("H", "G", "U", "dG", "dU"), got, refs):
        _close(name, a, b)
    assert all(torch.equal(a, b) for a, b in zip(got, run()))


def test_second_stages_against_float64():
    """Sums of 2 to 16 partial results (every remainder of the groups that are in flight together) and
    column sums at the edges of their row ranges and of a workgroup's 256 columns.  fp16 results of
    float32 sums: half an ulp, 2^-11, beside the sums' own rounding."""
    from triton_gated_mlp import _cabi
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(12)
    rnd = lambda *shape: torch.randn(*shape, generator=g).half().to(dev)
    seen = set()
    for red in range(512, 4608, 256):
        M, C = 40, 520
        a, w = rnd(M, red), rnd(C, red) * 0.03
        nbytes = _cabi.lib().gmlp_workspace_bytes(_cabi.GMLP_OP_LINEAR_FWD, M, red, C, _cabi.dtype_code(a.dtype))
        seen.add(nbytes // (4 * M * C))
        ref = a.double() @ w.double().T
        err = ((ops_fwd.linear_fwd(a, w).double() - ref).norm() / ref.norm()).item()
        print(f"reduction {red}: {nbytes // (4 * M * C)} splits, rel {err:.2e}", flush=True)
        assert err < 2.0**-11
    assert len(seen) >= 4 and max(seen) >= 9, seen
    for M, C in ((1, 8), (63, 264), (64, 256), (65, 248), (513, 1032), (1357, 3096)):
        a = rnd(M, C)
        ref = a.double().sum(0)
        for out in ops_bwd.colsum_grouped([a, a, a]):
            rel = ((out.double() - ref).norm() / ref.norm()).item()
            print(f"column sums {M} x {C}: rel {rel:.2e}", flush=True)
            assert rel < 2.0**-11


@pytest.mark.parametrize(
    "M,K,N",
    [
        (1, 8, 8),           # one tile, a quarter of a reduction tile
        (65, 40, 136),       # one row and 8 columns beyond a 64x64 tile; reduction tails
        (130, 1544, 264),    # few tiles, long reductions: split, ragged last split
        (4100, 72, 200),     # long reduction of the weight gradients only: grouped launch, split
        (2300, 1048, 4200),  # 128-row tiles (two reduction segments of unequal last tiles in dX)
    ],
)
def test_fp32_every_operator_against_float64_products(M, K, N):
    """float32 kernels: every tile class, split reductions, edges.  Bound: a sum of R products in float32,
    in any order, is off by at most (R + 2) 2^-24 sum |a||b| (first order in 2^-24), element by element."""
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    print(f"fp32 operators: M={M} K={K} N={N}", flush=True)
    g = torch.Generator().manual_seed(3)
    rnd = lambda *shape, s=1.0: (s * torch.randn(*shape, generator=g)).to(dev)
    d = lambda t: t.double()

    def check(name, got, pairs):
        ref = sum(a @ b for a, b in pairs)
        terms = sum(a.abs() @ b.abs() for a, b in pairs)
        R = sum(a.shape[1] for a, _ in pairs)
        assert torch.isfinite(got).all(), name
        worst = ((got.double() - ref).abs() / ((R + 2) * 2.0**-24 * terms).clamp_min(1e-300)).max().item()
        print(f"  {name}: largest error {worst:.3f} of its bound", flush=True)
        assert worst <= 1.0, name

    x, dy, h, dg, du = rnd(M, K), rnd(M, K), rnd(M, N), rnd(M, N), rnd(M, N)
    wg, wu, wd = rnd(N, K, s=0.03), rnd(N, K, s=0.03), rnd(K, N, s=0.03)
    hs = ops_fwd.gateup_fwd(x, wg, None, wu, None, save_activations=True)
    check("G", hs.gate, [(d(x), d(wg).T)])
    check("U", hs.up, [(d(x), d(wu).T)])
    check("Y", ops_fwd.linear_fwd(h, wd), [(d(h), d(wd).T)])
    ones = torch.ones_like(hs.up)
    check("dH", ops_bwd.dh_bwd(dy, wd, ones, ones, act_fn="no_act")[1], [(d(dy), d(wd))])
    check("dX", ops_bwd.dx_bwd(dg, du, wg, wu), [(d(dg), d(wg)), (d(du), d(wu))])
    lhs_rhs = [(dg, x), (du, x), (dy, h)]
    for name, got, (a, b) in zip(("dW_gate", "dW_up", "dW_down"), ops_bwd.dw_bwd_grouped(lhs_rhs), lhs_rhs):
        check(name, got, [(d(a).T, d(b))])
    check("dW alone", ops_bwd.dw_bwd(dy, h), [(d(dy).T, d(h))])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M", [1, 63, 64, 65, 700, 2560, 2561])  # row ranges empty, of one row, uneven; one launch and two
def test_column_sums_against_float64(M, dtype):
    """Column sums of three arrays, one strip of 64 columns to several with a ragged last one.  Bound: a
    float32 sum of M terms in any order, (M + 2) 2^-24 sum |a|, and half a unit of the stored type."""
    from triton_gated_mlp.ops import bwd as ops_bwd

    dev = _dev()
    g = torch.Generator().manual_seed(M)
    arrays = [torch.randn(M, C, generator=g).to(dtype).to(dev) for C in (8, 72, 264)]
    half_unit = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8, torch.float32: 2.0**-24}[dtype]
    for a, got in zip(arrays, ops_bwd.colsum_grouped(arrays)):
        ref = a.double().sum(0)
        bound = (M + 2) * 2.0**-24 * a.double().abs().sum(0) + half_unit * ref.abs()
        assert ((got.double() - ref).abs() <= bound * (1 + half_unit) + 2.0**-25).all(), (M, a.shape[1], dtype)
        assert torch.equal(got, ops_bwd.colsum(a))


@pytest.mark.parametrize("M,K,N", [(1, 8, 8), (65, 40, 136), (1, 1544, 264), (1, 2056, 4104)])  # both tile classes, splits
def test_fp32_products_of_single_terms_are_rounded_once(M, K, N):
    """Sums of which one term alone is not zero, with significands that leave all three bf16 parts of both operands as
    large as they get (1 + 2^-8 - 2^-17: parts 1, 2^-8, -2^-17) and random ones.  Bound: half a unit of the result, 2^-24,
    for the last addition; those before it add up what is below 2^-7 of the product, rounded to 2^-24 of that
    each, and the part that no product covers (third parts with each other) is below 2^-34: 2^-24 (1 + 2^-5)."""
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(23)

    def full(*shape):
        """Signs, exponents of 2^-6 to 2^6, 24 significant bits, every fourth one the worst."""
        t = 1 + torch.rand(shape, generator=g)
        t[torch.rand(shape, generator=g) < 0.25] = 1 + 2.0**-8 - 2.0**-17
        return t * 2.0 ** torch.randint(-6, 7, shape, generator=g) * (1 - 2.0 * torch.randint(0, 2, shape, generator=g))

    def lone(rows, red):
        """One nonzero element to a row."""
        t = torch.zeros(rows, red)
        at = torch.randint(0, red, (rows, 1), generator=g)
        return t.scatter_(1, at, full(rows, 1))

    def check(name, got, ref):
        worst = ((got.double() - ref).abs() / ref.abs().clamp_min(1e-300)).max().item() * 2.0**24
        print(f"  {name}: largest error {worst:.3f} of half a unit", flush=True)
        assert worst <= 1 + 2.0**-5, name

    d = lambda *ts: [t.to(dev) for t in ts]
    print(f"fp32 single terms: M={M} K={K} N={N}", flush=True)
    x, h, wg, wu, wd = d(lone(M, K), lone(M, N), full(N, K), full(N, K), full(K, N))
    hs = ops_fwd.gateup_fwd(x, wg, None, wu, None, save_activations=True)
    check("G", hs.gate, x.double() @ wg.double().T)
    check("U", hs.up, x.double() @ wu.double().T)
    check("Y", ops_fwd.linear_fwd(h, wd), h.double() @ wd.double().T)
    ones = torch.ones(M, N, device=dev)
    check("dH", ops_bwd.dh_bwd(x, wd, ones, ones, act_fn="no_act")[1], x.double() @ wd.double())
    check("dX", ops_bwd.dx_bwd(h, torch.zeros_like(h), wg, wu), h.double() @ wg.double())
    lhs, rhs = d(lone(N, M).T.contiguous(), full(M, K))  # the weight gradients of one token are such sums
    (dw,) = ops_bwd.dw_bwd_grouped([(lhs, rhs)])
    check("dW", dw, lhs.double().T @ rhs.double())


@pytest.mark.parametrize(
    "M,K,N",
    [(72, 40, 136), (130, 1544, 264),         # one 64-row tile and a bit; split reductions
     (1050, 1144, 1096), (1403, 352, 2816)],  # 128-row tiles, with and without splits
)
def test_fp32_extreme_operands_against_float64_products(M, K, N):
    """Operands that three bf16 parts of 2^16 x do not hold (infinities, NaNs, 2^111 and more), products
    that overflow on the way, and subnormal ones, in rows and columns of their own beside ordinary ones: NaNs
    and infinities where IEEE sums in float32 have them, and everything finite within the bound of a float32
    sum, (R + 2) 2^-24 sum |a||b|, beside half the spacing of subnormal results per term."""
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(17)
    rnd = lambda *shape: torch.randn(*shape, generator=g)
    inf, nan = float("inf"), float("nan")

    def extreme(t):
        """t [rows, red]: extremes in rows 3 to 13, at the start and at the end of the reduction."""
        t = t.clone()
        t[3, 1], t[4, -1], t[5, 2], t[5, -2] = inf, -inf, inf, -inf
        t[6, 0], t[7, 3], t[8, -1] = nan, 3.4e38, -(2.0**112)
        t[9] = 2.0**-140 * t[9].sign()
        t[10] *= 2.0**-120
        t[11] *= 2.0**100
        t[12] = 0.0
        t[13] = 2.0**-149
        return t

    def check(name, got, pairs):
        ref = sum(a.double() @ b.double() for a, b in pairs)
        terms = sum(a.double().abs() @ b.double().abs() for a, b in pairs)
        # what float32 makes of the float64 sum: out of range is infinite (no sum here is within rounding of it)
        ref = torch.where(ref.abs() >= 3.4028236e38, ref.sign() * inf, ref)
        got = got.double().cpu()
        assert torch.equal(torch.isnan(got), torch.isnan(ref)), name
        assert torch.equal(torch.isinf(got), torch.isinf(ref)) and torch.equal(got[torch.isinf(ref)], ref[torch.isinf(ref)]), name
        R = sum(a.shape[1] for a, _ in pairs)
        ok = torch.isfinite(ref)
        bound = (R + 2) * (2.0**-24 * terms + 2.0**-149)
        worst = ((got - ref).abs()[ok] / bound[ok]).max().item()
        print(f"  {name}: largest error {worst:.3f} of its bound, {int((~ok).sum())} not finite", flush=True)
        assert worst <= 1.0, name

    print(f"fp32 extremes: M={M} K={K} N={N}", flush=True)
    # weights that bf16 holds exactly (their second and third parts are zero), zeros among them
    exact = lambda *shape: (rnd(*shape) * 2).round() / 2
    d = lambda t: t.to(dev)
    x, w = extreme(rnd(M, K)), exact(N, K)
    hs = ops_fwd.gateup_fwd(d(x), d(w), None, d(exact(N, K)), None, save_activations=True)
    check("G", hs.gate, [(x, w.T)])
    h, wd = extreme(rnd(M, N)), exact(K, N)
    check("Y", ops_fwd.linear_fwd(d(h), d(wd)), [(h, wd.T)])
    a, we = exact(M, N), extreme(rnd(K, N))
    check("Y, extreme weights", ops_fwd.linear_fwd(d(a), d(we)), [(a, we.T)])
    ones = torch.ones(M, N)
    check("dH", ops_bwd.dh_bwd(d(x), d(wd), d(ones), d(ones), act_fn="no_act")[1], [(x, wd)])
    wg, wu = exact(N, K), exact(N, K)
    h2 = rnd(M, N)
    check("dX", ops_bwd.dx_bwd(d(h), d(h2), d(wg), d(wu)), [(h, wg), (h2, wu)])
    lhs = extreme(rnd(N, M)).T.contiguous()  # reduction over the rows: extremes in columns
    e = exact(M, K)
    check("dW", ops_bwd.dw_bwd(d(lhs), d(e)), [(lhs.T, e)])


@pytest.mark.parametrize(
    "M,K,N,halves",  # out [M, K], reduction N
    [(1, 8, 256, True), (1, 8, 248, True), (64, 72, 264, True), (33, 1024, 2816, True), (65, 136, 272, True),  # 8, 9 and 88 tiles
     (1, 16384, 256, True), (64, 8, 224, False), (1, 16392, 256, False)],  # a workgroup on every CU, 7 tiles, one more tile
)
def test_fp32_down_projections_in_two_halves(M, K, N, halves):
    """Down projections of few rows: both halves of the reduction in one workgroup, odd numbers of reduction tiles and
    ragged last ones included, without a workspace; elementwise within the bound of a float32 sum, and the kernel by name
    (on a whole MI355X).  An infinity in either half comes out as such."""
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator(device=dev).manual_seed(37)
    rnd = lambda *shape: torch.empty(shape, device=dev).normal_(generator=g)
    h, w, b = rnd(M, N), rnd(K, N), rnd(K)
    names, out = _launched(lambda: ops_fwd.linear_fwd(h, w, b))
    ref, terms = h.double() @ w.double().T + b.double(), h.double().abs() @ w.double().abs().T + b.double().abs()
    worst = ((out.double() - ref).abs() / ((N + 3) * 2.0**-24 * terms)).max().item()
    print(f"M={M} K={K} N={N}: largest error {worst:.3f} of its bound", flush=True)
    assert worst <= 1.0
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert any("halves" in n for n in names) == halves, names
    for k in (0, N - 1):
        t = h.clone()
        t[0, k] = float("inf")
        got = ops_fwd.linear_fwd(t, w, b)
        assert torch.equal(got[0], w[:, k].sign() * float("inf")) and torch.equal(got[1:], out[1:])


def test_fp32_operands_that_are_not_finite_cost_a_few_launches_at_most():
    """A single infinity makes a whole row or column of a product non-finite, a row of them all of a weight gradient: those
    outputs are computed a second time.  On the fp32 matrix cores that makes it up to three times the usual time here;
    element by element, as it was, 5 to 43 times.  Bound: twice what is measured."""
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    M, K, N = 2048, 1024, 2816
    g = torch.Generator(device=dev).manual_seed(29)
    rnd = lambda *shape: torch.empty(shape, device=dev).normal_(generator=g)
    x, dy, h, G, U, wg, wu = rnd(M, K), rnd(M, K), rnd(M, N), rnd(M, N), rnd(M, N), rnd(N, K), rnd(N, K)
    row, one, w = x.clone(), x.clone(), wg.clone()
    row[5], one[5, 7], w[3, 9] = float("inf"), float("inf"), float("inf")

    def us(run):
        times = []
        for _ in range(4):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(5):
                run()
            end.record()
            torch.cuda.synchronize()
            times.append(200 * start.elapsed_time(end))
        return min(times)

    grads = lambda t: ops_bwd.dw_bwd_grouped([(G, t), (U, t), (dy, h)])
    gates = lambda t: ops_fwd.gateup_fwd(x, t, None, wu, None, save_activations=True)
    for name, run, finite, extremes in (("weight gradients", grads, x, (row, one)), ("gate/up", gates, wg, (w, wg * 2.0**100))):
        usual = us(lambda: run(finite))
        for t in extremes:
            slow = us(lambda: run(t))
            print(f"{name}: {usual:.0f} us, with operands that are not finite or near it {slow:.0f}", flush=True)
            assert slow < 6 * usual, name


def test_random_modules_through_the_one_call_entries_no_worse_than_torch_16bit():
    """Four dozen seeded random modules (token counts 1 to 6144, widths that are multiples of 8, 64
    or 256, both 16-bit dtypes, biases, dropout, five activations) through FusedGatedMLP, i.e. through
    gmlp_mlp_fwd / gmlp_mlp_bwd, against fp32 formulas on the same rounded inputs with the library's
    own keep mask.  Weights ~ N(0, 0.03) and biases ~ U(-0.1, 0.1): harsher than the baseline's
    distributions, so that 16-bit rounding of G, U, H and of the outputs shows as a few elements
    beyond the element-wise band of `_close` (bf16 resolves 2^-9).  Those are counted, not waved
    through: the fused path may
    leave the band at most twice as often as the same formulas run through torch's own 16-bit
    operators on the same inputs with the same mask (plus 16 elements + 2e-5 of the tensor).  The
    relative Frobenius error stays below 1e-2 throughout.  The activations are the smooth ones: a
    relu whose fp32 pre-activation lies within 1e-6 of zero falls on either side of the kink
    depending on the summation order of whoever computes it, the fp32 reference included, and then
    moves a whole row of dW_gate (relu and leaky_relu are held to the CPU oracle in
    test_other_activations_*)."""
    import random

    from triton_gated_mlp import FusedGatedMLP
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    rng = random.Random(1)
    acts = {"silu": torch.nn.functional.silu, "gelu": torch.nn.functional.gelu, "tanh": torch.tanh,
            "sigmoid": torch.sigmoid, "no_act": lambda t: t}

    def outside(got, ref):
        got, ref = got.float(), ref.float()
        assert torch.isfinite(got).all()
        atol = ATOL * max(1.0, ref.abs().mean().item())
        fro = ((got - ref).norm() / ref.norm().clamp_min(1e-30)).item()
        return int(((got - ref).abs() > atol + RTOL * ref.abs()).sum()), fro

    for case in range(48):
        dt = rng.choice([torch.float16, torch.bfloat16])
        unit = rng.choice([64, 64, 64, 8, 256])
        M = rng.choice([1, 3, 16, 17, 33, 100, 255, 256, 257, 511, 700, 1024, 1500, 2048, 2304, 3000, 4097, 6144])
        K = rng.randint(1, 4096 // unit) * unit
        N = rng.randint(1, 6144 // unit) * unit
        bias = rng.random() < 0.5
        p = rng.choice([0.0, 0.0, 0.1, 0.3])
        act = rng.choice(list(acts))
        print(f"random module {case}: M={M} K={K} N={N} {dt} bias={bias} p={p} act={act}", flush=True)
        g = torch.Generator(device=dev).manual_seed(case)
        mlp = FusedGatedMLP(K, N, bias=bias, dropout_p=p, hidden_act=act).to(dev).to(dt)
        with torch.no_grad():
            for lin in (mlp.gate_proj, mlp.up_proj, mlp.down_proj):
                lin.weight.copy_(torch.empty(lin.weight.shape, device=dev).normal_(0, 0.03, generator=g))
                if bias:
                    lin.bias.copy_(torch.empty(lin.bias.shape, device=dev).uniform_(-0.1, 0.1, generator=g))
        mlp.train(p > 0)
        mlp.dropout_seed = 99
        x = torch.empty(M, K, device=dev).normal_(0, 1, generator=g).to(dt)
        dy = torch.empty(M, K, device=dev).normal_(0, 1, generator=g).to(dt)
        xs = x.clone().requires_grad_(True)
        y = mlp(xs)
        fused = [y] + list(torch.autograd.grad(y, [xs] + list(mlp.parameters()), dy))
        # fp32 formulas, the same keep mask
        xf = x.float().requires_grad_(True)
        ps = [q.detach().float().requires_grad_(True) for q in mlp.parameters()]
        if bias:
            Wg, bg, Wu, bu, Wd, bd = ps
        else:
            (Wg, Wu, Wd), bg, bu, bd = ps, None, None, None
        H = acts[act](torch.nn.functional.linear(xf, Wg, bg)) * torch.nn.functional.linear(xf, Wu, bu)
        if p > 0:
            seed, off = mlp.last_dropout_state
            keep = ops_fwd.dropout_mask(M, N, p, seed, off, device=dev).float()
            H = H * keep / (1 - p)
        yr = torch.nn.functional.linear(H, Wd, bd)
        ref = [yr] + list(torch.autograd.grad(yr, [xf] + ps, dy.float()))
        # yardstick: the same formulas through torch's own 16-bit operators, same keep mask
        xe = x.clone().requires_grad_(True)
        pe = [q.detach().clone().requires_grad_(True) for q in mlp.parameters()]
        if bias:
            Wg, bg, Wu, bu, Wd, bd = pe
        else:
            (Wg, Wu, Wd), bg, bu, bd = pe, None, None, None
        He = acts[act](torch.nn.functional.linear(xe, Wg, bg)) * torch.nn.functional.linear(xe, Wu, bu)
        if p > 0:
            He = He * (keep.to(dt) * (1.0 / (1 - p)))
        ye = torch.nn.functional.linear(He, Wd, bd)
        yard = [ye] + list(torch.autograd.grad(ye, [xe] + pe, dy))
        names = ["Y", "dX"] + [n for n, _ in mlp.named_parameters()]
        for i, n in enumerate(names):
            bad, fro = outside(fused[i], ref[i])
            allowed = 16 + 2e-5 * ref[i].numel() + 2 * outside(yard[i], ref[i])[0]
            assert fro < 1e-2, f"{n}: relative Frobenius error {fro:.3e}"
            assert bad <= allowed, f"{n}: {bad} elements outside the band, {allowed:.0f} allowed"


def test_grouped_weight_gradients_equal_single_launches():
    """gmlp_dw_bwd_grouped (one grid) is bit-identical to three gmlp_dw_bwd launches."""
    from triton_gated_mlp.ops import bwd as ops_bwd

    dev = _dev()
    g = torch.Generator().manual_seed(9)
    for M, K, N in [(2048, 2048, 5632), (512, 256, 520)]:  # full-tile class and predicated class
        x = torch.randn(M, K, generator=g).half().to(dev)
        dg = torch.randn(M, N, generator=g).half().to(dev)
        du = torch.randn(M, N, generator=g).half().to(dev)
        dy = torch.randn(M, K, generator=g).half().to(dev)
        h = torch.randn(M, N, generator=g).half().to(dev)
        pairs = [(dg, x), (du, x), (dy, h)]
        grouped = ops_bwd.dw_bwd_grouped(pairs)
        for (a, b), got in zip(pairs, grouped):
            assert torch.equal(got, ops_bwd.dw_bwd(a, b))  # (neither form shares out tiles at these shapes)
        _close("dW_gate grouped", grouped[0], dg.float().cpu().T @ x.float().cpu())


@pytest.mark.parametrize(
    "M,K,N,dtype,trained",
    [
        (380, 152, 136, torch.float32, ("gate_proj", "up_proj")),
        (708, 96, 912, torch.float16, ("gate_proj", "down_proj")),
        (5857, 1752, 6576, torch.float16, ("gate_proj", "up_proj")),  # stream-K
        (3776, 2720, 136, torch.bfloat16, ("gate_proj",)),
        (3115, 64, 7328, torch.float16, ("down_proj",)),
    ],
)
def test_some_weight_gradients_run_as_planned_for_them(M, K, N, dtype, trained):
    """A step that trains some of the weights gives their gradients the workspace that they use by
    themselves, which here is more than that of a step that trains all: bit-identical to the grouped launch
    (whose plan's order of additions differs from the one that a smaller workspace forces)."""
    from triton_gated_mlp import FusedGatedMLP, _cabi
    from triton_gated_mlp.ops import bwd as ops_bwd
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    torch.manual_seed(14)
    mlp = FusedGatedMLP(K, N, bias=False).to(dev).to(dtype)
    mlp.requires_grad_(False)
    weights = [getattr(mlp, name).weight.requires_grad_(True) for name in trained]
    x, dy = torch.randn(M, K, device=dev).to(dtype), torch.randn(M, K, device=dev).to(dtype)
    Wg, Wu, Wd = mlp.gate_proj.weight, mlp.up_proj.weight, mlp.down_proj.weight
    with torch.no_grad():
        hs = ops_fwd.gateup_fwd(x, Wg, None, Wu, None, save_activations=True)
        dg, du = ops_bwd.dh_bwd(dy, Wd, hs.gate, hs.up)
        operands = {"gate_proj": (dg, x), "up_proj": (du, x), "down_proj": (dy, hs.hidden)}
        want = ops_bwd.dw_bwd_grouped([operands[name] for name in trained])
        need = [False] * 7
        for name in trained:
            need[{"gate_proj": 1, "up_proj": 3, "down_proj": 5}[name]] = True
        used = ops_bwd._mlp_bwd_workspace_bytes(M, K, N, _cabi.dtype_code(dtype), need)
        assert used > _cabi.lib().gmlp_mlp_workspace_bytes(_cabi.GMLP_PASS_BWD, M, K, N, _cabi.dtype_code(dtype))
        one_call = ops_bwd.mlp_bwd(dy, x, Wg, Wu, Wd, hs.gate, hs.up, hs.hidden, need)
    mlp(x).backward(dy)
    for w, a, b in zip(weights, want, (t for t in one_call if t is not None)):
        assert torch.equal(w.grad, a) and torch.equal(b, a)


def test_one_call_backward_hands_its_launches_whatever_workspace_there_is():
    """gmlp_mlp_bwd for one weight gradient with the workspace of a pass that computes all three, which holds
    some of its ten splits: the value of gmlp_dw_bwd with that workspace, not the one of an unsplit launch
    (another order of additions)."""
    from triton_gated_mlp import _cabi

    dev, lib = _dev(), _cabi.lib()
    M, K, N, code = 3776, 2720, 136, _cabi.GMLP_BF16
    g = torch.Generator(device=dev).manual_seed(16)
    rnd = lambda *shape: torch.empty(shape, device=dev).normal_(generator=g).bfloat16()
    dy, x, wd, G, U = rnd(M, K), rnd(M, K), rnd(K, N) * 0.02, rnd(M, N), rnd(M, N)
    dg, du, dw, alone, unsplit = rnd(M, N), rnd(M, N), rnd(N, K), rnd(N, K), rnd(N, K)
    nbytes = lib.gmlp_mlp_workspace_bytes(_cabi.GMLP_PASS_BWD, M, K, N, code)
    assert 2 * 4 * N * K <= nbytes < lib.gmlp_workspace_bytes(_cabi.GMLP_OP_DW_BWD, M, N, K, code)
    ws = torch.empty(nbytes, device=dev, dtype=torch.uint8)
    p, stream = (lambda t: t.data_ptr()), _cabi.stream_ptr(dev)
    _cabi.check(lib.gmlp_mlp_bwd(
        p(dy), p(x), None, None, p(wd), p(G), p(U), None, p(dg), p(du), None, p(dw), None, None, None, None, None,
        M, K, N, code, _cabi.act_code("silu"), 0.0, 0, 0, p(ws), nbytes, stream))
    _cabi.check(lib.gmlp_dw_bwd(p(dg), p(x), p(alone), M, N, K, code, p(ws), nbytes, stream))
    _cabi.check(lib.gmlp_dw_bwd(p(dg), p(x), p(unsplit), M, N, K, code, None, 0, stream))
    assert torch.equal(dw, alone) and not torch.equal(dw, unsplit)
    _close("dW_gate", dw, dg.float().T @ x.float())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,K,N", [(4100, 72, 200), (9000, 264, 520)])
def test_grouped_weight_gradients_use_what_fits_of_a_smaller_workspace(M, K, N, dtype):
    """A workspace that does not hold the planned partial sums is used for as many splits as it holds, never
    beyond its end, and none is needed."""
    import ctypes

    from triton_gated_mlp import _cabi

    dev, lib, code = _dev(), _cabi.lib(), _cabi.dtype_code(dtype)
    g = torch.Generator(device=dev).manual_seed(15)
    rnd = lambda *shape: torch.empty(shape, device=dev).normal_(generator=g).to(dtype)
    pairs = [(rnd(M, N), rnd(M, K)), (rnd(M, N), rnd(M, K)), (rnd(M, K), rnd(M, N))]
    outs = [torch.empty(a.shape[1], b.shape[1], device=dev, dtype=dtype) for a, b in pairs]
    array = lambda kind, values: ctypes.cast((kind * 3)(*values), ctypes.c_void_p)
    lhs, rhs, dws = (array(ctypes.c_void_p, [t.data_ptr() for t in ts]) for ts in (*zip(*pairs), outs))
    R, C = array(ctypes.c_int64, [N, N, K]), array(ctypes.c_int64, [K, K, N])
    need = lib.gmlp_dw_bwd_grouped_workspace_bytes(3, M, R, C, code)
    one_split = 4 * 3 * N * K
    assert need >= 4 * one_split and need % one_split == 0
    for nbytes in (need, need - one_split, need // 2, 2 * one_split, 2 * one_split - 16, 0):
        buffer = torch.full((need,), 0xA5, device=dev, dtype=torch.uint8)
        _cabi.check(lib.gmlp_dw_bwd_grouped(
            3, lhs, rhs, dws, M, R, C, code, buffer.data_ptr() if nbytes else None, nbytes, _cabi.stream_ptr(dev)))
        assert (buffer[nbytes:] == 0xA5).all(), nbytes
        used = nbytes - int((buffer[:nbytes] == 0xA5).all()) * nbytes
        assert (used > 0) == (nbytes >= 2 * one_split), nbytes
        for (a, b), dw in zip(pairs, outs):
            _close(f"dW with {nbytes} of {need} bytes", dw, a.float().T @ b.float())


def test_grouped_weight_gradients_of_mixed_sizes_equal_single_launches():
    """One problem of a group beyond the pipelined kernels' 32-bit operand offsets takes the predicated
    kernel alone: the others run as they do by themselves (here with a split reduction), bit for bit."""
    from triton_gated_mlp.ops import bwd as ops_bwd

    dev = _dev()
    g = torch.Generator(device=dev).manual_seed(13)
    rnd = lambda *shape: torch.empty(shape, dtype=torch.float16, device=dev).normal_(generator=g)
    M = 66048
    big, small, thin = rnd(M, 16384), rnd(M, 520), rnd(M, 8)  # 2.16e9 bytes, 69 MB, 1 MB
    pairs = [(small, rnd(M, 520)), (big, thin), (thin, small)]
    got = ops_bwd.dw_bwd_grouped(pairs)
    for (a, b), dw in zip(pairs, got):
        assert torch.equal(dw, ops_bwd.dw_bwd(a, b)), (a.shape, b.shape)
        _close("dW", dw, sum(p.float().T @ q.float() for p, q in zip(a.split(8256), b.split(8256))))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_decode_matches_general_path(dtype):
    """Skinny-M kernels against the oracle and the general path: both layouts of the intermediate H
    (row-major up to M = 10, fragment order above, with token slots past M), both streaming variants
    of the down projection, and shapes that only the register-streaming kernels take."""
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(2)
    for M, K, N, bias in [(16, 1024, 2048, True), (3, 256, 512, False), (1, 4096, 11008, True), (5, 768, 1792, True),
                          (16, 4096, 11008, False), (12, 1024, 2048, True), (11, 768, 1792, False), (10, 8192, 512, True)]:
        x = torch.randn(M, K, generator=g).to(dtype).to(dev)
        Wg = (0.02 * torch.randn(N, K, generator=g)).to(dtype).to(dev)
        Wu = (0.02 * torch.randn(N, K, generator=g)).to(dtype).to(dev)
        Wd = (0.02 * torch.randn(K, N, generator=g)).to(dtype).to(dev)
        bg = bu = bd = None
        if bias:
            bg = (0.01 * torch.randn(N, generator=g)).to(dtype).to(dev)
            bu = (0.01 * torch.randn(N, generator=g)).to(dtype).to(dev)
            bd = (0.01 * torch.randn(K, generator=g)).to(dtype).to(dev)
        y = ops_fwd.decode_fwd(x, Wg, bg, Wu, bu, Wd, bd)
        f = lambda t: None if t is None else t.float().cpu()
        ref = oracle.forward(f(x), f(Wg), f(bg), f(Wu), f(bu), f(Wd), f(bd))
        _close(f"decode Y M={M}", y, ref["Y"])
        h = ops_fwd.gateup_fwd(x, Wg, bg, Wu, bu).hidden
        y_general = ops_fwd.linear_fwd(h, Wd, bd)
        _close(f"general Y M={M}", y_general, ref["Y"])


# Streaming kernels by (16-row regions per matrix, token tiles, bytes of a row per stage); what a case names
# is what its launches are held to.  K and N with a row tail unless marked: of 512-byte stages a width that
# is not a multiple of 256 elements, of 256-byte ones (rows of whole 128-byte lines only) 64 mod 128.
_DECODE_CASES = [
    # M, K, N, gate/up, down
    (1, 776, 1032, (1, 1, 512), (1, 1, 512)),      # least widths, one 16-byte piece in the last chunk of each
    (3, 2200, 4608, (1, 1, 512), (1, 1, 512)),     # no tail in the down projection
    (16, 4096, 4104, (2, 1, 256), (1, 1, 512)),    # none in gate/up; full tile of tokens
    (11, 4496, 9472, (1, 1, 512), (2, 1, 256)),    # H in fragment order; no tail in the down projection
    (17, 1016, 888, (1, 2, 512), (1, 2, 512)),     # last chunks short by one piece
    (24, 4104, 1160, (1, 2, 512), (2, 2, 512)),
    (20, 2056, 8200, (1, 2, 512), (1, 2, 512)),
    (7, 5192, 1160, (1, 1, 512), (2, 1, 512)),
    (29, 5192, 1160, (1, 2, 512), (2, 2, 512)),
    (32, 12568, 1032, (1, 2, 512), (2, 2, 512)),
    (18, 12544, 1280, (1, 2, 512), (4, 2, 256)),   # no tails
    (12, 1088, 4160, (2, 1, 256), (1, 1, 512)),
    (12, 4160, 1088, (1, 1, 512), (2, 1, 256)),
    (24, 4160, 4160, (2, 2, 256), (2, 2, 256)),
    (24, 4160, 1088, (2, 2, 256), (2, 2, 256)),
    (18, 12352, 1088, (1, 2, 512), (4, 2, 256)),
]


def _decode_tails():
    width = lambda kernel: kernel[2] // 2
    return {("gate/up", g) for _, K, _, g, _ in _DECODE_CASES if K % width(g)} | {
        ("down", d) for _, _, N, _, d in _DECODE_CASES if N % width(d)}


@pytest.mark.parametrize("bias", [True, False], ids=["biases", "plain"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["fp16", "bf16"])
@pytest.mark.parametrize("M,K,N,gated,down", _DECODE_CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_decode_streaming_kernels_at_any_width(M, K, N, gated, down, dtype, bias):
    """Streaming kernels whose last chunk of a row is partly beyond it, where the next row begins with
    large values, against float64 products; twice, bit-identical, the second time with the launched kernels'
    names (on a whole MI355X: the choice goes by rows per compute unit)."""
    import re

    from torch.profiler import ProfilerActivity, profile
    from triton_gated_mlp import _cabi

    dev = _dev()
    print(f"decode, any width: M={M} K={K} N={N} {dtype} bias={bias}", flush=True)
    g = torch.Generator(device=dev).manual_seed(21)
    rnd = lambda *shape, s=1.0: torch.empty(shape, device=dev).normal_(0.0, s, generator=g).to(dtype)
    x, wg, wu, wd = rnd(M, K, s=0.5), rnd(N, K, s=0.02), rnd(N, K, s=0.02), rnd(K, N, s=0.02)
    bg, bu, bd = (rnd(N, s=0.1), rnd(N, s=0.1), rnd(K, s=0.1)) if bias else (None, None, None)
    x[:, :8] *= 16
    for w in (wg, wu, wd):
        w[:, :8] *= 16

    def run():
        h = torch.full((16 if M <= 16 else 32, N), float("nan"), dtype=dtype, device=dev)
        y = torch.full((M, K), float("nan"), dtype=dtype, device=dev)
        _cabi.check(_cabi.lib().gmlp_decode_stream_fwd(
            *(_cabi.ptr(t) for t in (x, wg, wu, wd, bg, bu, bd, h, y)), M, K, N, _cabi.dtype_code(dtype),
            _cabi.act_code("silu"), _cabi.stream_ptr(dev)))
        return y

    y = run()
    d = lambda t: 0.0 if t is None else t.double()
    hidden = torch.nn.functional.silu(d(x) @ d(wg).T + d(bg)) * (d(x) @ d(wu).T + d(bu))
    ref = hidden.to(dtype).double() @ d(wd).T + d(bd)
    _close("Y", y, ref)
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as prof:
        again = run()
        torch.cuda.synchronize()
    assert torch.equal(y, again)
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        # (names come mangled or, bfloat16's, halfway demangled)
        name = r"decode_stream_kernel.*?(?:ELi|, )(\d+)(?:ELi|, )(\d+)(?:ELi|, )(\d+)(?:ELi|, )\d+(?:ELb|, )(0|1|false|true)"
        found = [m.groups() for m in (re.search(name, e.name) for e in prof.events()) if m]
        launched = [(*map(int, g[:3]), g[3] in ("1", "true")) for g in found]
        tail = lambda kernel, red: red % (kernel[2] // 2) != 0
        assert launched == [(*gated, tail(gated, K)), (*down, tail(down, N))], launched


def test_decode_cases_cover_every_row_tail():
    """Every block shape that launch_decode_stream chooses among occurs with a row tail."""
    assert _decode_tails() == {("gate/up", (h, t, s)) for h, s in ((1, 512), (2, 256)) for t in (1, 2)} | {
        ("down", k) for k in ((1, 1, 512), (2, 1, 256), (2, 1, 512), (1, 2, 512), (2, 2, 256), (2, 2, 512), (4, 2, 256))}


@pytest.mark.parametrize(
    "M,K,N,gated,down",  # on a whole MI355X, as above; rows per compute unit in brackets
    [
        (1, 768, 2048, (1, 1, 128), (1, 1, 128)),      # fewer stages than ring slots, half a block [8] and a quarter [3]
        (16, 1024, 5632, (2, 1, 128), (1, 1, 128)),    # [22] H in fragment order
        (5, 4352, 2112, (1, 1, 128), (2, 1, 256)),     # [8.25] K [17]; N no multiple of 256
        (9, 4352, 2048, (1, 1, 128), (2, 1, 128)),
        (17, 1280, 3904, (1, 2, 128), (1, 2, 512)),    # [15.25]
        (24, 768, 8256, (3, 2, 128), (1, 2, 512)),     # [32.25]
        (32, 768, 7744, (2, 2, 128), (1, 2, 512)),     # [30.25]
        (20, 768, 14336, (4, 2, 128), (1, 2, 512)),    # [56]
        (32, 768, 18944, (5, 2, 128), (1, 2, 512)),    # [74]
        (32, 768, 45056, (4, 2, 128), (1, 2, 512)),    # [176]: two whole blocks and most of a third
    ],
)
def test_decode_streaming_kernels_short_segments(M, K, N, gated, down):
    """Every block height of the kernels that stream 128-byte segments, with partly empty blocks, against
    float64 products; twice, bit-identical, the second time with the launched kernels' names."""
    test_decode_streaming_kernels_at_any_width(M, K, N, gated, down, torch.bfloat16 if M % 2 else torch.float16, M > 16)


@pytest.mark.parametrize(
    "M,K,N,down",  # down: token tiles, bytes of a row per stage, ring slots, row tails, rows of a region, wavefronts (on a whole MI355X)
    [
        (1, 768, 1024, (1, 128, 8, 0, 8, 4)),     # 96 workgroups; four chunks a wavefront
        (16, 2048, 1280, (1, 128, 8, 0, 8, 4)),   # 256 workgroups of 8 rows
        (1, 2048, 8192, (1, 512, 3, 0, 8, 3)),    # more weights than short segments take at this M; ten or eleven chunks
        (11, 2040, 2048, (1, 512, 3, 0, 8, 3)),   # 255 workgroups, fewer chunks than slots; H in fragment order
        (1, 776, 768, (1, 512, 3, 0, 8, 3)),      # one chunk a wavefront
        (3, 1984, 776, (1, 512, 3, 1, 8, 3)),     # 248; one 16-byte piece in the last chunk, rows across 128-byte lines
        (11, 1000, 4104, (1, 512, 3, 1, 8, 3)),
        (17, 2040, 768, (2, 512, 3, 0, 8, 3)),    # two token tiles, a chunk a wavefront
        (32, 2048, 1032, (2, 512, 3, 1, 8, 3)),
        (5, 2112, 4096, (1, 128, 8, 0, 16, 4)),   # 8.25 rows a share
        (9, 3328, 2048, (1, 128, 8, 0, 16, 4)),   # 13
        (2, 3392, 2048, (1, 128, 8, 0, 16, 3)),   # 13.25
    ],
    ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v),
)
def test_decode_down_projection_of_small_shares(M, K, N, down):
    """Regions of 8 rows and four wavefronts, at the ends of the widths that take them, against float64
    products; twice, bit-identical; with the launched kernel's name."""
    import re

    dev = _dev()
    dtype = torch.bfloat16 if M % 2 else torch.float16
    print(f"decode, small shares: M={M} K={K} N={N} {dtype}", flush=True)
    from triton_gated_mlp import _cabi

    g = torch.Generator(device=dev).manual_seed(22)
    rnd = lambda *shape, s=1.0: torch.empty(shape, device=dev).normal_(0.0, s, generator=g).to(dtype)
    x, wg, wu, wd, bd = rnd(M, K, s=0.5), rnd(N, K, s=0.02), rnd(N, K, s=0.02), rnd(K, N, s=0.02), rnd(K, s=0.1)
    wd[:, :8] *= 16

    def run():
        h = torch.full((16 if M <= 16 else 32, N), float("nan"), dtype=dtype, device=dev)
        y = torch.full((M, K), float("nan"), dtype=dtype, device=dev)
        _cabi.check(_cabi.lib().gmlp_decode_stream_fwd(
            *(_cabi.ptr(t) for t in (x, wg, wu, wd, None, None, bd, h, y)), M, K, N, _cabi.dtype_code(dtype),
            _cabi.act_code("silu"), _cabi.stream_ptr(dev)))
        return y

    names, y = _launched(run)
    hidden = torch.nn.functional.silu(x.double() @ wg.double().T) * (x.double() @ wu.double().T)
    _close("Y", y, hidden.to(dtype).double() @ wd.double().T + bd.double())
    assert torch.equal(y, run())
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        numbers = r"(?:ELi|, )(\d+)" * 4 + r"(?:ELb|, )(0|1|false|true)" + r"(?:ELi|, )(\d+)" * 2
        found = [m.groups() for m in (re.search(r"decode_stream_kernel.*?" + numbers, n) for n in names) if m]
        _, tiles, segment, slots, tail, rows, waves = found[-1]
        assert (*map(int, (tiles, segment, slots)), int(tail in ("1", "true")), int(rows), int(waves)) == down, found


def test_decode_streaming_entry_refuses_what_its_kernels_do_not_take():
    from triton_gated_mlp import _cabi

    a = torch.zeros(4096, dtype=torch.float16, device=_dev())
    call = lambda M, K, N, code=0: _cabi.lib().gmlp_decode_stream_fwd(
        *[a.data_ptr()] * 4, None, None, None, a.data_ptr(), a.data_ptr(), M, K, N, code, 0, None)
    for M, K, N in ((33, 1024, 1024), (0, 1024, 1024), (1, 760, 1024), (1, 1024, 760), (1, 1028, 1024), (1, 1024, 1028), (1, 32768, 32768)):
        assert call(M, K, N) == -2, (M, K, N)
    assert call(1, 1024, 1024, 2) == -2  # float32


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_decode_with_two_token_tiles(dtype):
    """16 < M <= 32 on the streaming kernels (two MFMAs per weight fragment, H for 32 token slots):
    full and partly filled second tiles, both block heights of the down projection, widths whose
    rows do not fill a last round of blocks, with and without biases."""
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    g = torch.Generator().manual_seed(5)
    for M, K, N, bias in [(32, 1024, 2048, True), (17, 768, 1792, False), (24, 8192, 768, True), (31, 4096, 11008, True),
                          (20, 4352, 1024, False), (32, 5120, 13824, False)]:
        assert ops_fwd.decode_supported(M, K, N, dtype)
        print(f"decode two tiles {dtype} M={M} K={K} N={N} bias={bias}", flush=True)
        x = torch.randn(M, K, generator=g).to(dtype).to(dev)
        Wg = (0.02 * torch.randn(N, K, generator=g)).to(dtype).to(dev)
        Wu = (0.02 * torch.randn(N, K, generator=g)).to(dtype).to(dev)
        Wd = (0.02 * torch.randn(K, N, generator=g)).to(dtype).to(dev)
        bg = bu = bd = None
        if bias:
            bg = (0.01 * torch.randn(N, generator=g)).to(dtype).to(dev)
            bu = (0.01 * torch.randn(N, generator=g)).to(dtype).to(dev)
            bd = (0.01 * torch.randn(K, generator=g)).to(dtype).to(dev)
        y = ops_fwd.decode_fwd(x, Wg, bg, Wu, bu, Wd, bd)
        f = lambda t: None if t is None else t.float().cpu()
        ref = oracle.forward(f(x), f(Wg), f(bg), f(Wu), f(bu), f(Wd), f(bd))
        _close(f"decode Y M={M}", y, ref["Y"])
    # shapes the streaming kernels do not take keep the limit of 16 rows
    assert not ops_fwd.decode_supported(17, 512, 1024, dtype)
    with pytest.raises(NotImplementedError):
        ops_fwd.decode_fwd(torch.zeros(17, 512, dtype=dtype, device=dev), *[t for _ in range(2) for t in (torch.zeros(1024, 512, dtype=dtype, device=dev), None)],
                           torch.zeros(512, 1024, dtype=dtype, device=dev), None)


@pytest.mark.parametrize(
    "M,K,N,streams,dtype",
    [(8, 2048, 4096, True, torch.float16), (24, 3584, 4096, True, torch.float16), (64, 1024, 4096, False, torch.float16),
     (33, 1024, 2816, False, torch.float32)],
)
def test_inference_forward_under_hip_graph_replay(M, K, N, streams, dtype):
    """Serving loops replay a captured forward: the skinny-M streaming path (one and two token
    tiles) and the general path (split reductions; float32, whose down projection here is reduced in
    two halves by one workgroup) are captured once and replayed with new
    inputs written into the captured input buffer; every replay must equal the eager result for
    that input, with eager work and synchronisations in between."""
    from triton_gated_mlp import FusedGatedMLP
    from triton_gated_mlp.ops import fwd as ops_fwd

    dev = _dev()
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    assert ops_fwd.decode_preferred(M, K, N, dtype, cus) == streams
    mlp = FusedGatedMLP(K, N, bias=True).to(dev).to(dtype).eval()
    g = torch.Generator().manual_seed(41)
    inputs = [torch.randn(M, K, generator=g).to(dtype).to(dev) for _ in range(3)]
    with torch.no_grad():
        eager = [mlp(v).clone() for v in inputs]
        x = inputs[0].clone()
        side = torch.cuda.Stream(device=dev)
        side.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(side):  # warm-up on a side stream, as torch's graph recipe asks
            mlp(x)
        torch.cuda.current_stream(dev).wait_stream(side)
        torch.cuda.synchronize(dev)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = mlp(x)
        for rep in (1, 2, 0, 1):
            x.copy_(inputs[rep])
            y.fill_(float("nan"))
            _ = (torch.randn(256, 256, device=dev) @ torch.randn(256, 256, device=dev)).sum().item()
            graph.replay()
            torch.cuda.synchronize(dev)
            assert torch.equal(y, eager[rep]), f"replay with input {rep} differs from the eager forward"


def test_native_autograd_nodes_keep_pytorchs_contracts():
    """What torch.autograd.Function gives for free, from the native nodes: N-D and non-contiguous inputs,
    partial gradients, errors on a second backward and on operands changed in place, saved-tensor hooks
    (non-reentrant checkpointing), steps from several threads at once on streams of their own."""
    import threading

    from torch.utils.checkpoint import checkpoint
    from triton_gated_mlp import FusedGatedMLP, FusedGatedMLPFunction

    dev = _dev()
    torch.manual_seed(6)
    mlp = FusedGatedMLP(256, 512, bias=True).to(dev).half()
    base = torch.randn(256, 3, 5, device=dev, dtype=torch.float16)
    x = base.permute(2, 1, 0).detach().requires_grad_(True)  # [5, 3, 256], not contiguous
    dy = torch.randn(5, 3, 256, device=dev, dtype=torch.float16)
    y = mlp(x)
    assert y.shape == x.shape and not y._is_view()
    y.backward(dy, retain_graph=True)
    ref = {n: p.grad.clone() for n, p in mlp.named_parameters()}
    ref_x = x.grad.clone()
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        with torch.no_grad():
            mlp.up_proj.weight.mul_(1.0)
        y.backward(dy)
    y = mlp(x)
    (gx,) = torch.autograd.grad(y, [x], dy)
    assert gx.shape == x.shape and torch.equal(gx, ref_x)
    with pytest.raises(RuntimeError, match="second time"):
        y.backward(dy)
    # frozen parameters get nothing, the others the same
    for n, p in mlp.named_parameters():
        p.requires_grad_(n.startswith("down"))
        p.grad = None
    mlp(x.detach()).backward(dy)
    for n, p in mlp.named_parameters():
        assert torch.equal(p.grad, ref[n]) if n.startswith("down") else p.grad is None
        p.requires_grad_(True)
        p.grad = None
    # saved-tensor hooks: the whole node is recomputed, same gradients
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(tuple(t.shape)) or t, lambda t: t):
        y = mlp(x)
    assert (3, 15, 512) in packed  # G, U, H
    y.backward(dy)
    assert all(torch.equal(p.grad, ref[n]) for n, p in mlp.named_parameters())
    for lean in (False, True):
        mlp.recompute_activations = lean
        mlp.zero_grad()
        checkpoint(mlp, x, use_reentrant=False).backward(dy)
        assert all(torch.equal(p.grad, ref[n]) for n, p in mlp.named_parameters())
    # the hidden-state operator: dY of a sum is an expanded scalar
    xs = x.detach().reshape(-1, 256).requires_grad_(True)
    W = [mlp.up_proj.weight.detach().requires_grad_(True), mlp.gate_proj.weight.detach()]
    FusedGatedMLPFunction.apply(xs, W[0], None, W[1], None).sum().backward()
    assert xs.grad.shape == xs.shape and W[0].grad.shape == W[0].shape and W[1].grad is None
    # two threads, a module and a stream each
    results = {}

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            m = FusedGatedMLP(256, 512, bias=True).to(dev).half()
            m.load_state_dict(mlp.state_dict())
            t = x.detach().clone().requires_grad_(True)
            for _ in range(20):
                m.zero_grad()
                t.grad = None
                m(t).backward(dy)
            torch.cuda.current_stream().synchronize()
            results[k] = (t.grad, {n: p.grad for n, p in m.named_parameters()})

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(results) == 2
    for gx, grads in results.values():
        assert torch.equal(gx, ref_x) and all(torch.equal(g, ref[n]) for n, g in grads.items())


def test_native_autograd_nodes_refuse_what_they_cannot_differentiate():
    """Forward mode and functorch transforms raise (a result without its tangent would be wrong), unpack
    hooks that change a saved tensor's type, size or device raise before a kernel reads it, and a
    checkpoint that holds other operators beside the module recomputes them with autograd recording."""
    import torch.autograd.forward_ad as fw
    from torch.utils.checkpoint import checkpoint

    from triton_gated_mlp import FusedGatedMLP, FusedGatedMLPFunction

    dev = _dev()
    torch.manual_seed(7)
    mlp = FusedGatedMLP(256, 512, bias=True).to(dev).half()
    x = torch.randn(24, 256, device=dev, dtype=torch.float16, requires_grad=True)
    W = [mlp.up_proj.weight, mlp.gate_proj.weight]
    calls = {256: mlp, 512: lambda t: FusedGatedMLPFunction.apply(t, W[0], None, W[1], None)}
    for width, call in calls.items():
        dy = torch.randn(24, width, device=dev, dtype=torch.float16)
        with fw.dual_level(), pytest.raises(NotImplementedError, match="forward-mode"):
            call(fw.make_dual(x, torch.ones_like(x)))
        with pytest.raises(RuntimeError):
            torch.vmap(call)(x[None])
        with pytest.raises(RuntimeError):
            torch.func.grad(lambda t: call(t).sum())(x.detach())
        for unpack in (lambda t: t.cpu(), lambda t: t.float(), lambda t: t.reshape(-1)[:-8]):
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
                y = call(x)
            with pytest.raises(RuntimeError, match="saved tensor came back"):
                y.backward(dy)
        block = torch.nn.Linear(256, 256, bias=False).to(dev).half()
        segment = lambda t: torch.tanh(call(torch.tanh(block(t))))
        (want,) = torch.autograd.grad(segment(x), [x], dy)
        (got,) = torch.autograd.grad(checkpoint(segment, x, use_reentrant=False), [x], dy)
        assert torch.equal(got, want)


@pytest.mark.parametrize("how", ["no_grad", "frozen"])
def test_forward_mode_and_functorch_are_refused_where_reverse_mode_records_nothing(how):
    """A dual tensor does not require grad and torch.no_grad() leaves forward mode on: an inference forward
    that dropped its tangent would answer wrongly.  Where forward mode is off it is a plain forward."""
    import torch.autograd.forward_ad as fw

    from triton_gated_mlp import FusedGatedMLP

    dev = _dev()
    torch.manual_seed(8)
    mlp = FusedGatedMLP(1024, 2048, bias=True).to(dev).half().requires_grad_(how == "no_grad")
    for M in (4, 200):  # the streaming and the general kernels
        x = torch.randn(M, 1024, device=dev, dtype=torch.float16)
        with torch.set_grad_enabled(how != "no_grad"):
            want = mlp(x)
            with fw.dual_level():
                dual = fw.make_dual(x, torch.ones_like(x))
                with pytest.raises(NotImplementedError, match="forward-mode"):
                    mlp(dual)
                with torch.inference_mode():
                    assert torch.equal(mlp(dual), want)
            with fw.dual_level(), pytest.raises(NotImplementedError, match="forward-mode"):
                bias = mlp.down_proj.bias
                torch.func.functional_call(mlp, {"down_proj.bias": fw.make_dual(bias.detach(), torch.ones_like(bias))}, (x,))
            for transform in (torch.vmap(mlp), lambda t: torch.func.jvp(mlp, (t,), (t,))):
                with pytest.raises(RuntimeError, match="functorch"):
                    transform(x[None])


@pytest.mark.parametrize("recompute", [False, True])
def test_missing_incoming_gradient_counts_as_zeros(recompute):
    """An operator behind the module whose backward returns None for it: every gradient is zeros (as from a
    torch.autograd.Function), not None, which an optimiser with momentum or weight decay would skip."""
    from triton_gated_mlp import FusedGatedMLP, FusedGatedMLPFunction

    class NoGradient(torch.autograd.Function):
        @staticmethod
        def forward(ctx, t):
            return t.clone()

        @staticmethod
        def backward(ctx, grad):
            return None

    dev = _dev()
    mlp = FusedGatedMLP(64, 128, bias=True).to(dev).half()
    mlp.recompute_activations = recompute
    x = torch.randn(2, 12, 64, device=dev, dtype=torch.float16, requires_grad=True)
    leaves = [x, *mlp.parameters()]
    NoGradient.apply(mlp(x)).sum().backward()
    assert all(t.grad is not None and t.grad.shape == t.shape and not t.grad.any() for t in leaves)
    up, gate = mlp.up_proj, mlp.gate_proj
    leaves = [up.weight, up.bias, gate.weight, gate.bias]
    mlp.zero_grad()
    NoGradient.apply(FusedGatedMLPFunction.apply(x.flatten(0, 1), *leaves)).sum().backward()
    assert all(t.grad is not None and not t.grad.any() for t in leaves)


@pytest.mark.parametrize("which", ["module", "hidden"])
def test_second_derivatives_raise_instead_of_being_dropped(which):
    """create_graph: the gradients are the usual ones, and a derivative through them raises, whatever it is
    asked for and whatever other terms a loss has (a penalty on the gradient would otherwise count as a
    constant).  What does not pass through them is differentiated."""
    from triton_gated_mlp import FusedGatedMLP, FusedGatedMLPFunction

    dev = _dev()
    torch.manual_seed(10)
    mlp = FusedGatedMLP(256, 512, bias=True).to(dev).half()
    W = [mlp.up_proj.weight, mlp.gate_proj.weight]
    call = mlp if which == "module" else lambda t: FusedGatedMLPFunction.apply(t, W[0], None, W[1], None)
    a = torch.randn(24, 256, device=dev, dtype=torch.float16, requires_grad=True)
    scale = torch.ones((), device=dev, dtype=torch.float16, requires_grad=True)
    x = a * 1.0
    plain = torch.autograd.grad(call(x).sum(), [x, *W])
    with_graph = torch.autograd.grad((call(x) * scale).sum(), [x, *W], create_graph=True)
    assert all(torch.equal(g, h) and h.requires_grad for g, h in zip(plain, with_graph))
    for gradient in with_graph:
        penalty = gradient.float().square().sum()
        for loss in (penalty, penalty + x.float().square().sum()):
            for wanted in (a, x, W[0], scale):
                with pytest.raises(RuntimeError, match="no second derivative"):
                    torch.autograd.grad(loss, wanted, retain_graph=True, allow_unused=True)
            with pytest.raises(RuntimeError, match="no second derivative"):
                loss.backward(retain_graph=True)
        # a weight of the other gradients only
        factor = torch.ones_like(gradient, requires_grad=True)
        assert torch.equal(torch.autograd.grad((gradient * factor).sum(), factor, retain_graph=True)[0], gradient)
    # an optimiser step on gradients that carry a graph
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")  # torch's, once per process, that such gradients are a reference cycle
        call(x).sum().backward(create_graph=True)
    torch.optim.SGD(W, lr=0.0).step()
    for w, g in zip(W, plain[1:]):
        assert torch.equal(w.grad, g)
        w.grad = None


@pytest.mark.parametrize("grad", [True, False], ids=["records a graph", "nothing to differentiate"])
def test_traced_forwards_run_the_kernels(grad):
    """torch.jit.trace of the module and of the hidden-state operator records the call, not the allocation
    of its output: the traced graph gives the eager result on other inputs and other numbers of tokens, bit
    for bit, and the eager gradients; with dropout the mask of the seed that was drawn while tracing."""
    from triton_gated_mlp import FusedGatedMLP, FusedGatedMLPFunction
    from triton_gated_mlp.gated_mlp import FusedGatedMLPFullFunction

    dev = _dev()
    torch.manual_seed(9)
    mlp = FusedGatedMLP(1024, 2048, bias=True).to(dev).half().requires_grad_(grad)
    W = [mlp.up_proj.weight, mlp.gate_proj.weight]
    hidden = lambda t, wu, wg: FusedGatedMLPFunction.apply(t, wu, None, wg, None)
    example = torch.randn(2, 3, 1024, device=dev, dtype=torch.float16)  # without a graph: the decode kernels
    traced = torch.jit.trace(mlp, (example,))
    traced_hidden = torch.jit.trace(hidden, (example.flatten(0, 1), *W))
    for shape in ((2, 3), (2, 3), (5, 40)):  # (the second and later runs are the executor's optimised graph)
        x = torch.randn(*shape, 1024, device=dev, dtype=torch.float16)
        got, want = traced(x), mlp(x)
        assert got.requires_grad == grad and torch.equal(got, want)
        got_h, want_h = (call(x.flatten(0, 1), *W) for call in (traced_hidden, hidden))
        assert got_h.requires_grad == grad and torch.equal(got_h, want_h)
        if grad:
            dy, dh = torch.randn_like(want), torch.randn_like(want_h)
            params = list(mlp.parameters())
            for a, b in zip(torch.autograd.grad(got, params, dy), torch.autograd.grad(want, params, dy)):
                assert torch.equal(a, b)
            for a, b in zip(torch.autograd.grad(got_h, W, dh), torch.autograd.grad(want_h, W, dh)):
                assert torch.equal(a, b)
    if grad:
        mlp.dropout.p = 0.25
        traced = torch.jit.trace(mlp, (example,), check_trace=False)
        seed, offset = mlp.last_dropout_state
        x = torch.randn_like(example)
        want = FusedGatedMLPFullFunction.apply(
            x, W[1], mlp.gate_proj.bias, W[0], mlp.up_proj.bias, mlp.down_proj.weight, mlp.down_proj.bias, 0.25, seed, offset
        )
        assert torch.equal(traced(x), want)


def test_training_step_under_stream_capture_is_refused(monkeypatch):
    """A forward that records an autograd graph while its stream is being captured raises a
    RuntimeError (no kernel is enqueued, nothing is captured); the capture state is simulated on
    the host, no stream is actually captured here."""
    from triton_gated_mlp import FusedGatedMLP

    dev = _dev()
    mlp = FusedGatedMLP(256, 512, bias=False).to(dev).half()
    x = torch.randn(64, 256, device=dev, dtype=torch.float16, requires_grad=True)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    with pytest.raises(RuntimeError, match="autograd graph"):
        mlp(x)
    with torch.no_grad():
        assert mlp(x).shape == (64, 256)  # inference is not affected


@pytest.mark.skip(
    reason="capturing the step with torch.cuda.graph ended in a host-side segmentation fault inside "
    "capture_end (hipStreamEndCapture) on this image; cause not established, so the case stays off the GPU"
)
def test_forward_backward_under_hip_graph_replay():
    """The entry points only enqueue kernels on the caller's stream (no allocation, no memset), so a
    training step can be captured once and replayed; every replay must equal the eager result."""
    from triton_gated_mlp import FusedGatedMLP

    dev = _dev()
    c = Case("graph", 512, 256, 768, torch.float16, bias=True, p=0.1, backward=True, seed=31)
    t = make_inputs(c)
    mlp = FusedGatedMLP(c.K, c.N, bias=True, dropout_p=c.p).to(dev).to(c.dtype).train()
    mlp.dropout_seed = 99
    x = t["x"].to(dev).requires_grad_(True)
    dY = t["dY"].to(dev)
    params = [x] + list(mlp.parameters())

    def step():
        mlp._dropout_calls = 0  # same mask stream for every step
        y = mlp(x)
        return (y,) + torch.autograd.grad(y, params, grad_outputs=dY)

    eager = [v.clone() for v in step()]
    side = torch.cuda.Stream(device=dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):  # warm-up on the capture stream, as torch's graph recipe asks
        step()
    torch.cuda.current_stream(dev).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step()
    for rep in range(3):
        for o in outs:
            o.fill_(float("nan"))
        _ = (torch.randn(256, 256, device=dev) @ torch.randn(256, 256, device=dev)).sum().item()  # eager work between replays
        graph.replay()
        torch.cuda.synchronize(dev)
        for name, got, ref in zip(["Y", "dX"] + [n for n, _ in mlp.named_parameters()], outs, eager):
            assert torch.equal(got, ref), f"replay {rep}: {name} differs from the eager step"


@pytest.mark.parametrize("amp_dtype", [torch.float16, torch.bfloat16])
def test_autocast_with_fp32_master_weights(amp_dtype):
    """Mixed-precision training: fp32 parameters, torch.autocast picks the kernel dtype; gradients
    come back in fp32 and match the oracle evaluated on the rounded operands."""
    from triton_gated_mlp import FusedGatedMLP

    dev = _dev()
    c = Case("amp", 384, 256, 640, amp_dtype, bias=True, backward=True, seed=41)
    t = make_inputs(c)  # values already representable in amp_dtype
    mlp = FusedGatedMLP(c.K, c.N, bias=True).to(dev).float()
    with torch.no_grad():
        for name, key in (("gate_proj", "gate"), ("up_proj", "up"), ("down_proj", "down")):
            getattr(mlp, name).weight.copy_(t[f"W_{key}"].float())
            getattr(mlp, name).bias.copy_(t[f"b_{key}"].float())
    x = t["x"].float().to(dev).requires_grad_(True)
    with torch.autocast("cuda", dtype=amp_dtype):
        y = mlp(x)
    assert y.dtype == amp_dtype
    params = [x] + list(mlp.parameters())
    grads = torch.autograd.grad(y, params, grad_outputs=t["dY"].to(dev))
    assert all(g.dtype == torch.float32 for g in grads), "master-weight gradients must stay fp32"
    o = _oracle_inputs(t)
    ref = oracle.backward(o["x"], o["W_gate"], o["b_gate"], o["W_up"], o["b_up"], o["W_down"], o["b_down"], o["dY"])
    _close("Y", y, ref["Y"])
    names = ["dX", "dW_gate", "db_gate", "dW_up", "db_up", "dW_down", "db_down"]
    for n, g in zip(names, grads):
        _close(n, g, ref[n])
