"""CPU checks of the host-side mirror of the reference interface (no GPU)."""

import math

import pytest
import torch


def test_constants_match_reference_defaults():
    from defmuon_amd.optim import deflation_batched as DB
    assert DB.DIVISOR_PAD == 1.01 and DB.RSVD_NITER == 1 and DB.CHOLQR_PASSES == 1
    assert DB.GRAM_DTYPE is torch.float64
    assert DB.GATE_WINDOW == DB.SKETCH_FRAC == DB.OVERSAMPLE_FRAC == 0.025
    assert DB.GATE_RATIO == DB.DEFLATE_THRESH == 0.10
    assert DB.DeflatedPEPolar.PAD == 1.1 and DB.DeflatedNSPolar.PAD == 1.01
    assert DB.DeflatedNSPolar.NS_ABC == (3.4445, -4.7750, 2.0315)


def test_pe_schedule_matches_oracle():
    from defmuon_amd.optim import polar_express as PE
    from oracle import polar_oracle as O
    assert PE.coeffs_list == O.PE_COEFFS
    assert PE.pe_schedule(11) == O.pe_schedule(11)


@pytest.mark.parametrize("m", [64, 80, 768, 1024, 1280])
def test_sketch_dims_match_oracle(m):
    from defmuon_amd.optim import deflation_batched as DB
    from oracle import polar_oracle as O
    assert DB.sketch_dims(m) == O.sketch_dims(m)


def test_polar_stats_schema():
    from defmuon_amd.optim import deflation_batched as DB
    DB._GATE_ACC[0] = torch.tensor([10, 4, 9])
    st = DB.polar_stats()
    assert st == dict(fired=4, total=10, k_mean=9 / 4, degenerate=0, parachute=0)
    DB._GATE_ACC[0] = None
    assert DB.polar_stats() == dict(fired=0, total=0, k_mean=0.0, degenerate=0, parachute=0)


def test_timing_accumulator():
    from defmuon_amd.optim import deflation_batched as DB

    class Ev:
        def __init__(self, t):
            self.t = t

        def elapsed_time(self, other):
            return other.t - self.t

    DB._PENDING.append((Ev(0.0), Ev(2.0), Ev(5.0)))
    st = DB.timing_stats()
    assert st == {"clip_ms": 2.0, "iter_ms": 3.0, "calls": 1}
    assert DB.timing_stats() == {"clip_ms": 0.0, "iter_ms": 0.0, "calls": 0}


def test_no_cpu_fallback():
    """The product path runs only through the HIP library."""
    from defmuon_amd import _native
    from defmuon_amd.optim import deflation_batched as DB
    from defmuon_amd.optim import muon
    G = torch.randn(16, 32)
    with pytest.raises(_native.NativeError):
        muon.zeropower_via_newtonschulz5(G, 5)
    with pytest.raises(_native.NativeError):
        DB.batched_rmfro_clip(torch.randn(1, 64, 32), Omega=torch.randn(1, 32, 2))


def test_muon_routing_and_arms(capsys):
    from defmuon_amd.optim import deflation_batched as DB
    from defmuon_amd.optim import deflation_cutoff as C
    from defmuon_amd.optim import muon
    C.install()
    C.install()           # idempotent
    params = [("wte.weight", torch.nn.Parameter(torch.zeros(10, 4))),
              ("h.0.attn.c_attn.weight", torch.nn.Parameter(torch.zeros(12, 4))),
              ("h.0.mlp.c_fc.weight", torch.nn.Parameter(torch.zeros(16, 4))),
              ("h.0.ln_1.weight", torch.nn.Parameter(torch.zeros(4)))]
    opt = muon.Muon(params, polar_method="deflated_ns_cut")
    assert isinstance(opt.polar_factorizer, C.CutoffDeflatedNSPolar)
    assert isinstance(opt.polar_factorizer, DB._DeflatedPolarBase)
    assert opt.batched_deflation and opt._bd_step == 0
    st = opt.state
    assert st[params[0][1]]["use_muon"] is False
    assert st[params[1][1]]["use_muon"] and st[params[1][1]]["is_W_QKV"]
    assert st[params[2][1]]["use_muon"] and "is_W_QKV" not in st[params[2][1]]
    assert st[params[3][1]]["use_muon"] is False
    assert opt._qkv_split(params[1][1], params[1][1]).shape == (3, 4, 4)
    opt2 = muon.Muon(params, polar_method="deflated_pe_cut")
    assert isinstance(opt2.polar_factorizer, C.CutoffDeflatedPEPolar)
    assert opt2.polar_factorizer.POST == "polarexpress"
    assert muon.Muon(params, polar_method="ns5").polar_factorizer is muon.zeropower_via_newtonschulz5
    with pytest.raises(ValueError):
        muon.Muon(params, polar_method="nope")
    # CPU parameters: the warm-up reports the missing GPU path and carries on
    assert "warm-up failed" in capsys.readouterr().out


def test_adjust_lr():
    from defmuon_amd.optim import muon
    opt = muon.Muon([("w", torch.nn.Parameter(torch.zeros(8, 2)))], polar_method="ns5")
    assert opt.adjust_lr_for_muon(0.1, True, False, (8, 2), None, None) == pytest.approx(0.2)
    assert opt.adjust_lr_for_muon(0.1, False, False, (8, 2), None, None) == 0.1
    g = torch.eye(3)
    assert opt.adjust_lr_for_muon(1.0, False, True, (3, 3), g, 2 * g) == pytest.approx(6.0)


class _Fake:
    """What _fused_glue_ok looks at of a tensor: a GPU tensor without a GPU."""

    def __init__(self, shape, device="cuda:0", dtype=torch.float32, contiguous=True):
        self.shape, self.ndim, self.dtype = torch.Size(shape), len(shape), dtype
        self.device, self.is_cuda = torch.device(device), device.startswith("cuda")
        self.is_contiguous = lambda: contiguous
        self.grad = None


@pytest.mark.parametrize("which", ["grad", "momentum_buffer"])
@pytest.mark.parametrize("bad", [dict(shape=(6, 3)), dict(shape=(3,)), dict(shape=(4, 6)),
                                 dict(shape=(6, 4), device="cuda:1"), dict(shape=(6, 4), device="cpu"),
                                 dict(shape=(6, 4), dtype=torch.bfloat16),
                                 dict(shape=(6, 4), contiguous=False)])
def test_fused_glue_takes_tensors_of_the_parameters_shape_alone(which, bad):
    """The fused glue reads and writes rows * cols elements of the gradient and the momentum
    buffer: a buffer of another shape (a state dict of another model) or device goes to the
    torch ops, which refuse it."""
    from defmuon_amd.optim import muon
    opt = muon.Muon([("w", torch.nn.Parameter(torch.zeros(8, 2)))], polar_method="ns5")
    p = _Fake((6, 4))
    p.grad = _Fake((6, 4))
    group = {"nuclear_scaling": False}
    opt.state[p]["momentum_buffer"] = _Fake((6, 4))
    assert opt._fused_glue_ok(group, [p])
    if which == "grad":
        p.grad = _Fake(**bad)
    else:
        opt.state[p]["momentum_buffer"] = _Fake(**bad)
    assert not opt._fused_glue_ok(group, [p])


def test_plain_buckets_keep_shared_memory_apart():
    """Parameters that share memory never share a bucket (its launches update all of them at
    once); neighbours in one buffer do."""
    from defmuon_amd.optim import muon
    flat = torch.zeros(40, 8)
    P = torch.nn.Parameter
    a, b, c = P(flat[:8]), P(flat[8:24]), P(flat[24:])
    tied, inner, row = P(flat[8:24]), P(flat[10:12]), P(flat[23:25])
    flipped = P(flat[:8].T)
    empty = P(torch.zeros(0, 8))
    opt = muon.Muon([("w", P(torch.zeros(8, 2)))], polar_method="ns5")

    def buckets(*params):
        for p in params:
            p.grad = torch.zeros_like(p)
        return [[id(e["p"]) for e in b] for b in opt._plain_buckets(params, 1)]

    def ids(*groups):
        return [[id(p) for p in g] for g in groups]

    assert buckets(c, a, b, empty, empty) == ids((c, a, b, empty, empty))
    assert buckets(a, b, a, c) == ids((a, b), (a, c))
    assert buckets(a, b, tied, c) == ids((a, b), (tied, c))
    assert buckets(a, inner, b, c) == ids((a, inner), (b, c))
    assert buckets(a, b, c, row) == ids((a, b, c), (row,))
    assert buckets(b, c, flipped, a) == ids((b, c, flipped), (a,))


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("shape", [(4096, 8), (16, 4096), (64, 64), (768, 3072), (3 * 256, 256)])
def test_plain_buckets_count_padded_bytes(shape, mode):
    """A bucket's stack, polar factors and chain workspaces, as they are allocated, stay within
    PLAIN_BUCKET (a parameter above it is alone), and a bucket is not broken while the next
    parameter still fits; no limit under grouped_plain."""
    from defmuon_amd import _native
    from defmuon_amd.optim import muon
    name = "attn.c_attn.weight" if shape[0] == 3 * shape[1] else "mlp.weight"
    params = [torch.nn.Parameter(torch.zeros(shape)) for _ in range(10)]
    opt = muon.Muon([(f"{i}.{name}", p) for i, p in enumerate(params)],
                    polar_method="ns5" if mode == 1 else "polarexpress")
    for p in params:
        p.grad = torch.zeros_like(p)
    nb = 3 if "c_attn" in name else 1
    rows, cols = shape[0] // nb, shape[1]
    tall = rows > cols if nb == 1 or mode == 2 else 3 > rows

    def allocated(n):    # fp32 momentum and stack, bf16 polar factors, one workspace
        return (n * params[0].numel() * (4 + 4 + 2)
                + _native.ns_workspace_bytes(n * nb, rows, cols, tall))

    for limit in (0, allocated(1), allocated(3) + 100000, allocated(10) + 100000):
        opt.PLAIN_BUCKET = limit
        bs = opt._plain_buckets(params, mode)
        assert [id(e["p"]) for b in bs for e in b] == [id(p) for p in params]
        for b in bs:
            assert len(b) == 1 or allocated(len(b)) <= limit
        assert all(allocated(len(b) + 1) > limit - 10 * 4096 for b in bs[:-1])
    opt.GROUPED_PLAIN, opt.PLAIN_BUCKET = True, 0
    assert len(opt._plain_buckets(params, mode)) == 1


@pytest.mark.parametrize("arm", ["ns5", "polarexpress", "deflated_ns_cut"])
def test_warm_up_runs_the_batches_of_the_step(monkeypatch, arm):
    """The polar kernels are chosen by their batch: the construction-time warm-up of the plain
    arms (and of the arm behind a deflation cutoff) runs the stacks that the step will run."""
    from defmuon_amd.optim import deflation_cutoff as C
    from defmuon_amd.optim import muon
    calls = []

    def chains(stacks, talls, mode, sched):
        calls.append(([(tuple(X.shape), X.dtype) for X in stacks], list(talls), mode, list(sched)))
        return [torch.zeros(X.shape, dtype=torch.bfloat16) for X in stacks]

    monkeypatch.setattr(muon, "plain_group_chains", chains)
    C.install()
    if arm.startswith("deflated"):
        monkeypatch.setattr(C, "CUTOFF_STEPS", 0)
    P = torch.nn.Parameter
    params = [("wte.weight", P(torch.zeros(16, 8)))]
    for i in range(3):
        params += [(f"{i}.attn.c_attn.weight", P(torch.zeros(24, 8))),
                   (f"{i}.mlp.c_fc.weight", P(torch.zeros(32, 8))),
                   (f"{i}.mlp.c_proj.weight", P(torch.zeros(8, 32, dtype=torch.bfloat16)))]
    monkeypatch.setattr(muon.Muon, "PLAIN_BUCKET", 5 << 20)
    opt = muon.Muon(params, polar_method=arm)
    warm = list(calls)
    calls.clear()
    for _, p in params:
        p.grad = torch.randn_like(p)
    opt.step()
    assert len(calls) > 1 and warm == calls
