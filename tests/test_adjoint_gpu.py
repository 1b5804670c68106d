"""Reverse mode on the GPU (pga_forward_tape / pga_backward and the
torch.autograd binding) against the oracle's FP64 adjoint twin: dL/dparams
within 1e-4 relative, the tape's derivation identical to the plain one, and
central finite differences of the FP64 twin (decisions frozen)."""
import numpy as np
import pytest

from operatorgraph_amd import abi, axioms, grammars
from operatorgraph_amd.grammars import op
from operatorgraph_amd.program import AxiomParam, DispatchTable, Entry, Program, Scalar
from tests.helpers import assert_same_multiset

pytestmark = pytest.mark.gpu

B, Q = abi.BOX, abi.QUAD


def _note(msg):
    print(msg, flush=True)


def _weights(inst):
    """A fixed pseudo-random dL/dmodel row per instance, keyed by (axiom, path)
    so that the GPU and oracle orders get the same rows."""
    key = inst["axiom"].astype(np.float64) * 7919.0 + (inst["path"] % 100003).astype(np.float64)
    k = np.arange(12, dtype=np.float64)
    return np.sin(key[:, None] * 0.013 + k[None, :] * 1.7)


def _diff_grammar():
    """Every differentiable operator with per-axiom parameters:
        A   = Rotate(p0, p1, p2) S;  S = Scale(-1, p3, -1) C;
        C   = CompSplit() { Top | Bot | Side };
        Side = Repeat(X, p4, ANCHOR_TO_START) T;  T = Translate(0, 0, p5) G0;
        Top = SubDiv(Y) { p6: G1 | -1: G1 | -1.5: G0 };
        Bot = Extrude(Z, p7) G2;  G0/G1 = Generate(0/1) (Quad), G2 = Generate(2) (Box)."""
    A, S, C, SIDE, T, TOP, BOT, G0, G1, G2 = range(10)
    table = DispatchTable([
        Entry(op(abi.ROTATE, B), [AxiomParam(0), AxiomParam(1), AxiomParam(2)], [(S, 0)]),
        Entry(op(abi.SCALE, B), [Scalar(-1.0), AxiomParam(3), Scalar(-1.0)], [(C, 0)]),
        Entry(op(abi.COMPSPLIT, B), [], [(TOP, 0), (BOT, 0), (SIDE, 0)]),
        Entry(op(abi.REPEAT, Q), [Scalar(abi.X), AxiomParam(4), Scalar(abi.ANCHOR_TO_START)], [(T, 0)]),
        Entry(op(abi.TRANSLATE, Q), [Scalar(0.0), Scalar(0.0), AxiomParam(5)], [(G0, 0)]),
        Entry(op(abi.SUBDIV, Q), [Scalar(abi.Y), AxiomParam(6), Scalar(-1.0), Scalar(-1.5)],
              [(G1, 0), (G1, 0), (G0, 0)]),
        Entry(op(abi.EXTRUDE, Q), [Scalar(abi.Z), AxiomParam(7)], [(G2, 0)]),
        Entry(op(abi.GENERATE, Q, 1), [Scalar(0)], []),
        Entry(op(abi.GENERATE, Q, 1), [Scalar(1)], []),
        Entry(op(abi.GENERATE, B, 1), [Scalar(2)], []),
    ])
    return Program(grammars.INTERPRETER_PROCEDURES, table, "diff_kitchen_sink")


def _diff_axioms(n, seed=21):
    rng = np.random.default_rng(seed)
    ax = axioms.empty(n)
    ax["size"] = rng.uniform(4.0, 9.0, size=(n, 3)).astype(np.float32)
    ax["model"][:, [3, 7, 11]] = rng.uniform(-20, 20, size=(n, 3)).astype(np.float32)
    ax["entry_index"] = 0
    ax["shape_type"] = B
    params = np.stack([rng.uniform(-30, 30, n), rng.uniform(-30, 30, n), rng.uniform(-30, 30, n),
                       rng.uniform(-1.2, -0.6, n), rng.uniform(0.9, 1.7, n), rng.uniform(-0.3, 0.3, n),
                       rng.uniform(0.5, 1.5, n), rng.uniform(0.5, 2.0, n)], axis=1).astype(np.float32)
    return ax, params


def _gpu_run(program, ax, params, n_terms, tape=True):
    import torch
    from operatorgraph_amd import engine
    eng = engine.Engine(queue_capacity=1 << 20)
    eng.load(program).set_axioms(ax).set_axiom_params(params)
    for t in range(n_terms):
        eng.bind(t, 1 << 18)
    if tape:
        eng.tape_reserve(1 << 20, 1 << 21)
        eng.forward_tape()
    else:
        eng.execute()
    return eng


def _adjoint_pair(program, ax, params, n_terms, weights=_weights):
    import torch
    from oracle import oracle as O
    eng = _gpu_run(program, ax, params, n_terms)
    got = [eng.instances(t) for t in range(n_terms)]
    dl = {}
    for t in range(n_terms):
        g = np.zeros((len(got[t]), 16), dtype=np.float32)
        g[:, :12] = weights(got[t])
        dl[t] = torch.from_numpy(g).cuda()
    grad = eng.backward(dl).cpu().numpy().astype(np.float64)
    r = O.derive(program, ax, params=params, twins=O.TWIN_F64 | O.TWIN_ADJ)
    ref_inst = [r.instances(t) for t in range(n_terms)]
    for t in range(n_terms):
        assert_same_multiset(got[t], ref_inst[t], f"terminal {t}")
    ref = r.backward([weights(ref_inst[t]) for t in range(n_terms)])
    eng.close()
    return grad, ref, r


def _assert_close(grad, ref, rel=1e-4, entry_rel=1e-3, floor=1e-6):
    """dL/dparams of each axiom within `rel` of the FP64 adjoint, normwise
    relative (max-norm of the row error over the max-norm of the row), the
    way instance transforms are checked; and every entry within `entry_rel`
    relative to itself, except entries more than six orders of magnitude
    below the largest of their parameter column, which are measured against
    that floor. An entry is a sum of per-terminal terms of both signs, so
    FP32 rounding of the terms can leave a larger relative error on a sum
    that cancels than on the row."""
    row = np.abs(ref).max(axis=1)
    live = row > 0
    row_err = np.abs(grad - ref).max(axis=1)[live] / row[live]
    col = np.maximum(np.abs(ref).max(axis=0, keepdims=True), 1e-30)
    err = np.abs(grad - ref) / np.maximum(np.abs(ref), floor * col)
    _note(f"  dL/dparams: max normwise error per axiom {row_err.max() if row_err.size else 0.0:.3e}, "
          f"max entry error {err.max():.3e} over {err.size} entries")
    assert np.all(grad[~live] == 0.0)
    assert row_err.size == 0 or row_err.max() <= rel, (row_err.max(), np.argmax(row_err))
    assert err.max() <= entry_rel, (err.max(), np.unravel_index(err.argmax(), err.shape))


def test_tape_forward_matches_plain_forward():
    _note("tape forward vs plain forward")
    ax, params = axioms.param_lots(24, perturb=0.05)
    prog = grammars.facade_params()
    a = _gpu_run(prog, ax, params, 2, tape=True)
    b = _gpu_run(prog, ax, params, 2, tape=False)
    for t in range(2):
        assert_same_multiset(a.instances(t), b.instances(t), f"terminal {t}")
    a.close()
    b.close()


def test_adjoint_facade_params_vs_fp64():
    _note("adjoint facade_params vs FP64 adjoint")
    ax, params = axioms.param_lots(16, perturb=0.05)
    grad, ref, _ = _adjoint_pair(grammars.facade_params(), ax, params, 2)
    # repetition counts are frozen: the repeat extents get no gradient
    assert np.all(grad[:, 2] == 0.0) and np.all(grad[:, 3] == 0.0)
    _assert_close(grad, ref)


def test_adjoint_every_operator_vs_fp64():
    _note("adjoint rotate/scale/compsplit/repeat/translate/subdiv/extrude vs FP64 adjoint")
    ax, params = _diff_axioms(12)
    grad, ref, _ = _adjoint_pair(_diff_grammar(), ax, params, 3)
    assert np.all(np.abs(ref[:, [0, 1, 2, 3, 4, 5, 6, 7]]).max(axis=0) > 0.0)
    _assert_close(grad, ref)


def test_adjoint_against_central_differences():
    """dL/dparams of the GPU adjoint against central differences (h = 1e-3)
    of the oracle's FP64 twin with the FP32 pass's decisions frozen."""
    from oracle import oracle as O
    _note("adjoint vs central differences")
    ax, params = axioms.param_lots(3, perturb=0.05)
    prog = grammars.facade_params()
    grad, _, r = _adjoint_pair(prog, ax, params, 2)
    g = [_weights(r.instances(t)) for t in range(2)]

    def loss(p):
        rr = O.derive(prog, ax, params=p, twins=O.TWIN_F64)
        assert rr.count(0) == r.count(0) and rr.count(1) == r.count(1)
        return sum(float(np.sum(rr.instances_f64(t)[:, :12] * g[t])) for t in range(2))

    for lot in range(3):
        for k in (0, 1, 4, 5, 6, 7):
            pp, pm = params.copy(), params.copy()
            pp[lot, k] += 1e-3
            pm[lot, k] -= 1e-3
            hh = (float(pp[lot, k]) - float(pm[lot, k])) / 2.0
            fd = (loss(pp) - loss(pm)) / (2 * hh)
            assert abs(fd - grad[lot, k]) <= 2e-3 * max(1.0, abs(fd)), (lot, k, fd, grad[lot, k])


def _keys(inst):
    """(axiom << 32) | path of a (count, 16) instance tensor, as int64."""
    import torch
    ax = inst[:, 13].contiguous().view(torch.int32).long() & 0xFFFFFFFF
    pa = inst[:, 14].contiguous().view(torch.int32).long() & 0xFFFFFFFF
    return (ax << 32) | pa


@pytest.mark.parametrize("fused", [False, True])
def test_autograd_function_matches_fp64_adjoint(fused):
    """C4-style loss through torch.autograd: MSE of instance centres and
    sizes against targets derived with perturbed split parameters (same
    topology), written with torch ops or as the fused loss kernel, checked
    against the FP64 adjoint of the same dL/dinstance."""
    import torch
    from oracle import oracle as O
    from operatorgraph_amd import engine
    from operatorgraph_amd.autograd import center_size_mse, centers_and_sizes, derive_instances
    _note(f"autograd function, fused loss={fused}")
    ax, params = axioms.param_lots(32)
    rng = np.random.default_rng(4)
    tparams = params.copy()
    tparams[:, [0, 1, 4, 5, 6, 7]] += rng.normal(0, 0.05, size=(32, 6)).astype(np.float32)
    prog = grammars.facade_params()
    tgt_eng = _gpu_run(prog, ax, tparams, 2, tape=False)
    targets = [tgt_eng.buffer(t)[: int(tgt_eng.counts(2)[t])].clone() for t in range(2)]
    tgt_eng.close()
    eng = engine.Engine(queue_capacity=1 << 20)
    eng.load(prog).set_axioms(ax).set_axiom_params(params)
    eng.bind(0, 1 << 19)
    eng.bind(1, 1 << 19)
    eng.tape_reserve(1 << 20, 1 << 21)
    p = torch.from_numpy(params).cuda().requires_grad_(True)
    outs = derive_instances(p, eng, (0, 1))
    loss = 0.0
    for inst, tgt in zip(outs, targets):
        assert inst.shape == tgt.shape
        oi, ot = torch.argsort(_keys(inst)), torch.argsort(_keys(tgt))
        assert torch.equal(_keys(inst)[oi], _keys(tgt)[ot])
        ct, st = centers_and_sizes(tgt[ot])
        if fused:
            loss = loss + center_size_mse(inst[oi], ct, st)
        else:
            c, sz = centers_and_sizes(inst[oi])
            loss = loss + ((c - ct) ** 2).sum(1).mean() + ((sz - st) ** 2).sum(1).mean()
    g_inst = torch.autograd.grad(loss, outs, retain_graph=True)
    loss.backward()
    r = O.derive(prog, ax, params=params, twins=O.TWIN_F64 | O.TWIN_ADJ)
    dl = []
    for t in range(2):
        keys = _keys(outs[t]).cpu().numpy()
        row = {int(k): i for i, k in enumerate(keys)}
        ri = r.instances(t)
        rk = (ri["axiom"].astype(np.int64) << 32) | ri["path"].astype(np.int64)
        g = g_inst[t][:, :12].double().cpu().numpy()
        dl.append(np.stack([g[row[int(k)]] for k in rk]))
    ref = r.backward(dl)
    _assert_close(p.grad.double().cpu().numpy(), ref)
    eng.close()


def test_fused_center_size_loss_matches_torch():
    """pga_center_size_mse (one kernel: loss and gradient rows) against the
    same loss written with torch ops and differentiated by autograd, FP32
    tolerance 1e-5; zero-norm columns get a zero gradient, as torch's norm
    backward gives."""
    import torch
    from operatorgraph_amd.autograd import center_size_mse, centers_and_sizes
    _note("fused centre/size loss")
    gen = torch.Generator().manual_seed(3)
    n = 100_003
    inst = torch.randn(n, 16, generator=gen)
    inst[:7, 0] = inst[:7, 4] = inst[:7, 8] = 0.0
    inst = inst.cuda()
    tc = torch.randn(n, 3, generator=gen).cuda()
    ts = torch.rand(n, 3, generator=gen).cuda()
    for mean in (True, False):
        x = inst.clone().requires_grad_(True)
        c, s = centers_and_sizes(x)
        ref = ((c - tc) ** 2).sum(1) + ((s - ts) ** 2).sum(1)
        ref = ref.mean() if mean else ref.sum()
        (3.0 * ref).backward()
        y = inst.clone().requires_grad_(True)
        got = center_size_mse(y, tc, ts, mean=mean)
        (3.0 * got).backward()
        assert abs(got.item() - ref.item()) <= 1e-5 * abs(ref.item())
        gx, gy = x.grad.double(), y.grad.double()
        assert torch.all(gy[:, 12:] == 0)
        assert torch.all(gy[:7, [0, 4, 8]] == 0)
        err = (gx - gy).abs().max().item()
        assert err <= 1e-5 * gx.abs().max().item(), err


def test_backward_waits_for_torch_stream():
    """dL/dinstance written on torch's stream behind a busy kernel reaches
    the adjoint: the engine's own stream is ordered after torch's current
    stream (regression test: the engine stream does not wait for torch's
    default stream by itself)."""
    import torch
    _note("backward ordered after torch's stream")
    ax, params = axioms.param_lots(16)
    eng = _gpu_run(grammars.facade_params(), ax, params, 2)
    got = [eng.instances(t) for t in range(2)]
    want = {}
    for t in range(2):
        g = np.zeros((len(got[t]), 16), dtype=np.float32)
        g[:, :12] = _weights(got[t])
        want[t] = torch.from_numpy(g).cuda()
    ref = eng.backward(want).cpu().numpy()
    dl = {t: torch.zeros_like(want[t]) for t in range(2)}
    torch.cuda.synchronize()
    torch.cuda._sleep(50_000_000)          # a bounded spin on torch's stream
    for t in range(2):
        dl[t].copy_(want[t])               # queued behind the spin
    grad = eng.backward(dl).cpu().numpy()
    assert np.abs(ref).max() > 0
    np.testing.assert_array_equal(grad, ref)
    eng.close()


def test_adjoint_mixed_menger_and_lots_vs_fp64():
    """The mixed batch's forward + backward at reduced size: a Menger sponge
    (8,000 cubes) and 16 parameterised facade lots in one program
    (grammars.combine), one tape forward and one adjoint, against the FP64
    adjoint; the sponge's axiom reads no parameter and gets none."""
    _note("adjoint mixed menger-3 + 16 parameterised lots vs FP64 adjoint")
    prog, starts = grammars.combine((grammars.facade_params(), 0), (grammars.menger_interpreter(1.0), 2))
    lots, lparams = axioms.param_lots(16, perturb=0.05)
    ax = np.concatenate([axioms.menger_axiom(9.0, starts[1]), lots])
    params = np.zeros((len(ax), lparams.shape[1]), dtype=np.float32)
    params[1:] = lparams
    grad, ref, r = _adjoint_pair(prog, ax, params, 3)
    assert r.count(2) == 8000
    assert np.all(grad[0] == 0.0) and np.all(ref[0] == 0.0)
    assert np.abs(ref[1:]).max() > 0.0
    _assert_close(grad, ref)


def test_backward_refuses_a_replaced_tape():
    """A backward replays the engine's current tape: after another forward,
    or new parameters or axioms, the earlier forward's backward raises
    instead of returning another derivation's gradients."""
    import torch
    from operatorgraph_amd.autograd import derive_instances
    from operatorgraph_amd.engine import PGAError
    _note("backward after the tape changed")
    ax, params = axioms.param_lots(8, perturb=0.05)
    eng = _gpu_run(grammars.facade_params(), ax, params, 2)
    g0 = eng.tape_generation()
    assert g0 > 0
    p = torch.from_numpy(params).cuda()
    q1 = p.clone().requires_grad_(True)
    outs1 = derive_instances(q1, eng, (0, 1))
    q2 = p.clone().requires_grad_(True)
    outs2 = derive_instances(q2, eng, (0, 1))
    assert eng.tape_generation() > g0
    with pytest.raises(RuntimeError, match="tape changed"):
        sum(o[:, :12].sum() for o in outs1).backward()
    sum(o[:, :12].sum() for o in outs2).backward()     # the current tape replays
    assert q2.grad is not None and torch.isfinite(q2.grad).all()
    dl = {t: torch.ones((int(eng.counts(2)[t]), 16), dtype=torch.float32, device="cuda") for t in range(2)}
    for change in ("params", "axioms"):
        eng.forward_tape()
        assert eng.tape_generation() > 0
        if change == "params":
            eng.set_axiom_params(params)
        else:
            eng.set_axioms(ax)
        assert eng.tape_generation() == 0
        with pytest.raises(PGAError) as e:
            eng.backward(dl)
        assert e.value.status == abi.ERR_NOT_INITIALIZED
    eng.close()


@pytest.mark.parametrize("n", [1, 2, 21, 43, 64])
def test_adjoint_wave_edges_vs_fp64(n):
    """Levels whose children end inside a wave (3 children a box face, the
    adjoint's slots leave 64 at a time), every operator."""
    _note(f"adjoint at the edges of a wave n={n}")
    ax, params = _diff_axioms(n, seed=100 + n)
    grad, ref, _ = _adjoint_pair(_diff_grammar(), ax, params, 3)
    _assert_close(grad, ref)


@pytest.mark.parametrize("children", [1, 2, 7, 8, 9, 33])
def test_adjoint_axioms_sharing_a_wave(children):
    """A wave with the children of several axioms sums the parameters axiom by
    axiom, from eight children of one on: Repeat(X, 1) Translate(p0, p1, 0)
    Scale(p2, -1, -1) Generate(0) over `children` tiles each. FP32 terms of
    both signs, whose sum can cancel: their rounding is held against the
    largest parameter of the axiom, and an entry only loosely against itself
    (the next test holds the sums exactly)."""
    _note(f"adjoint of {children} children an axiom")
    table = DispatchTable([
        Entry(op(abi.REPEAT, Q), [Scalar(abi.X), Scalar(1.0), Scalar(abi.ADJUST_TO_FILL)], [(1, 0)]),
        Entry(op(abi.TRANSLATE, Q), [AxiomParam(0), AxiomParam(1), Scalar(0.0)], [(2, 0)]),
        Entry(op(abi.SCALE, Q), [AxiomParam(2), Scalar(-1.0), Scalar(-1.0)], [(3, 0)]),
        Entry(op(abi.GENERATE, Q, 1), [Scalar(0)], []),
    ])
    n = 37
    rng = np.random.default_rng(children)
    ax = axioms.empty(n)
    ax["size"] = np.stack([np.full(n, children + 0.25), rng.uniform(1, 2, n), np.zeros(n)], axis=1)
    ax["model"][:, [3, 7, 11]] = rng.uniform(-5, 5, size=(n, 3)).astype(np.float32)
    ax["shape_type"] = Q
    params = rng.uniform(0.2, 0.8, size=(n, 3)).astype(np.float32)
    grad, ref, r = _adjoint_pair(Program(grammars.INTERPRETER_PROCEDURES, table, "tiles"), ax, params, 1)
    assert r.count(0) == n * children
    _assert_close(grad, ref, rel=1e-4, entry_rel=5e-2)


def _whole_weights(inst):
    """Whole numbers from -2 to 2 by (axiom, path), none of a row's zero."""
    key = inst["axiom"].astype(np.int64)[:, None] * 31 + (inst["path"].astype(np.int64) % 97)[:, None] * 7
    w = (key + np.arange(12)[None, :] * 3) % 4 - 2
    return np.where(w >= 0, w + 1, w).astype(np.float64)


@pytest.mark.parametrize("children", [1, 2, 7, 8, 9, 33, 64, 65])
@pytest.mark.parametrize("slots", [3, 8, 9])
def test_adjoint_axioms_sharing_a_wave_exactly(children, slots):
    """The same sums with every term exact: sizes, positions and parameters
    are multiples of 1/8, weights are whole numbers, so that FP32 terms and
    FP64 sums have no rounding and the gradients are the oracle's to the last
    bit. A term lost, doubled or given to another axiom shows. slots: three
    parameters that are used, at the ends of a row of `slots` (more than eight
    go past the sums in LDS)."""
    _note(f"adjoint of {children} children an axiom, {slots} parameters, exactly")
    last = slots - 1
    table = DispatchTable([
        Entry(op(abi.REPEAT, Q), [Scalar(abi.X), Scalar(1.0), Scalar(abi.ADJUST_TO_FILL)], [(1, 0)]),
        Entry(op(abi.TRANSLATE, Q), [AxiomParam(0), AxiomParam(last), Scalar(0.0)], [(2, 0)]),
        Entry(op(abi.SCALE, Q), [AxiomParam(1), Scalar(-1.0), Scalar(-1.0)], [(3, 0)]),
        Entry(op(abi.GENERATE, Q, 1), [Scalar(0)], []),
    ])
    n = 37
    rng = np.random.default_rng(children)
    ax = axioms.empty(n)
    ax["size"] = np.stack([np.full(n, float(children)), rng.integers(8, 17, n) / 8.0, np.zeros(n)], axis=1)
    ax["model"][:, [3, 7, 11]] = rng.integers(-40, 41, size=(n, 3)) / 8.0
    ax["shape_type"] = Q
    params = (rng.integers(2, 8, size=(n, slots)) / 8.0).astype(np.float32)
    grad, ref, r = _adjoint_pair(Program(grammars.INTERPRETER_PROCEDURES, table, "tiles"), ax, params, 1,
                                 weights=_whole_weights)
    assert r.count(0) == n * children and np.abs(ref).max() > 0
    assert np.array_equal(grad, ref), np.abs(grad - ref).max()


@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 513, 512 * 512 - 1, 512 * 512 + 65])
def test_fused_loss_tile_edges(n):
    """The fused loss at the edges of a wave's tile, a workgroup and the
    whole grid (then a workgroup takes a second tile), against FP64 torch."""
    import torch
    from operatorgraph_amd.autograd import center_size_mse, centers_and_sizes
    _note(f"fused loss tiles n={n}")
    gen = torch.Generator(device="cuda").manual_seed(n)
    inst = torch.randn(n, 16, generator=gen, device="cuda").requires_grad_(True)
    tc = torch.randn(n, 3, generator=gen, device="cuda")
    ts = torch.rand(n, 3, generator=gen, device="cuda")
    loss = center_size_mse(inst, tc, ts, mean=False)
    (g,) = torch.autograd.grad(loss, inst)
    ref = inst.detach().double().requires_grad_(True)
    c, s = centers_and_sizes(ref)
    rl = ((c - tc) ** 2).sum() + ((s - ts) ** 2).sum()
    (rg,) = torch.autograd.grad(rl, ref)
    # FP32 terms of order 1 a row, summed in FP64
    assert abs(loss.item() - rl.item()) <= 1e-5 * rl.item()
    assert float((g - rg).abs().max()) <= 1e-5 * float(rg.abs().max())


def test_axiom_params_from_device_tensors():
    """Device tensors (any layout, float64 too) bind the same values as a
    numpy array, and are copied before the call returns."""
    import torch
    from operatorgraph_amd import engine
    _note("axiom parameters from device tensors")
    ax, params = axioms.param_lots(24, perturb=0.05)
    ref = _gpu_run(grammars.facade_params(), ax, params, 2, tape=False)
    want = [ref.instances(t) for t in range(2)]
    ref.close()
    dev = torch.from_numpy(params).cuda()
    forms = [dev.clone(), dev.double(), dev.t().contiguous().t(), torch.cat([dev, dev], dim=1)[:, :8]]
    eng = engine.Engine(queue_capacity=1 << 20)
    eng.load(grammars.facade_params()).set_axioms(ax)
    for t in range(2):
        eng.bind(t, 1 << 18)
    for p in forms:
        eng.set_axiom_params(p)
        p.zero_()
        eng.execute()
        for t in range(2):
            assert_same_multiset(eng.instances(t), want[t], f"terminal {t}")
    eng.close()


@pytest.mark.parametrize("form", ["negative", "imaginary"])
def test_axiom_params_from_lazy_views(form):
    """Device tensors whose memory does not hold their values (torch's negative
    views, the imaginary part of a conjugate) bind their values, too."""
    import torch
    from operatorgraph_amd import engine
    _note(f"axiom parameters from a {form} view")
    ax, params = axioms.param_lots(24, perturb=0.05)
    dev = torch.from_numpy(params).cuda()
    if form == "negative":
        view = torch._neg_view(-dev)
    else:
        view = torch.complex(torch.zeros_like(dev), -dev).conj().imag
    assert view.is_neg() and torch.equal(view, dev)
    eng = engine.Engine(queue_capacity=1 << 20)
    eng.load(grammars.facade_params()).set_axioms(ax).set_axiom_params(view)
    for t in range(2):
        eng.bind(t, 1 << 18)
    eng.execute()
    got = [eng.instances(t) for t in range(2)]
    eng.set_axiom_params(params)
    eng.execute()
    for t in range(2):
        assert_same_multiset(got[t], eng.instances(t), f"terminal {t}")
    eng.close()
