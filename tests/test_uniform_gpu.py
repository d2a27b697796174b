"""GPU parity of the uniform periodic multigrid (mg.F90 path) against the CPU oracle.

FP64 kernels and the plain FP64 solve must be bit-for-bit equal to the oracle (same operand
order, no FMA contraction on either side).  FP32 kernels are compared within FP32 rounding, and
the mixed-precision solve is checked by its FP64 residual (recomputed here with numpy) and by its
distance to the FFT solution."""
import numpy as np
import pytest
import torch

import oracle
from oracle import fft_poisson as fp
from code_only_amd import problems
from code_only_amd._lib import SgError
from code_only_amd.uniform import (SG_COARSE_EXACT, SG_COARSE_VCYCLE, SG_PREC_FP64, SG_PREC_MIXED,
                                   SG_STOP_REFERENCE, SG_STOP_TRUE_RESIDUAL, UniformSolver)

pytestmark = pytest.mark.gpu


def rand(n, seed):
    return np.random.default_rng(seed).standard_normal((n, n, n))


def T(a, dev, dtype=torch.float64):
    return torch.tensor(a, dtype=dtype, device=dev).contiguous()


@pytest.fixture(scope="module")
def solver64(gpu):
    s = UniformSolver(64, precisions=SG_PREC_FP64 | SG_PREC_MIXED)
    yield s
    s.close()


@pytest.mark.parametrize("n", [1, 2, 4, 16, 64])
def test_relax_bitwise(solver64, gpu, n):
    h = 1.0 / n
    u = rand(n, 10 + n)
    f = rand(n, 20 + n)
    ug = T(u, gpu)
    rm = solver64.relax(ug, T(f, gpu), h)
    rm_ref = oracle.relax(u, f, h)
    assert np.array_equal(ug.cpu().numpy(), u)
    assert rm == rm_ref


@pytest.mark.parametrize("n", [2, 8, 64])
def test_resid_bitwise(solver64, gpu, n):
    h = 1.0 / n
    u, f = rand(n, 1), rand(n, 2)
    res = solver64.resid(T(u, gpu), T(f, gpu), h).cpu().numpy()
    assert np.array_equal(res, oracle.resid(u, f, h))


@pytest.mark.parametrize("nc", [1, 4, 32])
def test_restrict_bitwise(solver64, gpu, nc):
    uf = rand(2 * nc, 3)
    assert np.array_equal(solver64.restrict(T(uf, gpu)).cpu().numpy(), oracle.restrict(uf))


@pytest.mark.parametrize("nc", [1, 2, 3, 16, 32])
@pytest.mark.parametrize("cubic", [False, True])
def test_interp_bitwise(solver64, gpu, nc, cubic):
    if nc == 3:
        pytest.skip("odd coarse sizes do not occur on power-of-two hierarchies")
    uc = rand(nc, 4)
    got = solver64.interp(T(uc, gpu), cubic).cpu().numpy()
    assert np.array_equal(got, oracle.interp(uc, cubic))


@pytest.mark.parametrize("cubic", [False, True])
def test_fp32_kernels_within_rounding(solver64, gpu, cubic):
    n, h = 32, 1.0 / 32
    u, f = rand(n, 5), rand(n, 6)
    r32 = solver64.resid(T(u, gpu, torch.float32), T(f, gpu, torch.float32), h, prec=SG_PREC_MIXED).double().cpu().numpy()
    r64 = oracle.resid(u.astype(np.float32).astype(np.float64), f.astype(np.float32).astype(np.float64), h)
    assert np.max(np.abs(r32 - r64)) <= 2e-6 * np.max(np.abs(r64))
    ug = T(u, gpu, torch.float32)
    solver64.relax(ug, T(f, gpu, torch.float32), h, prec=SG_PREC_MIXED)
    u64 = u.astype(np.float32).astype(np.float64)
    oracle.relax(u64, f.astype(np.float32).astype(np.float64), h)
    assert np.max(np.abs(ug.double().cpu().numpy() - u64)) <= 2e-6 * np.max(np.abs(u64))
    uc = rand(16, 7)
    i32 = solver64.interp(T(uc, gpu, torch.float32), cubic, prec=SG_PREC_MIXED).double().cpu().numpy()
    i64 = oracle.interp(uc.astype(np.float32).astype(np.float64), cubic)
    assert np.max(np.abs(i32 - i64)) <= 1e-6 * np.max(np.abs(i64))


@pytest.mark.parametrize("n", [16, 64])
def test_plain_fp64_cycle_bitwise(gpu, n):
    f = problems.clumpy_rhs(n, seed=3)
    h = 1.0 / n
    s = UniformSolver(n, precisions=SG_PREC_FP64)
    psi = torch.zeros((n, n, n), dtype=torch.float64, device=gpu)
    st = s.cycle(psi, T(f, gpu), tol=1e-10, maxit=30, precision=SG_PREC_FP64)
    ref, st_ref = oracle.mg_cycle(f, h, tol=1e-10, maxit=30)
    assert st["iterations"] == st_ref["iterations"]
    assert np.array_equal(psi.cpu().numpy(), ref)
    assert st["rel_linf"] == st_ref["rel_linf"] and st["rel_linf"] < 1e-10
    g = s.gradient(psi).cpu().numpy()
    assert np.array_equal(g, oracle.gradient(ref, h))
    s.close()


def test_plain_fp64_reference_stop_mode(gpu):
    n = 32
    f = problems.clumpy_rhs(n, seed=4)
    s = UniformSolver(n, precisions=SG_PREC_FP64)
    psi = torch.zeros((n, n, n), dtype=torch.float64, device=gpu)
    st = s.cycle(psi, T(f, gpu), tol=1e-2, maxit=10, stop_mode=SG_STOP_REFERENCE, precision=SG_PREC_FP64)
    ref, st_ref = oracle.mg_cycle(f, 1.0 / n, tol=1e-2, maxit=10, mode=oracle.STOP_REFERENCE)
    assert st["iterations"] == st_ref["iterations"]
    assert st["resmaxg"] == st_ref["resmaxg"]
    assert np.array_equal(psi.cpu().numpy(), ref)
    s.close()


@pytest.mark.parametrize("use_graph", [False, True])
def test_mixed_cycle_converges_and_matches_oracle(gpu, use_graph):
    n = 64
    h = 1.0 / n
    f = problems.clumpy_rhs(n, seed=0)
    s = UniformSolver(n, precisions=SG_PREC_MIXED)
    psi = torch.zeros((n, n, n), dtype=torch.float64, device=gpu)
    st = s.cycle(psi, T(f, gpu), tol=1e-10, maxit=30, precision=SG_PREC_MIXED, use_graph=use_graph)
    p = psi.cpu().numpy()
    r = f - fp.apply_laplacian(p, h)
    assert np.max(np.abs(r)) / np.max(np.abs(f)) < 1e-10
    assert abs(np.max(np.abs(r)) / np.max(np.abs(f)) - st["rel_linf"]) < 1e-12
    ref = fp.solve(f, h)
    err = np.linalg.norm((p - p.mean()) - ref) / np.linalg.norm(ref)
    assert err < 1e-9
    # replaying the captured graph a second time gives the same answer
    psi2 = torch.zeros_like(psi)
    st2 = s.cycle(psi2, T(f, gpu), tol=1e-10, maxit=30, precision=SG_PREC_MIXED, use_graph=use_graph)
    assert st2["iterations"] == st["iterations"]
    assert torch.equal(psi, psi2)
    s.close()


def test_host_pointer_entry_matches_device_entry(gpu):
    """sg_uniform_cycle_host takes the reference's ghosted u(-1:n,...) layout."""
    import ctypes
    from code_only_amd import _lib
    n = 16
    h = 1.0 / n
    f = problems.clumpy_rhs(n, seed=9)
    s = UniformSolver(n, precisions=SG_PREC_FP64)
    fg = np.pad(f, 1, mode="wrap")
    pg = np.zeros_like(fg)
    p = _lib.default_params(tol=1e-10, maxit=30, stop_mode=SG_STOP_TRUE_RESIDUAL, precision=SG_PREC_FP64)
    st = _lib.SgStats()
    dp = ctypes.POINTER(ctypes.c_double)
    rc = s._lib.sg_uniform_cycle_host(s._ctx, pg.ctypes.data_as(dp), fg.ctypes.data_as(dp), ctypes.byref(p),
                                      ctypes.byref(st))
    _lib.check(rc)
    ref, _ = oracle.mg_cycle(f, h, tol=1e-10, maxit=30)
    assert np.array_equal(pg, np.pad(ref, 1, mode="wrap"))
    s.close()


def test_full_size_256_mixed_vs_plain(gpu):
    """256^3 (the benchmark workload): both solvers reach 1e-10 by an independent FP64 residual
    and agree with each other; the FFT solution pins both."""
    n = 256
    h = 1.0 / n
    f = problems.clumpy_rhs(n, seed=0)
    ft = T(f, gpu)
    s = UniformSolver(n)
    out = {}
    for prec in (SG_PREC_FP64, SG_PREC_MIXED):
        psi = torch.zeros_like(ft)
        st = s.cycle(psi, ft, tol=1e-10, maxit=40, precision=prec)
        # independent residual with torch.roll in FP64
        lap = -6.0 * psi
        for ax in range(3):
            lap = lap + torch.roll(psi, 1, ax) + torch.roll(psi, -1, ax)
        r = ft - lap / (h * h)
        rel = (r.abs().max() / ft.abs().max()).item()
        assert rel < 1e-10, (prec, rel, st)
        out[prec] = psi - psi.mean()
    d = (out[SG_PREC_FP64] - out[SG_PREC_MIXED]).norm() / out[SG_PREC_FP64].norm()
    assert d.item() < 1e-9
    ref = torch.tensor(fp.solve(f, h), device=gpu)
    e = (out[SG_PREC_FP64] - ref).norm() / ref.norm()
    assert e.item() < 1e-9
    s.close()


@pytest.mark.parametrize("n", [16, 32, 64, 128])
@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("coarse", [SG_COARSE_EXACT, SG_COARSE_VCYCLE])
def test_fused_mixed_equals_unfused_bitwise(gpu, n, use_graph, coarse):
    """The fused FP32 kernels (LDS tiles, single-workgroup coarse solve) reproduce the
    one-kernel-per-loop FP32 inner solve bit for bit, including Resmaxg, with either coarse-grid
    solve (exact at 16^3, or the reference's levels down to 1^3)."""
    f = problems.clumpy_rhs(n, seed=11)
    s = UniformSolver(n, precisions=SG_PREC_MIXED)
    ft = T(f, gpu)
    out = []
    for fused in (False, True):
        psi = torch.zeros_like(ft)
        st = s.cycle(psi, ft, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, fused=fused, use_graph=use_graph,
                     coarse=coarse)
        out.append((psi, st))
    (p0, s0), (p1, s1) = out
    assert s0["iterations"] == s1["iterations"]
    assert s0["resmaxg"] == s1["resmaxg"]
    assert torch.equal(p0, p1)
    s.close()


def test_fused_mixed_equals_unfused_bitwise_256(gpu):
    """At 256^3 the fused update + residual step runs in 256 x 4 patches (grid-wide rows); it still
    reproduces the separate update, residual and restriction kernels bit for bit."""
    n = 256
    f = problems.clumpy_rhs(n, seed=3)
    s = UniformSolver(n, precisions=SG_PREC_MIXED)
    ft = T(f, gpu)
    out = []
    for fused in (False, True):
        psi = torch.zeros_like(ft)
        st = s.cycle(psi, ft, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, fused=fused)
        out.append((psi, st))
    (p0, s0), (p1, s1) = out
    assert s0["iterations"] == s1["iterations"]
    assert s0["resmaxg"] == s1["resmaxg"]
    assert torch.equal(p0, p1)
    s.close()


@pytest.mark.parametrize("n", [64, 128])
def test_repeated_fused_solves_bitwise(gpu, n):
    """Consecutive fused mixed solves on one context start their phi ping-pong from psi or from its
    copy in the second buffer (chosen by the previous solve's iteration parity, so that an odd count
    ends in psi); every solve gives the same phi, statistics and Resmaxg bit for bit, from a zero
    and from a non-zero initial guess."""
    f = problems.clumpy_rhs(n, seed=5)
    ft = T(f, gpu)
    g0 = T(0.01 * rand(n, 6), gpu)
    s = UniformSolver(n, precisions=SG_PREC_MIXED)
    for init in (torch.zeros_like(ft), g0):
        outs = []
        for _ in range(3):
            psi = init.clone()
            st = s.cycle(psi, ft, tol=1e-10, maxit=30, precision=SG_PREC_MIXED)
            outs.append((psi, st))
        (p0, s0) = outs[0]
        assert s0["status"] == 0
        for p1, s1 in outs[1:]:
            assert s1["iterations"] == s0["iterations"]
            assert s1["resmaxg"] == s0["resmaxg"] and s1["rel_linf"] == s0["rel_linf"]
            assert torch.equal(p1, p0)
    s.close()


@pytest.mark.parametrize("n", [32, 128])
def test_exact_coarse_solve_contracts_at_least_as_well(gpu, n):
    """Solving the 16^3 level exactly (instead of the V-cycle below it) keeps the mixed solve's
    contraction: the first outer iteration reduces the residual at least as much (up to 5 %) as
    with the reference's coarse levels (later ones sit at the FP32 inner solve's round-off level),
    it takes no more iterations, and the result matches the FP64 solve."""
    f = problems.clumpy_rhs(n, seed=21)
    s = UniformSolver(n, precisions=SG_PREC_MIXED | SG_PREC_FP64)
    ft = T(f, gpu)
    hs = {}
    for coarse in (SG_COARSE_EXACT, SG_COARSE_VCYCLE):
        psi = torch.zeros_like(ft)
        st = s.cycle(psi, ft, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, coarse=coarse)
        hs[coarse] = (st, psi - psi.mean())
    p64 = torch.zeros_like(ft)
    s.cycle(p64, ft, tol=1e-12, maxit=30, precision=SG_PREC_FP64)
    p64 -= p64.mean()
    ex, vc = hs[SG_COARSE_EXACT][0], hs[SG_COARSE_VCYCLE][0]
    print("exact", ex["iterations"], ex["hist"], "vcycle", vc["iterations"], vc["hist"], flush=True)
    assert ex["iterations"] <= vc["iterations"]
    assert ex["hist"][1] <= 1.05 * vc["hist"][1]
    e = ((hs[SG_COARSE_EXACT][1] - p64).norm() / p64.norm()).item()
    assert e < 1e-9, e
    s.close()


STREAM_CFGS = list(range(5, 14))   # streaming sweep shapes


@pytest.mark.parametrize("n", [32, 64, 128])
@pytest.mark.parametrize("cfg", STREAM_CFGS + [0, 4])
def test_every_sweep_shape_bitwise(gpu, n, cfg):
    """Each sweep configuration, forced on every fused level where it fits, reproduces the unfused
    FP32 solve bit for bit (its plain, zero-start, prolongation and residual variants all run)."""
    f = problems.clumpy_rhs(n, seed=13)
    s = UniformSolver(n, precisions=SG_PREC_MIXED)
    ft = T(f, gpu)
    forced = 0
    lev, m = 0, n
    while m > 16:
        try:
            s.set_tile(lev, cfg, 1, 0)
            forced += 1
        except Exception:
            pass
        lev += 1
        m //= 2
    if not forced:
        pytest.skip(f"configuration {cfg} fits no level of n = {n}")
    res = []
    for fused in (False, True):
        psi = torch.zeros_like(ft)
        st = s.cycle(psi, ft, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, fused=fused,
                     stop_mode=SG_STOP_REFERENCE, raise_on_fail=False)
        res.append((psi, st))
    assert torch.equal(res[0][0], res[1][0])
    assert res[0][1]["resmaxg"] == res[1][1]["resmaxg"]
    s.close()


@pytest.mark.parametrize("cfg", STREAM_CFGS)
def test_stream_numbers_keep_their_widths(gpu, cfg):
    """A streaming shape's number takes every level width it has taken, whatever shape stands behind it."""
    narrowest = {5: 64, 6: 64, 7: 64, 8: 32, 9: 64, 10: 32, 11: 32, 12: 32, 13: 32}[cfg]
    s = UniformSolver(128, precisions=SG_PREC_MIXED)
    for lev, m in ((0, 128), (1, 64), (2, 32)):
        if m >= narrowest:
            s.set_tile(lev, cfg, 1, 0)
            assert s.tile_info(lev)["cfg"] == cfg
        else:
            with pytest.raises(SgError):
                s.set_tile(lev, cfg, 1, 0)
    s.close()


@pytest.mark.parametrize("npre,npost", [(2, 2), (3, 1)])
@pytest.mark.parametrize("n", [32, 64, 128])
@pytest.mark.parametrize("cfg", STREAM_CFGS + [14, 15, 16])
def test_streams_of_two_sweeps_bitwise(gpu, n, cfg, npre, npost):
    """The streaming shapes with two sweeps per launch (and the odd sweep alone), forced where they
    fit, against the unfused FP32 solve, bit for bit; columns that meet their own periodic images
    (n equal to the shape's width) included."""
    s = UniformSolver(n, precisions=SG_PREC_MIXED)
    ft = T(problems.clumpy_rhs(n, seed=14), gpu)
    forced, lev, m = 0, 0, n
    while m > 16:
        try:
            s.set_tile(lev, cfg, 2, 0)
            forced += 1
        except Exception:
            pass
        lev += 1
        m //= 2
    if not forced:
        pytest.skip(f"configuration {cfg} fits no level of n = {n}")
    res = []
    for fused in (False, True):
        psi = torch.zeros_like(ft)
        st = s.cycle(psi, ft, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, fused=fused, npre=npre, npost=npost,
                     stop_mode=SG_STOP_REFERENCE, raise_on_fail=False)
        res.append((psi, st))
    assert torch.equal(res[0][0], res[1][0])
    assert res[0][1]["resmaxg"] == res[1][1]["resmaxg"]
    s.close()


@pytest.mark.parametrize("npre,npost,ncycle", [(1, 1, 1), (3, 2, 2), (2, 3, 1)])
def test_fused_other_cycle_shapes_bitwise(gpu, npre, npost, ncycle):
    n = 64
    f = problems.clumpy_rhs(n, seed=12)
    s = UniformSolver(n, precisions=SG_PREC_MIXED)
    ft = T(f, gpu)
    res = []
    for fused in (False, True):
        psi = torch.zeros_like(ft)
        st = s.cycle(psi, ft, tol=1e-10, maxit=40, precision=SG_PREC_MIXED, fused=fused, npre=npre, npost=npost,
                     ncycle=ncycle, stop_mode=SG_STOP_REFERENCE, raise_on_fail=False)
        res.append((psi, st))
    assert torch.equal(res[0][0], res[1][0])
    assert res[0][1]["resmaxg"] == res[1][1]["resmaxg"]
    s.close()


@pytest.mark.parametrize("cycle", [(2, 2, 2), (1, 3, 1), (2, 1, 2)])
@pytest.mark.parametrize("n", [2, 4, 8, 16, 32, 64, 128, 256])
def test_fp64_fused_equals_plain(n, cycle, gpu):
    """The fused FP64 solve (one launch for n <= 16, k_coarse from the 16^3 level down for the others, of
    the rule's sweep shapes the 8^3 tile at 32, the 16 x 8 x 8 tile at 64 and the streams of 32 x 16 columns
    in chunks of 16 planes at 128 and 64 at 256; odd sweep counts) against one kernel per loop nest,
    bit for bit, in both stopping modes, and again with other phi and source arrays (the graph is
    the context's own)."""
    import torch
    s = UniformSolver(n, 1.0 / n, precisions=SG_PREC_FP64)
    try:
        for seed, stop in ((3, SG_STOP_TRUE_RESIDUAL), (4, SG_STOP_REFERENCE), (5, SG_STOP_TRUE_RESIDUAL)):
            f = torch.tensor(problems.clumpy_rhs(n, seed=seed), device=gpu)
            out = []
            for fused in (True, False):
                psi = torch.zeros_like(f)
                st = s.cycle(psi, f, tol=1e-9, maxit=4, stop_mode=stop, precision=SG_PREC_FP64, ncycle=cycle[0],
                             npre=cycle[1], npost=cycle[2], fused=fused, raise_on_fail=False)
                out.append((psi, st))
            (a, sa), (b, sb) = out
            assert torch.equal(a, b)
            assert sa["iterations"] == sb["iterations"] and sa["rel_linf"] == sb["rel_linf"]
            assert sa["resmaxg"] == sb["resmaxg"] if stop == SG_STOP_REFERENCE else True
    finally:
        s.close()


@pytest.mark.parametrize("n", [2, 4, 8, 16])
def test_small_grid_mixed_equals_unfused(n, gpu):
    """The one-launch mixed solve of n <= 16 against one kernel per loop nest, bit for bit, from a
    non-zero guess, with maxit 0, a zero source and a NaN in it."""
    import torch
    s = UniformSolver(n, 1.0 / n, precisions=SG_PREC_MIXED)
    f = torch.tensor(problems.clumpy_rhs(n, seed=8), device=gpu)
    guess = torch.tensor(np.random.default_rng(9).standard_normal((n, n, n)), device=gpu)
    bad = f.clone()
    bad[0, 0, 0] = float("nan")
    try:
        for src, start, kw in ((f, None, {}), (f, guess, {}), (f, guess, dict(stop_mode=SG_STOP_REFERENCE, tol=1e-2)),
                               (f, guess, dict(maxit=0)), (torch.zeros_like(f), None, {}), (bad, None, {})):
            out = []
            for fused in (True, False):
                psi = torch.zeros_like(f) if start is None else start.clone()
                st = s.cycle(psi, src, precision=SG_PREC_MIXED, fused=fused, raise_on_fail=False,
                             **dict(dict(tol=1e-9, maxit=6), **kw))
                out.append((psi, st))
            (a, sa), (b, sb) = out
            assert torch.equal(torch.nan_to_num(a, nan=7.0), torch.nan_to_num(b, nan=7.0))
            assert sa["iterations"] == sb["iterations"] and sa["status"] == sb["status"]
            assert sa["hist"] == sb["hist"] or sa["status"] == 4
    finally:
        s.close()


@pytest.mark.parametrize("prec,word", [(SG_PREC_FP64, 8), (SG_PREC_MIXED, 4)])
def test_context_memory(prec, word, gpu):
    """A context holds three arrays per level and a second phi: 3 x 8/7 words and 8 bytes per cell."""
    n = 256
    UniformSolver(n, precisions=prec).close()   # the runtime's own memory (code, queues) is there from here on
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    s = UniformSolver(n, precisions=prec)
    used = free0 - torch.cuda.mem_get_info()[0]
    s.close()
    print(used / n ** 3, flush=True)
    # 0.2 bytes per cell of norm partials, and 16 MiB for the allocator's granularity and small tables
    assert used <= (3 * 8 / 7 * word + 8 + 0.2) * n ** 3 + (16 << 20)
