"""GPU parity of the AMR solve (fmg.F90 / vmg.F90 path) against the CPU oracle (oracle/amr.c).

Operator by operator: the oracle and the GPU library start from the same random state -- every
array of every code at every FMG level, ghosts included -- run one reference operation, and every
array must then be bit-for-bit equal.  The full solve is compared bit for bit as well (FP64, same
operand order, no FMA contraction, fixed summation orders), up to a 2048-block sphere hierarchy.
The mixed-precision solve is compared with the oracle's converged FP64 solution on the small
hierarchies, and on the 20 480-block sphere hierarchy with a tightly converged FP64 GPU solve."""
import numpy as np
import pytest

import oracle
from code_only_amd import amr_hierarchy as ah
from code_only_amd import problems
from code_only_amd.amr import SG_PREC_MIXED, AmrSolver

pytestmark = pytest.mark.gpu

OPS = oracle


def hierarchies():
    return {
        "periodic": ah.random_hierarchy(4, 3, 0.35, seed=7, bc=ah.PERIODIC),
        "sphere": ah.nested(base=4, levels=3, bc=ah.SPHERE),
    }


@pytest.fixture(scope="module")
def pair(gpu):
    out = {}
    for name, h in hierarchies().items():
        out[name] = (h, oracle.Amr(h), AmrSolver(h))
    yield out
    for h, o, g in out.values():
        o.close()
        g.close()


def randomize(h, o, g, seed):
    rng = np.random.default_rng(seed)
    for L in range(3):
        n = 8 >> L
        for code in range(6):
            a = rng.standard_normal((h.nblk, n + 2, n + 2, n + 2))
            o.set(L, code, a)
            g.set(L, code, a)


def assert_same_state(h, o, g, what):
    for L in range(3):
        for code in range(6):
            a, b = o.get(L, code), g.get(L, code)
            if not np.array_equal(a, b):
                bad = np.argwhere(a != b)
                d = np.abs(a - b).max()
                raise AssertionError(f"{what}: FMG level {L} code {code}: {len(bad)} elements differ "
                                     f"(first {bad[0].tolist()}, max |diff| {d:.3e})")


CASES = [
    ("c2p", OPS.OP_C2P, dict(L=0, a=OPS.U, flag=0)),
    ("c2p-cubic", OPS.OP_C2P, dict(L=0, a=OPS.U, flag=1)),
    ("c2p-L1-cubic", OPS.OP_C2P, dict(L=1, a=OPS.RES, flag=1)),
    ("c2p-L2", OPS.OP_C2P, dict(L=2, a=OPS.RHS, flag=0)),
    ("ghostfix-L0", OPS.OP_GHOSTFIX, dict(L=0, a=OPS.U, flag=0)),
    ("ghostfix-L1-cubic", OPS.OP_GHOSTFIX, dict(L=1, a=OPS.U, flag=1)),
    ("ghostfix-L0-cubic", OPS.OP_GHOSTFIX, dict(L=0, a=OPS.PSI, flag=1)),
    ("ghostfix-L2", OPS.OP_GHOSTFIX, dict(L=2, a=OPS.U, flag=1)),
    # one launch per level (the inner solve's form), same values as the staged passes
    ("ghostfix-onepass-L0", OPS.OP_GHOSTFIX, dict(L=0, a=OPS.U, flag=2)),
    ("ghostfix-onepass-L1-cubic", OPS.OP_GHOSTFIX, dict(L=1, a=OPS.U, flag=3)),
    ("ghostfix-onepass-L0-cubic", OPS.OP_GHOSTFIX, dict(L=0, a=OPS.PSI, flag=3)),
    ("ghostfix-onepass-L2", OPS.OP_GHOSTFIX, dict(L=2, a=OPS.RES, flag=3)),
    ("fill0-L0", OPS.OP_FILL0, dict(L=0, a=OPS.U)),
    ("extrap-L1", OPS.OP_EXTRAP, dict(L=1, a=OPS.U)),
    ("relax-L0", OPS.OP_RELAX, dict(L=0, a=OPS.U, b=OPS.RHS, flag=0)),
    ("relax-L0-fill0", OPS.OP_RELAX, dict(L=0, a=OPS.U, b=OPS.RHS, flag=1)),
    ("relax-L1-fill0", OPS.OP_RELAX, dict(L=1, a=OPS.U, b=OPS.RHS, flag=1)),
    ("resid-L0", OPS.OP_RESID, dict(L=0, a=OPS.RHO, b=OPS.PSI, c=OPS.SRC, flag=0)),
    ("resid-L1-fill0", OPS.OP_RESID, dict(L=1, a=OPS.RES, b=OPS.U, c=OPS.RHS, flag=1)),
    ("rstrct-L1", OPS.OP_RSTRCT, dict(L=1, a=OPS.RHO, b=OPS.RHO)),
    ("rstrct-L2", OPS.OP_RSTRCT, dict(L=2, a=OPS.RHS, b=OPS.RES)),
    ("interp-L1-cubic", OPS.OP_INTERP, dict(L=1, a=OPS.U, b=OPS.U, flag=1)),
    ("interp-L0-cubic", OPS.OP_INTERP, dict(L=0, a=OPS.U, b=OPS.U, flag=1)),
    ("interp-L0-linear", OPS.OP_INTERP, dict(L=0, a=OPS.RES, b=OPS.U, flag=0)),
    ("addint-L1", OPS.OP_ADDINT, dict(L=1, a=OPS.U, b=OPS.U, c=OPS.RES)),
    ("vmg-fas-rho", OPS.OP_VMG_FAS, dict(a=OPS.RHO)),
    ("vmg-fas-rhs", OPS.OP_VMG_FAS, dict(a=OPS.RHS)),
    ("vmg-tau-l0", OPS.OP_VMG_TAU, dict(L=2, a=OPS.RES, b=OPS.U, flag=0)),
    ("vmg-tau-l1", OPS.OP_VMG_TAU, dict(L=2, a=OPS.RES, b=OPS.U, flag=1)),
    ("fmg-lin", OPS.OP_FMG_LIN, dict()),
]


@pytest.mark.parametrize("name", ["periodic", "sphere"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_operator_bitwise(pair, name, case):
    label, opc, kw = case
    h, o, g = pair[name]
    randomize(h, o, g, seed=hash(label) % 1000)
    for fl in (-1, kw.get("L", 0)) if opc == OPS.OP_RELAX else (-1,):
        o.fill0_level = fl
        g.fill0_level = fl
        ro = o.op(opc, **kw)
        rg = g.op(opc, **kw)
        assert ro == rg, f"{label}: returned {ro!r} vs {rg!r}"
        assert o.fill0_level == g.fill0_level
        assert_same_state(h, o, g, f"{name}/{label}/fill0_level={fl}")


def test_sphere_bc_bitwise(pair):
    h, o, g = pair["sphere"]
    randomize(h, o, g, seed=99)
    src = ah.to_blocks(h, lambda x, y, z: 1.0 / (x * x + y * y + z * z + 1e-3))
    pad = np.zeros((h.nblk, 10, 10, 10))
    pad[:, 1:-1, 1:-1, 1:-1] = src
    o.set(0, OPS.SRC, pad)
    g.set(0, OPS.SRC, pad)
    o.op(OPS.OP_SPHERE_BC, 0, OPS.PSI, OPS.SRC)
    g.op(OPS.OP_SPHERE_BC, 0, OPS.PSI, OPS.SRC)
    assert_same_state(h, o, g, "sphere_bc")


def test_remove_mean_bitwise(pair):
    h, o, g = pair["periodic"]
    randomize(h, o, g, seed=5)
    o.op(OPS.OP_REMOVE_MEAN, 0, OPS.RHO)
    g.op(OPS.OP_REMOVE_MEAN, 0, OPS.RHO)
    assert_same_state(h, o, g, "remove_mean")


@pytest.mark.parametrize("name", ["periodic", "sphere"])
@pytest.mark.parametrize("mode", [OPS.STOP_TRUE_RESIDUAL, OPS.STOP_REFERENCE])
def test_solve_bitwise(pair, name, mode):
    h, o, g = pair[name]
    src = problems.amr_source(h, seed=11)
    tol = 1e-10 if mode == OPS.STOP_TRUE_RESIDUAL else 1e-3
    po, go_, so = o.solve(src, tol=tol, maxit=20, mode=mode)
    pg, gg, sg = g.solve_host(src, tol=tol, maxit=20, stop_mode=mode)
    print(name, mode, so["iterations"], so["rel_linf"], sg["iterations"], sg["rel_linf"], flush=True)
    assert so["iterations"] == sg["iterations"] and so["status"] == sg["status"] == 0
    assert so["rel_linf"] == sg["rel_linf"]
    assert np.array_equal(po, pg)
    assert np.array_equal(go_, gg)
    if mode == OPS.STOP_TRUE_RESIDUAL:
        assert sg["rel_linf"] < 1e-10


def test_mid_size_sphere_parity(gpu):
    """8^3 base blocks, four levels (2048 blocks)."""
    h = ah.nested(base=8, levels=4, bc=ah.SPHERE)
    src = problems.sis_source(h, seed=3)
    o = oracle.Amr(h)
    po, go_, so = o.solve(src, tol=1e-10, maxit=20)
    g = AmrSolver(h)
    pg, gg, sg = g.solve_host(src, tol=1e-10, maxit=20)
    print("mid", so["iterations"], sg["iterations"], sg["rel_linf"], sg["ms"], flush=True)
    assert so["iterations"] == sg["iterations"]
    assert np.array_equal(po, pg) and np.array_equal(go_, gg)


@pytest.mark.parametrize("name", ["periodic", "sphere"])
@pytest.mark.parametrize("graph", [False, True])
def test_mixed_solve_against_oracle(pair, name, graph):
    """FP32 inner fmg_lin (exact base-grid transform solve) inside FP64 defect correction: the
    FP64 composite residual reaches 1e-10, and potential / acceleration stay within 1e-9 (relative
    L2) of the FP64 oracle's converged solution (periodic: potentials compared without their mean)."""
    h, o, g = pair[name]
    src = problems.amr_source(h, seed=12)
    po, go_, so = o.solve(src, tol=1e-12, maxit=30)
    pm, gm, sm = g.solve_host(src, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, use_graph=graph)
    print(name, graph, sm["iterations"], sm["rel_linf"], sm["hist"], flush=True)
    assert sm["status"] == 0 and sm["rel_linf"] < 1e-10
    # the inner solve follows the reference's ghost state: its first outer iteration contracts
    # the residual as the FP64 solve's does (a stale ghost state after the VMG smoother once
    # weakened it five-fold on the sphere)
    _, _, s1 = o.solve(src, tol=0.0, maxit=1)
    assert sm["hist"][1] < 1.05 * s1["hist"][1]
    if name == "periodic":
        po = po - po.mean()
        pm = pm - pm.mean()
    e_psi = np.linalg.norm(pm - po) / np.linalg.norm(po)
    e_g = np.linalg.norm(gm - go_) / np.linalg.norm(go_)
    print("mixed vs oracle", e_psi, e_g, flush=True)
    assert e_psi < 1e-9 and e_g < 1e-8


def test_mixed_full_sphere_hierarchy(gpu):
    """16^3 base blocks, five levels (20 480 blocks), singular isothermal sphere source.  A composite
    residual of 1e-10 bounds the solution error only to ~1e-9 at this resolution (finest h = L/2048),
    so both the FP64 and the mixed solve at tol 1e-10 are measured against an FP64 GPU solve
    converged to 1e-12 (the FP64 GPU path is bitwise equal to the oracle): the mixed error must stay
    below 1e-8 (potential) / 1e-7 (acceleration) and within 4x of the FP64 solve's own error at the
    same tolerance, and a mixed solve to 1e-12 must agree with the reference to 1e-10 / 1e-9."""
    h = ah.nested(base=16, levels=5, bc=ah.SPHERE)
    src = problems.sis_source(h, seed=1)
    g = AmrSolver(h)
    pr, gr, sr = g.solve_host(src, tol=1e-12, maxit=40)
    print("reference fp64", sr["iterations"], sr["status"], sr["rel_linf"], flush=True)
    assert sr["rel_linf"] < 1e-11

    def err(p, a):
        return np.linalg.norm(p - pr) / np.linalg.norm(pr), np.linalg.norm(a - gr) / np.linalg.norm(gr)

    p64, g64, s64 = g.solve_host(src, tol=1e-10, maxit=30)
    pm, gm, sm = g.solve_host(src, tol=1e-10, maxit=30, precision=SG_PREC_MIXED)
    e64, em = err(p64, g64), err(pm, gm)
    print("tol 1e-10: fp64", s64["iterations"], s64["ms"], e64, "mixed", sm["iterations"], sm["ms"],
          sm["rel_linf"], em, flush=True)
    assert sm["status"] == 0 and sm["rel_linf"] < 1e-10
    assert em[0] < 1e-8 and em[1] < 1e-7
    assert em[0] < 4 * e64[0] + 1e-11 and em[1] < 4 * e64[1] + 1e-10
    pt, gt, st = g.solve_host(src, tol=1e-12, maxit=40, precision=SG_PREC_MIXED)
    et = err(pt, gt)
    print("tol 1e-12: mixed", st["iterations"], st["rel_linf"], et, flush=True)
    assert st["rel_linf"] < 1e-11
    assert et[0] < 1e-10 and et[1] < 1e-9


# ---- failure paths: ordinary arithmetic outcomes reported through the status codes ----

@pytest.mark.parametrize("precision", [1, SG_PREC_MIXED])
def test_nonfinite_source_is_reported(pair, precision):
    """A NaN in the source: fmax-based maxima drop it, the sum of squares keeps it; the solve must
    return SG_ERR_NONFINITE instead of 'converged'."""
    from code_only_amd import _lib
    h, o, g = pair["periodic"]
    src = problems.amr_source(h, seed=13)
    # a leaf block: a covered block's source is overwritten by the restriction of its children
    b = int(np.flatnonzero(h.leaf)[0])
    src[b, 2, 1, 0] = np.nan
    psi, _, st = g.solve_host(src, tol=1e-10, maxit=5, precision=precision, raise_on_fail=False)
    print("nan", precision, st["status"], st["iterations"], st["rel_linf"], flush=True)
    assert st["status"] == _lib.SG_ERR_NONFINITE
    with pytest.raises(_lib.SgError) as e:
        g.solve_host(src, tol=1e-10, maxit=5, precision=precision)
    assert e.value.code == _lib.SG_ERR_NONFINITE


@pytest.mark.parametrize("precision", [1, SG_PREC_MIXED])
def test_maxit_reached_is_reported(pair, precision):
    from code_only_amd import _lib
    h, o, g = pair["sphere"]
    src = problems.amr_source(h, seed=14)
    _, _, st = g.solve_host(src, tol=1e-10, maxit=1, precision=precision, raise_on_fail=False)
    assert st["status"] == _lib.SG_ERR_NOT_CONVERGED and st["iterations"] == 1
    assert st["rel_linf"] > 1e-10
    if precision == 1:
        _, _, so = o.solve(src, tol=1e-10, maxit=1)
        assert so["status"] == _lib.SG_ERR_NOT_CONVERGED and so["rel_linf"] == st["rel_linf"]


def test_stall_exit_is_reported(pair):
    """Periodic hierarchy, zero averaging off, source with a non-zero mean: the singular problem
    has no solution, Resh2maxg stops falling and fmg_cycle's stall test (fmg.F90:193) ends the
    loop before maxit; oracle and GPU agree on where and report SG_ERR_NOT_CONVERGED."""
    from code_only_amd import _lib
    h, o, g = pair["periodic"]
    src = problems.amr_source(h, seed=15) + 1.0
    o.set_zero_average(False)
    g.set_zero_average(False)
    try:
        _, _, so = o.solve(src, tol=1e-12, maxit=20, mode=OPS.STOP_REFERENCE)
        _, _, sg = g.solve_host(src, tol=1e-12, maxit=20, stop_mode=OPS.STOP_REFERENCE, raise_on_fail=False)
    finally:
        o.set_zero_average(True)
        g.set_zero_average(True)
    print("stall", so["iterations"], so["status"], sg["iterations"], sg["status"], flush=True)
    assert so["status"] == sg["status"] == _lib.SG_ERR_NOT_CONVERGED
    assert so["iterations"] == sg["iterations"] < 20


def test_zero_average_toggle_recaptures_the_graph(pair):
    """The mixed iteration's graph bakes in vmg_fas's zero-average step: after toggling the
    setting, graph replay must give the eager result for the new setting."""
    h, o, g = pair["periodic"]
    src = problems.amr_source(h, seed=16)
    g.solve_host(src, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, use_graph=True)
    g.set_zero_average(False)
    try:
        pe, _, se = g.solve_host(src, tol=0.0, maxit=2, precision=SG_PREC_MIXED, use_graph=False,
                                 raise_on_fail=False)
        pg, _, sg = g.solve_host(src, tol=0.0, maxit=2, precision=SG_PREC_MIXED, use_graph=True,
                                 raise_on_fail=False)
    finally:
        g.set_zero_average(True)
    assert se["iterations"] == sg["iterations"] == 2
    assert np.array_equal(pe, pg)


# ---- fused refresh of the mixed solve ----

@pytest.mark.parametrize("which", ["nested-sphere", "nested-periodic", "random-periodic", "random-sphere"])
@pytest.mark.parametrize("graph", [False, True])
def test_fused_refresh_equals_staged(which, graph, gpu):
    """The mixed solve with one-launch refreshes (k_prep + halo-free colour passes) against the
    same solve with the staged refresh launches: bit for bit the same iterates (potential,
    acceleration, residual history), since every cell a colour pass or residual reads gets the
    value the staged fill gives it.  The nested hierarchies must admit the fused form."""
    h = {"nested-sphere": lambda: ah.nested(base=4, levels=3, bc=ah.SPHERE),
         "nested-periodic": lambda: ah.nested(base=4, levels=3, bc=ah.PERIODIC),
         "random-periodic": lambda: ah.random_hierarchy(4, 3, 0.35, seed=7, bc=ah.PERIODIC),
         # refinement reaching the domain boundary: physical faces on fine blocks
         "random-sphere": lambda: ah.random_hierarchy(4, 3, 0.35, seed=3, bc=ah.SPHERE)}[which]()
    g = AmrSolver(h)
    info = g.info()
    print(which, info, flush=True)
    if which.startswith("nested"):
        assert info["fused_levels"] == 3
    # the base level's fmg_ghostcell_fix at FMG levels 1 and 2 as one gather
    assert info["base_gather_levels"] == 6
    src = problems.amr_source(h, seed=17)
    ps, gs, ss = g.solve_host(src, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, use_graph=graph, fused=False)
    pf, gf, sf = g.solve_host(src, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, use_graph=graph, fused=True)
    print(ss["iterations"], sf["iterations"], ss["hist"], sf["hist"], flush=True)
    assert ss["iterations"] == sf["iterations"] and ss["hist"] == sf["hist"]
    assert np.array_equal(ps, pf) and np.array_equal(gs, gf)
    g.close()


@pytest.mark.parametrize("which", ["sphere-4", "periodic-4", "sphere-16"])
def test_mixed_base_solve_chip_equals_one_workgroup(which, gpu):
    """The inner solve's exact base solve as six chip-wide transform passes equals the one-workgroup
    form bit for bit (each output summed over the same terms in the same order): the whole mixed
    solve, graphed, is the same either way (8^3 and 32^3 base grids; DST and Hartley bases)."""
    base, bc = {"sphere-4": (4, ah.SPHERE), "periodic-4": (4, ah.PERIODIC), "sphere-16": (16, ah.SPHERE)}[which]
    h = ah.nested(base=base, levels=3, bc=bc)
    g = AmrSolver(h)
    try:
        src = problems.amr_source(h, seed=23)
        pc, gc, sc = g.solve_host(src, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, use_graph=True)
        g.set_base_solver(False)
        pw, gw, sw = g.solve_host(src, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, use_graph=True)
        g.set_base_solver(True)
        print(which, sc["iterations"], sw["iterations"], flush=True)
        assert sc["iterations"] == sw["iterations"] and sc["hist"] == sw["hist"]
        assert np.array_equal(pc, pw) and np.array_equal(gc, gw)
    finally:
        g.close()


def test_fused_refresh_full_sphere_hierarchy_launches(gpu):
    """16^3 base blocks, five levels: the fused form applies at FMG levels 0 and 1, reproduces
    the staged mixed solve bit for bit, and needs fewer kernel nodes per outer iteration."""
    h = ah.nested(base=16, levels=5, bc=ah.SPHERE)
    src = problems.sis_source(h, seed=1)
    g = AmrSolver(h)
    ps, gs, ss = g.solve_host(src, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, fused=False)
    n_staged = g.info()["graph_nodes"]
    pf, gf, sf = g.solve_host(src, tol=1e-10, maxit=30, precision=SG_PREC_MIXED, fused=True)
    info = g.info()
    print("nodes staged", n_staged, "fused", info["graph_nodes"], "ms", ss["ms"], sf["ms"], flush=True)
    assert info["fused_levels"] == 3
    assert info["vmg_fill_levels"] == (1 << h.nlev) - 1
    assert ss["iterations"] == sf["iterations"] and ss["hist"] == sf["hist"]
    assert np.array_equal(ps, pf) and np.array_equal(gs, gf)
    assert info["graph_nodes"] < n_staged


def _zero_physical_ghosts(h, a, L):
    """Zero the ghost layers on physical faces (what every refresh of the inner solve leaves)."""
    n = 8 >> L
    for b in range(h.nblk):
        for f in range(6):
            if h.nbr[b, f] >= 0:
                continue
            d, lr = f // 2, f % 2
            sl = [slice(None)] * 3
            sl[2 - d] = n + 1 if lr else 0   # arrays are [k][j][i]
            a[(b,) + tuple(sl)] = 0.0


@pytest.mark.parametrize("which", ["nested-sphere", "nested-periodic", "random-periodic", "nested-8-4", "nested-16-5"])
@pytest.mark.parametrize("L", [0, 1])
@pytest.mark.parametrize("opname", ["relax", "resid"])
def test_fused_operator_equals_staged(which, L, opname, gpu):
    """One fmg_poisson_relax / fmg_poisson_resid with the fused refresh against the oracle's staged
    one, from a random state whose physical ghosts are zero: the interiors of the leaf blocks (and
    the residual) must agree bit for bit."""
    h = {"nested-sphere": lambda: ah.nested(base=4, levels=3, bc=ah.SPHERE),
         "nested-periodic": lambda: ah.nested(base=4, levels=3, bc=ah.PERIODIC),
         "random-periodic": lambda: ah.random_hierarchy(4, 3, 0.35, seed=7, bc=ah.PERIODIC),
         "nested-8-4": lambda: ah.nested(base=8, levels=4, bc=ah.SPHERE),
         "nested-16-5": lambda: ah.nested(base=16, levels=5, bc=ah.SPHERE)}[which]()
    o, g = oracle.Amr(h), AmrSolver(h)
    try:
        if not (g.info()["fused_levels"] >> L) & 1:
            pytest.skip("hierarchy does not admit the fused form at this level")
        rng = np.random.default_rng(3 + L)
        n = 8 >> L
        for code in range(6):
            a = rng.standard_normal((h.nblk, n + 2, n + 2, n + 2))
            _zero_physical_ghosts(h, a, L)
            o.set(L, code, a)
            g.set(L, code, a)
        if opname == "relax":
            o.op(OPS.OP_RELAX, L, OPS.U, OPS.RHS, 0, 1)
            g.op(OPS.OP_RELAX, L, OPS.U, OPS.RHS, 0, 1 | 4)
            code = OPS.U
        else:
            o.op(OPS.OP_RESID, L, OPS.RES, OPS.U, OPS.RHS, 1)
            g.op(OPS.OP_RESID, L, OPS.RES, OPS.U, OPS.RHS, 1 | 4)
            code = OPS.RES
        a, b = o.get(L, code)[:, 1:-1, 1:-1, 1:-1], g.get(L, code)[:, 1:-1, 1:-1, 1:-1]
        leaf = np.asarray(h.leaf, bool)
        bad = np.argwhere((a != b) & leaf[:, None, None, None])
        if len(bad):
            lines = []
            for blk, k, j, i in bad[:12]:
                kinds = ["-" if h.nbr[blk, f] < 0 else ("S" if h.level[h.nbr[blk, f]] == h.level[blk] else "P")
                         for f in range(6)]
                lines.append(f"blk {blk} lev {h.level[blk]} cell ({i},{j},{k}) faces {''.join(kinds)} "
                             f"oracle {a[blk, k, j, i]:.6e} gpu {b[blk, k, j, i]:.6e}")
            blocks = sorted(set(int(x) for x in bad[:, 0]))
            raise AssertionError(f"{len(bad)} leaf cells differ in {len(blocks)} blocks {blocks[:20]}\n" + "\n".join(lines))
    finally:
        o.close()
        g.close()


@pytest.mark.parametrize("which", ["nested-periodic", "random-periodic"])
def test_fused_fmg_lin_equals_staged(which, gpu):
    """A whole fmg_lin with the fused refreshes at FMG levels 0 and 1 against the oracle's staged
    fmg_lin, from a random state with zero physical ghosts: the leaf interiors of every code at every
    FMG level agree bit for bit."""
    h = {"nested-periodic": lambda: ah.nested(base=4, levels=3, bc=ah.PERIODIC),
         "random-periodic": lambda: ah.random_hierarchy(4, 3, 0.35, seed=7, bc=ah.PERIODIC)}[which]()
    o, g = oracle.Amr(h), AmrSolver(h)
    try:
        rng = np.random.default_rng(11)
        for L in range(3):
            n = 8 >> L
            for code in range(6):
                a = rng.standard_normal((h.nblk, n + 2, n + 2, n + 2))
                _zero_physical_ghosts(h, a, L)
                o.set(L, code, a)
                g.set(L, code, a)
        o.fill0_level = -1
        g.fill0_level = -1
        ro = o.op(OPS.OP_FMG_LIN)
        rg = g.op(OPS.OP_FMG_LIN, flag=4)
        leaf = np.asarray(h.leaf, bool)
        report = []
        for L in range(3):
            for code in range(6):
                a = o.get(L, code)[:, 1:-1, 1:-1, 1:-1]
                b = g.get(L, code)[:, 1:-1, 1:-1, 1:-1]
                bad = np.argwhere((a != b) & leaf[:, None, None, None])
                if len(bad):
                    report.append(f"L{L} code {code}: {len(bad)} leaf cells in {len(set(bad[:, 0].tolist()))} blocks, "
                                  f"max {np.abs(a - b)[leaf].max():.3e}")
        print("\n".join(report), ro, rg, flush=True)
        assert not report, "\n".join(report)
        assert ro == rg
    finally:
        o.close()
        g.close()


SEQUENCES = {
    "relax-relax-resid-L0": [("relax", 0), ("relax", 0), ("resid", 0)],
    "relax-relax-resid-L1": [("relax", 1), ("relax", 1), ("resid", 1)],
    "interp-relax-L0": [("interp", 0), ("relax", 0), ("relax", 0)],
    "addint-relax-L1": [("addint", 1), ("relax", 1), ("relax", 1)],
    "addint-relax-L0": [("addint", 0), ("relax", 0), ("relax", 0)],
    "down-leg-L0": [("relax", 0), ("relax", 0), ("resid", 0), ("rstrct", 1), ("fill0U", 1), ("relax", 1),
                    ("relax", 1), ("resid", 1)],
    "down-vmg-up-L1": [("relax", 1), ("relax", 1), ("resid", 1), ("rstrct", 2), ("fill0U", 2), ("vmg", 2),
                       ("addint", 1), ("relax", 1), ("relax", 1)],
}


@pytest.mark.parametrize("seq", sorted(SEQUENCES))
def test_fused_sequence_equals_staged(seq, gpu):
    """Short sequences of fmg_lin's operations, the relaxations and residuals with the fused refresh,
    against the oracle's staged ones: leaf interiors of every array after every step."""
    h = ah.nested(base=4, levels=3, bc=ah.PERIODIC)
    o, g = oracle.Amr(h), AmrSolver(h)
    try:
        rng = np.random.default_rng(21)
        for L in range(3):
            n = 8 >> L
            for code in range(6):
                a = rng.standard_normal((h.nblk, n + 2, n + 2, n + 2))
                o.set(L, code, a)
                g.set(L, code, a)
        leaf = np.asarray(h.leaf, bool)
        for step, (what, L) in enumerate(SEQUENCES[seq]):
            if what == "relax":
                o.op(OPS.OP_RELAX, L, OPS.U, OPS.RHS, 0, 1)
                g.op(OPS.OP_RELAX, L, OPS.U, OPS.RHS, 0, 1 | 4)
            elif what == "resid":
                o.op(OPS.OP_RESID, L, OPS.RES, OPS.U, OPS.RHS, 1)
                g.op(OPS.OP_RESID, L, OPS.RES, OPS.U, OPS.RHS, 1 | 4)
            elif what == "interp":
                o.op(OPS.OP_INTERP, L, OPS.U, OPS.U, 0, 1)
                g.op(OPS.OP_INTERP, L, OPS.U, OPS.U, 0, 1)
            elif what == "addint":
                o.op(OPS.OP_ADDINT, L, OPS.U, OPS.U, OPS.RES)
                g.op(OPS.OP_ADDINT, L, OPS.U, OPS.U, OPS.RES)
            elif what == "rstrct":
                o.op(OPS.OP_RSTRCT, L, OPS.RHS, OPS.RES)
                g.op(OPS.OP_RSTRCT, L, OPS.RHS, OPS.RES)
            elif what == "fill0U":
                # fmg_fill0 (whole arrays of the non-skipped blocks) and the FmgLevel_fill0 mark
                a = o.get(L, OPS.U)
                a[leaf] = 0.0
                o.set(L, OPS.U, a)
                g.set(L, OPS.U, a)
                o.fill0_level = L
                g.fill0_level = L
            elif what == "vmg":
                o.op(OPS.OP_VMG_FAS, L, OPS.RHS)
                g.op(OPS.OP_VMG_FAS, L, OPS.RHS)
            report = []
            for LL in range(3):
                for code in range(6):
                    a = o.get(LL, code)[:, 1:-1, 1:-1, 1:-1]
                    b = g.get(LL, code)[:, 1:-1, 1:-1, 1:-1]
                    bad = np.argwhere((a != b) & leaf[:, None, None, None])
                    if len(bad):
                        report.append(f"L{LL} code {code}: {len(bad)} cells, blocks {sorted(set(bad[:, 0].tolist()))[:8]}, "
                                      f"first {bad[0].tolist()}")
            assert not report, f"{seq} step {step} ({what} L{L}):\n" + "\n".join(report)
    finally:
        o.close()
        g.close()


@pytest.mark.parametrize("which", ["nested-sphere", "random-periodic"])
def test_base_solver_chip_equals_one_workgroup(which, gpu):
    """The plain FP64 solve with the base grid's mg_cycle spread over the chip and in one
    workgroup: the same values bit for bit (and the oracle's, which the other solve tests check)."""
    h = {"nested-sphere": lambda: ah.nested(base=8, levels=3, bc=ah.SPHERE),
         "random-periodic": lambda: ah.random_hierarchy(4, 3, 0.35, seed=7, bc=ah.PERIODIC)}[which]()
    g = AmrSolver(h)
    src = problems.amr_source(h, seed=23)
    try:
        g.set_base_solver(True)
        pc, gc, sc = g.solve_host(src, tol=1e-10, maxit=30)
        g.set_base_solver(False)
        pw, gw, sw = g.solve_host(src, tol=1e-10, maxit=30)
        print(which, sc["iterations"], sc["ms"], sw["ms"], flush=True)
        assert sc["iterations"] == sw["iterations"] and sc["hist"] == sw["hist"]
        assert np.array_equal(pc, pw) and np.array_equal(gc, gw)
    finally:
        g.close()


@pytest.mark.parametrize("which", ["nested-sphere", "nested-periodic", "random-periodic", "random-sphere"])
def test_fp64_fused_refresh_equals_staged(which, gpu):
    """The plain FP64 solve with the mixed solve's launch structure (fused refresh, halo-free colour
    passes, merged VMG steps) against the reference's staged sequence: the same iterates bit for
    bit."""
    h = {"nested-sphere": lambda: ah.nested(base=4, levels=3, bc=ah.SPHERE),
         "nested-periodic": lambda: ah.nested(base=4, levels=3, bc=ah.PERIODIC),
         "random-periodic": lambda: ah.random_hierarchy(4, 3, 0.35, seed=7, bc=ah.PERIODIC),
         # refinement reaching the domain boundary: physical faces on fine blocks
         "random-sphere": lambda: ah.random_hierarchy(4, 3, 0.35, seed=3, bc=ah.SPHERE)}[which]()
    g = AmrSolver(h)
    src = problems.amr_source(h, seed=29)
    try:
        ps, gs, ss = g.solve_host(src, tol=1e-10, maxit=30)
        g.set_fp64_refresh(True)
        pf, gf, sf = g.solve_host(src, tol=1e-10, maxit=30)
        g.set_fp64_refresh(False)
        print(which, ss["iterations"], ss["ms"], sf["ms"], flush=True)
        assert ss["iterations"] == sf["iterations"] and ss["hist"] == sf["hist"]
        assert np.array_equal(ps, pf) and np.array_equal(gs, gf)
    finally:
        g.close()


@pytest.mark.parametrize("bc", [ah.PERIODIC, ah.SPHERE])
@pytest.mark.parametrize("base", [1, 2, 4, 8, 16, 32])
def test_base_cycle_widths(base, bc, gpu):
    """The base-grid mg_cycle on the fused kernels against the one-workgroup form, bit for bit, for every
    width it dispatches on (2^3 ... 16^3 in one launch, 32^3 and 64^3 over the chip), both boundaries."""
    refine = [] if base < 4 else [{(1, 1, 1), (2, 1, 1)}]
    if base == 1 and bc == ah.PERIODIC:
        refine = []
    h = ah.build((base,) * 3, refine, bc=bc)
    src = problems.amr_source(h, seed=5)
    out = []
    g = AmrSolver(h)
    try:
        for chip in (True, False):
            g.set_base_solver(chip)
            out.append(g.solve_host(src, tol=1e-8, maxit=3, raise_on_fail=False))
    finally:
        g.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert out[0][2]["hist"] == out[1][2]["hist"]


@pytest.mark.parametrize("which", ["nested-sphere-8", "nested-sphere-16", "random-periodic", "random-sphere"])
def test_fp64_default_equals_staged(which, gpu):
    """The plain FP64 solve's default (fused refresh, fmg_lin replayed as graphs: one, or stretches
    between base solves at a 32^3 base grid) against the reference's staged sequence, bit for bit: as
    recorded and replayed, eagerly, with another source, and after the settings a graph holds changed."""
    h = {"nested-sphere-8": lambda: ah.nested(base=8, levels=3, bc=ah.SPHERE),
         "nested-sphere-16": lambda: ah.nested(base=16, levels=2, bc=ah.SPHERE),
         "random-periodic": lambda: ah.random_hierarchy(4, 3, 0.35, seed=7, bc=ah.PERIODIC),
         "random-sphere": lambda: ah.random_hierarchy(4, 3, 0.35, seed=3, bc=ah.SPHERE)}[which]()
    g = AmrSolver(h)
    kw = dict(tol=1e-9, maxit=4, raise_on_fail=False)
    try:
        for seed in (41, 42):
            src = problems.amr_source(h, seed=seed)
            g.set_fp64_refresh(False)
            ref = g.solve_host(src, **kw)
            g.set_fp64_refresh(True)
            runs = [g.solve_host(src, **kw), g.solve_host(src, use_graph=False, **kw)]
            g.set_base_solver(False)
            runs.append(g.solve_host(src, **kw))
            g.set_base_solver(True)
            runs.append(g.solve_host(src, **kw))
            for psi, acc, st in runs:
                assert st["hist"] == ref[2]["hist"] and st["resmaxg"] == ref[2]["resmaxg"]
                assert np.array_equal(psi, ref[0]) and np.array_equal(acc, ref[1])
    finally:
        g.close()
