"""GPU: the contraction's right operands built on the device.

Densities without any symmetry, so a swapped index, a wrong spin sign or a
misplaced element of the operand layouts changes the tensors, on bases whose
sizes fill, pad and overrun the 8- and 32-function groups; both storage
orders of the C ABI give the oracle's tensors.
"""
import numpy as np
import pytest

from conftest import rel_err
from oracle import oracle

pytestmark = pytest.mark.gpu

# shells per centre: nbf 1, 8, 31 (s, p, d on the last centre), 33 and 65
SHELLS = {1: [[0]], 8: [[0, 1], [0, 1]], 31: [[0, 1, 2], [0, 1, 2], [0, 2, 1, 0]],
          33: [[2, 2, 1], [2, 2, 1, 1]], 65: [[3, 3, 3, 2, 1], [2, 3, 2, 1, 0]]}


def _system(nbf):
    rng = np.random.default_rng(100 + nbf)
    shells = SHELLS[nbf]
    atoms = [a for a, ls in enumerate(shells) for _ in ls]
    ls = [l for ls in shells for l in ls]
    nprim = [1 + k % 3 for k in range(len(ls))]
    poff = np.concatenate([[0], np.cumsum(nprim)[:-1]])
    n = int(sum((l + 1) * (l + 2) // 2 for l in ls))
    assert n == nbf, n
    i32 = lambda v: np.asarray(v, dtype=np.int32)
    return dict(coords=rng.uniform(-2.0, 2.0, (len(shells), 3)), shell_atom=i32(atoms),
                shell_l=i32(ls), shell_nprim=i32(nprim), shell_poff=i32(poff),
                exps=rng.uniform(0.2, 4.0, sum(nprim)), coefs=rng.uniform(0.2, 1.0, sum(nprim)),
                turbomole=0), rng


@pytest.mark.parametrize("nbf", sorted(SHELLS))
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("mixed", 1e-5)])
def test_tensors_of_unsymmetric_densities(nbf, precision, tol):
    from gimic_amd import lib
    a, rng = _system(nbf)
    dens = rng.standard_normal((2, 4, nbf, nbf))
    pts = rng.uniform(-3.0, 3.0, (70, 3))
    ctx = lib.Context.from_arrays(a["coords"], a["shell_atom"], a["shell_l"], a["shell_nprim"],
                                  a["shell_poff"], a["exps"], a["coefs"], screening=1e-8)
    for order in ("rows", "columns"):
        if order == "rows":
            ctx.set_density(dens)
        else:
            cols = np.ascontiguousarray(dens.transpose(0, 1, 3, 2))
            lib.check(ctx._lib.gimic_ctx_set_density(ctx._h, 2, lib.ptr(cols)))
        for spin in ("alpha", "beta", "total", "spindens"):
            print("case operands", nbf, precision, order, spin, flush=True)
            J = ctx.jtensor(pts, spin=spin, precision=precision)
            ref = oracle.jtensor(a, dens, pts, screening=1e-8, spin=spin)
            assert rel_err(J, ref).max() <= tol, (order, spin, rel_err(J, ref).max())
    ctx.close()
