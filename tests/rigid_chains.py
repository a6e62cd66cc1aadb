"""Rigid zig-zag chains of any length and boxes of them on a jittered grid, for
tests of kinds other than one- and three-site ones."""
import numpy as np

from gomc_amd import systems


def chain_kind(atoms, types, seed=1, first_type=0):
    """A neutral chain; atom i is of type first_type + i % types."""
    rng = np.random.default_rng([seed, atoms])
    geo = np.zeros((atoms, 3))
    geo[:, 0] = 0.75 * np.arange(atoms)
    geo[:, 1] = 0.5 * (np.arange(atoms) % 2)
    geo -= geo.mean(0)
    q = 0.3 * rng.normal(size=atoms)
    q -= q.mean()
    return systems.MolKind(f"chain{atoms}", [first_type + i % types for i in range(atoms)],
                           [float(v) for v in q], geo)


def chain_box(kinds, mol_kind, edges, types, rcut=8.0, tolerance=1e-5, seed=3, **kw):
    """Molecules on a jittered grid in random orientations."""
    rng = np.random.default_rng(seed)
    edges = np.asarray(edges, float)
    mol_kind = np.asarray(mol_kind, np.int32)
    div = np.ones(3, int)
    while div.prod() < len(mol_kind):
        div[np.argmax(edges / div)] += 1
    grid = np.stack(np.meshgrid(*(np.arange(d) for d in div), indexing="ij"), -1).reshape(-1, 3)
    xyz = []
    for cell, k in zip(grid[rng.permutation(len(grid))], mol_kind):
        rot, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        at = (cell + 0.5 + rng.uniform(-0.1, 0.1, 3)) * edges / div
        xyz.append(at + kinds[k].geometry @ rot.T)
    return systems.System(
        box=tuple(edges), temperature=300.0, rcut=rcut, rcut_low=0.1, rcut_coulomb=rcut,
        tolerance=tolerance, kinds=kinds, mol_kind=mol_kind,
        xyz=np.mod(np.concatenate(xyz), edges), seed=seed,
        sigma=[1.6 + 0.05 * i for i in range(types)], epsilon=[40.0 + 3.0 * i for i in range(types)],
        n_rep=kw.pop("n_rep", [12.0] * types), **kw)
