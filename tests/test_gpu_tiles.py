"""HIP path vs the CPU oracle at the sizes where the kernels' work is cut: atom
counts at and beside the edges of their 16-atom tiles, on the fused and the
scalar filter kernels of the shipped model and on the generic widths; head
widths that leave a part of a 16-unit tile.  Bars as in test_gpu_edges.py:
energy 1e-10 relative, forces and virial 1e-9.
"""
import numpy as np
import pytest

import support
from oracle.oracle import Oracle
from test_gpu_edges import _both_paths, model, orc  # noqa: F401

pytestmark = pytest.mark.gpu


def _cluster(n, seed=3, spacing=1.7):
    """n H and O atoms on a jittered lattice, every pair of neighbours inside
    the short-range cutoff."""
    rng = np.random.default_rng([seed, n])
    g = int(np.ceil(n ** (1 / 3) - 1e-9))
    sites = np.array([[i, j, k] for i in range(g) for j in range(g) for k in range(g)], float)[:n]
    z = rng.choice([1, 8], size=n, p=[0.6, 0.4])
    return z, spacing * sites + rng.uniform(-0.2, 0.2, (n, 3)), 1.0 + float((z == 1).sum() % 2)


@pytest.mark.parametrize("n", [2, 15, 16, 17, 33, 65])
def test_atom_tiles(orc, model, n):  # noqa: F811
    z, x, m = _cluster(n)
    _both_paths(z, x, 0.0, m, orc, model)


@pytest.mark.parametrize("n", [499, 500, 2399, 2400])
def test_node_shares(orc, model, n):  # noqa: F811
    """Both sides of the atom counts at which 8, 4 and 1 wavefronts share a
    node's incidence list; nodes with fewer partners than wavefronts are at
    the cluster's corners."""
    z, x, m = _cluster(n, spacing=2.8)
    _both_paths(z, x, 0.0, m, orc, model)


@pytest.mark.parametrize("copies", [17, 86])
def test_partner_counts(orc, model, copies):  # noqa: F811
    """Separate groups of 1 to 7 atoms: nodes with 0 to 6 active partners, the
    remainders of the four entries the node-major sums read at a time, with
    the list shared by 8 wavefronts (476 atoms) and read by one (2,408)."""
    parts = [_cluster(1 + k % 7, seed=k) for k in range(7 * copies)]
    g = int(np.ceil(len(parts) ** (1 / 3) - 1e-9))
    at = 9.0 * np.array([[k // (g * g), k // g % g, k % g] for k in range(len(parts))], float)
    z = np.concatenate([p[0] for p in parts])
    x = np.concatenate([p[1] + o for p, o in zip(parts, at)])
    _both_paths(z, x, 0.0, 1.0 + float((z == 1).sum() % 2), orc, model)


@pytest.mark.parametrize("n", [85, 86, 1000])
def test_few_candidates(orc, model, n):  # noqa: F811
    """One candidate pair and the other atoms on a 7 A lattice without any:
    the launch that counts the candidates gathers 3 n coordinates beside it
    (255 and 258, on both sides of its blocks of 256, and many blocks)."""
    g = int(np.ceil(n ** (1 / 3) - 1e-9))
    sites = np.array([[i, j, k] for i in range(g) for j in range(g) for k in range(g)], float)[:n]
    x = 7.0 * sites + np.random.default_rng(n).uniform(-0.2, 0.2, (n, 3))
    x[1] = x[0] + [1.0, 0.3, -0.2]
    z = np.full(n, 8)
    z[:2] = 1
    _both_paths(z, x, 0.0, 1.0, orc, model)


@pytest.mark.parametrize("limit", ["0", "1000000"])
@pytest.mark.parametrize("n", [2, 3, 17, 65])
def test_few_pairs(monkeypatch, n, limit):
    """A pair or a handful per interval bucket (mostly padding slots) up to
    several buckets of 16, on the kernels for few pairs and on the scalar ones."""
    monkeypatch.setenv("SO3LR_SCALAR_FILTER_PAIRS", limit)
    z, x, m = _cluster(n)
    _both_paths(z, x, 0.0, m, Oracle(support.MODEL), support.MODEL)


@pytest.mark.parametrize("n", [146, 148, 268, 272])
def test_few_pairs_line(orc, model, n):  # noqa: F811
    """Pair counts beside the lines between the kernels for few pairs and
    those for many: 9/8 of the pairs plus 256 is 3,663, 3,709, 7,451 and 7,618
    (F = 256: 3,700; F = 128: 7,500)."""
    z, x, m = _cluster(n)
    _both_paths(z, x, 0.0, m, orc, model)


@pytest.mark.parametrize("width", [129, 200])
def test_head_width_remainder(tmp_path, width):
    """Energy and charge heads whose width is no multiple of 16 (the generic
    kernels pad their last tile)."""
    path = support.head_width_model(tmp_path / "heads.so3lr", width, live=True)
    z, x, m = _cluster(17)
    _both_paths(z, x, 0.0, m, Oracle(path), path)
