"""The Dense row kernel at the edges of its blocks: every lane count, row
widths that end inside and at a block, rows that end anywhere beside longer
ones, rows of wavefronts on and off the box faces, boxes whose faces are near in
some dimensions only, species parameters and box matrices.  Forces against the float64 sum over the same rows, with
the bars of test_gpu_pair.py (float32 pair terms: 1e-5 norm-wise, 5e-5 of the
rms for one particle, 1e-6 for the energy)."""

import dataclasses

import numpy as np
import pytest
import torch

from tests.test_gpu_pair import FORCE_RTOL, FORCE_WORST, _force_err

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _rows_fp64(R, sides, idx, species=None, sigma=1.0):
  """Energy and force of the switched Lennard-Jones rows in float64; sides is
  a vector, or a box matrix with R fractional."""
  x, L = R.astype(np.float64), np.asarray(sides, np.float64)
  n = len(x)
  i, k = np.nonzero(idx < n)
  j = idx[i, k]
  d = x[j] - x[i]
  if L.ndim == 2:
    d = (d - np.rint(d)) @ L.T
  else:
    d -= L * np.rint(d / L)
  s = (d ** 2).sum(1)
  c, o = 2.5 ** 2, 2.0 ** 2
  sig = sigma if species is None else np.asarray(sigma, np.float64)[species[i], species[j]]
  q6 = (sig ** 2 / s) ** 3.0
  V, dV = 4 * (q6 ** 2 - q6), -24 * (2 * q6 ** 2 - q6) / s
  S = np.where(s < o, 1.0, (c - s) ** 2 * (c + 2 * s - 3 * o) / (c - o) ** 3)
  dS = np.where(s < o, 0.0, 12 * (c - s) * (o - s) / (c - o) ** 3)
  inside = s < c
  g = np.where(inside, S * dV + dS * V, 0.0)
  F = np.zeros_like(x)
  np.add.at(F, i, g[:, None] * d)
  return 0.5 * np.where(inside, S * V, 0.0).sum(), F


def _system(dims, seed):
  rng = np.random.default_rng(seed)
  a = (1 / 0.8442) ** (1 / 3)
  sides = (np.array(dims) * a).astype(np.float32)
  g = np.stack(np.meshgrid(*[np.arange(d) for d in dims], indexing='ij'), -1).reshape(-1, 3)
  R = (g + 0.5) * (sides.astype(np.float64) / dims) + rng.normal(0, 0.05, g.shape)
  R = np.mod(R, sides.astype(np.float64)).astype(np.float32)
  return np.where(R >= sides, np.float32(0), R), sides


@pytest.mark.parametrize('lanes', [0, 2, 4, 8, 16])
@pytest.mark.parametrize('dims,multiplier,shortened', [
    ((8, 8, 8), 1.0, False),       # all pairs, rows end at their capacity
    ((9, 8, 14), 1.25, True),      # far faces in one dimension only
    ((11, 13, 10), 1.0, False),
    ((16, 9, 9), 1.5, True)])
def test_rows(lanes, dims, multiplier, shortened):
  import jax_md_amd as jmd
  R, sides = _system(dims, seed=sum(dims))
  disp, _ = jmd.space.periodic(sides)
  nfn, efn = jmd.energy.lennard_jones_neighbor_list(disp, sides, format=jmd.partition.Dense,
                                                    capacity_multiplier=multiplier)
  Rt = torch.as_tensor(R, device=DEV)
  nbrs = nfn.allocate(Rt)
  if shortened:  # rows of any length in one wavefront, empty ones among them
    keep = np.random.default_rng(1).integers(0, nbrs.idx.shape[1] + 1, (R.shape[0], 1))
    past = torch.arange(nbrs.idx.shape[1], device=DEV) >= torch.as_tensor(keep, device=DEV)
    nbrs.idx[past] = R.shape[0]
  E64, F64 = _rows_fp64(R, sides, nbrs.idx.cpu().numpy())
  lib = jmd._native.load()
  assert lib.jmd_set_threads_per_atom(lanes) == 0
  try:
    for in_box in (False, True):
      F = efn.force(Rt, nbrs, in_box=in_box)
      rel, worst = _force_err(F.cpu().numpy(), F64)
      print(f'rows {dims} lanes {lanes} in_box {in_box}: {rel:.2e} {worst:.2e}', flush=True)
      assert rel <= FORCE_RTOL and worst <= FORCE_WORST
    E, _ = efn.energy_and_force(Rt, nbrs)
    assert abs(float(E) - E64) <= 1e-6 * abs(E64)
  finally:
    lib.jmd_set_threads_per_atom(0)


@pytest.mark.parametrize('lanes', [0, 2, 4, 8, 16])
@pytest.mark.parametrize('species,matrix', [(True, False), (False, True), (True, True)])
def test_rows_with_species_and_box_matrix(lanes, species, matrix):
  """Parameters by species and fractional positions in a triclinic box, whose
  rows take their own instances and folds."""
  import jax_md_amd as jmd
  R, sides = _system((11, 9, 10), seed=3)
  n = R.shape[0]
  rng = np.random.default_rng(4)
  kw, sp, sig = {}, None, np.float32(1.0)
  if species:
    sp = rng.integers(0, 2, n).astype(np.int32)
    sig = np.array([[1.0, 0.95], [0.95, 0.9]], np.float32)
    kw = dict(species=torch.as_tensor(sp, device=DEV), sigma=torch.as_tensor(sig, device=DEV))
  box, disp = sides, jmd.space.periodic(sides)[0]
  if matrix:
    box = np.diag(sides) + np.array([[0, 1.1, 0.4], [0, 0, 0.9], [0, 0, 0]], np.float32)
    R = (R / sides).astype(np.float32)
    disp = jmd.space.periodic_general(box)[0]
    kw['fractional_coordinates'] = True
  nfn, efn = jmd.energy.lennard_jones_neighbor_list(disp, box, format=jmd.partition.Dense, **kw)
  Rt = torch.as_tensor(R, device=DEV)
  nbrs = nfn.allocate(Rt)
  E64, F64 = _rows_fp64(R, box, nbrs.idx.cpu().numpy(), sp, sig)
  lib = jmd._native.load()
  assert lib.jmd_set_threads_per_atom(lanes) == 0
  try:
    for in_box in (False, True):
      F = efn.force(Rt, nbrs, in_box=in_box)
      rel, worst = _force_err(F.cpu().numpy(), F64)
      print(f'rows species {species} matrix {matrix} lanes {lanes} in_box {in_box}: '
            f'{rel:.2e} {worst:.2e}', flush=True)
      assert rel <= FORCE_RTOL and worst <= FORCE_WORST
    E, _ = efn.energy_and_force(Rt, nbrs)
    assert abs(float(E) - E64) <= 1e-6 * abs(E64)
  finally:
    lib.jmd_set_threads_per_atom(0)


@pytest.mark.parametrize('lanes', [0, 2, 4, 8, 16])
@pytest.mark.parametrize('dim', [2, 3])
def test_rows_narrower_than_a_block(dim, lanes):
  """Soft-sphere rows cut to every width around a block of 4 entries a lane
  (fewer entries than lanes, a full block, one more), some rows ending before."""
  import jax_md_amd as jmd
  rng = np.random.default_rng(dim)
  n, L = 1500, np.float32(30.0 if dim == 2 else 10.0)
  R = rng.uniform(0, L, (n, dim)).astype(np.float32)
  disp, _ = jmd.space.periodic(L)
  nfn, efn = jmd.energy.soft_sphere_neighbor_list(disp, L, sigma=2.0, dr_threshold=0.2,
                                                  format=jmd.partition.Dense)
  Rt = torch.as_tensor(R, device=DEV)
  nbrs = nfn.allocate(Rt)
  lib = jmd._native.load()
  assert lib.jmd_set_threads_per_atom(lanes) == 0
  try:
    for width in (1, 2, 3, 5, 7, 8, 9, 15, 16, 17, 31, 32, 33):
      width = min(width, nbrs.idx.shape[1])
      rows = nbrs.idx[:, :width].contiguous()
      idx = rows.cpu().numpy()
      i, k = np.nonzero(idx < n)
      d = R[idx[i, k]].astype(np.float64) - R[i]
      d -= float(L) * np.rint(d / float(L))
      r = np.sqrt((d ** 2).sum(1))
      g = np.where(r < 2.0, -(1 - r / 2.0) / (2.0 * r), 0.0)
      F64 = np.zeros((n, dim))
      np.add.at(F64, i, g[:, None] * d)
      for in_box in (False, True):
        F = efn.force(Rt, dataclasses.replace(nbrs, idx=rows), in_box=in_box)
        rel, worst = _force_err(F.cpu().numpy(), F64)
        print(f'narrow rows {dim}-D lanes {lanes} width {width}: {rel:.2e} {worst:.2e}', flush=True)
        assert rel <= FORCE_RTOL and worst <= FORCE_WORST
  finally:
    lib.jmd_set_threads_per_atom(0)


@pytest.mark.parametrize('n', [1, 63, 4096, 32184, 70001, 98304, 98305, 131073, 262177, 600000])
def test_energy_total_is_the_sum_of_its_rows(n):
  """The total over block partials against the particles' own energies
  (float32 each, summed here in float64): 2^-24 of the sum of magnitudes.
  The last five have 3,072 partials, up to which a thread of the sum takes them
  one at a time, and 3,080, 4,104, 8,200 and 18,752, which it takes by fours."""
  import jax_md_amd as jmd
  g = torch.Generator(device=DEV).manual_seed(n)
  R = torch.rand((n, 3), generator=g, device=DEV) * 100.0
  disp, _ = jmd.space.periodic(100.0)
  nfn, efn = jmd.energy.soft_sphere_neighbor_list(disp, 100.0, sigma=2.0, dr_threshold=0.5,
                                                  format=jmd.partition.Dense)
  _, each_fn = jmd.energy.soft_sphere_neighbor_list(disp, 100.0, sigma=2.0, dr_threshold=0.5,
                                                    per_particle=True,
                                                    format=jmd.partition.Dense)
  nbrs = nfn.allocate(R)
  E, _ = efn.energy_and_force(R, nbrs)
  each = each_fn(R, nbrs).to(torch.float64)
  assert abs(float(E) - float(each.sum())) <= 2.0 ** -24 * float(each.abs().sum()) + 1e-30


@pytest.mark.parametrize('n', [8192, 8193, 12288, 12289, 20480, 20481, 24576, 24577])
@pytest.mark.parametrize('spacing,skin,species', [(1.06, 0.5, False), (1.06, 0.5, True),
                                                  (1.36, 0.3, False)])
def test_rows_on_both_sides_of_the_lane_rule(n, spacing, skin, species):
  """The built-in lanes at the row counts where they change: wide rows of
  scalar and of species parameters, narrow rows."""
  import jax_md_amd as jmd
  rng = np.random.default_rng(n)
  dims = (30, 29, 29)
  sides = (np.array(dims) * spacing).astype(np.float32)
  g = np.stack(np.meshgrid(*[np.arange(d) for d in dims], indexing='ij'), -1).reshape(-1, 3)
  R = ((g[:n] + 0.5) * spacing + rng.uniform(-0.08, 0.08, (n, 3))).astype(np.float32)
  sp, sig = None, np.float32(1.0)
  kw = {}
  if species:
    sp = rng.integers(0, 2, n).astype(np.int32)
    sig = np.array([[1.0, 0.95], [0.95, 0.9]], np.float32)
    kw = dict(species=torch.as_tensor(sp, device=DEV), sigma=torch.as_tensor(sig, device=DEV))
  disp, _ = jmd.space.periodic(sides)
  nfn, efn = jmd.energy.lennard_jones_neighbor_list(disp, sides, format=jmd.partition.Dense,
                                                    dr_threshold=skin, **kw)
  Rt = torch.as_tensor(R, device=DEV)
  nbrs = nfn.allocate(Rt)
  assert nbrs.idx.shape[1] >= 64 if spacing < 1.2 else 32 <= nbrs.idx.shape[1] < 64
  E64, F64 = _rows_fp64(R, sides, nbrs.idx.cpu().numpy(), sp, sig)
  E, F = efn.energy_and_force(Rt, nbrs)
  rel, worst = _force_err(F.cpu().numpy(), F64)
  print(f'lane rule n={n} width {nbrs.idx.shape[1]} species {species}: {rel:.2e} {worst:.2e}',
        flush=True)
  assert rel <= FORCE_RTOL and worst <= FORCE_WORST
  assert abs(float(E) - E64) <= 1e-6 * abs(E64)
