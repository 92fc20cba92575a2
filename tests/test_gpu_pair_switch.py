"""The switched Lennard-Jones pair term inside its window, pair by pair,
against float64 at the same float32 r^2.

The pairs lie along x with one particle at the origin, so that r^2 is one
rounded product and the window's squares are exact in float32: what is left is
the evaluation from r^2.  Bar: 64 x 2^-24 norm-wise, from the roundings of that
evaluation in units of 2^-24: 1/r^2 2 (one ulp), t = r^-6 11, 2 t - 1 at most 23
(r >= 1.18), the switch variable y 3 and y (3 - 2 y) 11, products and sums 5, in
all 56 of the pair's own force, and 3 of y for x = 1 - y, at most 7 of the
norm over a window.  None of them grows as the window narrows."""

import dataclasses

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _dimers(jmd, x, r_onset, r_cutoff):
  """Energy function, positions and list of pairs (2k, 2k+1) at separation x[k] along x."""
  n = 2 * len(x)
  R = np.zeros((n, 3), np.float32)
  R[1::2, 0] = x
  disp, _ = jmd.space.free()
  nfn, efn = jmd.energy.lennard_jones_neighbor_list(
      disp, 100.0, r_onset=r_onset, r_cutoff=r_cutoff, format=jmd.partition.Dense,
      disable_cell_list=True)
  apart = np.zeros((n, 3), np.float32)
  apart[:, 0] = 10.0 * np.arange(n)
  nbrs = nfn.allocate(torch.as_tensor(apart, device=DEV))
  idx = torch.full((n, 3), n, dtype=torch.int32, device=DEV)
  idx[:, 0] = torch.arange(n, device=DEV).to(torch.int32) ^ 1
  return efn, torch.as_tensor(R, device=DEV), dataclasses.replace(nbrs, idx=idx)


@pytest.mark.parametrize('r_onset,r_cutoff', [
    (2.0, 2.5), (1.1875, 1.25), (2.5 - 2 ** -7, 2.5), (2.5 - 2 ** -10, 2.5)])
def test_pair_term_inside_the_switch(r_onset, r_cutoff):
  import jax_md_amd as jmd
  assert all(float(np.float32(v * v)) == v * v for v in (r_onset, r_cutoff))
  rng = np.random.default_rng(7)
  x = rng.uniform(r_onset, r_cutoff, 1000).astype(np.float32)
  s = (x * x).astype(np.float64)  # the float32 r^2
  o, c = r_onset ** 2, r_cutoff ** 2
  V, dV = 4 * (s ** -6 - s ** -3), -24 * (2 * s ** -6 - s ** -3) / s
  S = np.where(s < o, 1.0, (c - s) ** 2 * (c + 2 * s - 3 * o) / (c - o) ** 3)
  dS = np.where(s < o, 0.0, 12 * (c - s) * (o - s) / (c - o) ** 3)
  U, f = np.where(s < c, S * V, 0.0), np.where(s < c, (S * dV + dS * V) * x, 0.0)
  efn, R, nbrs = _dimers(jmd, x, r_onset, r_cutoff)
  E, F = efn.energy_and_force(R, nbrs)
  F = F.cpu().numpy().astype(np.float64)
  assert np.array_equal(F[0::2], -F[1::2]) and not F[:, 1:].any()
  ef = np.linalg.norm(F[0::2, 0] - f) / np.linalg.norm(f)
  ee = abs(float(E) - U.sum()) / np.abs(U).sum()
  print(f'switch [{r_onset}, {r_cutoff}]: force {ef:.2e} energy {ee:.2e}', flush=True)
  assert ef <= 64 * 2.0 ** -24
  assert ee <= 64 * 2.0 ** -24


@pytest.mark.parametrize('fmt', ['Dense', 'OrderedSparse'])
@pytest.mark.parametrize('r_onset', [2.0, 2.5])
def test_coincident_particles_have_no_energy(r_onset, fmt):
  """r = 0: the terms r^-12 and -r^-6 are both infinite, so the energy, like
  the force, is not a number (with the switch and, r_onset = r_cutoff,
  without)."""
  import jax_md_amd as jmd
  disp, _ = jmd.space.free()
  R = torch.zeros((4, 3), device=DEV)
  R[2:, 0] = torch.tensor([10.0, 11.5], device=DEV)
  kw = dict(r_onset=r_onset, r_cutoff=2.5, format=getattr(jmd.partition, fmt),
            disable_cell_list=True)
  nfn, efn = jmd.energy.lennard_jones_neighbor_list(disp, 100.0, **kw)
  nbrs = nfn.allocate(R)
  print(f'case coincident r_onset={r_onset} {fmt}', flush=True)
  E, F = efn.energy_and_force(R, nbrs)
  assert torch.isnan(E).all()
  assert torch.isnan(F[:2]).all() and torch.isfinite(F[2:]).all()
