"""Dense rows over a position table beyond 2 GiB (512 x 512 x 513 particles,
rows of 16 bytes), whose gathers take another form: every row's force and the
energy against float64, with the bars of test_gpu_pair.py (1e-5 norm-wise,
5e-5 of the rms for one component, 1e-6 for the energy)."""

import dataclasses

import pytest
import torch

from tests.test_gpu_pair import FORCE_RTOL, FORCE_WORST

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'
SIDE = (512, 512, 513)
SPACING = 1.1
WIDTH = 7  # six lattice neighbours and a pad: a whole block and a short one


def _rows():
  """Jittered lattice and each particle's six neighbours (at a face the inner
  one twice, so that no pair crosses the box)."""
  from jax_md_amd import _native as nat
  X, Y, Z = SIDE
  n = X * Y * Z
  ids = torch.arange(n, device=DEV, dtype=torch.int32)
  cell = [ids % X, (ids // X) % Y, ids // (X * Y)]
  R = nat.padded_positions(n, DEV)
  idx = torch.full((n, WIDTH), n, dtype=torch.int32, device=DEV)
  g = torch.Generator(device=DEV).manual_seed(5)
  for c, (v, step) in enumerate(zip(cell, (1, X, X * Y))):
    R[:, c] = 5.0 + SPACING * v + (torch.rand((n,), generator=g, device=DEV) - 0.5) * 0.1
    idx[:, 2 * c] = ids + torch.where(v > 0, -step, step).to(torch.int32)
    idx[:, 2 * c + 1] = ids + torch.where(v < SIDE[c] - 1, step, -step).to(torch.int32)
  return R, idx


def _pair_fp64(kind, s, sig):
  """U and U'(r)/r from r^2 in float64."""
  if kind == 'soft':  # 1/2 (1 - r / sigma)^2
    r = s.sqrt()
    b = (1 - r / sig).clamp(min=0)
    return 0.5 * b * b, -b / (sig * r)
  q = (sig * sig / s) ** 3
  V, dV = 4 * (q * q - q), -24 * (2 * q * q - q) / s
  o, c = 2.0 ** 2, 2.5 ** 2
  S = torch.where(s < o, torch.ones_like(s), (c - s) ** 2 * (c + 2 * s - 3 * o) / (c - o) ** 3)
  dS = torch.where(s < o, torch.zeros_like(s), 12 * (c - s) * (o - s) / (c - o) ** 3)
  return torch.where(s < c, S * V, 0 * s), torch.where(s < c, S * dV + dS * V, 0 * s)


@pytest.mark.parametrize('kind', ['lj', 'lj species', 'lj matrix', 'soft'])
def test_rows_of_a_large_table(kind):
  import jax_md_amd as jmd
  if torch.cuda.get_device_properties(0).total_memory < 64 << 30:
    pytest.skip('needs 64 GiB of device memory')
  R, idx = _rows()
  n = R.shape[0]
  assert n * 16 > 2 ** 31
  print(f'case large table {kind} n={n}', flush=True)
  box = [SPACING * d + 20.0 for d in SIDE]
  disp, _ = jmd.space.periodic(box)
  T = torch.diag(torch.tensor(box, dtype=torch.float64, device=DEV))
  kw = dict(format=jmd.partition.Dense)
  if kind == 'lj matrix':  # fractional positions, the lattice sheared a little
    R /= torch.tensor(box, device=DEV)
    T[0, 1], T[1, 2] = 0.02 * T[1, 1], 0.03 * T[2, 2]
    T = T.float().double()
    box = T.cpu().numpy().astype('float32')
    disp, _ = jmd.space.periodic_general(box)
    kw['fractional_coordinates'] = True
  sig = torch.tensor([[1.0, 0.95], [0.95, 0.9]], device=DEV)
  if kind == 'soft':
    nfn, efn = jmd.energy.soft_sphere_neighbor_list(disp, box, sigma=1.2, **kw)
  elif kind != 'lj species':
    nfn, efn = jmd.energy.lennard_jones_neighbor_list(disp, box, **kw)
  else:
    species = torch.arange(n, device=DEV, dtype=torch.int32) % 2
    nfn, efn = jmd.energy.lennard_jones_neighbor_list(disp, box, species=species, sigma=sig, **kw)
  few = jmd.energy.lennard_jones_neighbor_list(disp, box, **kw)[0].allocate(
      R[:64].contiguous())
  E, F = efn.energy_and_force(R, dataclasses.replace(few, idx=idx))
  e64 = mag = err = ref = torch.zeros((), dtype=torch.float64, device=DEV)
  worst = 0.0
  for lo in range(0, n, 1 << 23):
    hi = min(lo + (1 << 23), n)
    j = idx[lo:hi, :6].long()
    d = R[j].double() - R[lo:hi, None].double()
    if kind == 'lj matrix':
      d = d @ T.T
    s = (d * d).sum(-1)
    sg = 1.2 if kind == 'soft' else 1.0
    if kind == 'lj species':
      sg = sig.double()[torch.arange(lo, hi, device=DEV)[:, None] % 2, j % 2]
    U, g = _pair_fp64(kind, s, sg)
    F64 = (g[..., None] * d).sum(1)
    diff = F[lo:hi].double() - F64
    e64, mag = e64 + 0.5 * U.sum(), mag + 0.5 * U.abs().sum()
    err, ref = err + (diff * diff).sum(), ref + (F64 * F64).sum()
    worst = max(worst, float(diff.abs().max()))
  rel, rms = float((err / ref).sqrt()), float((ref / (3 * n)).sqrt())
  print(f'  force {rel:.2e} worst/rms {worst / rms:.2e} energy {float(abs(E - e64) / mag):.2e}',
        flush=True)
  assert rel <= FORCE_RTOL and worst <= FORCE_WORST * rms
  assert float(abs(E - e64)) <= 1e-6 * float(mag)
