"""The native Dense-to-Sparse conversion against the same list written out on
the host: entry for entry, at the edges of its blocks of 64 rows and of its
64-entry chunks, with and without room for every entry."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = 'cuda:0'


def _expected(rows, ordered, cap):
  n = len(rows)
  idx = np.full((2, cap), n, np.int32)
  pairs = [(j, i) for i, row in enumerate(rows) for j in row
           if j < n and (not ordered or j < i)]
  if pairs[:cap]:
    idx[:, :min(cap, len(pairs))] = np.array(pairs[:cap], np.int32).T
  return idx, len(pairs)


@pytest.mark.parametrize('ordered', [False, True])
@pytest.mark.parametrize('n,width', [(1, 1), (63, 5), (64, 63), (65, 64), (130, 65), (257, 141),
                                     (2000, 17), (70000, 3)])
def test_rows_to_sparse(n, width, ordered):
  from jax_md_amd import _native as nat
  lib = nat.load()
  rng = np.random.default_rng(n * 1000 + width)
  rows = rng.integers(0, n, (n, width)).astype(np.int32)
  count = rng.integers(0, width + 1, n)
  rows[np.arange(width)[None, :] >= count[:, None]] = n
  want_all, total = _expected(rows, ordered, n * width)
  rows_d = torch.as_tensor(rows, device=DEV)
  ws = torch.empty((lib.jmd_dense_rows_to_sparse_workspace_bytes(n),), dtype=torch.uint8,
                   device=DEV)
  for cap in sorted({max(total // 2, 1), total, total + 100}):
    print(f'rows to sparse n={n} width={width} ordered={ordered} cap={cap}', flush=True)
    idx = torch.full((2, cap), -7, dtype=torch.int32, device=DEV)
    err = torch.full((), 4, dtype=torch.uint8, device=DEV)
    rc = lib.jmd_dense_rows_to_sparse(
        nat.ptr(rows_d), n, width, nat.ORDERED_SPARSE if ordered else nat.SPARSE, nat.ptr(idx),
        cap, nat.ptr(err), nat.ptr(ws), nat.stream_handle(torch.device(DEV)))
    assert rc == nat.JMD_OK
    want = np.full((2, cap), n, np.int32)
    m = min(cap, total)
    want[:, :m] = want_all[:, :m]
    assert np.array_equal(idx.cpu().numpy(), want)
    assert int(err) == (5 if total > cap else 4)


def test_a_block_leaves_what_was_derived_from_the_list_behind():
  """After a block over a Sparse-format list the forces follow the list the
  block wrote, not the rows that came with the list before it."""
  import jax_md_amd as jmd
  from oracle import jaxmd_oracle as O
  R, P, L = O.lj_lattice(12, seed=3)
  disp, shift = jmd.space.periodic(L)
  nfn, efn = jmd.energy.lennard_jones_neighbor_list(disp, L,
                                                    format=jmd.partition.OrderedSparse)
  Rt = torch.as_tensor(R, device=DEV)
  nbrs = nfn.allocate(Rt, extra_capacity=16)
  init, _ = jmd.simulate.nve(efn, shift, 5e-3)
  st = init(0, Rt, 0.0, momenta=torch.as_tensor(P, device=DEV), neighbor=nbrs)
  loop = jmd.simulate.NVELoop(efn, shift, 5e-3)
  loop.prime(st, nbrs)
  assert jmd.partition.current_shadow(nbrs) is not None
  loop.run(st, nbrs, 30)
  assert jmd.partition.current_shadow(nbrs) is None
  F = efn.force(st.position, nbrs)
  m = O.PairModel('lj')
  _, _, F64 = O.energy_force_brute(m, O.Space(np.float64(L)),
                                   st.position.cpu().numpy().astype(np.float64))
  assert np.linalg.norm(F.cpu().numpy() - F64) <= 1e-5 * np.linalg.norm(F64)
