"""The shapes that tests/test_hip_gemm_f32.py runs against the rules that give a
float32 product its kernel and its tile (no GPU)."""

import os
import re

from tests import test_hip_gemm_f32 as gemm_f32

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "mesh_amd", "csrc")
COMPUTE_UNITS = 256     # of one MI355X


def _tiles():
  """[(rows, columns, k of a K tile, a, b, c, d)] of the table in gemm_f32.hip."""
  with open(os.path.join(CSRC, "gemm_f32.hip")) as f:
    found = re.findall(r"split_tile<([\d, ]+)>\(([\d., ]+)\)", f.read())
  tiles = []
  for sizes, costs in found:
    tm, tn, wn, wk, _ = [int(s) for s in sizes.split(",")]
    tiles.append((16 * tm, 16 * tn * wn, 32 * wk) +
                 tuple(float(c) for c in costs.split(",")))
  return tiles


def _picked(tiles, e, r, n, k):
  def cost(tile):
    rows, cols, tile_k, a, b, c, d = tile
    blocks = e * -(-r // rows) * -(-n // cols)
    per_unit = -(-blocks // COMPUTE_UNITS)
    return a + per_unit * b + -(-k // tile_k) * (c + per_unit * d)
  return min((t for t in tiles if t[2] <= k), key=cost)


def _in_terms(e, r, n, k):
  """Not one of the short reductions of little work that stay on float32 MFMAs."""
  with open(os.path.join(CSRC, "ffn.hip")) as f:
    (most_k, most_work), = re.findall(
        r"if \(K < (\d+) && \(double\)E \* R \* N \* K < ([\d.e]+)\)", f.read())
  return k >= int(most_k) or e * r * n * k >= float(most_work)


def test_every_tile_is_run_with_remainders():
  tiles = _tiles()
  assert len(tiles) == len(gemm_f32.TILE_SHAPES) == 13
  for tile, (e, r, n, k) in zip(tiles, gemm_f32.TILE_SHAPES):
    assert _in_terms(e, r, n, k)
    assert _picked(tiles, e, r, n, k) == tile
    assert _picked(tiles, e, r, n, k + 1) == tile       # a weight gradient
    assert r % tile[0] and n % tile[1] and k % tile[2] and (k + 1) % tile[2]


def test_which_products_are_short():
  """Seven of SHAPES run on float32 MFMAs as products, and one of
  NON_FINITE_SHAPES."""
  assert sum(not _in_terms(*s) for s in gemm_f32.SHAPES) == 7
  assert [_in_terms(*s) for s in gemm_f32.NON_FINITE_SHAPES] == [False, True, True]
