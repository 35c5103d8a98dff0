"""float32 products in three bf16 terms per operand, against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
  from mesh_amd import moe_hip
  moe_hip.load_library()
  return moe_hip


def _values(gen, *sizes):
  """Sixteen binary orders of magnitude, signs mixed."""
  exponent = torch.randint(-8, 8, sizes, generator=gen, device="cuda")
  return torch.ldexp(torch.randn(sizes, generator=gen, device="cuda"), exponent)


def _assert_close(got, a, b):
  """got [E,R,N] against a [E,R,K] . b [E,K,N].  Per 32 k six matrix products of
  exact terms and one addition to the sum, and a handful of additions where
  wavefronts share k out; what the three dropped products of terms leave out is at
  most 2^-24 of |a b|, and far less for most values.  (The shapes on float32 MFMAs
  round once per k, up to 260 times, in either direction: their sums stay inside it
  too.)"""
  a, b = a.double(), b.double()
  roundings = a.shape[2] // 32 + 20
  bound = roundings * 2.0 ** -24 * (a.abs() @ b.abs())
  assert (((got.double() - a @ b).abs()) <= bound).all()


# rows and columns around the tiles' edges (16 to 160 rows, 32 to 256 columns), k
# below, at and above one K tile of 32 to 256 and with remainders, few and many
# tiles.  (Seven of them are products short enough for float32 MFMAs; TILE_SHAPES has
# one for every tile in terms.)
SHAPES = [
    (1, 32, 32, 32), (1, 33, 36, 36), (1, 33, 68, 60), (3, 47, 132, 64),
    (1, 64, 512, 512), (2, 65, 260, 100), (1, 37, 64, 2052), (1, 100, 96, 1028),
    (8, 161, 1028, 196), (8, 320, 2048, 256), (8, 320, 512, 1028), (7, 95, 508, 260),
    (4, 330, 516, 644), (16, 97, 1024, 100), (30, 129, 1028, 68), (24, 255, 772, 36),
    (9, 161, 4096, 64), (1, 2000, 640, 320), (1, 5000, 36, 96), (12, 427, 1024, 128)]


# [experts, rows, columns, k]: one for each tile of the table, in its order, as a
# product and as a weight gradient summed over k + 1 rows (128 x 256, 160 x 256, 160 x
# 128, 64 x 128, 80 x 64, 96 x 64, 32 x 32, 16 x 32, 32 x 64, 96 x 256, 64 x 256, 64 x
# 128 with K tiles of 32, 16 x 128); rows, columns and k all leave a remainder
TILE_SHAPES = [
    (7, 1760, 280, 36), (16, 2276, 72, 48), (24, 1400, 72, 72), (24, 36, 660, 228),
    (4, 2224, 68, 204), (16, 1288, 32, 220), (1, 2084, 40, 348), (1, 36, 40, 332),
    (7, 36, 584, 328), (3, 2028, 548, 36), (4, 692, 1084, 40), (2, 712, 916, 92),
    (8, 36, 1040, 328)]


@pytest.mark.parametrize("shape", SHAPES + TILE_SHAPES)
def test_products(hip, shape):
  e, r, n, k = shape
  gen = torch.Generator(device="cuda").manual_seed(sum(shape))
  a, w = _values(gen, e, r, k), _values(gen, e, n, k)
  got = hip.expert_linear(a, w, "linear")
  _assert_close(got, a, w.transpose(1, 2).contiguous())


@pytest.mark.parametrize("shape", SHAPES + TILE_SHAPES)
def test_products_summed_over_rows(hip, shape):
  """Weight gradients: both operands with the reduction outermost, any length."""
  e, m, n, rows = shape
  m, rows = (m + 3) // 4 * 4, rows + 1
  gen = torch.Generator(device="cuda").manual_seed(sum(shape))
  a, dy = _values(gen, e, rows, m), _values(gen, e, rows, n)
  w = torch.empty(e, m, n, device="cuda")
  _, got = hip.expert_linear_backward(a, dy, w, want_da=False)
  _assert_close(got, a.transpose(1, 2).contiguous(), dy)


# (the first is short enough for float32 MFMAs)
NON_FINITE_SHAPES = [(2, 70, 260, 100), (8, 320, 512, 1028), (2, 70, 260, 1028)]


@pytest.mark.parametrize("shape", NON_FINITE_SHAPES)
@pytest.mark.parametrize("activation", ["linear", "relu"])
def test_infinities_nan_and_overflow(hip, shape, activation):
  """What an infinity, a NaN or an overflow does to a sum is what it does in
  float32 arithmetic; the rest of its tile keeps its values."""
  e, r, n, k = shape
  gen = torch.Generator(device="cuda").manual_seed(5)
  a, w = _values(gen, e, r, k), _values(gen, e, n, k)
  a[0, 3, 7] = float("inf")
  w[0, 9, 7] = -2.0            # -inf
  w[0, 10, 7] = 1.0            # +inf: no remainder of 1.0 times infinity
  w[0, 11, 7] = 0.0            # NaN
  a[0, 5, 1] = float("nan")
  a[1, 0, 2], a[1, 0, 3] = 3e38, -3e38
  w[1, 4, 2], w[1, 4, 3] = 2.0, -2.0    # overflows in any order
  a[1, 1, 0] = 3.402823e38              # rounds to infinity in bf16
  w[1, :, 0] = 2.0 ** -20
  got = hip.expert_linear(a, w, activation).double()
  wt = w.double().transpose(1, 2).contiguous()
  want, absolute = a.double() @ wt, a.double().abs() @ wt.abs()
  # (an element of a tile that is computed again is added k by k)
  bound = (k + 20) * 2.0 ** -24 * absolute
  want = want.float().double()
  if activation == "relu":
    # NaN and negative sums become 0, as in every other kernel here
    want = torch.where(want > 0, want, torch.zeros_like(want))
  sure = absolute < 3.4e38              # no partial sum can overflow
  assert ((got - want).abs() <= bound)[sure].all()
  sure = ~absolute.isfinite()
  sure[1, 0, 4] = True
  assert torch.equal(got[sure].nan_to_num(7.0, 1e300, -1e300),
                     want[sure].nan_to_num(7.0, 1e300, -1e300))


@pytest.mark.parametrize("form", ["product", "masked", "weight gradient"])
@pytest.mark.parametrize("shape", TILE_SHAPES)
def test_infinities_and_nan_in_every_tile(hip, shape, form):
  """Non-finite values in both operands, at the k that the last K tile takes twice
  among others, do to every sum what they do in float64; the other sums of their
  tiles keep their values."""
  e, r, n, k = shape
  gen = torch.Generator(device="cuda").manual_seed(sum(shape))
  if form == "weight gradient":
    k += 1
  a, w = _values(gen, e, r, k), _values(gen, e, n, k)
  for t in (a, w):
    for at, value in enumerate(("inf", "-inf", "nan") * 2):
      row = int(torch.randint(t.shape[1], (), generator=gen, device="cuda"))
      back = int(torch.randint(min(k, 300), (), generator=gen, device="cuda"))
      t[at % e, row, k - 1 - back] = float(value)
  wt = w.transpose(1, 2).contiguous()
  want = a.double() @ wt.double()
  if form == "product":
    got = hip.expert_linear(a, w, "linear")
  elif form == "masked":
    mask = torch.randn((e, r, n), generator=gen, device="cuda")
    got, _ = hip.expert_linear_backward(torch.zeros_like(mask), a, w,
                                        da_relu_mask=mask)
    want = torch.where(mask > 0, want, torch.zeros_like(want))
  else:
    _, got = hip.expert_linear_backward(
        a.transpose(1, 2).contiguous(), wt, torch.empty(e, r, n, device="cuda"),
        want_da=False)
  finite = want.isfinite()
  assert not finite.all() and finite.any()
  # (a tile that is made again is added k by k; what the mask clears is 0)
  bound = (k + 20) * 2.0 ** -24 * (a.double().abs() @ wt.double().abs())
  bound = bound.nan_to_num(0.0, 0.0)
  assert ((got.double() - want).abs() <= bound)[finite].all()
  assert torch.equal(got.double()[~finite].nan_to_num(7.0, 1e300, -1e300),
                     want[~finite].nan_to_num(7.0, 1e300, -1e300))


def _time_us(call, reps=5):
  call()
  times = []
  for _ in range(reps):
    start, end = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    start.record()
    call()
    end.record()
    end.synchronize()
    times.append(start.elapsed_time(end) * 1e3)
  return sorted(times)[reps // 2]


@pytest.mark.parametrize("kmajor", [False, True])
def test_products_of_nan_take_no_more_than_a_few_times_as_long(hip, kmajor):
  """A diverged step, all of whose gradients are NaN, still ends in time."""
  e, r, n, k = 8, 1024, 512, 2048
  gen = torch.Generator(device="cuda").manual_seed(6)
  if kmajor:
    a, dy = _values(gen, e, k, r), _values(gen, e, k, n)
    w = torch.empty(e, r, n, device="cuda")
    call = lambda t: hip.expert_linear_backward(a, t, w, want_da=False)[1]
  else:
    a, dy = _values(gen, e, r, k), _values(gen, e, n, k)
    call = lambda t: hip.expert_linear(a, t, "linear")
  finite = _time_us(lambda: call(dy))
  dy = torch.full_like(dy, float("nan"))
  assert call(dy).isnan().all()
  # (the products in terms, then on float32 MFMAs at less than half their rate)
  nan = _time_us(lambda: call(dy))
  print("finite %.1f us, NaN %.1f us" % (finite, nan))
  assert nan < 10 * finite


@pytest.mark.parametrize("kmajor", [False, True])
@pytest.mark.parametrize("exponent", [-60, -100, -109, -112, -118, -124, -135])
@pytest.mark.parametrize("shape", [(1, 40, 64, 1028), (3, 164, 260, 324),
                                   (8, 320, 512, 2048)])
def test_tiny_values_keep_their_bits(hip, shape, exponent, kmajor):
  """A product with a selection of the columns gives back every value exactly, also
  where its third term would lie below the last bit of a bf16 denormal; as either
  operand, and with one tiny value in a thousand."""
  e, r, n, k = shape
  gen = torch.Generator(device="cuda").manual_seed(r - exponent)
  scale = 2.0 ** 60                    # (the results are no denormals)
  for share in (1.0, 1e-3):
    a = torch.randn((e, r, k), generator=gen, device="cuda")
    tiny = torch.rand((e, r, k), generator=gen, device="cuda") < share
    a = torch.where(tiny, (a.double() * 2.0 ** exponent).float(), a)
    at = torch.randint(0, k, (e, n), generator=gen, device="cuda")
    pick = torch.zeros((e, n, k), device="cuda").scatter_(2, at[..., None], scale)
    want = (a.double() * scale).float().gather(
        2, at[:, None].expand(e, r, n).contiguous())
    for first, second, result in ((a, pick, want),
                                  (pick, a, want.transpose(1, 2).contiguous())):
      if kmajor:
        first, second = [t.transpose(1, 2).contiguous() for t in (first, second)]
        _, got = hip.expert_linear_backward(
            first, second, torch.empty_like(result), want_da=False)
      else:
        got = hip.expert_linear(first, second, "linear")
      assert torch.equal(got, result)


@pytest.mark.parametrize("kmajor", [False, True])
def test_products_of_many_rows_stay_on_the_matrix_cores(hip, kmajor):
  """More than 2^22 rows (of a weight gradient: to sum over) cost per row what fewer
  do."""
  n = 256
  gen = torch.Generator(device="cuda").manual_seed(7)

  def run(rows):
    a = torch.randn((1, rows, n), generator=gen, device="cuda")
    if not kmajor:
      w = torch.randn((1, n, n), generator=gen, device="cuda")
      call = lambda: hip.expert_linear(a, w, "linear")
      _assert_close(call()[:, -100:], a[:, -100:], w.transpose(1, 2).contiguous())
    else:
      w = torch.empty(1, n, n, device="cuda")
      dy = torch.randn((1, rows, n), generator=gen, device="cuda")
      call = lambda: hip.expert_linear_backward(a, dy, w, want_da=False)[1]
      _assert_close(call(), a.transpose(1, 2).contiguous(), dy)
    return _time_us(call)
  few, many = run(1 << 22), run((1 << 22) + 4)
  torch.cuda.empty_cache()
  assert many < 1.5 * few


def test_long_reductions(hip):
  """A reduction of more than 2^25 elements, which no tile in terms takes."""
  r, n, k = 33, 36, (1 << 25) + 4
  gen = torch.Generator(device="cuda").manual_seed(8)
  a = torch.zeros((1, r, k), device="cuda")
  at = torch.randint(0, k, (64,), generator=gen, device="cuda")
  at[0] = k - 1
  a[0, :, at] = _values(gen, r, 64)
  w = torch.zeros((1, n, k), device="cuda")
  w[0, :, at] = _values(gen, n, 64)
  got = hip.expert_linear(a, w, "linear")
  x, y = a[:, :, at.unique()], w[:, :, at.unique()].transpose(1, 2)
  # (64 sums that are not of zeros)
  bound = 84 * 2.0 ** -24 * (x.double().abs() @ y.double().abs().contiguous())
  assert ((got.double() - x.double() @ y.double().contiguous()).abs() <= bound).all()


def test_weight_gradients_of_long_rows(hip):
  """Rows too long for 32-bit offsets inside a K tile of 32."""
  m, n, rows = 89478488, 32, 33
  gen = torch.Generator(device="cuda").manual_seed(9)
  a = torch.randn((1, rows, m), generator=gen, device="cuda")
  dy = _values(gen, 1, rows, n)
  _, got = hip.expert_linear_backward(a, dy, torch.empty(1, m, n, device="cuda"),
                                      want_da=False)
  at = torch.randint(0, m, (1000,), generator=gen, device="cuda")
  at[:40] = torch.arange(m - 40, m, device="cuda")
  x = a[:, :, at].transpose(1, 2).contiguous()
  bound = (rows + 20) * 2.0 ** -24 * (x.double().abs() @ dy.double().abs())
  close = (got[:, at].double() - x.double() @ dy.double()).abs() <= bound
  del a, got
  torch.cuda.empty_cache()
  assert close.all()
