"""GPU parity of each C-ABI entry point against the CPU oracle."""

import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
  from mesh_amd import moe_hip
  moe_hip.load_library()
  return moe_hip


# (G, S, E, C) -- the first three are the routing shapes of the benchmark
# configurations 1-3; the rest are ragged / odd shapes and the wide-E paths.
GATING_SHAPES = [
    (2, 1024, 8, 160), (16, 1024, 32, 40), (16, 2048, 64, 32),
    (3, 77, 5, 7), (1, 1, 2, 1), (2, 300, 128, 6), (2, 130, 200, 4),
    (1, 257, 300, 3), (5, 64, 16, 64), (1, 4096, 64, 128),
]


@pytest.mark.parametrize("shape", GATING_SHAPES)
def test_gating_random_logits(hip, shape):
  g, s, e, c = shape
  rng = np.random.default_rng(hash(shape) % (2 ** 31))
  bias = H.zipf_bias(rng, e) if shape == (16, 2048, 64, 32) else None
  logits = H.safe_logits(rng, g, s, e, scale=1.5, bias=bias)
  assert H.min_relative_gap(O.softmax(logits), min(3, e)) > 2e-5
  want = O.top_2_gating(logits, c)
  r = hip.top2_gating(torch.from_numpy(logits).cuda(), c)
  got = H.routing_to_np(r)
  H.assert_routing_equal(got, want)
  np.testing.assert_allclose(got["loss"], want["loss"], rtol=2e-5)


# group sizes around the 64-token blocks and the eight ids of a wide read, expert
# counts around the 16 lanes of a token and the groups of four of its sums, the
# most experts and a group whose ids fill most of LDS
@pytest.mark.parametrize("shape", [
    (2, 63, 17, 5), (1, 64, 16, 6), (3, 65, 3, 30), (1, 129, 33, 8),
    (2, 71, 512, 2), (1, 1500, 16, 100), (1, 15999, 6, 3000)])
@pytest.mark.parametrize("second_place_loss", [False, True])
def test_gating_edges(hip, shape, second_place_loss):
  g, s, e, c = shape
  rng = np.random.default_rng(sum(shape))
  logits = H.safe_logits(rng, g, s, e, scale=1.5)
  want = O.top_2_gating(logits, c, use_second_place_loss=second_place_loss)
  r = hip.top2_gating(torch.from_numpy(logits).cuda(), c,
                      use_second_place_loss=second_place_loss)
  got = H.routing_to_np(r)
  H.assert_routing_equal(got, want)
  np.testing.assert_allclose(got["loss"], want["loss"], rtol=2e-5)


@pytest.mark.parametrize("shape", [(2, 256, 8, 40), (3, 500, 64, 9)])
def test_gating_exact_ties(hip, shape):
  """Logits on a coarse grid: many exact ties, where the lowest index must win
  both times; unequal logits differ by >= 0.25 so nothing is a near-tie."""
  g, s, e, c = shape
  rng = np.random.default_rng(7)
  logits = H.random_logits(rng, g, s, e, scale=0.6, quantum=0.25)
  want = O.top_2_gating(logits, c)
  got = H.routing_to_np(hip.top2_gating(torch.from_numpy(logits).cuda(), c))
  H.assert_routing_equal(got, want)


@pytest.mark.parametrize("imp_dtype", ["float32", "bfloat16"])
def test_gating_importance(hip, imp_dtype):
  g, s, e, c = 4, 320, 16, 24
  rng = np.random.default_rng(11)
  logits = H.safe_logits(rng, g, s, e)
  imp = rng.choice(np.array([0.0, 0.5, 1.0], np.float32), size=(g, s),
                   p=[0.2, 0.3, 0.5])
  assert H.min_relative_gap(O.softmax(logits)) > 1e-5
  want = O.top_2_gating(logits, c, importance=imp, use_second_place_loss=True)
  r = hip.top2_gating(torch.from_numpy(logits).cuda(), c,
                      importance=H.to_gpu(imp, imp_dtype),
                      use_second_place_loss=True)
  got = H.routing_to_np(r)
  H.assert_routing_equal(got, want)
  np.testing.assert_allclose(got["loss"], want["loss"], rtol=2e-5)
  # importance 0.5 rows go to their best expert as a second-priority choice
  half = imp == 0.5
  assert (got["index_1"][half] == got["index_2"][half]).all()
  assert not got["kept_1"][half].any()
  assert not got["kept_1"][imp == 0].any() and not got["kept_2"][imp == 0].any()


@pytest.mark.parametrize("policy", ["none", "threshold", "random"])
def test_gating_second_policy(hip, policy):
  g, s, e, c = 3, 512, 8, 200
  rng = np.random.default_rng(13)
  logits = H.safe_logits(rng, g, s, e)
  u = rng.random((g, s)).astype(np.float32)
  thr = 0.3
  ref_all = O.top_2_gating(logits, 10 ** 6)  # uncapped: raw normalised gates
  g2 = ref_all["gate_2"]
  if policy == "threshold":
    assert np.abs(g2 - np.float32(thr)).min() > 1e-6
  if policy == "random":
    assert np.abs(u - g2 * np.float32(1.0 / thr)).min() > 1e-6
  want = O.top_2_gating(logits, c, policy=policy, threshold=thr,
                        second_uniform=u, use_second_place_loss=True,
                        num_microbatches=4)
  r = hip.top2_gating(torch.from_numpy(logits).cuda(), c, policy=policy,
                      threshold=thr, second_uniform=torch.from_numpy(u).cuda(),
                      use_second_place_loss=True, num_microbatches=4)
  got = H.routing_to_np(r)
  H.assert_routing_equal(got, want)
  np.testing.assert_allclose(got["loss"], want["loss"], rtol=2e-5)


# token, expert and column counts around the 16 x 16 tiles, the groups of 16
# columns and the 128 that are on their way, rows of 16-byte pieces and others
@pytest.mark.parametrize("shape", [
    (1, 1, 1, 2), (1, 15, 3, 16), (1, 17, 15, 17), (2, 33, 17, 3), (1, 16, 130, 64),
    (3, 5, 128, 128), (1, 1000, 255, 33), (1, 40, 256, 8), (2, 70, 260, 100),
    (1, 31, 516, 15), (1, 300, 63, 1)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_router_logits_edges(hip, shape, dtype):
  b, t, m, e = shape
  gen = torch.Generator(device="cuda").manual_seed(sum(shape))
  x = torch.randn((b, t, m), generator=gen, device="cuda").to(H.ACT_TORCH[dtype])
  w = torch.randn((b, m, e), generator=gen, device="cuda").to(H.ACT_TORCH[dtype])
  bias = torch.randn((e,), generator=gen, device="cuda")
  got = hip.router_logits(x, w, bias).double()
  want = x.double() @ w.double() + bias.double()
  # a rounding per column and one for the bias
  bound = (m + 1) * 2.0 ** -24 * (
      x.double().abs() @ w.double().abs() + bias.double().abs())
  assert ((got - want).abs() <= bound).all()


@pytest.mark.parametrize("s,e", [(1, 2), (3, 512), (17, 5), (63, 16), (64, 64)])
@pytest.mark.parametrize("router", ["top2", "switch"])
def test_small_groups_gating(hip, router, s, e):
  """Groups of at most 64 tokens are gated by one launch where they are few: the bits
  of the launch per step that many groups take (more than 2048; slots by gate: more
  than 128)."""
  gen = torch.Generator(device="cuda").manual_seed(s + e)
  groups = 2100
  logits = torch.randn((groups, s, e), generator=gen, device="cuda")
  logits[0, s // 2] = 0.25                      # equal probabilities
  importance = torch.randint(0, 3, (groups, s), generator=gen, device="cuda") / 2
  capacity = max(1, s // 4)
  for imp in (None, importance):
    def gating(g):
      some = None if imp is None else imp[:g].contiguous()
      if router == "switch":
        return hip.switch_gating(logits[:g].contiguous(), capacity, importance=some,
                                 z_loss=0.01, slots_by_gate=e % 2 == 0)
      return hip.top2_gating(logits[:g].contiguous(), capacity, importance=some,
                             policy="threshold", use_second_place_loss=True)
    many = gating(groups)
    for g in (1, 2, 128):
      few = gating(g)
      for name in ("idx", "pos", "gate", "kept", "fill"):
        assert torch.equal(getattr(few, name), getattr(many, name)[:g]), name


def _gating(hip, router, logits, importance, capacity):
  if router == "switch":
    return hip.switch_gating(logits, capacity, importance=importance, z_loss=0.01)
  return hip.top2_gating(logits, capacity, importance=importance, policy="threshold",
                         use_second_place_loss=True)


# groups of one block of 64 tokens, of one and a token, of whole blocks, of more blocks
# than are read together (16), the most experts; groups that are one launch however
# many blocks they have, with an expert that most tokens choose
@pytest.mark.parametrize("s,e", [(64, 16), (65, 5), (128, 64), (1000, 8), (1100, 33),
                                 (130, 512), (8192, 16), (16384, 4)])
@pytest.mark.parametrize("router", ["top2", "switch"])
def test_gating_in_one_launch(hip, router, s, e):
  """Few groups are gated by one launch, many by one per step: the same bits.  Twice,
  since the launch's counters are left for the next call.  The many are the few over
  and over, whose loss is the same mean: but for a rounding per group, and (both sides,
  which may cut a group into blocks of 64 and of 128 tokens) per block and per token of
  a block."""
  gen = torch.Generator(device="cuda").manual_seed(s + e)
  nblk = (s + 63) // 64
  cus = torch.cuda.get_device_properties(0).multi_processor_count
  # more than 2048 single blocks; tokens from which a block is 128 of them; else more
  # than 5 / 4 blocks per compute unit
  least = (2049 if nblk == 1 else -(-65536 // s) if s >= 8192 else
           (5 * cus // 4) // nblk + 1)
  copies = -(-least // 3)
  few_logits = torch.randn((3, s, e), generator=gen, device="cuda")
  few_logits[0, s // 2] = 0.25                  # equal probabilities
  if s >= 8192:
    few_logits[..., 0] += 2.5
  few_importance = torch.randint(0, 3, (3, s), generator=gen, device="cuda") / 2
  capacity = max(1, s // 4)
  rel = 2 * (3 * copies + nblk + 128) * 2.0 ** -24
  for with_importance in (False, True):
    def gating(logits, importance):
      return _gating(hip, router, logits, importance if with_importance else None,
                     capacity)
    many = gating(few_logits.repeat(copies, 1, 1), few_importance.repeat(copies, 1))
    for g in (1, 3, 3):
      few = gating(few_logits[:g].contiguous(), few_importance[:g].contiguous())
      for name in ("idx", "pos", "gate", "kept", "fill"):
        assert torch.equal(getattr(few, name), getattr(many, name)[:g]), name
      if g == 3:
        assert abs(float(few.loss) - float(many.loss)) <= rel * abs(float(many.loss))


@pytest.mark.parametrize("router", ["top2", "switch"])
def test_gating_loss_of_one_launch(hip, router):
  """The loss of the launch that finishes groups in their last blocks, of 1, 16, 17 and
  18 blocks (16 are added at a time), against the oracle's."""
  for g, s, e in ((3, 50, 8), (2, 1024, 8), (2, 1025, 16), (3, 1100, 33)):
    rng = np.random.default_rng(s + e)
    logits = H.safe_logits(rng, g, s, e)
    importance = (rng.integers(0, 3, (g, s)) / 2).astype(np.float32)
    capacity = max(1, s // 4)
    got = _gating(hip, router, torch.from_numpy(logits).cuda(),
                  torch.from_numpy(importance).cuda(), capacity)
    if router == "switch":
      want = O.switch_gating(logits, capacity, importance=importance, train=True,
                             z_loss=0.01, num_microbatches=1)
    else:
      want = O.top_2_gating(logits, capacity, importance=importance,
                            policy="threshold", use_second_place_loss=True)
    np.testing.assert_allclose(H.routing_to_np(got)["loss"], want["loss"], rtol=2e-5)


@pytest.mark.parametrize("router", ["top2", "switch"])
def test_gating_of_2048_groups(hip, router):
  """2048 groups of one block are the most that one launch gates; 2049 take the launch
  per step.  Every group is the same, so the loss is one group's, but for a rounding per
  group."""
  gen = torch.Generator(device="cuda").manual_seed(5)
  logits = torch.randn((1, 40, 8), generator=gen, device="cuda").repeat(2049, 1, 1)
  got = {g: _gating(hip, router, logits[:g].contiguous(), None, 10)
         for g in (2, 2048, 2049)}
  for g in (2, 2048):
    for name in ("idx", "pos", "gate", "kept", "fill"):
      assert torch.equal(getattr(got[g], name), getattr(got[2049], name)[:g]), name
    want = float(got[2049].loss)
    assert abs(float(got[g].loss) - want) <= 2 * 2049 * 2.0 ** -24 * abs(want)


@pytest.mark.parametrize("s,e", [(64, 16), (256, 8), (1024, 32), (8192, 4)])
def test_gating_with_any_workspace(hip, monkeypatch, s, e):
  """The launches that finish a group in its last block count arrivals in a workspace
  that may hold anything: zeros, ones, what another call left.  One group and several,
  from logits and beside the projection: the same bits."""
  gen = torch.Generator(device="cuda").manual_seed(s + e)
  m, capacity = 64, max(1, s // 4)
  x = torch.randn((1, 3 * s, m), generator=gen, device="cuda").bfloat16()
  w = hip.pack_weights(torch.randn((1, m, e), generator=gen, device="cuda").bfloat16(),
                       torch.bfloat16)
  logits = torch.randn((3, s, e), generator=gen, device="cuda")
  plain, workspaces = torch.empty, []

  def empty(*size, **kw):
    t = plain(*size, **kw)
    if kw.get("dtype") == torch.uint8 and t.dim() == 1:
      if isinstance(held, int):
        t.fill_(held)
      else:
        n = min(t.numel(), held.numel())
        t[:n] = held[:n]
      workspaces.append(t)
    return t
  monkeypatch.setattr(torch, "empty", empty)

  def calls(g):
    yield hip.top2_gating(logits[:g].contiguous(), capacity, policy="threshold",
                          use_second_place_loss=True)
    yield hip.switch_gating(logits[:g].contiguous(), capacity, z_loss=0.01)
    if s % 128 == 0:
      yield hip.router_top2_gating(x[:, :g * s].contiguous(), w, s, capacity)
  for g in (1, 3):
    held = 0
    want = list(calls(g))
    left = workspaces[-1].clone()
    for held in (255, 1, 0x5a, left):
      for got, right in zip(calls(g), want):
        for name in ("idx", "pos", "gate", "kept", "fill", "loss"):
          assert torch.equal(getattr(got, name), getattr(right, name)), name


def test_recorded_gating_with_any_workspace(hip):
  """A recorded launch carries one call number into every replay, and its workspace is
  written over between two of them (all of the recorded step's memory that is not an
  output)."""
  gen = torch.Generator(device="cuda").manual_seed(3)
  g, s, e, c = 3, 1024, 8, 300
  logits = torch.randn((g, s, e), generator=gen, device="cuda")
  workspaces, plain = [], torch.empty

  def empty(*size, **kw):
    t = plain(*size, **kw)
    if kw.get("dtype") == torch.uint8 and t.dim() == 1:
      workspaces.append(t)
    return t
  want = hip.top2_gating(logits, c)               # (also loads what a launch needs)
  torch.cuda.synchronize()
  graph = torch.cuda.CUDAGraph()
  torch.empty = empty
  try:
    with torch.cuda.graph(graph):
      got = hip.top2_gating(logits, c)
  finally:
    torch.empty = plain
  assert len(workspaces) == 1
  for held in (0, 255, 1, None, 0x5a):
    if held is not None:
      workspaces[0].fill_(held)
    for t in (got.idx, got.pos, got.gate, got.kept, got.fill, got.loss):
      t.zero_()
    graph.replay()
    eager = hip.top2_gating(logits, c)
    for name in ("idx", "pos", "gate", "kept", "fill", "loss"):
      assert torch.equal(getattr(got, name), getattr(want, name)), (held, name)
      assert torch.equal(getattr(eager, name), getattr(want, name)), (held, name)


# a reduction of one K tile, of whole and of partly filled batches of tiles; tokens and
# experts around the 32 of a wavefront; the row that the K tiles' rotation restarts at
@pytest.mark.parametrize("tokens", [1, 31, 33, 200])
@pytest.mark.parametrize("m,e", [(64, 4), (256, 36), (320, 32), (512, 64),
                                 (576, 128), (1088, 100)])
def test_router_logits_few_tokens(hip, tokens, m, e):
  """Few tokens take a kernel of their own, with the bits that the same rows have in
  a call with many."""
  gen = torch.Generator(device="cuda").manual_seed(tokens + m + e)
  x = torch.randn((40000, m), generator=gen, device="cuda").bfloat16()
  w = torch.randn((m, e), generator=gen, device="cuda").bfloat16()
  bias = torch.randn((e,), generator=gen, device="cuda")
  packed = w.t().contiguous()
  few = hip.router_logits(x[:tokens].clone(), w, bias, w_packed=packed)
  assert torch.equal(few, hip.router_logits(x, w, bias, w_packed=packed)[:tokens])
  batched = hip.router_logits(torch.stack([x[:tokens], x[:tokens] + 1]),
                              torch.stack([w, w]), w_packed=torch.stack([packed] * 2))
  assert torch.equal(batched[0], hip.router_logits(x, w, w_packed=packed)[:tokens])


@pytest.mark.parametrize("act_dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("shape", [(2, 1024, 512, 8), (3, 100, 72, 5),
                                   (1, 640, 1024, 128), (1, 15, 4, 17),
                                   (1, 16401, 40, 5)])
def test_router_logits(hip, act_dtype, shape):
  g, s, m, e = shape
  rng = np.random.default_rng(17)
  x = O.cast_act(rng.standard_normal((g * s, m)).astype(np.float32), act_dtype)
  w = O.cast_act(rng.standard_normal((m, e)).astype(np.float32) / np.sqrt(m),
                 act_dtype)
  bias = rng.standard_normal(e).astype(np.float32)
  want = (x.astype(np.float64) @ w.astype(np.float64))
  got = H.to_np(hip.router_logits(H.to_gpu(x, act_dtype), H.to_gpu(w, act_dtype)))
  np.testing.assert_allclose(got, want, rtol=1e-5, atol=2e-5)
  got_b = H.to_np(hip.router_logits(H.to_gpu(x, act_dtype),
                                    H.to_gpu(w, act_dtype),
                                    bias=torch.from_numpy(bias).cuda()))
  np.testing.assert_allclose(got_b, want + bias, rtol=1e-5, atol=2e-5)
  # packed router weights: the matrix-core path for bf16 (when M % 64 == 0 and
  # E % 4 == 0), the same FMA kernel otherwise
  wg = H.to_gpu(w, act_dtype)
  wp = hip.pack_weights(wg.unsqueeze(0), wg.dtype)[0]
  got_p = H.to_np(hip.router_logits(H.to_gpu(x, act_dtype), wg, w_packed=wp,
                                    bias=torch.from_numpy(bias).cuda()))
  np.testing.assert_allclose(got_p, want + bias, rtol=1e-5, atol=2e-5)


def test_router_logits_mfma_shapes(hip):
  """Matrix-core router: ragged token counts, E = 4 .. 128, batched weights."""
  rng = np.random.default_rng(31)
  for b, t, m, e in [(1, 1, 64, 4), (1, 127, 128, 32), (3, 300, 192, 20),
                     (2, 129, 64, 128), (1, 2048, 1024, 64)]:
    x = O.round_bf16(rng.standard_normal((b, t, m)).astype(np.float32))
    w = O.round_bf16((rng.standard_normal((b, m, e)) / np.sqrt(m)).astype(np.float32))
    want = np.matmul(x.astype(np.float64), w.astype(np.float64))
    wg = H.to_gpu(w, "bfloat16")
    got = H.to_np(hip.router_logits(H.to_gpu(x, "bfloat16"), wg,
                                    w_packed=hip.pack_weights(wg, wg.dtype)))
    np.testing.assert_allclose(got, want, rtol=1e-5, atol=2e-5,
                               err_msg=str((b, t, m, e)))


def test_router_logits_batched(hip):
  b, t, m, e = 4, 150, 64, 16
  rng = np.random.default_rng(19)
  x = rng.standard_normal((b, t, m)).astype(np.float32)
  w = rng.standard_normal((b, m, e)).astype(np.float32)
  want = np.matmul(x.astype(np.float64), w.astype(np.float64))
  got = H.to_np(hip.router_logits(H.to_gpu(x), H.to_gpu(w)))
  np.testing.assert_allclose(got, want, rtol=1e-5, atol=2e-5)


@pytest.mark.parametrize("act_dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("shape", [(2, 256, 8, 40, 64), (3, 77, 5, 7, 36),
                                   (4, 128, 16, 8, 1024)])
def test_dispatch_combine(hip, act_dtype, shape):
  g, s, e, c, m = shape
  rng = np.random.default_rng(23)
  logits = H.safe_logits(rng, g, s, e)
  x = O.cast_act(rng.standard_normal((g, s, m)).astype(np.float32), act_dtype)
  want_r = O.top_2_gating(logits, c)
  r = hip.top2_gating(torch.from_numpy(logits).cuda(), c)
  H.assert_routing_equal(H.routing_to_np(r), want_r)
  ein, slot_gate = hip.dispatch(H.to_gpu(x, act_dtype), r, want_slot_gate=True)
  want_ein = O.dispatch_gather(x, want_r, e, c, act_dtype)
  np.testing.assert_array_equal(H.to_np(ein), want_ein)
  # slot weights: the dense combine tensor summed over the group-size dim
  dense = O.top_2_gating(logits, c, act_dtype=act_dtype, dense=True)
  want_sg = dense["combine"].sum(axis=1).transpose(1, 0, 2)       # [E,G,C]
  np.testing.assert_allclose(H.to_np(slot_gate), want_sg, rtol=1e-5, atol=1e-7)
  # the gather form equals the reference's dense einsum
  dense_ein = np.einsum("gsm,gsec->egcm", x, dense["dispatch"])
  np.testing.assert_array_equal(want_ein, dense_ein.astype(np.float32))
  # combine
  y = O.cast_act(rng.standard_normal((e, g, c, m)).astype(np.float32), act_dtype)
  got_out = H.to_np(hip.combine(H.to_gpu(y, act_dtype), r, s))
  gpu_r = H.routing_to_np(r)
  want_out = O.combine_gather(y, gpu_r, act_dtype)
  np.testing.assert_array_equal(got_out, want_out)
  dense_out = O.cast_act(np.einsum("egcn,gsec->gsn", y, dense["combine"]),
                         act_dtype)
  tol = dict(rtol=2e-2, atol=1e-2) if act_dtype == "bfloat16" else dict(
      rtol=1e-4, atol=1e-5)
  np.testing.assert_allclose(got_out, dense_out, **tol)


@pytest.mark.parametrize("act_dtype,activation", [
    ("float32", "relu"), ("bfloat16", "relu"), ("bfloat16", "gelu"),
    ("float32", "linear")])
@pytest.mark.parametrize("shape", [(3, 320, 64, 128, 64), (2, 100, 72, 200, 40),
                                   (2, 1100, 128, 1152, 1024),
                                   (1, 40, 30, 50, 20),
                                   # 256-row tiles with 1, 2, 3 and 5 K tiles,
                                   # ragged rows and a ragged last column tile
                                   (2, 512, 64, 256, 256), (1, 256, 128, 320, 256),
                                   (2, 700, 192, 256, 512),
                                   # last row tiles with 5, 4, 8 and 1 of their
                                   # eight 32-row pieces in use (the kernel
                                   # skips the others), rows not a multiple
                                   # of 32
                                   (2, 400, 128, 512, 256), (3, 640, 64, 256, 256),
                                   (1, 510, 128, 256, 256), (2, 770, 64, 256, 256)])
def test_expert_ffn(hip, act_dtype, activation, shape):
  e, rows, m, hdim, n = shape
  rng = np.random.default_rng(29)
  ein = O.cast_act(rng.standard_normal((e, rows, m)).astype(np.float32), act_dtype)
  wi = (rng.standard_normal((e, m, hdim)) / np.sqrt(m)).astype(np.float32)
  wo = (rng.standard_normal((e, hdim, n)) / np.sqrt(hdim)).astype(np.float32)
  dt = H.ACT_TORCH[act_dtype]
  wi_p = hip.pack_weights(torch.from_numpy(wi).cuda(), dt)
  wo_p = hip.pack_weights(torch.from_numpy(wo).cuda(), dt)
  np.testing.assert_array_equal(
      H.to_np(wi_p), O.cast_act(wi, act_dtype).transpose(0, 2, 1))
  got = H.to_np(hip.expert_ffn(H.to_gpu(ein, act_dtype), wi_p, wo_p, activation))
  want = O.expert_ffn(ein, O.cast_act(wi, act_dtype), O.cast_act(wo, act_dtype),
                      activation, act_dtype)
  tol = dict(rtol=2e-2, atol=1e-2) if act_dtype == "bfloat16" else dict(
      rtol=1e-4, atol=1e-5)
  np.testing.assert_allclose(got, want, **tol)


def test_expert_ffn_and_backward_random_shapes(hip):
  """expert_ffn and expert_ffn_backward over 300 random shapes (1-6 experts,
  8-1100 rows, widths that are and are not multiples of the tile sizes, both
  dtypes: every grouped-GEMM kernel and tile choice is hit) against float64
  products in torch.  y and the gradients are compared from the kernel's own
  hidden tensor, so a rounding flip in h does not count twice.  (5600 seeds of
  this sweep passed when it was written.)"""
  row_choices = [8, 40, 100, 128, 160, 256, 320, 384, 400, 510, 512, 640, 770,
                 1024, 1100]
  for seed in range(300):
    rng = np.random.default_rng(5000 + seed)
    gen = torch.Generator(device="cuda").manual_seed(5000 + seed)
    dt = [torch.float32, torch.bfloat16][int(rng.integers(2))]
    e = int(rng.integers(1, 7))
    rows = int(rng.choice(row_choices))
    m = int(rng.choice([16, 24, 30, 64, 72, 128, 192, 256, 320, 512]))
    hdim = int(rng.choice([20, 40, 64, 128, 200, 256, 320, 512, 1024, 1152]))
    n = int(rng.choice([16, 20, 40, 64, 128, 256, 320, 512]))
    case = (seed, str(dt), e, rows, m, hdim, n)
    ein = torch.randn((e, rows, m), generator=gen, device="cuda").to(dt)
    wi = torch.randn((e, m, hdim), generator=gen, device="cuda") / m ** 0.5
    wo = torch.randn((e, hdim, n), generator=gen, device="cuda") / hdim ** 0.5
    wi_d, wo_d = wi.to(dt), wo.to(dt)
    h = torch.empty((e, rows, hdim), dtype=dt, device="cuda")
    y = hip.expert_ffn(ein, hip.pack_weights(wi, dt), hip.pack_weights(wo, dt),
                       "relu", h=h)
    tol = (dict(rtol=2e-2, atol=1e-2) if dt == torch.bfloat16
           else dict(rtol=1e-4, atol=1e-5))

    def close(got, want, name):
      scale = max(1.0, float(want.abs().max()))
      torch.testing.assert_close(
          got.double(), want, rtol=tol["rtol"], atol=tol["atol"] * scale,
          msg=lambda text: "%s %s: %s" % (name, case, text))

    close(h, torch.relu(torch.matmul(ein.double(), wi_d.double())), "h")
    close(y, torch.matmul(h.double(), wo_d.double()), "y")
    dy = torch.randn((e, rows, n), generator=gen, device="cuda").to(dt)
    dxe, dwi, dwo = hip.expert_ffn_backward(ein, h, dy, wi_d, wo_d, "relu")
    dh = (torch.matmul(dy.double(), wo_d.double().transpose(1, 2))
          * (h > 0)).to(dt).double()
    close(dwo, torch.matmul(h.double().transpose(1, 2), dy.double()), "dwo")
    close(dwi, torch.matmul(ein.double().transpose(1, 2), dh), "dwi")
    close(dxe, torch.matmul(dh, wi_d.double().transpose(1, 2)), "dxe")


def test_rejects_bad_arguments(hip):
  logits = torch.zeros((1, 8, 4), device="cuda")
  with pytest.raises(ValueError):
    hip.top2_gating(logits, 2, policy="sometimes")
  with pytest.raises(hip.MoeHipError):
    hip.top2_gating(logits, 2, policy="random")          # no samples given
  with pytest.raises(hip.MoeHipError):
    hip.top2_gating(torch.zeros((1, 8, 1), device="cuda"), 2)   # E < 2
  with pytest.raises(hip.MoeHipError):
    hip.router_logits(torch.zeros((4, 8), device="cuda"),
                      torch.zeros((9, 2), device="cuda"))


def test_gating_hand_worked_case(hip):
  """One group, S = 6, E = 3, C = 2, worked by hand from
  transformer/moe.py:1472-1496 (no oracle involved): first choices in token
  order, then second choices behind the kept first ones; token 3 loses both
  choices; the loss from its definition (:1420-1442) in float64."""
  idx1 = [0, 0, 1, 0, 2, 1]
  idx2 = [1, 2, 0, 1, 0, 0]
  logits = np.zeros((1, 6, 3), np.float32)
  for t, (a, b) in enumerate(zip(idx1, idx2)):
    logits[0, t, a], logits[0, t, b] = 5.0, 3.0
  got = H.routing_to_np(hip.top2_gating(torch.from_numpy(logits).cuda(), 2))
  np.testing.assert_array_equal(got["index_1"][0], idx1)
  np.testing.assert_array_equal(got["index_2"][0], idx2)
  np.testing.assert_array_equal(got["pos_1"][0], [0, 1, 0, 2, 0, 1])
  np.testing.assert_array_equal(got["kept_1"][0], [1, 1, 1, 0, 1, 1])
  np.testing.assert_array_equal(got["pos_2"][0], [2, 1, 2, 3, 3, 4])
  np.testing.assert_array_equal(got["kept_2"][0], [0, 1, 0, 0, 0, 0])
  np.testing.assert_array_equal(got["fill"][0], [2, 2, 2])
  e = np.exp(np.array([5.0, 3.0, 0.0]))
  g1, g2 = e[0] / (e[0] + e[1]), e[1] / (e[0] + e[1])   # normalised top-2 gates
  np.testing.assert_allclose(got["gate_1"][0], [g1, g1, g1, 0, g1, g1], rtol=1e-5)
  np.testing.assert_allclose(got["gate_2"][0], [0, g2, 0, 0, 0, 0], rtol=1e-5)
  prob = np.exp(logits[0].astype(np.float64))
  prob /= prob.sum(-1, keepdims=True)
  density = np.array([3, 2, 1]) / 6.0               # first choices, before drops
  want_loss = (prob.mean(0) * density).mean() * 9
  np.testing.assert_allclose(got["loss"], want_loss, rtol=2e-5)


def test_gating_golden_fixture(hip):
  """The committed golden vectors (tests/golden/top2_gating_small.json)."""
  import json
  import os
  path = os.path.join(os.path.dirname(__file__), "golden",
                      "top2_gating_small.json")
  with open(path) as f:
    gold = json.load(f)
  logits = np.array(gold["logits"], np.float32)
  got = H.routing_to_np(hip.top2_gating(torch.from_numpy(logits).cuda(),
                                        gold["capacity"]))
  for k in ("index_1", "index_2", "pos_1", "pos_2"):
    np.testing.assert_array_equal(got[k], np.array(gold[k]), err_msg=k)
  for k in ("kept_1", "kept_2"):
    np.testing.assert_array_equal(got[k], np.array(gold[k], bool), err_msg=k)
  np.testing.assert_allclose(got["gate_1"], np.array(gold["gate_1"]), rtol=1e-5)
  np.testing.assert_allclose(got["gate_2"], np.array(gold["gate_2"]), rtol=1e-5,
                             atol=1e-7)
  np.testing.assert_allclose(got["loss"], gold["loss"], rtol=2e-5)


# Full benchmark sizes: (G, S, E, C, M) of configurations 3 and 4.  The oracle
# is too slow here, so the checks are size-independent properties.
FULL_SIZES = [(16, 2048, 64, 32, 1024, True), (32, 2048, 64, 64, 4096, False)]


@pytest.mark.parametrize("size", FULL_SIZES, ids=["cfg3", "cfg4"])
def test_full_size_routing_properties(hip, size):
  g, s, e, c, m, skew = size
  gen = torch.Generator(device="cuda")
  gen.manual_seed(5)
  logits = torch.randn((g, s, e), generator=gen, device="cuda")
  if skew:
    ranks = torch.randperm(e, generator=gen, device="cuda").double() + 1
    logits = logits + (3.0 * ranks ** -1.2).float()
  r = hip.top2_gating(logits, c)
  want_used = H.assert_routing_properties(r, logits)
  kept = r.kept.bool()
  if skew:
    assert float(kept.float().mean()) < 0.8       # the drop path is exercised

  # dispatch -> combine with identity experts: out = (w1 + w2) * x
  x = torch.randn((g, s, m), generator=gen, device="cuda").to(torch.bfloat16)
  ein, slot_gate = hip.dispatch(x, r, want_slot_gate=True)
  w = r.gate.to(torch.bfloat16).float() * kept.float()
  # checksum: every kept choice copies its row exactly once
  n_copies = (kept & (w != 0)).sum(-1).double()
  want_sum = (x.double().sum(-1) * n_copies).sum()
  got_sum = ein.double().sum()
  assert abs(float(got_sum - want_sum)) <= 1e-6 * float(x.double().abs().sum())
  assert torch.equal(ein.view(e, g, c, m)[~want_used.permute(1, 0, 2)],
                     torch.zeros((), dtype=torch.bfloat16, device="cuda").expand(
                         int((~want_used).sum()), m))
  assert abs(float(slot_gate.double().sum() - w.double().sum())) < 1e-3
  out = hip.combine(ein, r, s)
  want = (w[..., 0:1] * x.float() + w[..., 1:2] * x.float()).to(torch.bfloat16)
  assert torch.equal(out, want)


@pytest.mark.parametrize("case", [
    # routers, groups per router, S, M, E, C
    (1, 2, 256, 128, 8, 70), (1, 3, 128, 64, 64, 5), (2, 2, 384, 192, 20, 40),
    (4, 1, 128, 64, 128, 3), (1, 16, 1024, 1024, 32, 40),
    (1, 32, 2048, 4096, 64, 64)],
    ids=["e8", "e64", "two_routers", "e128", "cfg2", "cfg4"])
def test_router_top2_gating_fused(hip, case):
  """The fused router + gating entry point against the oracle (and against the
  two-call path): bf16 tokens whose router logits do not nearly tie.  The last
  two cases are the full routing shapes of benchmark configurations 2 and 4;
  the logits the oracle is fed are the float64 product rounded to float32."""
  b, gpr, s, m, e, c = case
  rng = np.random.default_rng(41)
  w = O.round_bf16((rng.standard_normal((b, m, e)) / np.sqrt(m)).astype(np.float32))
  x = np.stack([H.safe_tokens(rng, gpr * s, m, w[i], "bfloat16") for i in range(b)])
  imp = rng.choice(np.array([0.0, 0.5, 1.0], np.float32), size=(b * gpr, s),
                   p=[0.1, 0.2, 0.7])
  logits = np.concatenate([
      np.matmul(x[:, r0:r0 + 8192].astype(np.float64), w.astype(np.float64))
      for r0 in range(0, gpr * s, 8192)], axis=1)
  logits = logits.astype(np.float32).reshape(b * gpr, s, e)
  xg, wg = H.to_gpu(x, "bfloat16"), H.to_gpu(w, "bfloat16")
  wp = hip.pack_weights(wg, wg.dtype)
  assert hip.fused_gating_supported(xg, e, s)
  for importance in (None, imp):
    want = O.top_2_gating(logits, c, importance=importance,
                          use_second_place_loss=True, num_microbatches=2)
    r, got_logits = hip.router_top2_gating(
        xg, wp, s, c, importance=None if importance is None else H.to_gpu(importance),
        use_second_place_loss=True, num_microbatches=2, want_logits=True)
    np.testing.assert_allclose(H.to_np(got_logits), logits, rtol=1e-5, atol=2e-5)
    got = H.routing_to_np(r)
    H.assert_routing_equal(got, want, gate_rtol=2e-5)
    np.testing.assert_allclose(got["loss"], want["loss"], rtol=5e-5)
    # same record as the two separate calls fed the fused kernel's logits
    r2 = hip.top2_gating(got_logits, c,
                         importance=None if importance is None else H.to_gpu(importance),
                         use_second_place_loss=True, num_microbatches=2)
    for a_, b_ in ((r.idx, r2.idx), (r.pos, r2.pos), (r.kept, r2.kept),
                   (r.fill, r2.fill), (r.gate, r2.gate)):
      assert torch.equal(a_, b_)


def test_router_gating_largest_group_one_popular_expert(hip):
  """The largest group the gating entries take (S = 16384, 128 blocks of the
  one-launch kernel) with 4 experts and a router bias that sends most first
  choices to expert 0: the per-block slot prefixes of the group tail grow to
  thousands (they are kept in 16 bits, which the group-size limit makes
  safe).  One-launch entry against the logits-in entry, bit for bit, and both
  against the oracle; both capacities, nothing dropped and almost all dropped.
  A larger group is refused by name."""
  g, s, m, e = 2, 16384, 64, 4
  rng = np.random.default_rng(77)
  w = O.round_bf16((rng.standard_normal((1, m, e)) / np.sqrt(m)).astype(np.float32))
  x = H.safe_tokens(rng, g * s, m, w[0], "bfloat16",
                    bias=np.array([2.5, 0.0, 0.0, 0.0], np.float32))[None]
  bias = np.array([2.5, 0.0, 0.0, 0.0], np.float32)
  xg, wg = H.to_gpu(x, "bfloat16"), H.to_gpu(w, "bfloat16")
  wp = hip.pack_weights(wg, wg.dtype)
  assert hip.fused_gating_supported(xg, e, s)
  bg = torch.from_numpy(bias).cuda()
  for c in (s, 300):
    r, got_logits = hip.router_top2_gating(xg, wp, s, c, bias=bg,
                                           want_logits=True)
    r2 = hip.top2_gating(got_logits, c)
    for name in ("idx", "pos", "kept", "fill", "gate"):
      assert torch.equal(getattr(r, name), getattr(r2, name)), name
    # (the two entries sum the loss's column sums over blocks of different
    # sizes at this expert count)
    torch.testing.assert_close(r.loss, r2.loss, rtol=2e-6, atol=0)
    want = O.top_2_gating(H.to_np(got_logits), c)
    got = H.routing_to_np(r)
    H.assert_routing_equal(got, want, gate_rtol=2e-5)
    # raw positions (kept or not): expert 0's last first-choice position
    np.testing.assert_array_equal(got["pos_1"], want["pos_1"])
    first0 = (got["index_1"] == 0).sum(axis=1)
    assert (first0 > 9000).all()                  # prefixes in the thousands
    assert got["pos_1"].max() == first0.max() - 1
  too_big = torch.zeros((1, 2 * (s + 128), m), dtype=torch.bfloat16, device="cuda")
  with pytest.raises(Exception, match="group size S=16512 > 16384"):
    hip.router_top2_gating(too_big, wp, s + 128, 8)
  with pytest.raises(Exception, match="group size S=16512 > 16384"):
    hip.top2_gating(torch.zeros((2, s + 128, e), device="cuda"), 8)


@pytest.mark.parametrize("policy", ["all", "none", "threshold", "random"])
@pytest.mark.parametrize("second_place_loss", [False, True])
def test_router_top2_gating_fused_policies(hip, policy, second_place_loss):
  """Every second-place policy, with a router bias and importance, through the
  one-launch entry point: the same record, to the bit, as the logits-in entry
  point fed the logits the fused kernel reports (the two select the experts
  in different code: accumulator registers against one thread per token)."""
  b, gpr, s, m, e, c = 2, 3, 256, 128, 16, 30
  gen = torch.Generator(device="cuda").manual_seed(7)
  x = torch.randn((b, gpr * s, m), generator=gen, device="cuda").to(torch.bfloat16)
  w = (torch.randn((b, m, e), generator=gen, device="cuda") / m ** 0.5).to(
      torch.bfloat16)
  wp = hip.pack_weights(w, w.dtype)
  bias = torch.randn((e,), generator=gen, device="cuda") * 0.1
  u = torch.rand((b * gpr, s), generator=gen, device="cuda")
  imp = torch.tensor([0.0, 0.5, 1.0], device="cuda")[
      torch.randint(0, 3, (b * gpr, s), generator=gen, device="cuda")]
  kw = dict(policy=policy, threshold=0.25, second_uniform=u, importance=imp,
            use_second_place_loss=second_place_loss, num_microbatches=3)
  r, logits = hip.router_top2_gating(x, wp, s, c, bias=bias, want_logits=True,
                                     **kw)
  r2 = hip.top2_gating(logits, c, **kw)
  for name in ("idx", "pos", "kept", "fill", "gate", "loss"):
    assert torch.equal(getattr(r, name), getattr(r2, name)), name
  if policy == "all":
    H.assert_routing_properties(r, logits, importance=imp)
  # and without reporting the logits (they then never leave the chip)
  r3 = hip.router_top2_gating(x, wp, s, c, bias=bias, **kw)
  for name in ("idx", "pos", "kept", "fill", "gate", "loss"):
    assert torch.equal(getattr(r, name), getattr(r3, name)), name


def test_stage_timer_keeps_calls_for_back_to_back_timing(hip):
  """StageTimer(keep_calls=True) keeps the router and combine library calls;
  launching them again back to back gives a positive time and rewrites the
  outputs with the same bits."""
  b, gpr, s, m, e, c = 1, 2, 256, 128, 8, 70
  gen = torch.Generator(device="cuda").manual_seed(3)
  x = torch.randn((b, gpr * s, m), generator=gen, device="cuda").to(torch.bfloat16)
  w = (torch.randn((b, m, e), generator=gen, device="cuda") / m ** 0.5).to(
      torch.bfloat16)
  wp = hip.pack_weights(w, w.dtype)
  y = torch.randn((e, gpr, c, m), generator=gen, device="cuda").to(torch.bfloat16)
  with hip.StageTimer(keep_calls=True) as timer:
    r = hip.router_top2_gating(x, wp, s, c)
    out = hip.combine(y, r, s)
  assert set(timer.calls) == {"router_top2_gating", "combine"}
  before = {k: getattr(r, k).clone() for k in ("idx", "pos", "kept", "fill", "gate", "loss")}
  out_before = out.clone()
  for name, call in timer.calls.items():
    assert hip.back_to_back_ms(call, reps=5, warmup=1) > 0.0, name
  for k, v in before.items():
    assert torch.equal(getattr(r, k), v), k
  assert torch.equal(out, out_before)
  # without keep_calls nothing is kept
  with hip.StageTimer() as timer:
    hip.router_top2_gating(x, wp, s, c)
  assert timer.calls == {}


def test_router_gating_fused_random_shapes(hip):
  """Differential sweep of the one-launch entries over random shapes (groups,
  group sizes that are multiples of 128, expert counts that are multiples of 4,
  capacities from starved to ample, one or several routers, both routers'
  modes): the routing record must equal, to the bit, what the logits-in
  entries make of the logits the fused kernel reports.  Shapes with many groups also
  exercise blocks of different groups finishing in any order."""
  rng = np.random.default_rng(1234)
  gen = torch.Generator(device="cuda").manual_seed(99)
  for trial in range(36):
    b = int(rng.choice([1, 1, 2, 3]))
    gpr = int(rng.integers(1, 9))
    s = 128 * int(rng.integers(1, 9))
    m = 64 * int(rng.integers(1, 5))
    e = 4 * int(rng.integers(1, 33))
    c = int(rng.choice([1, 2, max(1, s // e), max(1, 2 * s // e), s]))
    c = min(c, s)
    x = torch.randn((b, gpr * s, m), generator=gen, device="cuda").to(torch.bfloat16)
    w = (torch.randn((b, m, e), generator=gen, device="cuda") * (2.0 / m ** 0.5)
         ).to(torch.bfloat16)
    wp = hip.pack_weights(w, w.dtype)
    if not hip.fused_gating_supported(x, e, s):
      continue
    imp = None
    if trial % 3 == 1:
      imp = torch.tensor([0.0, 0.5, 1.0], device="cuda")[
          torch.randint(0, 3, (b * gpr, s), generator=gen, device="cuda")]
    tag = "trial %d: b=%d gpr=%d s=%d m=%d e=%d c=%d" % (trial, b, gpr, s, m, e, c)
    if trial % 2 == 0:
      kw = dict(importance=imp, use_second_place_loss=trial % 4 == 0,
                num_microbatches=2)
      r, logits = hip.router_top2_gating(x, wp, s, c, want_logits=True, **kw)
      r2 = hip.top2_gating(logits, c, **kw)
    else:
      kw = dict(importance=imp, num_microbatches=3)
      r, logits = hip.router_switch_gating(x, wp, s, c, want_logits=True, **kw)
      r2 = hip.switch_gating(logits, c, **kw)
    for name in ("idx", "pos", "kept", "fill", "gate"):
      assert torch.equal(getattr(r, name), getattr(r2, name)), (tag, name)
    # (the loss's float32 partial sums are grouped differently in the two
    # paths: 4 row ranges per block against one sum per block)
    torch.testing.assert_close(r.loss, r2.loss, rtol=1e-5, atol=1e-7, msg=tag)


def test_router_top2_gating_rejects_unsupported(hip):
  x = torch.zeros((1, 96, 64), dtype=torch.bfloat16, device="cuda")
  wp = torch.zeros((1, 8, 64), dtype=torch.bfloat16, device="cuda")
  assert not hip.fused_gating_supported(x, 8, 96)
  with pytest.raises(hip.MoeHipError, match="fused kernel needs"):
    hip.router_top2_gating(x, wp, 96, 4)


# ---- switch (top-1) gating ------------------------------------------------------
@pytest.mark.parametrize("shape", [(2, 1024, 8, 160), (16, 2048, 64, 32),
                                   (3, 77, 5, 7), (1, 1, 2, 1),
                                   (2, 130, 200, 4), (1, 4096, 64, 70),
                                   (32, 2048, 64, 64)])
def test_switch_gating_random_logits(hip, shape):
  g, s, e, c = shape
  rng = np.random.default_rng(1000 + hash(shape) % 1000)
  logits = H.safe_logits(rng, g, s, e, scale=1.5)
  want = O.switch_gating(logits, c)
  got = H.routing_to_np(hip.switch_gating(torch.from_numpy(logits).cuda(), c))
  H.assert_routing_equal(got, want)
  np.testing.assert_allclose(got["loss"], want["loss"], rtol=2e-5)


def test_switch_gating_choice_logits(hip):
  """Policy "sample": experts from the arg-max of separate choice logits, gates
  from the probabilities, for both slot orders."""
  g, s, e, c = 3, 400, 16, 30
  rng = np.random.default_rng(14)
  logits = H.safe_logits(rng, g, s, e)
  u = rng.random((g, s, e)).astype(np.float32)
  choice = O.sample_choice_logits(logits, 1.0, u)
  imp = rng.choice(np.array([0.0, 1.0], np.float32), size=(g, s), p=[0.2, 0.8])
  lg, ch = torch.from_numpy(logits).cuda(), torch.from_numpy(choice).cuda()
  want = O.switch_gating(logits, c, importance=imp, choice_logits=choice)
  assert (want["index_1"] != logits.argmax(-1)).mean() > 0.2
  got = H.routing_to_np(hip.switch_gating(lg, c, importance=H.to_gpu(imp),
                                          choice_logits=ch))
  H.assert_routing_equal(got, want)
  np.testing.assert_allclose(got["loss"], want["loss"], rtol=2e-5)
  with pytest.raises(hip.MoeHipError, match="choice_logits"):
    hip.switch_gating(lg, c, choice_logits=ch[:, :, :8].contiguous())


def test_switch_gating_exact_ties(hip):
  g, s, e, c = 3, 500, 64, 9
  rng = np.random.default_rng(8)
  logits = H.random_logits(rng, g, s, e, scale=0.6, quantum=0.25)
  want = O.switch_gating(logits, c)
  got = H.routing_to_np(hip.switch_gating(torch.from_numpy(logits).cuda(), c))
  H.assert_routing_equal(got, want)


@pytest.mark.parametrize("imp_dtype", ["float32", "bfloat16"])
def test_switch_gating_importance_and_z_loss(hip, imp_dtype):
  g, s, e, c = 4, 320, 16, 24
  rng = np.random.default_rng(12)
  logits = H.safe_logits(rng, g, s, e)
  imp = rng.choice(np.array([0.0, 0.5, 1.0], np.float32), size=(g, s),
                   p=[0.2, 0.2, 0.6])
  lg = torch.from_numpy(logits).cuda()
  for z, mb in ((None, None), (1e-3, 1), (0.5, 4)):
    want = O.switch_gating(logits, c, importance=imp, train=True, z_loss=z,
                           num_microbatches=mb)
    got = H.routing_to_np(hip.switch_gating(
        lg, c, importance=H.to_gpu(imp, imp_dtype), z_loss=z,
        num_microbatches=mb))
    H.assert_routing_equal(got, want)
    np.testing.assert_allclose(got["loss"], want["loss"], rtol=2e-5)
  # only importance == 1 rows are routed
  assert not got["kept_1"][imp != 1.0].any()
  assert (got["gate_1"][imp != 1.0] == 0).all()
  # z-loss closed form through the kernel: constant logits c0 give
  # (c0 + log E)^2 / microbatches whatever the mask
  const = torch.full((g, s, e), 1.5, dtype=torch.float32, device="cuda")
  a = hip.switch_gating(const, c, importance=H.to_gpu(imp), z_loss=0.1,
                        num_microbatches=2).loss.item()
  b = hip.switch_gating(const, c, importance=H.to_gpu(imp),
                        num_microbatches=2).loss.item()
  np.testing.assert_allclose(a - b, 0.1 * (1.5 + np.log(e)) ** 2 / 2, rtol=1e-4)


@pytest.mark.parametrize("case", [
    (1, 2, 256, 128, 8, 70), (2, 2, 384, 192, 20, 40), (1, 16, 1024, 1024, 32, 40)])
def test_router_switch_gating_fused(hip, case):
  b, gpr, s, m, e, c = case
  rng = np.random.default_rng(43)
  w = O.round_bf16((rng.standard_normal((b, m, e)) / np.sqrt(m)).astype(np.float32))
  x = np.stack([H.safe_tokens(rng, gpr * s, m, w[i], "bfloat16") for i in range(b)])
  imp = rng.choice(np.array([0.0, 1.0], np.float32), size=(b * gpr, s),
                   p=[0.2, 0.8])
  logits = np.matmul(x, w).astype(np.float32).reshape(b * gpr, s, e)
  xg, wg = H.to_gpu(x, "bfloat16"), H.to_gpu(w, "bfloat16")
  wp = hip.pack_weights(wg, wg.dtype)
  for importance, z in ((None, None), (imp, 1e-2)):
    want = O.switch_gating(logits, c, importance=importance, train=True,
                           z_loss=z, num_microbatches=2)
    gi = None if importance is None else H.to_gpu(importance)
    r, got_logits = hip.router_switch_gating(
        xg, wp, s, c, importance=gi, z_loss=z, num_microbatches=2,
        want_logits=True)
    np.testing.assert_allclose(H.to_np(got_logits), logits, rtol=1e-5, atol=2e-5)
    got = H.routing_to_np(r)
    H.assert_routing_equal(got, want, gate_rtol=2e-5)
    np.testing.assert_allclose(got["loss"], want["loss"], rtol=5e-5)
    r2 = hip.switch_gating(got_logits, c, importance=gi, z_loss=z,
                           num_microbatches=2)
    for a_, b_ in ((r.idx, r2.idx), (r.pos, r2.pos), (r.kept, r2.kept),
                   (r.fill, r2.fill), (r.gate, r2.gate)):
      assert torch.equal(a_, b_)


def test_switch_dispatch_combine_roundtrip(hip):
  """Switch routing record through the unchanged dispatch / combine kernels."""
  g, s, e, c, m = 2, 256, 8, 40, 64
  rng = np.random.default_rng(44)
  logits = H.safe_logits(rng, g, s, e)
  x = rng.standard_normal((g, s, m)).astype(np.float32)
  want_r = O.switch_gating(logits, c)
  r = hip.switch_gating(torch.from_numpy(logits).cuda(), c)
  xg = H.to_gpu(x)
  expert_in = hip.dispatch(xg, r)
  np.testing.assert_array_equal(H.to_np(expert_in),
                                O.dispatch_gather(x, want_r, e, c, "float32"))
  out = hip.combine(expert_in, r, s)
  np.testing.assert_allclose(
      H.to_np(out), O.combine_gather(H.to_np(expert_in), want_r, "float32"),
      rtol=1e-6, atol=1e-7)


def test_switch_gating_golden_fixture(hip):
  """The committed golden vectors (tests/golden/switch_gating_small.json)."""
  import json
  import os
  path = os.path.join(os.path.dirname(__file__), "golden",
                      "switch_gating_small.json")
  with open(path) as f:
    gold = json.load(f)
  logits = np.array(gold["logits"], np.float32)
  imp = np.array(gold["importance"], np.float32)
  got = H.routing_to_np(hip.switch_gating(
      torch.from_numpy(logits).cuda(), gold["capacity"],
      importance=H.to_gpu(imp), z_loss=gold["z_loss"],
      num_microbatches=gold["num_microbatches"]))
  for k in ("index_1", "pos_1"):
    np.testing.assert_array_equal(got[k], np.array(gold[k]), err_msg=k)
  np.testing.assert_array_equal(got["kept_1"], np.array(gold["kept_1"], bool))
  np.testing.assert_allclose(got["gate_1"], np.array(gold["gate_1"]), rtol=1e-5,
                             atol=1e-7)
  np.testing.assert_allclose(got["loss"], gold["loss"], rtol=2e-5)


# ---- switch_max gating ----------------------------------------------------------
def _assert_switch_max_equal(got, want):
  for k in ("index_1", "kept_1", "kept_2", "fill"):
    np.testing.assert_array_equal(got[k], want[k], err_msg=k)
  kept = want["kept_1"]
  np.testing.assert_array_equal(got["pos_1"][kept], want["pos_1"][kept])
  np.testing.assert_allclose(got["gate_1"], want["gate_1"], rtol=1e-5, atol=1e-7)
  assert not got["gate_2"].any()


# ---- ntlb ("no token left behind") gating ---------------------------------------
@pytest.mark.parametrize("shape", [(2, 1024, 8, 100, 2), (8, 2048, 64, 30, 4),
                                   (3, 77, 5, 12, 3), (1, 1, 2, 1, 1),
                                   (2, 131, 200, 1, 4), (1, 4096, 64, 60, 8),
                                   (2, 512, 16, 512, 4), (4, 300, 6, 40, 6),
                                   (32, 2048, 64, 64, 4)])
def test_ntlb_gating_random_logits(hip, shape):
  """Skewed router (a Zipf bias) so that the popular experts overflow in pass
  0 and the later passes route what is left."""
  g, s, e, c, k = shape
  rng = np.random.default_rng(3000 + sum(shape))
  logits = H.safe_logits(rng, g, s, e, scale=1.5,
                         bias=H.zipf_bias(rng, e, scale=2.0), top=k + 1)
  imp = rng.choice(np.array([0.0, 0.5, 1.0], np.float32), size=(g, s),
                   p=[0.1, 0.1, 0.8])
  lg = torch.from_numpy(logits).cuda()
  for importance, mb in ((None, None), (imp, 2)):
    want = O.ntlb_gating(logits, c, k, importance=importance,
                         num_microbatches=mb)
    got = H.routing_to_np(hip.ntlb_gating(
        lg, c, k, importance=None if importance is None else H.to_gpu(importance),
        num_microbatches=mb))
    H.assert_routing_equal(got, want)
    np.testing.assert_allclose(got["loss"], want["loss"], rtol=2e-5)
  if s > 64 and k > 1 and c * e < s:
    assert (want["taken_in_pass"] > 0).any()       # the later passes did something
  assert not got["kept_1"][imp != 1.0].any()


@pytest.mark.parametrize("shape", [(2, 1024, 8, 100, 2), (8, 2048, 64, 30, 4),
                                   (3, 77, 5, 12, 3), (1, 1, 2, 1, 1),
                                   (2, 131, 200, 1, 4), (2, 512, 16, 512, 4),
                                   (32, 2048, 64, 64, 4)])
def test_ntlb_gating_bfloat16_softmax(hip, shape):
  """bfloat16 activations: the reference rounds the projection's result and
  every op of the softmax to bfloat16 before the cast to float32
  (moe.py:825-836).  Record and loss against the oracle's bfloat16 chain; the
  float32 logits fed here are NOT bfloat16 values (the kernel rounds them).
  Equal probabilities are common in bfloat16 and go to the lower index."""
  g, s, e, c, k = shape
  rng = np.random.default_rng(3100 + sum(shape))
  logits = H.bf16_softmax_safe_logits(rng, g, s, e, scale=1.5,
                                      bias=H.zipf_bias(rng, e, scale=2.0))
  imp = rng.choice(np.array([0.0, 0.5, 1.0], np.float32), size=(g, s),
                   p=[0.1, 0.1, 0.8])
  lg = torch.from_numpy(logits).cuda()
  ties = 0
  for importance, mb in ((None, None), (imp, 2)):
    want = O.ntlb_gating(logits, c, k, importance=importance,
                         num_microbatches=mb, act_dtype="bfloat16")
    got = H.routing_to_np(hip.ntlb_gating(
        lg, c, k, importance=None if importance is None else H.to_gpu(importance),
        num_microbatches=mb, softmax_dtype=torch.bfloat16))
    H.assert_routing_equal(got, want)
    # the gates are bfloat16 values, bit for bit
    np.testing.assert_array_equal(got["gate_1"], want["gate_1"])
    assert not (got["gate_1"].view(np.uint32) & 0xFFFF).any()
    np.testing.assert_allclose(got["loss"], float(want["loss"]), rtol=1e-2)
    p = O.softmax_bf16(logits)
    top = -np.sort(-p, axis=-1)[..., :min(k + 1, e)]
    ties += int((top[..., :-1] == top[..., 1:]).sum())
  if s * g > 1000:
    assert ties > 0                     # the tie rule was exercised
    # and the float32 chain would have routed differently somewhere
    f32 = O.ntlb_gating(logits, c, k)
    assert (f32["topk_index"] != want["topk_index"]).any()


def test_ntlb_gating_bfloat16_hand_case(hip):
  """[0, 0, 0, -1] four times, capacity 1, k = 3 (worked by hand in the
  oracle's tests): tokens 0, 1, 2 land on experts 0, 1, 2 in passes 0, 1, 2
  with the bfloat16 probability 0.294921875; token 3 is left out."""
  logits = np.tile(np.array([0, 0, 0, -1], np.float32), (1, 4, 1))
  got = H.routing_to_np(hip.ntlb_gating(torch.from_numpy(logits).cuda(), 1, 3,
                                        softmax_dtype=torch.bfloat16))
  np.testing.assert_array_equal(got["kept_1"][0], [True, True, True, False])
  np.testing.assert_array_equal(got["index_1"][0][:3], [0, 1, 2])
  np.testing.assert_array_equal(got["gate_1"][0], [0.294921875] * 3 + [0.0])
  # a float32 difference that bfloat16 does not see: tie, lower index first
  two = np.array([[[1.0, 1.001, -3.0]]], np.float32)
  r32 = H.routing_to_np(hip.ntlb_gating(torch.from_numpy(two).cuda(), 4, 2))
  r16 = H.routing_to_np(hip.ntlb_gating(torch.from_numpy(two).cuda(), 4, 2,
                                        softmax_dtype=torch.bfloat16))
  assert (r32["index_1"][0, 0], r16["index_1"][0, 0]) == (1, 0)


def test_ntlb_gating_exact_ties(hip):
  """Logits on a coarse grid: equal probabilities within a row go to the lower
  expert index first (repeated first-arg-max, ops.py:5009-5014)."""
  g, s, e, c, k = 3, 500, 16, 20, 4
  rng = np.random.default_rng(31)
  logits = H.random_logits(rng, g, s, e, scale=0.6, quantum=0.25)
  want = O.ntlb_gating(logits, c, k)
  got = H.routing_to_np(hip.ntlb_gating(torch.from_numpy(logits).cuda(), c, k))
  H.assert_routing_equal(got, want)
  np.testing.assert_allclose(got["loss"], want["loss"], rtol=2e-5)


def test_ntlb_dispatch_combine_roundtrip(hip):
  """The record drives the unchanged dispatch / combine kernels: with identity
  experts the output is gate * x for routed tokens and 0 for the others."""
  g, s, e, c, m, k = 2, 256, 8, 24, 64, 3
  rng = np.random.default_rng(32)
  logits = H.safe_logits(rng, g, s, e, scale=1.5,
                         bias=H.zipf_bias(rng, e, scale=2.0), top=k + 1)
  x = rng.standard_normal((g, s, m)).astype(np.float32)
  r = hip.ntlb_gating(torch.from_numpy(logits).cuda(), c, k)
  xe = hip.dispatch(H.to_gpu(x), r)
  out = H.to_np(hip.combine(xe, r, s))
  rec = H.routing_to_np(r)
  want = x * (rec["gate_1"] * rec["kept_1"])[..., None]
  np.testing.assert_allclose(out, want, rtol=1e-6, atol=1e-7)
  ref = O.ntlb_gating(logits, c, k)
  np.testing.assert_array_equal(
      H.to_np(xe), O.dispatch_gather(x, ref, e, c, "float32"))


# ---- training-time summaries of the f1 routers --------------------------------
@pytest.mark.parametrize("shape", [(2, 256, 8, 40), (32, 2048, 64, 64),
                                   (3, 77, 5, 12), (1, 1, 2, 1),
                                   (2, 131, 200, 3)])
@pytest.mark.parametrize("gating", ["switch", "switch_max", "ntlb", "ntlb_bf16"])
def test_router_summaries(hip, gating, shape):
  """entropy, expert_gate, per-expert shares, fraction_routed and z-loss as the
  reference hands them to mtf.scalar_summary, against the oracle.  The shares
  are ratios of integer counts; the float32 sums over tokens agree to
  rounding (rtol 2e-5, stated here)."""
  g, s, e, c = shape
  k = min(3, e)
  rng = np.random.default_rng(4100 + sum(shape))
  bf16 = gating == "ntlb_bf16"
  name = "ntlb" if bf16 else gating
  if bf16:
    logits = H.bf16_softmax_safe_logits(rng, g, s, e, scale=1.5,
                                        bias=H.zipf_bias(rng, e, scale=2.0))
  else:
    logits = H.safe_logits(rng, g, s, e, scale=1.5,
                           bias=H.zipf_bias(rng, e, scale=2.0), top=k + 1)
  imp = rng.choice(np.array([0.0, 0.5, 1.0], np.float32), size=(g, s),
                   p=[0.1, 0.1, 0.8])
  imp[0, 0] = 1.0
  act = "bfloat16" if bf16 else "float32"
  lg = torch.from_numpy(logits).cuda()
  for importance, mb in ((None, None), (imp, 2)):
    ip = None if importance is None else H.to_gpu(importance)
    if name == "switch":
      want_r = O.switch_gating(logits, c, importance=importance)
      r = hip.switch_gating(lg, c, importance=ip)
    elif name == "switch_max":
      want_r = O.switch_max_gating(logits, c, importance=importance)
      r = hip.switch_gating(lg, c, importance=ip, slots_by_gate=True)
    else:
      want_r = O.ntlb_gating(logits, c, k, importance=importance, act_dtype=act)
      r = hip.ntlb_gating(lg, c, k, importance=ip,
                          softmax_dtype=torch.bfloat16 if bf16 else torch.float32)
    want = O.router_summaries(logits, name, want_r, importance=importance,
                              top_k=k, num_microbatches=mb, act_dtype=act)
    got = H.to_np(hip.router_summaries(
        lg, name, c, importance=ip, kept=r.kept, top_k=k, num_microbatches=mb,
        softmax_dtype=torch.bfloat16 if bf16 else torch.float32))
    assert got.shape == (4 + e,)
    np.testing.assert_allclose(got[0], want["entropy"], rtol=2e-5)
    np.testing.assert_allclose(got[1], want["expert_gate"], rtol=2e-5)
    np.testing.assert_allclose(got[4:], want["experts"], rtol=1e-6)
    np.testing.assert_allclose(got[4:].sum(), 1.0, rtol=1e-5)
    if name != "ntlb":
      np.testing.assert_allclose(got[2], want["fraction_routed"], rtol=1e-6)
      np.testing.assert_allclose(got[3], want["z_loss"], rtol=2e-5)
    # the same bits on every run
    again = H.to_np(hip.router_summaries(
        lg, name, c, importance=ip, kept=r.kept, top_k=k, num_microbatches=mb,
        softmax_dtype=torch.bfloat16 if bf16 else torch.float32))
    np.testing.assert_array_equal(got, again)


@pytest.mark.parametrize("shape", [(2, 256, 8, 40), (32, 2048, 64, 64),
                                   (3, 77, 5, 12), (2, 131, 200, 3)])
def test_router_summaries_expert_selection(hip, shape):
  g, s, e, c = shape
  rng = np.random.default_rng(4200 + sum(shape))
  logits = H.random_logits(rng, g, s, e, scale=1.5)
  imp = rng.choice(np.array([0.0, 1.0], np.float32), size=(g, s), p=[0.1, 0.9])
  lg, ip = torch.from_numpy(logits).cuda(), H.to_gpu(imp)
  r = hip.expert_choice_gating(lg, c, importance=ip)
  want_r = dict(slot_token=H.to_np(r.slot_token).astype(np.int64))
  want = O.router_summaries(logits, "expert_selection", want_r, importance=imp)
  got = H.to_np(hip.router_summaries(lg, "expert_selection", c, importance=ip,
                                     tok_slot=r.tok_slot))
  assert got.shape == (4 + s,)
  np.testing.assert_allclose(got[0], want["entropy"], rtol=2e-5)
  np.testing.assert_array_equal(got[4:], want["group_token"])
  assert got[4:].sum() == float(g * e * c) * e * c


def test_router_summaries_rejections(hip):
  lg = torch.zeros((1, 8, 4), device="cuda")
  with pytest.raises(hip.MoeHipError, match="need kept"):
    hip.router_summaries(lg, "switch", 2)
  with pytest.raises(hip.MoeHipError, match="tok_slot"):
    hip.router_summaries(lg, "expert_selection", 2)
  with pytest.raises(hip.MoeHipError, match="top_k"):
    hip.router_summaries(lg, "ntlb", 2, top_k=9)
  kept = torch.zeros((1, 8, 2), dtype=torch.uint8, device="cuda")
  with pytest.raises(hip.MoeHipError, match="bfloat16"):
    hip.router_summaries(lg, "switch", 2, kept=kept,
                         softmax_dtype=torch.bfloat16)


def test_ntlb_gating_rejections(hip):
  lg = torch.zeros((1, 8, 4), dtype=torch.float32, device="cuda")
  with pytest.raises(hip.MoeHipError, match="top_k=5 with 4 experts"):
    hip.ntlb_gating(lg, 2, 5)
  with pytest.raises(hip.MoeHipError, match="top_k=0"):
    hip.ntlb_gating(lg, 2, 0)
  big = torch.zeros((1, 8, 16), dtype=torch.float32, device="cuda")
  with pytest.raises(hip.MoeHipError, match="top_k=9 > 8"):
    hip.ntlb_gating(big, 2, 9)


@pytest.mark.parametrize("shape", [(2, 1024, 8, 160), (16, 2048, 64, 32),
                                   (3, 77, 5, 7), (1, 1, 2, 1),
                                   (2, 131, 200, 4), (1, 4096, 64, 40),
                                   (32, 2048, 64, 64)])
def test_switch_max_gating(hip, shape):
  """Slots by descending gate.  The oracle ranks NumPy's softmax values and the
  kernel its own: the generator keeps the top logits apart, and gates of
  different tokens that tie to the last bit would need the same expf -- the
  comparison below is therefore on inputs where, per expert, no two choosers'
  gates are closer than 1e-6 relative (checked)."""
  g, s, e, c = shape
  rng = np.random.default_rng(2000 + hash(shape) % 1000)
  for attempt in range(20):
    logits = H.safe_logits(rng, g, s, e, scale=1.5)
    p = O.softmax(logits)
    top = p.max(-1)
    idx = p.argmax(-1)
    ok = True
    for gi in range(g):
      for ex in range(e):
        v = np.sort(top[gi][idx[gi] == ex])
        if len(v) > 1 and (np.diff(v) < 1e-6 * v[1:]).any():
          ok = False
    if ok:
      break
  assert ok
  imp = rng.choice(np.array([0.0, 1.0], np.float32), size=(g, s), p=[0.15, 0.85])
  for importance in (None, imp):
    want = O.switch_max_gating(logits, c, importance=importance,
                               num_microbatches=2)
    r = hip.switch_gating(torch.from_numpy(logits).cuda(), c,
                          importance=None if importance is None else H.to_gpu(importance),
                          num_microbatches=2, slots_by_gate=True)
    got = H.routing_to_np(r)
    _assert_switch_max_equal(got, want)
    np.testing.assert_allclose(got["loss"], want["loss"], rtol=2e-5)


def test_switch_max_exact_ties_token_order(hip):
  """Equal gates: the lower token index gets the lower slot (tf.math.top_k).
  Logits on a coarse grid, rows repeated so that whole rows tie exactly."""
  g, s, e, c = 2, 300, 6, 20
  rng = np.random.default_rng(9)
  base = H.random_logits(rng, g, 12, e, scale=0.6, quantum=0.25)
  logits = np.tile(base, (1, s // 12, 1)).astype(np.float32)
  want = O.switch_max_gating(logits, c)
  got = H.routing_to_np(hip.switch_gating(torch.from_numpy(logits).cuda(), c,
                                          slots_by_gate=True))
  # identical rows give bit-identical gates in either implementation, so the
  # tie order is exercised and the ranks must agree exactly
  _assert_switch_max_equal(got, want)
  assert not want["kept_1"].all()


def test_router_switch_max_fused(hip):
  b, gpr, s, m, e, c = 1, 4, 256, 128, 8, 40
  rng = np.random.default_rng(45)
  w = O.round_bf16((rng.standard_normal((b, m, e)) / np.sqrt(m)).astype(np.float32))
  x = np.stack([H.safe_tokens(rng, gpr * s, m, w[i], "bfloat16") for i in range(b)])
  xg, wg = H.to_gpu(x, "bfloat16"), H.to_gpu(w, "bfloat16")
  wp = hip.pack_weights(wg, wg.dtype)
  r, got_logits = hip.router_switch_gating(xg, wp, s, c, want_logits=True,
                                           slots_by_gate=True)
  r2 = hip.switch_gating(got_logits, c, slots_by_gate=True)
  for a_, b_ in ((r.idx, r2.idx), (r.pos, r2.pos), (r.kept, r2.kept),
                 (r.fill, r2.fill), (r.gate, r2.gate)):
    assert torch.equal(a_, b_)
  got = H.routing_to_np(r)
  # invariants of the by-gate order on the kernel's own gates
  p = O.softmax(H.to_np(got_logits))
  for gi in range(b * gpr):
    for ex in range(e):
      mine = (got["index_1"][gi] == ex)
      kept = mine & got["kept_1"][gi]
      assert kept.sum() == min(mine.sum(), c) == got["fill"][gi, ex]
      if kept.any() and (mine & ~kept).any():
        assert p[gi][kept, ex].min() >= p[gi][mine & ~kept, ex].max() * (1 - 1e-6)
      order = np.argsort(got["pos_1"][gi][kept])
      assert (np.diff(got["gate_1"][gi][kept][order]) <= 0).all()


# ---- expert FFN at the full benchmark sizes ---------------------------------------
@pytest.mark.parametrize("size", [(64, 512, 1024, 4096), (64, 2048, 4096, 16384)],
                         ids=["cfg3", "cfg4"])
def test_full_size_expert_ffn_properties(hip, size):
  """(E, rows per expert, M, H) of configurations 3 and 4.  The oracle is too
  slow here: row blocks sampled from the first, a middle and the last expert
  are checked against float32 matmuls of the same bf16 operands (tile mapping,
  K loop, epilogue at the real grid size), and two exact properties hold on the
  whole output: scaling the tokens by 2 scales the output by 2 bit for bit,
  and an expert whose token rows are zero outputs zeros."""
  e, r, m, hdim = size
  gen = torch.Generator(device="cuda")
  gen.manual_seed(17)
  x = torch.randn((e, r, m), generator=gen, device="cuda").to(torch.bfloat16)
  wi = torch.empty((e, hdim, m), dtype=torch.bfloat16, device="cuda")
  wo = torch.empty((e, m, hdim), dtype=torch.bfloat16, device="cuda")
  for i in range(e):                         # packed layout [E, N, K] directly
    wi[i] = (torch.randn((hdim, m), generator=gen, device="cuda") / m ** 0.5).to(torch.bfloat16)
    wo[i] = (torch.randn((m, hdim), generator=gen, device="cuda") / hdim ** 0.5).to(torch.bfloat16)
  x[e // 2 + 1].zero_()
  y = hip.expert_ffn(x, wi, wo, "relu")
  assert bool(torch.isfinite(y.float()).all())
  for ei, r0 in ((0, 0), (e // 2, r // 2 - 37), (e - 1, r - 64), (e - 1, 0)):
    xs = x[ei, r0:r0 + 64].float()
    h_ref = torch.relu(xs @ wi[ei].float().t()).to(torch.bfloat16).float()
    y_ref = h_ref @ wo[ei].float().t()
    err = (y[ei, r0:r0 + 64].float() - y_ref).abs().max().item()
    scale = y_ref.abs().max().item()
    assert err <= 2e-2 * scale, (ei, r0, err, scale)
  assert not bool(y[e // 2 + 1].any())
  y2 = hip.expert_ffn(x * 2, wi, wo, "relu")
  assert torch.equal(y2, y * 2)


# ---- expert-selection (expert choice) gating ---------------------------------------
def _column_gaps_ok(logits, imp, min_gap=1e-4):
  """No two unmasked tokens of a group have logits for the same expert closer
  than min_gap: their probabilities then rank the same way whatever the last
  ulp of exp/log."""
  g, s, e = logits.shape
  for gi in range(g):
    keep = imp[gi] != 0
    col = np.sort(logits[gi][keep], axis=0)
    if (np.diff(col, axis=0) < min_gap).any():
      return False
  return True


@pytest.mark.parametrize("shape", [(2, 64, 4, 8), (3, 77, 5, 20), (2, 1024, 8, 256),
                                   (16, 2048, 64, 32), (1, 300, 130, 7),
                                   (32, 2048, 64, 64)])
def test_expert_choice_gating(hip, shape):
  g, s, e, c = shape
  rng = np.random.default_rng(3000 + hash(shape) % 1000)
  # per (group, expert) a shuffled grid of logits with spacing 6 / S plus a
  # jitter below a quarter of it: no two tokens of a column nearly tie
  step = 6.0 / s
  grid = (np.arange(s) - s / 2) * step
  logits = np.empty((g, s, e), np.float32)
  for gi in range(g):
    for ex in range(e):
      logits[gi, :, ex] = rng.permutation(grid) + rng.uniform(-step / 4, step / 4, s)
  imp = rng.choice(np.array([0.0, 0.5, 1.0], np.float32), size=(g, s),
                   p=[0.1, 0.1, 0.8])
  assert _column_gaps_ok(logits, imp, min_gap=step / 4)
  want = O.expert_selection_gating(logits, c, imp, num_microbatches=2)
  for imp_dtype in ("float32", "bfloat16"):
    r = hip.expert_choice_gating(torch.from_numpy(logits).cuda(), c,
                                 importance=H.to_gpu(imp, imp_dtype),
                                 num_microbatches=2)
    np.testing.assert_array_equal(H.to_np(r.slot_token), want["slot_token"])
    np.testing.assert_allclose(H.to_np(r.slot_weight), want["slot_weight"],
                               rtol=2e-5, atol=1e-30)
    np.testing.assert_allclose(H.to_np(r.loss)[0], want["loss"], rtol=5e-5)
    # tok_slot is the inverse of slot_token
    ts = H.to_np(r.tok_slot)
    inv = np.full((g, s, e), -1, np.int16)
    for gi in range(g):
      for ex in range(e):
        inv[gi, want["slot_token"][gi, ex], ex] = np.arange(c)
    np.testing.assert_array_equal(ts, inv)


def test_expert_choice_exact_ties_token_order(hip):
  g, s, e, c = 2, 96, 4, 30
  rng = np.random.default_rng(10)
  logits = (np.round(rng.standard_normal((g, s, e)) * 2) / 2).astype(np.float32)
  imp = np.ones((g, s), np.float32)
  want = O.expert_selection_gating(logits, c, imp)
  r = hip.expert_choice_gating(torch.from_numpy(logits).cuda(), c,
                               importance=H.to_gpu(imp))
  # equal logits give bit-equal probabilities in either implementation and
  # unequal ones differ by >= 0.5, so the slots must agree exactly
  np.testing.assert_array_equal(H.to_np(r.slot_token), want["slot_token"])


@pytest.mark.parametrize("act_dtype", ["float32", "bfloat16"])
def test_slot_dispatch_combine(hip, act_dtype):
  g, s, e, c, m = 2, 128, 8, 40, 72
  rng = np.random.default_rng(11)
  logits = (rng.standard_normal((g, s, e)) * 1.5).astype(np.float32)
  imp = np.ones((g, s), np.float32)
  want_r = O.expert_selection_gating(logits, c, imp)
  r = hip.expert_choice_gating(torch.from_numpy(logits).cuda(), c,
                               importance=H.to_gpu(imp))
  assert np.array_equal(H.to_np(r.slot_token), want_r["slot_token"])
  x = O.cast_act(rng.standard_normal((g, s, m)).astype(np.float32), act_dtype)
  ein = hip.slot_dispatch(H.to_gpu(x, act_dtype), r)
  np.testing.assert_array_equal(H.to_np(ein), O.slot_dispatch(x, want_r))
  y = O.cast_act(rng.standard_normal((e, g, c, m)).astype(np.float32), act_dtype)
  out = hip.slot_combine(H.to_gpu(y, act_dtype), r, s)
  # the kernel's own weights (they match the oracle's to float32 round-off;
  # a bf16 rounding boundary could otherwise flip a weight by one bf16 ulp)
  r_np = dict(slot_token=want_r["slot_token"], slot_weight=H.to_np(r.slot_weight))
  np.testing.assert_allclose(H.to_np(out), O.slot_combine(y, r_np, s, act_dtype),
                             **H.value_tolerance(act_dtype))
  chosen = np.zeros((g, s), bool)
  for gi in range(g):
    chosen[gi][want_r["slot_token"][gi].reshape(-1)] = True
  assert (H.to_np(out)[~chosen] == 0).all()


@pytest.mark.parametrize("shape", [(4, 512, 8, 128, 256, 512, 256),
                                   (2, 1024, 16, 128, 128, 384, 128),
                                   (5, 300, 4, 180, 64, 256, 64),
                                   # 400 and 640 rows per expert: a last row
                                   # tile of 144 / 128 rows
                                   (5, 512, 8, 80, 128, 512, 256),
                                   (16, 256, 8, 40, 64, 256, 256)])
def test_dispatched_expert_ffn_equals_two_calls(hip, shape):
  """The dispatch folded into the first expert GEMM gives bit-identical h-free
  outputs to mesh_moe_dispatch + mesh_moe_expert_ffn (same kernel, same
  operands, rows fetched through the slot map), including empty slots and
  kept choices whose bf16 gate is 0."""
  g, s, e, c, m, hdim, n = shape
  rng = np.random.default_rng(sum(shape))
  logits = H.safe_logits(rng, g, s, e, scale=1.5,
                         bias=H.zipf_bias(rng, e, scale=2.0))
  x = H.to_gpu(rng.standard_normal((g, s, m)).astype(np.float32), "bfloat16")
  wi = H.to_gpu(H.normal_weights(rng, (e, m, hdim), m), "bfloat16")
  wo = H.to_gpu(H.normal_weights(rng, (e, hdim, n), hdim), "bfloat16")
  wi_p = hip.pack_weights(wi, torch.bfloat16)
  wo_p = hip.pack_weights(wo, torch.bfloat16)
  r = hip.top2_gating(torch.from_numpy(logits).cuda(), c)
  r.gate[0, 0, 0] = 0.0            # a kept choice with gate 0: dispatches zeros
  assert int((r.fill < c).sum()) > 0                   # some empty slots
  want = hip.expert_ffn(hip.dispatch(x, r).reshape(e, g * c, m), wi_p, wo_p,
                        "relu")
  got = hip.dispatched_expert_ffn(x, r, wi_p, wo_p, "relu")
  assert got is not None
  assert torch.equal(got, want)
  # float32, and row counts whose whole 256-row tiles would be more than a fifth
  # padding: the library declines and the caller makes the two calls
  assert hip.dispatched_expert_ffn(x.float(), r, wi_p.float(), wo_p.float(),
                                   "relu") is None
  if g * c == 256:
    r2 = hip.top2_gating(torch.from_numpy(logits).cuda(), c + 32)
    assert hip.dispatched_expert_ffn(x, r2, wi_p, wo_p, "relu") is None


@pytest.mark.parametrize("m", [64, 128, 192, 320])
@pytest.mark.parametrize("g,c", [(5, 80), (7, 91)])
def test_dispatched_expert_ffn_tile_after_tile(hip, g, c, m):
  """Rows fetched through the slot map by blocks that go from tile to tile (1024 of
  them), whose map entries they ask for a tile ahead: row tiles of fewer than 256 rows,
  the last one partly empty; reductions of one to five K tiles.  The second product's
  weights are the identity, so that the result is the hidden tensor.  The bits of the
  two calls, and against float64: one bf16 rounding, and K / 2 ulps of the sum of
  magnitudes for the float32 sum of K products."""
  s, e, h = 2048, 64, 2048
  gen = torch.Generator(device="cuda").manual_seed(g + c + m)
  mk = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
  r = hip.top2_gating(mk(g, s, e), c)
  assert int((r.fill < c).sum()) > 0                   # some empty slots
  x = mk(g, s, m).to(torch.bfloat16)
  wi = mk(e, h, m).to(torch.bfloat16)
  wo = torch.eye(h, device="cuda", dtype=torch.bfloat16).repeat(e, 1, 1)
  got = hip.dispatched_expert_ffn(x, r, wi, wo, "relu")
  assert got is not None
  xe = hip.dispatch(x, r).reshape(e, g * c, m)
  assert torch.equal(got, hip.expert_ffn(xe, wi, wo, "relu"))
  for i in range(0, e, 7):
    t = wi[i].double().t().contiguous()
    want = (xe[i].double() @ t).clamp(min=0)
    magnitude = xe[i].double().abs() @ t.abs()
    bound = 2.0 ** -8 * want + m * 2.0 ** -25 * magnitude
    assert bool(((got[i].double() - want).abs() <= bound).all())


@pytest.mark.parametrize("case", [
    # G, S, E, C, M, H, N, router
    (4, 512, 8, 128, 256, 512, 256, "switch"),
    (8, 1024, 16, 128, 128, 256, 256, "switch"),
    (4, 512, 8, 256, 256, 512, 256, "top_2"),
    (32, 2048, 64, 64, 1024, 2048, 1024, "switch")],
    ids=["small", "mid", "top2_record", "cfg4_routing"])
def test_compact_expert_ffn_equals_two_calls(hip, case):
  """mesh_moe_compact_expert_ffn + mesh_moe_combine_compact (occupied slots
  first, only the tiles that hold them multiplied) give the same layer output,
  bit for bit, as dispatch + expert FFN + combine on every slot: a slot's
  result depends on its own row only, wherever the row sits."""
  g, s, e, c, m, hdim, n, router = case
  rng = np.random.default_rng(sum(case[:7]))
  logits = torch.from_numpy(H.safe_logits(
      rng, g, s, e, scale=1.5, bias=H.zipf_bias(rng, e, scale=1.0))).cuda()
  x = H.to_gpu(rng.standard_normal((g, s, m)).astype(np.float32), "bfloat16")
  wi_p = hip.pack_weights(H.to_gpu(H.normal_weights(rng, (e, m, hdim), m),
                                   "bfloat16"), torch.bfloat16)
  wo_p = hip.pack_weights(H.to_gpu(H.normal_weights(rng, (e, hdim, n), hdim),
                                   "bfloat16"), torch.bfloat16)
  r = (hip.switch_gating(logits, c) if router == "switch"
       else hip.top2_gating(logits, c))
  r.gate[0, 0, 0] = 0.0             # a kept choice with gate 0
  fill = r.fill.long()
  assert int((fill < c).sum()) > 0 and int(fill.sum()) < 0.8 * g * e * c
  y_all = hip.expert_ffn(hip.dispatch(x, r).reshape(e, g * c, m), wi_p, wo_p,
                         "relu")
  want = hip.combine(y_all.reshape(e, g, c, n), r, s)
  got = hip.compact_expert_ffn(x, r, wi_p, wo_p, "relu")
  assert got is not None
  y, row_offsets = got
  # row_offsets[e][g] = occupied slots of expert e in earlier groups
  want_off = (fill.t().cumsum(1) - fill.t()).to(torch.int32)
  assert torch.equal(row_offsets, want_off)
  out = hip.combine(y.reshape(e, g, c, n), r, s, row_offsets=row_offsets)
  assert torch.equal(out, want)
  # the occupied rows themselves, slot by slot
  for ei in (0, e // 2, e - 1):
    for gi in (0, g - 1):
      k = int(fill[gi, ei])
      o = int(row_offsets[ei, gi])
      assert torch.equal(y[ei, o:o + k], y_all[ei, gi * c:gi * c + k])


@pytest.mark.parametrize("case", [
    (1, 300, 2, 256, 64, 256, 256), (300, 16, 8, 2, 64, 256, 264),
    (257, 16, 65, 2, 64, 320, 256), (2, 1024, 512, 128, 64, 4352, 256)],
    ids=lambda c: "x".join(map(str, c)))
def test_compact_rows_map_and_lists(hip, case):
  """The compacted rows' offsets, map and tile lists at their edges: one group
  and two experts, more groups than a block has threads, more experts than a
  wavefront, more tiles than one block lists, experts without a token."""
  g, s, e, c, m, h, n = case
  gen = torch.Generator(device="cuda")
  gen.manual_seed(sum(case))
  mk = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
  logits = mk(g, s, e)
  logits[..., e // 2] -= 100.0
  r = hip.switch_gating(logits, c)
  x = mk(g, s, m).to(torch.bfloat16)
  wi = mk(e, h, m).to(torch.bfloat16) / m ** 0.5
  wo = mk(e, n, h).to(torch.bfloat16) / h ** 0.5
  y, row_offsets = hip.compact_expert_ffn(x, r, wi, wo, "relu")
  fill = r.fill.long()
  assert torch.equal(row_offsets, (fill.t().cumsum(1) - fill.t()).to(torch.int32))
  want = hip.expert_ffn(hip.dispatch(x, r).reshape(e, g * c, m), wi, wo, "relu")
  assert torch.equal(
      hip.combine(y.reshape(e, g, c, n), r, s, row_offsets=row_offsets),
      hip.combine(want.reshape(e, g, c, n), r, s))


def test_dispatched_expert_ffn_equals_two_calls_cfg4(hip):
  """The same identity at the full size of benchmark configuration 4 (32 groups
  of 2048 tokens, 64 experts, capacity 64, d_model 4096, hidden 16384), where
  the gathered GEMM is the kernel the benchmark times: hidden and output
  tensors bit for bit equal to dispatch + expert FFN, with empty slots (a
  biased router leaves some experts short) and kept choices of gate 0."""
  g, s, e, c, m, hdim = 32, 2048, 64, 64, 4096, 16384
  gen = torch.Generator(device="cuda")
  gen.manual_seed(23)
  logits = torch.randn((g, s, e), generator=gen, device="cuda")
  ranks = torch.randperm(e, generator=gen, device="cuda").double() + 1
  logits = logits + (1.5 * ranks ** -1.2).float()
  x = torch.randn((g, s, m), generator=gen, device="cuda").to(torch.bfloat16)
  wi = torch.empty((e, hdim, m), dtype=torch.bfloat16, device="cuda")
  wo = torch.empty((e, m, hdim), dtype=torch.bfloat16, device="cuda")
  for i in range(e):                         # packed layout [E, N, K] directly
    wi[i] = (torch.randn((hdim, m), generator=gen, device="cuda") / m ** 0.5).to(torch.bfloat16)
    wo[i] = (torch.randn((m, hdim), generator=gen, device="cuda") / hdim ** 0.5).to(torch.bfloat16)
  r = hip.top2_gating(logits, c)
  r.gate[0, 0, 0] = 0.0
  r.gate[g - 1, s - 1, 1] = 0.0
  assert int((r.fill < c).sum()) > 0 and int((r.fill == c).sum()) > 0
  h_want = torch.empty((e, g * c, hdim), dtype=torch.bfloat16, device="cuda")
  h_got = torch.empty_like(h_want)
  want = hip.expert_ffn(hip.dispatch(x, r).reshape(e, g * c, m), wi, wo, "relu",
                        h=h_want)
  got = hip.dispatched_expert_ffn(x, r, wi, wo, "relu", h=h_got)
  assert got is not None
  assert torch.equal(h_got, h_want)
  assert torch.equal(got, want)
  assert bool(torch.isfinite(got.float()).all())
  # and on compacted rows, the layout the layer uses for two choices per token
  # when an expert's slot rows are whole tiles (2048 here): the same layer
  # output bit for bit
  del h_got, h_want
  out_want = hip.combine(want.reshape(e, g, c, m), r, s)
  del want, got
  compact = hip.compact_expert_ffn(x, r, wi, wo, "relu")
  assert compact is not None
  y, row_offsets = compact
  fill = r.fill.long()
  assert torch.equal(row_offsets,
                     (fill.t().cumsum(1) - fill.t()).to(torch.int32))
  out = hip.combine(y.reshape(e, g, c, m), r, s, row_offsets=row_offsets)
  assert torch.equal(out, out_want)


@pytest.mark.parametrize("act_dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("activation", ["relu", "linear"])
def test_hidden_product_and_dropout_backward(hip, act_dtype, activation):
  """mesh_moe_hidden_product (a second factor, then dropout) and the backward
  of the expert einsums with the dropout noise, against the oracle."""
  e, rows, m, hdim, n = 3, 70, 24, 40, 16
  keep = 0.7
  rng = np.random.default_rng(17)
  cast = lambda a: O.cast_act(a.astype(np.float32), act_dtype)
  xe = cast(rng.standard_normal((e, rows, m)))
  wi = cast(H.normal_weights(rng, (e, m, hdim), m))
  wi2 = cast(H.normal_weights(rng, (e, m, hdim), m))
  wo = cast(H.normal_weights(rng, (e, hdim, n), hdim))
  dy = cast(rng.standard_normal((e, rows, n)))
  u = cast(rng.random((e, rows, hdim)))
  u = np.minimum(u, np.float32(0.99))          # bf16 rounding may reach 1.0
  u[0, 0, 0] = O.cast_act(np.float32(keep), act_dtype)   # the threshold itself
  dt = H.ACT_TORCH[act_dtype]
  g = lambda a: H.to_gpu(a, act_dtype)
  wi_p, wi2_p = hip.pack_weights(g(wi), dt), hip.pack_weights(g(wi2), dt)
  noise_want = O.hidden_dropout_noise(u, keep, act_dtype)
  assert noise_want[0, 0, 0] == 0
  tol = H.value_tolerance(act_dtype)

  # two factors and dropout, forward
  h = hip.expert_linear(g(xe), wi_p, activation)
  f = hip.expert_linear(g(xe), wi2_p, "sigmoid")
  assert hip.hidden_product(h, factor=f) is None
  noise = hip.hidden_product(h, uniform=g(u), keep_prob=keep, want_noise=True)
  np.testing.assert_array_equal(H.to_np(noise), noise_want)
  h_want = O.expert_hidden(xe, [wi, wi2], [activation, "sigmoid"], act_dtype,
                           noise_want)
  np.testing.assert_allclose(H.to_np(h), h_want, **tol)
  assert (H.to_np(h)[noise_want == 0] == 0).all()

  # one factor and dropout, forward and backward
  h = hip.expert_linear(g(xe), wi_p, activation)
  noise = hip.hidden_product(h, uniform=g(u), keep_prob=keep, want_noise=True)
  dxe, dwi, dwo = hip.expert_ffn_backward(g(xe), h, g(dy), g(wi), g(wo),
                                          activation, dh_scale=noise)
  want = O.expert_ffn_backward(xe, wi, wo, dy, activation, act_dtype,
                               noise_want)
  plain = O.expert_ffn_backward(xe, wi, wo, dy, activation, act_dtype)
  assert np.abs(want[1] - plain[1]).max() > 0.05
  for got_, want_, name in zip((dxe, dwi, dwo), want, ("dxe", "dwi", "dwo")):
    np.testing.assert_allclose(
        H.to_np(got_), want_, rtol=tol["rtol"],
        atol=tol["atol"] * max(1.0, np.abs(want_).max()), err_msg=name)
  # nothing to do / bad arguments
  h0 = h.clone()
  hip.hidden_product(h)
  assert torch.equal(h, h0)
  with pytest.raises(hip.MoeHipError):
    hip.hidden_product(h, uniform=g(u), keep_prob=0.0)
  with pytest.raises(hip.MoeHipError):
    hip.hidden_product(h, factor=f[:, :1])


@pytest.mark.parametrize("shape", [(2, 128, 256, 512, 256), (3, 192, 136, 264, 136),
                                   (1, 2048, 512, 1024, 256), (2, 64, 256, 256, 128),
                                   (2, 96, 256, 256, 256),
                                   # rows that end inside a K tile of 64
                                   (2, 400, 256, 512, 256), (3, 8, 128, 128, 128),
                                   (1, 1000, 128, 256, 128)])
def test_expert_ffn_backward_weight_gradients_bf16(hip, shape):
  """bf16 weight gradients dwi = expert_in^T . dh and dwo = h^T . dy: the
  reduction runs over token rows.  The kernel reads both operands as they lie
  in memory (transposing LDS reads); row counts that end inside its K tile of
  64 (96, 400, 8, 1000) take the rest of the tile from a zero buffer; kernel
  dimensions that are not multiples of 8 (136, 264) go through transposed
  copies.  All against float32 matmuls of the same bf16 operands."""
  e, rows, m, hdim, n = shape
  rng = np.random.default_rng(sum(shape))
  g = lambda a: H.to_gpu(O.cast_act(a.astype(np.float32), "bfloat16"), "bfloat16")
  xe = g(rng.standard_normal((e, rows, m)))
  wi = g(H.normal_weights(rng, (e, m, hdim), m))
  wo = g(H.normal_weights(rng, (e, hdim, n), hdim))
  dy = g(rng.standard_normal((e, rows, n)))
  wi_p = hip.pack_weights(wi, torch.bfloat16)
  h = hip.expert_linear(xe, wi_p, "relu")
  dxe, dwi, dwo = hip.expert_ffn_backward(xe, h, dy, wi, wo, "relu")
  dh = (torch.bmm(dy.float(), wo.float().transpose(1, 2)).to(torch.bfloat16).float()
        * (h > 0))
  want_dwo = torch.bmm(h.float().transpose(1, 2), dy.float())
  want_dwi = torch.bmm(xe.float().transpose(1, 2), dh)
  want_dxe = torch.bmm(dh, wi.float().transpose(1, 2))
  for got, want, name in ((dwo, want_dwo, "dwo"), (dwi, want_dwi, "dwi"),
                          (dxe, want_dxe, "dxe")):
    scale = float(want.abs().max())
    np.testing.assert_allclose(H.to_np(got), H.to_np(want), rtol=2e-2,
                               atol=1e-2 * scale, err_msg=name)


@pytest.mark.parametrize("shape", [(1, 4096, 256, 1024), (2, 6144, 128, 2048),
                                   (1, 4096 + 256, 128, 1024),
                                   (1, 512, 4096, 1024)],
                         ids=lambda s: "x".join(map(str, s)))
def test_expert_linear_many_row_tiles(hip, shape):
  """More than 8 row tiles of 256 per group (the dense layers of a transformer
  block: one group, every token a row): the tile order that keeps an XCD's
  resident tiles in blocks of 8 x 4, and a row-tile count that does not divide
  by 8 (plain order); forward and the weight gradient (row tiles = the columns
  of the first operand there) against float32 matmuls."""
  e, rows, k, n = shape
  rng = np.random.default_rng(sum(shape))
  g = lambda a: H.to_gpu(O.cast_act(a.astype(np.float32), "bfloat16"), "bfloat16")
  a = g(rng.standard_normal((e, rows, k)))
  w = g(H.normal_weights(rng, (e, k, n), k))
  dy = g(rng.standard_normal((e, rows, n)))
  y = hip.expert_linear(a, hip.pack_weights(w, torch.bfloat16))
  want = torch.bmm(a.float(), w.float())
  np.testing.assert_allclose(H.to_np(y), H.to_np(want), rtol=2e-2,
                             atol=1e-2 * float(want.abs().max()))
  da, dw = hip.expert_linear_backward(a, dy, w)
  want_da = torch.bmm(dy.float(), w.float().transpose(1, 2))
  want_dw = torch.bmm(a.float().transpose(1, 2), dy.float())
  for got, wnt, name in ((da, want_da, "da"), (dw, want_dw, "dw")):
    np.testing.assert_allclose(H.to_np(got), H.to_np(wnt), rtol=2e-2,
                               atol=1e-2 * float(wnt.abs().max()), err_msg=name)


@pytest.mark.parametrize("shape", [(64, 1024, 16), (66, 1001, 128), (9, 16384, 32),
                                   (130, 1009, 24), (1400, 97, 3), (2048, 64, 10)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("with_importance", [False, True])
def test_gating_of_many_tokens_equals_its_parts(hip, shape, with_importance):
  """Sixteen, eight or four lanes select for a token, by the number of tokens and
  experts: routing, gates and counts are bit for bit those of the groups gated in
  two calls of half the tokens.  The loss is the mean of theirs with its sums of
  positive terms in another order: at most 16 terms, 16 ranges, 256 blocks and 2048
  groups after each other, half a rounding of 2^-23 each."""
  g, s, e = shape
  half = 131072 if e <= 24 and g * s >= 131072 else 65536
  assert g * s >= half > (g - g // 2) * s or e == 32
  gen = torch.Generator(device="cuda")
  gen.manual_seed(sum(shape))
  logits = torch.randn((g, s, e), generator=gen, device="cuda")
  logits[::3, 5] = 1.0                           # ties
  imp = None
  if with_importance:
    imp = torch.tensor([0.0, 0.5, 1.0], device="cuda")[
        torch.randint(0, 3, (g, s), generator=gen, device="cuda")].to(torch.bfloat16)
  c = max(1, s // e)
  parts = [slice(0, g // 2), slice(g // 2, g)]
  choice = torch.randn((g, s, e), generator=gen, device="cuda")
  for run in (lambda p: hip.top2_gating(logits[p], c, use_second_place_loss=True,
                                        importance=None if imp is None else imp[p]),
              lambda p: hip.switch_gating(logits[p], c, z_loss=1e-3,
                                          importance=None if imp is None else imp[p]),
              lambda p: hip.switch_gating(logits[p], c, choice_logits=choice[p])):
    whole, halves = run(slice(0, g)), [run(p) for p in parts]
    for name in ("idx", "pos", "kept", "fill"):
      assert torch.equal(getattr(whole, name),
                         torch.cat([getattr(h, name) for h in halves])), name
    gates = torch.cat([h.gate for h in halves])
    assert torch.equal(whole.gate.view(torch.int32), gates.view(torch.int32))
    if imp is None:
      mean = sum(float(h.loss) * (p.stop - p.start)
                 for h, p in zip(halves, parts)) / g
      assert abs(float(whole.loss) - mean) <= 2336 * 2.0 ** -24 * mean



def _check_linear(hip, shape, activation):
  """expert_linear against float32 products.  The bound: one bf16 rounding and
  the float32 sums of K products in another order."""
  e, rows, k, n = shape
  gen = torch.Generator(device="cuda")
  gen.manual_seed(sum(shape))
  a = torch.randn((e, rows, k), generator=gen, device="cuda").to(torch.bfloat16)
  w = torch.randn((e, n, k), generator=gen, device="cuda").to(torch.bfloat16)
  y = hip.expert_linear(a, w, activation)
  assert torch.equal(y, hip.expert_linear(a, w, activation))
  for i in range(0, e, max(1, e // 4)):
    wt = w[i].float().t().contiguous()
    want = a[i].float() @ wt
    bound = 2.0 ** -8 * want.abs() + k * 2.0 ** -24 * (a[i].float().abs() @ wt.abs())
    want = want.relu() if activation == "relu" else want
    assert bool(((y[i].float() - want).abs() <= bound).all())


@pytest.mark.parametrize("shape", [
    (1, 1, 32, 16), (1, 17, 96, 48), (1, 33, 2080, 80), (2, 64, 512, 1040),
    (3, 65, 4096, 112), (1, 97, 1056, 2064), (1, 128, 768, 768),
    # 32 columns a block: one to eight tiles of rows, the last columns a half
    # block; the longest reduction with eight tiles (LDS holds 8 wavefronts' sums)
    (1, 1, 64, 8192), (3, 30, 480, 2736), (1, 40, 4128, 4112), (5, 64, 1024, 1616),
    (7, 96, 352, 1040), (1, 97, 1088, 8176), (1, 128, 8192, 4112),
    # more blocks of 32 columns than compute units, K % 64 != 0
    (1, 50, 96, 16000), (30, 64, 160, 400),
    # neither kernel's any more: too many columns for the rows
    (1, 65, 192, 10240), (1, 128, 256, 16000), (60, 100, 128, 256)],
    ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("activation", ["linear", "relu"])
def test_linear_of_few_rows_and_columns(hip, shape, activation):
  """Few rows, and fewer column tiles than compute units: the reduction is cut
  over the wavefronts of a block.  One to eight tiles of 16 rows; reductions of
  1 to 256 steps over 2 to 16 wavefronts; columns inside a block's 16 or 32."""
  _check_linear(hip, shape, activation)


@pytest.mark.parametrize("shape", [
    (130, 1, 64, 72), (64, 32, 192, 256), (43, 33, 320, 400), (128, 64, 1024, 128),
    (16, 5, 128, 1032), (160, 20, 4096, 256), (160, 64, 4160, 256),
    # fewer than 128 column tiles, more than 256 blocks of 32 columns
    (1, 64, 1024, 10248), (9, 17, 320, 936), (33, 48, 64, 256),
    # more blocks than compute units: 48 rows, 49, longer reductions, more columns
    (130, 48, 512, 264), (130, 49, 512, 264), (130, 49, 576, 264), (33, 64, 64, 1032)],
    ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("activation", ["linear", "relu"])
def test_linear_of_few_rows_many_experts(hip, shape, activation):
  """At most 64 rows for each of many column tiles: reductions shorter than the
  ring of K tiles, and ones that go round it many times while two blocks share a
  compute unit; columns that end inside a 128-column tile."""
  _check_linear(hip, shape, activation)


@pytest.mark.parametrize("case", [(1, 64, 64, 4, 256, 512), (3, 40, 32, 5, 128, 1088),
                                  (8, 32, 48, 8, 64, 384)],
                         ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("activation", ["relu", "gelu"])
def test_dispatched_ffn_of_few_rows(hip, case, activation):
  """dispatch + experts in one call with at most 64 rows per expert, some of
  the experts without a token: the slots that the combine reads equal those of
  the two calls bit for bit."""
  g, s, e, c, m, h = case
  gen = torch.Generator(device="cuda")
  gen.manual_seed(sum(case))
  mk = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
  logits = mk(g, s, e)
  logits[..., e // 2:e // 2 + 3] -= 100.0       # experts that nobody chooses
  r = hip.top2_gating(logits, c)
  x = mk(g, s, m).to(torch.bfloat16)
  wi = mk(e, h, m).to(torch.bfloat16) / m ** 0.5
  wo = mk(e, m, h).to(torch.bfloat16) / h ** 0.5
  y = hip.dispatched_expert_ffn(x, r, wi, wo, activation)
  assert y is not None
  want = hip.expert_ffn(hip.dispatch(x, r).reshape(e, g * c, m), wi, wo, activation)
  assert not bool((r.fill.sum(0) > 0).all())
  for gi in range(g):
    for ei in range(e):
      n = int(r.fill[gi, ei])
      at = slice(gi * c, gi * c + n)
      assert torch.equal(y[ei, at], want[ei, at])
  out = hip.combine(y.reshape(e, g, c, m), r, s)
  assert torch.equal(out, hip.combine(want.reshape(e, g, c, m), r, s))


@pytest.mark.parametrize("tokens", [512, 513])
def test_dispatched_ffn_of_few_rows_and_many_tokens(hip, tokens):
  """The map is made by a walk over all tokens for every expert: above 512 tokens
  the call is declined."""
  e, c, m, h = 64, 16, 64, 256
  gen = torch.Generator(device="cuda")
  gen.manual_seed(tokens)
  mk = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
  r = hip.top2_gating(mk(1, tokens, e), c)
  x = mk(1, tokens, m).to(torch.bfloat16)
  wi, wo = mk(e, h, m).to(torch.bfloat16), mk(e, m, h).to(torch.bfloat16)
  y = hip.dispatched_expert_ffn(x, r, wi, wo, "relu")
  assert (y is not None) == (tokens <= 512)
  if y is not None:
    want = hip.expert_ffn(hip.dispatch(x, r).reshape(e, c, m), wi, wo, "relu")
    assert torch.equal(hip.combine(y.reshape(e, 1, c, m), r, tokens),
                       hip.combine(want.reshape(e, 1, c, m), r, tokens))


@pytest.mark.parametrize("shape", [
    (3, 640, 128, 4096), (32, 640, 512, 1024), (5, 705, 192, 768), (1, 129, 64, 256),
    (2, 320, 1088, 264), (1, 2000, 256, 776), (1, 5000, 128, 1280), (7, 257, 64, 520),
    # tiles that are no multiple of the 8 XCDs, in one round and in two
    (42, 384, 1024, 512), (43, 400, 320, 512),
    # 128 x 128 tiles for short reductions and single row tiles, either side
    (30, 384, 64, 512), (30, 640, 128, 512), (1, 1100, 256, 1032), (1, 4096, 256, 1024),
    (64, 128, 1024, 1024), (130, 128, 576, 520)],
    ids=lambda s: "x".join(map(str, s)))
def test_linear_row_tiles(hip, shape):
  """Row counts that are spread over row tiles of 32 to 256 rows, the pieces of
  a tile dealt out between its two halves: plain, with ReLU, and with the ReLU
  mask of a gradient on the stores.  (The masked product always takes these
  tiles; where the plain one takes 128 x 128 tiles its bits are the same.)"""
  for activation in ("linear", "relu"):
    _check_linear(hip, shape, activation)
  e, rows, k, n = shape
  gen = torch.Generator(device="cuda")
  gen.manual_seed(1)
  dy = torch.randn((e, rows, k), generator=gen, device="cuda").to(torch.bfloat16)
  w = torch.randn((e, n, k), generator=gen, device="cuda").to(torch.bfloat16)
  mask = torch.randn((e, rows, n), generator=gen, device="cuda").to(torch.bfloat16)
  da, _ = hip.expert_linear_backward(mask, dy, w)
  masked, _ = hip.expert_linear_backward(mask, dy, w, da_relu_mask=mask)
  assert torch.equal(masked, da * (mask > 0))
  assert torch.equal(da, hip.expert_linear(dy, w))


def _off_16(t):
  moved = torch.empty(t.numel() + 4, dtype=t.dtype, device="cuda")
  moved = moved[1:1 + t.numel()].view(t.shape)
  moved.copy_(t)
  return moved


# one and two row tiles; one and two column tiles per wavefront; partial row and column
# tiles; reductions that end inside a group of 16 and are shorter than the loads ahead
@pytest.mark.parametrize("rows", [1, 3, 16, 17, 31])
@pytest.mark.parametrize("e,k,n", [(3, 16, 20), (2, 20, 16), (5, 52, 260), (2, 832, 132),
                                   (70, 192, 1000), (140, 100, 512)])
def test_float32_few_rows(hip, e, k, n, rows):
  """Fewer than 32 float32 rows per expert: products, masked ones and weight gradients
  have the bits of the kernel that takes operands off 16 bytes, which adds with one
  chain of multiply-adds; also where products underflow."""
  gen = torch.Generator(device="cuda").manual_seed(e + k + n + rows)
  mk = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
  for scale in (1.0, 2.0 ** -70):
    a, w, dy = mk(e, rows, k) * scale, mk(e, n, k) * scale, mk(e, rows, n) * scale
    for act in ("linear", "relu"):
      assert torch.equal(hip.expert_linear(a, w, act),
                         hip.expert_linear(_off_16(a), w, act))
    wt = w.transpose(1, 2).contiguous()
    mask = mk(e, rows, k)
    got = hip.expert_linear_backward(a, dy, wt, da_relu_mask=mask)
    want = hip.expert_linear_backward(_off_16(a), _off_16(dy), wt, da_relu_mask=mask)
    for g, x in zip(got, want):
      assert torch.equal(g, x)
    assert bool((got[0][mask <= 0] == 0).all())
  # (and they are the products: float32 sums of k and of the rows)
  a, w, dy = (t.double() for t in (a, w, dy))
  t = lambda x: x.transpose(1, 2).contiguous()
  y = hip.expert_linear(a.float(), w.float()).double()
  assert ((y - a @ t(w)).abs() <= k * 2.0 ** -24 * (a.abs() @ t(w).abs()) + 1e-43).all()
  dw = got[1].double()
  assert ((dw - t(a) @ dy).abs() <=
          rows * 2.0 ** -24 * (t(a).abs() @ dy.abs()) + 1e-43).all()


@pytest.mark.parametrize("k", [64, 128, 192, 448])
@pytest.mark.parametrize("e,rows,n", [(130, 129, 520), (200, 257, 520),
                                      (64, 260, 1024), (20, 290, 264), (9, 150, 264)])
def test_linear_three_token_slots(hip, e, rows, n, k):
  """Row tiles of 32 to 160 rows, whose token tiles have three slots: tiles of one
  to five pieces, last rows of a tile one and 97 to 129 rows in, fewer K tiles than
  slots, blocks with one tile and with several; with ReLU and with its mask."""
  _check_linear(hip, (e, rows, k, n), "relu")
  gen = torch.Generator(device="cuda").manual_seed(e + rows)
  dy, w, y = (torch.randn(s, generator=gen, device="cuda").to(torch.bfloat16)
              for s in ((e, rows, k), (e, n, k), (e, rows, n)))
  masked = hip.expert_linear_backward(y, dy, w, da_relu_mask=y)[0]
  assert torch.equal(masked, hip.expert_linear(dy, w) * (y > 0))


@pytest.mark.parametrize("e,g,c,h", [(32, 5, 128, 1024), (32, 5, 127, 1024),
                                     (16, 2, 128, 512)])
def test_gathered_rows_with_three_token_slots(hip, e, g, c, h):
  """The same tiles with rows fetched through the slot map: the bits of dispatch and
  two products."""
  s, m = 512, 1024
  gen = torch.Generator(device="cuda").manual_seed(g + c)
  mk = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
  r = hip.top2_gating(mk(g, s, e), c)
  x, wi, wo = (t.to(torch.bfloat16) for t in (mk(g, s, m), mk(e, h, m), mk(e, m, h)))
  got = hip.dispatched_expert_ffn(x, r, wi, wo, "relu")
  xe = hip.dispatch(x, r).reshape(e, g * c, m)
  assert torch.equal(got, hip.expert_ffn(xe, wi, wo, "relu"))


@pytest.mark.parametrize("e,g,c,outer", [(4, 6, 65, 2), (16, 40, 80, 8), (3, 12, 64, 4),
                                         (2, 4, 256, 1), (5, 9, 43, 3)])
def test_gathered_rows_of_kernels_per_part(hip, e, g, c, outer):
  """Several kernels per expert, each for a run of groups: the bits of dispatch and two
  products, rows that are dropped, empty or have a gate of zero among them."""
  s, m, h = 192, 256, 512
  gen = torch.Generator(device="cuda").manual_seed(g + c)
  mk = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
  importance = (mk(g, s) > -0.5).float()
  r = hip.top2_gating(mk(g, s, e), c, importance=importance)
  x, wi, wo = (t.to(torch.bfloat16) for t in (
      mk(g, s, m), mk(e * outer, h, m), mk(e * outer, m, h)))
  got = hip.dispatched_expert_ffn(x, r, wi, wo, "relu", outer=outer)
  xe = hip.dispatch(x, r).reshape(e * outer, g // outer * c, m)
  assert torch.equal(got, hip.expert_ffn(xe, wi, wo, "relu"))
  assert hip.dispatched_expert_ffn(x, r, wi, wo, "relu", outer=g + 1) is None


@pytest.mark.parametrize("c", [43, 64, 65, 700])
def test_gathered_rows_of_mostly_empty_slots(hip, c):
  """Experts without a token, with one and with as many as there are: every empty slot
  is known as one, whatever the map's memory held."""
  e, g, outer, s, m, h = 3, 6, 2, 96, 256, 512
  gen = torch.Generator(device="cuda").manual_seed(c)
  mk = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
  logits = mk(g, s, e) - 30.0 * torch.arange(e, device="cuda")
  importance = (mk(g, s) > 0).float()
  importance[1] = 0.0
  importance[2] = 0.0
  importance[2, 5] = 1.0
  r = hip.top2_gating(logits, c, importance=importance)
  x, wi, wo = (t.to(torch.bfloat16) for t in (
      mk(g, s, m), mk(e * outer, h, m), mk(e * outer, m, h)))
  xe = hip.dispatch(x, r).reshape(e * outer, g // outer * c, m)
  want = hip.expert_ffn(xe, wi, wo, "relu")
  for _ in range(2):
    # (memory that the call's workspace is likely to get)
    torch.full((1 << 20,), 7, dtype=torch.int32, device="cuda")
    assert torch.equal(hip.dispatched_expert_ffn(x, r, wi, wo, "relu", outer=outer),
                       want)


@pytest.mark.parametrize("shape", [(1, 4000, 264, 520), (1, 1025, 128, 256),
                                   (2, 6144, 776, 256), (29, 3000, 520, 760)],
                         ids=lambda s: "x".join(map(str, s)))
def test_weight_gradient_of_split_reductions(hip, shape):
  """Weight gradients whose last round of tiles is cut into parts along the
  reduction (few tiles, many rows; the last shape has whole tiles before the
  split ones; row counts that leave part of a K tile, edges of the output
  inside a tile).  The bound: one bf16 rounding, and for each of the two
  float32 sums of R products R / 2 ulps of the sum of magnitudes."""
  e, rows, k, n = shape
  gen = torch.Generator(device="cuda")
  gen.manual_seed(sum(shape))
  a, dy, w = (torch.randn(s, generator=gen, device="cuda").to(torch.bfloat16)
              for s in ((e, rows, k), (e, rows, n), (e, k, n)))
  dw = hip.expert_linear_backward(a, dy, w, want_da=False)[1]
  assert torch.equal(dw, hip.expert_linear_backward(a, dy, w, want_da=False)[1])
  for i in range(0, e, max(1, e // 3)):
    at = a[i].float().t().contiguous()
    want = at @ dy[i].float()
    magnitude = at.abs() @ dy[i].float().abs()
    bound = 2.0 ** -8 * want.abs() + rows * 2.0 ** -24 * magnitude
    assert bool(((dw[i].float() - want).abs() <= bound).all())


@pytest.mark.parametrize("shape", [
    # the width is cut into tiles of 32 (the last one 8), 64 (8), 96 (40), 128, 160
    # (104), 192, 224 and 256 rows
    (2, 64, 200, 136), (6, 200, 520, 776), (10, 200, 520, 776), (6, 70, 1000, 776),
    (90, 70, 264, 512), (16, 704, 768, 3072), (32, 160, 640, 1920),
    (64, 130, 1024, 1024)], ids=lambda s: "x".join(map(str, s)))
def test_weight_gradient_row_tiles(hip, shape):
  """Weight gradients whose output rows are spread over row tiles of 32 to 256.
  The bound: one bf16 rounding, and for each of the two float32 sums of R
  products R / 2 ulps of the sum of magnitudes."""
  e, rows, k, n = shape
  gen = torch.Generator(device="cuda")
  gen.manual_seed(sum(shape))
  a, dy, w = (torch.randn(s, generator=gen, device="cuda").to(torch.bfloat16)
              for s in ((e, rows, k), (e, rows, n), (e, k, n)))
  dw = hip.expert_linear_backward(a, dy, w, want_da=False)[1]
  for i in range(e):
    at = a[i].float().t().contiguous()
    want = at @ dy[i].float()
    magnitude = at.abs() @ dy[i].float().abs()
    bound = 2.0 ** -8 * want.abs() + rows * 2.0 ** -24 * magnitude
    assert bool(((dw[i].float() - want).abs() <= bound).all())


@pytest.mark.parametrize("k", [64, 128, 192, 256, 1024])
@pytest.mark.parametrize("e,rows,n", [(36, 300, 1288), (150, 130, 520),
                                      (3, 5376, 1536)])
def test_linear_tile_after_tile(hip, e, rows, n, k):
  """More tiles than compute units, so that blocks go from one to the next: with
  fewer K tiles than a block loads ahead, with rows and columns that end inside a
  tile (whose neighbours' rows must stay as they are), with the ReLU and with its
  mask.  The bound: one bf16 rounding, and for each of the two float32 sums of K
  products K / 2 ulps of the sum of magnitudes."""
  gen = torch.Generator(device="cuda")
  gen.manual_seed(e + rows + n + k)
  a, w, dy = (torch.randn(s, generator=gen, device="cuda").to(torch.bfloat16)
              for s in ((e, rows, k), (e, n, k), (e, rows, k)))
  y = hip.expert_linear(a, w, "relu")
  # dx = dy . v^T where y > 0, v [E, N, K]: the same product, masked
  v = w
  dx = hip.expert_linear_backward(y, dy, v, da_relu_mask=y)[0]
  for i in range(e):
    for got, lhs, keep in ((y, a, None), (dx, dy, y)):
      want = lhs[i].float() @ w[i].float().t().contiguous()
      magnitude = lhs[i].float().abs() @ w[i].float().abs().t().contiguous()
      want = want.clamp(min=0) if keep is None else want * (keep[i] > 0)
      bound = 2.0 ** -8 * want.abs() + k * 2.0 ** -24 * magnitude
      assert bool(((got[i].float() - want).abs() <= bound).all())


@pytest.mark.parametrize("rows", [1, 40, 64, 65, 128, 130, 192, 200])
@pytest.mark.parametrize("e,k,n", [(30, 264, 2568), (12, 1280, 1288)])
def test_weight_gradient_of_few_rows(hip, rows, e, k, n):
  """Reductions of one to four K tiles, more tiles than compute units; the bound as
  in the test above."""
  gen = torch.Generator(device="cuda")
  gen.manual_seed(rows + e)
  a, dy, w = (torch.randn(s, generator=gen, device="cuda").to(torch.bfloat16)
              for s in ((e, rows, k), (e, rows, n), (e, k, n)))
  dw = hip.expert_linear_backward(a, dy, w, want_da=False)[1]
  for i in range(e):
    at = a[i].float().t().contiguous()
    want = at @ dy[i].float()
    magnitude = at.abs() @ dy[i].float().abs()
    bound = 2.0 ** -8 * want.abs() + rows * 2.0 ** -24 * magnitude
    assert bool(((dw[i].float() - want).abs() <= bound).all())


@pytest.mark.parametrize("shape", [
    (8, 320, 2048, 512), (8, 320, 512, 2048), (2, 33, 36, 100), (1, 32, 32, 32),
    (1, 2000, 260, 1028), (40, 65, 68, 132), (3, 161, 1000, 64), (5, 97, 64, 300)],
    ids=lambda s: "x".join(map(str, s)))
def test_linear_float32_tiles(hip, shape):
  """The float32 kernel's block tiles, with their edges inside a tile and a last
  K tile that is partly there: products, with ReLU, with a gradient's ReLU mask
  on the stores, and weight gradients from rows as they lie.  The bound: K / 2
  ulps of the sum of magnitudes for a sum of K products."""
  e, rows, k, n = shape
  gen = torch.Generator(device="cuda")
  gen.manual_seed(sum(shape))
  a, dy, w = (torch.randn(s, generator=gen, device="cuda")
              for s in ((e, rows, n), (e, rows, k), (e, n, k)))

  def check(got, x, y, terms, keep=None):
    want = x.double() @ y.double()
    bound = terms * 2.0 ** -24 * (x.double().abs() @ y.double().abs())
    if keep is not None:
      want = want * keep
      assert not bool(got[~keep].any())
    assert bool(((got.double() - want).abs() <= bound).all())
  wt = w.transpose(1, 2)
  y = hip.expert_linear(dy, w)
  check(y, dy, wt, k)
  assert torch.equal(hip.expert_linear(dy, w, activation="relu"), y.clamp(min=0))
  da, dw = hip.expert_linear_backward(a, dy, w, da_relu_mask=a)
  check(da, dy, wt, k, a > 0)
  check(dw, a.transpose(1, 2), dy, rows)


@pytest.mark.parametrize("act_dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("shape", [(2, 256, 512, 128), (1, 100, 72, 40),
                                   (1, 4096, 1024, 256)],
                         ids=lambda s: "x".join(map(str, s)))
def test_expert_linear_backward_relu_mask(hip, shape, act_dtype):
  """da_relu_mask of mesh_moe_expert_linear_backward: da is the unmasked
  product with zeros wherever the mask is not positive, bit for bit, whether
  the mask rides on the GEMM's stores (bf16 shapes of the direct-to-LDS
  kernel) or is a pass of its own; dw is not touched."""
  e, rows, k, n = shape
  rng = np.random.default_rng(sum(shape))
  g = lambda a: H.to_gpu(O.cast_act(a.astype(np.float32), act_dtype), act_dtype)
  a = g(np.maximum(rng.standard_normal((e, rows, k)), 0))       # a = relu(...)
  w = g(H.normal_weights(rng, (e, k, n), k))
  dy = g(rng.standard_normal((e, rows, n)))
  da, dw = hip.expert_linear_backward(a, dy, w)
  da_m, dw_m = hip.expert_linear_backward(a, dy, w, da_relu_mask=a)
  assert torch.equal(dw, dw_m)
  assert torch.equal(da_m, da * (a > 0))
  assert float((a > 0).float().mean()) < 0.6 and da.abs().sum() > 0


@pytest.mark.parametrize("size", [(8, 512, 1024, 4096), (8, 2048, 4096, 16384)],
                         ids=["cfg3_slice", "cfg4_slice"])
def test_full_size_ffn_backward_properties(hip, size):
  """Eight experts of configurations 3 and 4 at their real (rows, M, H).  The
  weight gradients, which the library computes from operands with the reduction
  index outermost, equal bit for bit the same products taken through transposed
  copies and the row-major kernel (same K tiles, same order of summation);
  d(expert_in) and the masked dh are checked on sampled row blocks against
  float32 matmuls; an expert whose dy is zero gets zero gradients."""
  e, r, m, hdim = size
  gen = torch.Generator(device="cuda")
  gen.manual_seed(23)
  mk = lambda *s: torch.randn(s, generator=gen, device="cuda")
  xe = mk(e, r, m).to(torch.bfloat16)
  wi = (mk(e, m, hdim) / m ** 0.5).to(torch.bfloat16)
  wo = (mk(e, hdim, m) / hdim ** 0.5).to(torch.bfloat16)
  dy = mk(e, r, m).to(torch.bfloat16)
  dy[e // 2].zero_()
  wi_p = hip.pack_weights(wi, torch.bfloat16)
  h = hip.expert_linear(xe, wi_p, "relu")
  dxe, dwi, dwo = hip.expert_ffn_backward(xe, h, dy, wi, wo, "relu")
  for t in (dxe, dwi, dwo):
    assert bool(torch.isfinite(t.float()).all())
  # dwo = h^T . dy through transposed copies
  tr = lambda a: hip.pack_weights(a, torch.bfloat16)       # [E, R, X] -> [E, X, R]
  assert torch.equal(dwo, hip.expert_linear(tr(h), tr(dy), "linear"))
  # dh on sampled rows, then dwi from the library's own dh via the same route
  for ei, r0 in ((0, 0), (e - 1, r - 64), (e // 2 + 1, r // 2 - 13)):
    dh_ref = (dy[ei, r0:r0 + 64].float() @ wo[ei].float().t()).to(torch.bfloat16)
    dh_ref = dh_ref.float() * (h[ei, r0:r0 + 64] > 0)
    dxe_ref = dh_ref @ wi[ei].float().t()
    err = (dxe[ei, r0:r0 + 64].float() - dxe_ref).abs().max().item()
    scale = dxe_ref.abs().max().item()
    assert err <= 2e-2 * scale, (ei, r0, err, scale)
  dh = (torch.bmm(dy.float()[:2], wo.float()[:2].transpose(1, 2)).to(torch.bfloat16)
        .float() * (h[:2] > 0)).to(torch.bfloat16)
  want_dwi = hip.expert_linear(tr(xe[:2].contiguous()), tr(dh), "linear")
  err = (dwi[:2].float() - want_dwi.float()).abs().max().item()
  assert err <= 2e-2 * want_dwi.float().abs().max().item()
  assert not bool(dwo[e // 2].any()) and not bool(dwi[e // 2].any())
  assert not bool(dxe[e // 2].any())


@pytest.mark.parametrize("act_dtype", ["float32", "bfloat16"])
def test_expert_linear_backward_and_activations(hip, act_dtype):
  """mesh_moe_expert_linear_backward against float32 matmuls, and
  mesh_moe_activation / mesh_moe_activation_backward against the oracle's
  activation tables for every activation."""
  e, rows, k, n = 2, 192, 136, 264
  rng = np.random.default_rng(29)
  cast = lambda a: O.cast_act(a.astype(np.float32), act_dtype)
  g = lambda a: H.to_gpu(a, act_dtype)
  a = cast(rng.standard_normal((e, rows, k)))
  w = cast(H.normal_weights(rng, (e, k, n), k))
  dy = cast(rng.standard_normal((e, rows, n)))
  da, dw = hip.expert_linear_backward(g(a), g(dy), g(w))
  tol = H.value_tolerance(act_dtype)
  want_da = np.matmul(dy, w.transpose(0, 2, 1))
  want_dw = np.matmul(a.transpose(0, 2, 1), dy)
  for got, want, name in ((da, want_da, "da"), (dw, want_dw, "dw")):
    np.testing.assert_allclose(H.to_np(got), O.cast_act(want, act_dtype),
                               rtol=tol["rtol"],
                               atol=tol["atol"] * np.abs(want).max(), err_msg=name)
  none, dw2 = hip.expert_linear_backward(g(a), g(dy), g(w), want_da=False)
  assert none is None and torch.equal(dw2, dw)
  pre = cast(rng.standard_normal((e, rows, n)) * 2.0)
  f = cast(rng.standard_normal((e, rows, n)))
  for act in ("relu", "linear", "gelu", "sigmoid", "tanh", "swish"):
    out = hip.activation(g(pre), act)
    np.testing.assert_allclose(
        H.to_np(out), O.cast_act(O.ACTIVATIONS[act](pre), act_dtype),
        rtol=1e-2 if act_dtype == "bfloat16" else 1e-5, atol=1e-6, err_msg=act)
    # same values as the activation applied inside the projection
    assert torch.equal(out, hip.activation(g(pre), act))
    for factor in (None, f):
      got = hip.activation_backward(g(dy), g(pre), act, factor=None if factor
                                    is None else g(factor))
      want = dy * (1.0 if factor is None else factor) * O.ACTIVATION_GRADS[act](pre)
      np.testing.assert_allclose(
          H.to_np(got), O.cast_act(want.astype(np.float32), act_dtype),
          rtol=2e-2 if act_dtype == "bfloat16" else 1e-4,
          atol=(2e-2 if act_dtype == "bfloat16" else 1e-5) * np.abs(want).max(),
          err_msg=act)
  with pytest.raises(ValueError):
    hip.activation(g(pre), "softplus")


@pytest.mark.parametrize("act_dtype", ["float32", "bfloat16"])
def test_expert_choice_backward_stages(hip, act_dtype):
  """The three backward entry points of the per-slot record against the
  oracle: combine backward, dispatch backward (with and without the router's
  share), and d(logits) of the gating (importance 0 / 0.5 / 1, two
  microbatches)."""
  g, s, e, c, m = 3, 96, 6, 20, 40
  rng = np.random.default_rng(13)
  logits = (rng.standard_normal((g, s, e)) * 1.5).astype(np.float32)
  imp = rng.choice([0.0, 0.5, 1.0], size=(g, s), p=[0.15, 0.15, 0.7]).astype(np.float32)
  want_r = O.expert_selection_gating(logits, c, imp, num_microbatches=2)
  lg = torch.from_numpy(logits).cuda()
  r = hip.expert_choice_gating(lg, c, importance=H.to_gpu(imp), num_microbatches=2)
  assert np.array_equal(H.to_np(r.slot_token), want_r["slot_token"])
  r_np = dict(slot_token=want_r["slot_token"], slot_weight=H.to_np(r.slot_weight))
  cast = lambda a: O.cast_act(a.astype(np.float32), act_dtype)
  tol = H.value_tolerance(act_dtype)
  dout, y = cast(rng.standard_normal((g, s, m))), cast(rng.standard_normal((e, g, c, m)))
  dy, dw = hip.slot_combine_backward(H.to_gpu(dout, act_dtype),
                                     H.to_gpu(y, act_dtype), r)
  want_dy, want_dw = O.slot_combine_backward(dout, y, r_np, act_dtype)
  np.testing.assert_allclose(H.to_np(dy), want_dy, **tol)
  np.testing.assert_allclose(H.to_np(dw), want_dw, rtol=1e-4, atol=1e-4)
  dxe = cast(rng.standard_normal((e, g, c, m)))
  dx = hip.slot_dispatch_backward(H.to_gpu(dxe, act_dtype), r, s)
  want_dx = O.slot_dispatch_backward(dxe, r_np, s)
  np.testing.assert_allclose(H.to_np(dx), O.cast_act(want_dx, act_dtype),
                             rtol=tol["rtol"], atol=tol["atol"] * 4)
  held = np.zeros((g, s), bool)
  for gi in range(g):
    held[gi][want_r["slot_token"][gi].reshape(-1)] = True
  assert (~held).any() and (H.to_np(dx)[~held] == 0).all()
  dweight = rng.standard_normal((g, e, c)).astype(np.float32)
  want_dl = O.expert_selection_gating_backward(logits, r_np, imp, dweight, 0.7, 2)
  assert np.abs(want_dl).max() > 0
  dl = hip.expert_choice_backward(
      lg, r, torch.from_numpy(dweight).cuda(),
      torch.tensor([0.7], dtype=torch.float32, device="cuda"), 1.0,
      importance=H.to_gpu(imp), num_microbatches=2)
  np.testing.assert_allclose(H.to_np(dl), want_dl, rtol=1e-3,
                             atol=1e-5 * np.abs(want_dl).max())
  assert (H.to_np(dl)[imp == 0] == 0).all()          # masked tokens: p = 0
  # with the router's share
  wg = cast(H.normal_weights(rng, (m, e), m))
  wg_p = hip.pack_weights(H.to_gpu(wg, act_dtype).reshape(1, m, e),
                          H.ACT_TORCH[act_dtype]).reshape(e, m)
  dx2 = hip.slot_dispatch_backward(H.to_gpu(dxe, act_dtype), r, s, dl, wg_p)
  want2 = want_dx + np.matmul(H.to_np(dl), wg.T)
  np.testing.assert_allclose(H.to_np(dx2), O.cast_act(want2, act_dtype),
                             rtol=tol["rtol"], atol=tol["atol"] * 4)


@pytest.mark.parametrize("shape", [(2, 64, 16, 12, 512), (2, 128, 64, 5, 1024)],
                         ids=lambda s: "x".join(map(str, s)))
def test_expert_choice_backward_wide_rows(hip, shape):
  """The per-slot backward calls at row lengths their 16-byte and matrix-core
  kernels take (bf16): combine backward against the oracle; dispatch backward
  with the router's share on the matrix cores against float64 sums rounded
  once and against the call without the router kernel in its variable
  layout."""
  g, s, e, c, m = shape
  rng = np.random.default_rng(19)
  logits = (rng.standard_normal((g, s, e)) * 1.5).astype(np.float32)
  r = hip.expert_choice_gating(torch.from_numpy(logits).cuda(), c)
  r_np = dict(slot_token=r.slot_token.cpu().numpy(),
              slot_weight=H.to_np(r.slot_weight))
  cast = lambda a: O.cast_act(a.astype(np.float32), "bfloat16")
  tol = H.value_tolerance("bfloat16")
  dout, y = cast(rng.standard_normal((g, s, m))), cast(rng.standard_normal((e, g, c, m)))
  dy, dw = hip.slot_combine_backward(H.to_gpu(dout, "bfloat16"),
                                     H.to_gpu(y, "bfloat16"), r)
  want_dy, want_dw = O.slot_combine_backward(dout, y, r_np, "bfloat16")
  np.testing.assert_allclose(H.to_np(dy), want_dy, **tol)
  np.testing.assert_allclose(H.to_np(dw), want_dw, rtol=1e-4, atol=1e-3)
  dxe = cast(rng.standard_normal((e, g, c, m)))
  dl = (rng.standard_normal((g, s, e)) * 2.0).astype(np.float32)
  wg = cast(H.normal_weights(rng, (m, e), m))
  wg_g = H.to_gpu(wg, "bfloat16")
  wg_p = hip.pack_weights(wg_g.reshape(1, m, e), torch.bfloat16).reshape(e, m)
  dl_g = torch.from_numpy(dl).cuda()
  got = hip.slot_dispatch_backward(H.to_gpu(dxe, "bfloat16"), r, s, dl_g, wg_p,
                                   w_gate=wg_g)
  plain = hip.slot_dispatch_backward(H.to_gpu(dxe, "bfloat16"), r, s, dl_g, wg_p)
  want = (O.slot_dispatch_backward(dxe, r_np, s).astype(np.float64) +
          np.matmul(dl.astype(np.float64), wg.astype(np.float64).T))
  held = np.zeros((g, s), bool)
  for gi in range(g):
    held[gi][r_np["slot_token"][gi].reshape(-1)] = True
  assert held.any() and (~held).any()
  err = np.abs(H.to_np(got).astype(np.float64) - want)
  assert (err <= np.abs(want) * 2.0 ** -8 * 1.01 + 4e-5).all()
  step = np.abs(H.to_np(got) - H.to_np(plain))
  assert (step <= np.abs(H.to_np(plain)) * 2.0 ** -7 + 4e-5).all()


def test_dropout_noise_from_the_relu_mask(hip):
  """Backward of ReLU experts behind a hidden dropout: told the keep
  probability, the library takes the noise from the stored activation (kept
  where it is positive, 1 / keep_prob there) while the dh GEMM writes its
  tiles; told nothing it reads the noise tensor in a pass of its own.  Same
  bits either way, padded and compacted rows."""
  e, g, c, m, hdim, keep = 4, 2, 256, 256, 512, 0.75
  dt = torch.bfloat16
  gen = torch.Generator(device="cuda").manual_seed(77)
  mk = lambda *sh: torch.randn(sh, generator=gen, device="cuda")
  xe = mk(e, g * c, m).to(dt)
  wi = (mk(e, m, hdim) / m ** 0.5).to(dt)
  wo = (mk(e, hdim, m) / hdim ** 0.5).to(dt)
  dy = mk(e, g * c, m).to(dt)
  h = hip.expert_linear(xe, hip.pack_weights(wi, dt), "relu")
  u = torch.rand(h.shape, generator=gen, device="cuda").to(dt)
  noise = hip.hidden_product(h, uniform=u, keep_prob=keep, want_noise=True)
  assert 0.2 < float((noise == 0).float().mean()) < 0.3
  a = hip.expert_ffn_backward(xe, h, dy, wi, wo, "relu", dh_scale=noise,
                              keep_prob=keep)
  b = hip.expert_ffn_backward(xe, h, dy, wi, wo, "relu", dh_scale=noise)
  # (the noise tensor itself is then not needed)
  c_ = hip.expert_ffn_backward(xe, h, dy, wi, wo, "relu", keep_prob=keep)
  for x_, y_, z_ in zip(a, b, c_):
    assert torch.equal(x_, y_) and torch.equal(x_, z_)
  assert float(a[0].abs().sum()) > 0
  # float32, and rows the matrix-core kernels do not take: the same through
  # the element-wise pass
  f = lambda t: t[:, :40].float().contiguous()
  h32 = hip.expert_linear(f(xe), hip.pack_weights(wi.float(), torch.float32),
                          "relu")
  n32 = hip.hidden_product(h32, uniform=f(u.float().reshape(e, g * c, hdim)),
                           keep_prob=keep, want_noise=True)
  a32 = hip.expert_ffn_backward(f(xe), h32, f(dy), wi.float(), wo.float(),
                                "relu", dh_scale=n32)
  c32 = hip.expert_ffn_backward(f(xe), h32, f(dy), wi.float(), wo.float(),
                                "relu", keep_prob=keep)
  for x_, z_ in zip(a32, c32):
    assert torch.equal(x_, z_)
  # compacted rows: a switch routing that fills about half of the slots
  s = 1024
  r = hip.switch_gating(mk(g, s, e), c)
  xg = mk(g, s, m).to(dt)
  wi_p, wo_p = hip.pack_weights(wi, dt), hip.pack_weights(wo, dt)
  uc = torch.rand((e, g * c, hdim), generator=gen, device="cuda").to(dt)
  y_c, ro, h_c, noise_c = hip.compact_expert_ffn(
      xg, r, wi_p, wo_p, "relu", want_hidden=True, uniform=uc, keep_prob=keep,
      want_noise=True)
  xe_c = hip.dispatch(xg, r, row_offsets=ro).reshape(e, g * c, m)
  dy_c, _ = hip.combine_backward(mk(g, s, m).to(dt), y_c.reshape(e, g, c, m), r,
                                 row_offsets=ro)
  dy_c = dy_c.reshape(e, g * c, m)
  a = hip.compact_expert_ffn_backward(xe_c, h_c, dy_c, wi, wo, r, ro, "relu",
                                      dh_scale=noise_c, keep_prob=keep)
  b = hip.compact_expert_ffn_backward(xe_c, h_c, dy_c, wi, wo, r, ro, "relu",
                                      dh_scale=noise_c)
  fill = r.fill.cpu().numpy()
  used = fill.sum(0)
  for j, (x_, y_) in enumerate(zip(a, b)):
    if j == 0:      # d(expert_in): the occupied rows (the rest is unspecified)
      for ei in range(e):
        assert torch.equal(x_[ei, :used[ei]], y_[ei, :used[ei]]), ei
    else:
      assert torch.equal(x_, y_), j
  # a keep probability outside [0, 1] is refused by name, not taken for
  # "unknown"
  for bad in (-0.25, 1.5):
    with pytest.raises(Exception, match="dh_keep_prob"):
      hip.expert_ffn_backward(xe, h, dy, wi, wo, "relu", keep_prob=bad)
    with pytest.raises(Exception, match="dh_keep_prob"):
      hip.compact_expert_ffn_backward(xe_c, h_c, dy_c, wi, wo, r, ro, "relu",
                                      keep_prob=bad)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("g,s,n", [(1, 1, 8), (2, 130, 72), (3, 64, 20)])
def test_combine_with_loss(hip, dtype, g, s, n):
  """The layer's loss on the way out: the bits of a cast and a scalar product."""
  e, c = 6, 40
  gen = torch.Generator(device="cuda").manual_seed(s + n)
  logits = torch.randn((g, s, e), generator=gen, device="cuda")
  r = hip.top2_gating(logits, c)
  y = torch.randn((e, g, c, n), generator=gen, device="cuda").to(dtype)
  coef = torch.tensor(1e-2, dtype=dtype).item()
  out, loss, scaled = hip.combine(y, r, s, loss_coef=coef)
  assert torch.equal(out, hip.combine(y, r, s))
  want = r.loss.to(dtype).reshape(())
  assert torch.equal(loss, want) and torch.equal(scaled, want * coef)
