"""The workloads that this package is timed on: passes through its public entry
points (the Mixture-of-Experts layers, the transformer block around them, the
decoding step) with inputs that are already on the GPU, as a program that
serves or trains a model has them.

A case is a dict of plain values:

  kind       "layer" (transformer_moe_layer_v1), "hierarchical"
             (transformer_moe_layer_v2), "block" (a LayerStack with attention,
             experts and dense layers over whole sequences) or "decode" (the
             same stack, one position per sequence on the recurrent states)
  dtype      "bf16" or "f32": activations, and the dtype of the variables
  batch, length   sequences and positions (for "decode": of the memory)
  d_model, d_ff   model width; hidden width of the experts and dense layers
  experts    number of experts ("hierarchical": of both levels together,
             experts_outer groups of them)
  group, capacity_factor   the layer's group size and capacity factor
  gating     "top_2", "switch", "switch_max", "ntlb", "expert_selection"
  skewed     the router prefers some experts (Zipf s = 1.2 rank profile scaled
             to 3.0 on its logits), so that many tokens find no slot
  padded     sequences of unequal length ("layer": nonpadding; "block":
             sequence ids, several sequences in a row and padding at its end)
  train      training mode, and the pass returns the gradients of the tokens
             and of every variable too
  graph      the step is recorded once (Lowering.capture) and replayed
  d_kv, relative   attention head width; the shared relative position bias

The numbers are those of the benchmark's five layer configurations and of the
tests around them, and widths that follow from them.
"""

import math

import torch

import mesh_amd as mtf
from mesh_amd.transformer import moe, transformer, transformer_layers

# The residual stream a block gets in the middle of a deep stack: what a layer
# adds to it is small beside it.
STREAM_RMS = 8.0


def _layer(name, **kw):
  case = dict(name=name, kind="layer", dtype="bf16", gating="top_2",
              skewed=False, padded=False, train=False, graph=False)
  case.update(kw)
  return case


def _block(name, kind, **kw):
  case = dict(name=name, kind=kind, dtype="bf16", gating="top_2", padded=False,
              train=False, graph=False, relative=False, d_kv=128)
  case.update(kw)
  return case


def listed():
  return [
      # The benchmark's float32 configuration: a small model, or a big one
      # while it is being debugged.
      _layer("layer_f32_2k", dtype="f32", batch=2, length=1024, group=1024,
             d_model=512, d_ff=2048, experts=8, capacity_factor=1.25),
      # The same layer in training: forward, loss and all gradients.
      _layer("layer_f32_2k_train", dtype="f32", batch=2, length=1024,
             group=1024, d_model=512, d_ff=2048, experts=8,
             capacity_factor=1.25, train=True),
      # One layer of a decoding step of 64 sequences, recorded as a graph: every
      # expert's weights are read for a few rows.
      _layer("layer_64_graph", batch=64, length=1, group=1024, d_model=1024,
             d_ff=4096, experts=64, capacity_factor=2.0, graph=True),
      # An ordinary batch through an ordinary layer.
      _layer("layer_16k", batch=16, length=1024, group=1024, d_model=1024,
             d_ff=4096, experts=32, capacity_factor=1.25),
      # A router that overloads some experts: drops, and empty slots elsewhere.
      _layer("layer_skewed_32k", batch=16, length=2048, group=2048,
             d_model=1024, d_ff=4096, experts=64, capacity_factor=1.0,
             skewed=True),
      # The largest layer: 17 GB of weights, 65536 tokens.
      _layer("layer_64k", batch=32, length=2048, group=2048, d_model=4096,
             d_ff=16384, experts=64, capacity_factor=2.0),
      # Two-level gating over 8 x 16 experts.
      dict(name="hierarchical_32k", kind="hierarchical", dtype="bf16",
           gating="top_2", batch=32, length=1024, group=1024, d_model=2048,
           d_ff=8192, experts=128, experts_outer=8, capacity_factor=1.25,
           padded=False, train=False, graph=False),
      # Fine-tuning on texts of odd lengths: six sequences of up to 1500
      # tokens, padding masked out of the routing.
      _layer("layer_ragged_train", batch=6, length=1500, group=1500,
             d_model=768, d_ff=3072, experts=16, capacity_factor=1.25,
             padded=True, train=True),
      # Pre-training with one choice per token.
      _layer("layer_switch_32k_train", batch=32, length=1024, group=1024,
             d_model=1024, d_ff=4096, experts=64, capacity_factor=1.25,
             gating="switch", train=True),
      # A block (attention, experts, attention, dense layers) over whole
      # prompts.
      _block("block_prefill", "block", batch=8, length=2048, group=2048,
             d_model=1024, d_ff=4096, experts=32, capacity_factor=2.0),
      # A block in training on packed rows, with the relative position bias.
      _block("block_packed_train", "block", batch=16, length=1000, group=1000,
             d_model=768, d_ff=3072, experts=16, capacity_factor=1.25, d_kv=64,
             padded=True, relative=True, train=True),
      # One token for each of 32 sequences on their recurrent states.
      _block("block_decode", "decode", batch=32, length=1024, group=1024,
             d_model=1024, d_ff=4096, experts=32, capacity_factor=2.0),
  ]


def _log_int(rng, low, high):
  return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw(rng):
  kind = rng.choices(["layer", "block", "decode", "hierarchical"],
                     [6, 3, 2, 1])[0]
  train = kind != "decode" and rng.random() < 0.4
  case = dict(kind=kind, dtype="bf16", gating="top_2", train=train,
              graph=False, padded=False,
              capacity_factor=rng.choice([1.0, 1.25, 1.5, 2.0]))
  if kind == "layer":
    small = rng.random() < 0.25
    if small:
      case["dtype"] = "f32"
    case["gating"] = rng.choices(
        ["top_2", "switch", "switch_max", "ntlb", "expert_selection"],
        [8, 3, 1, 1, 1])[0]
    tokens = _log_int(rng, 64, 4096 if small else 32768)
    case["batch"] = rng.randint(1, min(16, tokens))
    case["length"] = min(2048, tokens // case["batch"])
    case["d_model"] = 64 * _log_int(rng, 4 if small else 8, 16 if small else 32)
    case["experts"] = rng.choice([8, 12, 16, 24, 32, 48, 64])
    case["skewed"] = case["gating"] == "top_2" and rng.random() < 0.25
    # the balancing loss of expert selection needs to know the padding
    case["padded"] = (case["gating"] == "expert_selection" or
                      rng.random() < 0.25)
    case["graph"] = not train and tokens <= 1024
  elif kind == "hierarchical":
    case["batch"] = rng.randint(2, 16)
    case["length"] = 4 * _log_int(rng, 32, 256)
    case["d_model"] = 128 * rng.randint(4, 16)
    case["experts_outer"] = rng.choice([2, 4, 8])
    case["experts"] = case["experts_outer"] * rng.choice([4, 8, 16])
  else:
    case["d_kv"] = rng.choice([64, 128])
    case["d_model"] = 128 * rng.randint(4, 12)
    case["experts"] = rng.choice([8, 16, 32])
    case["relative"] = rng.random() < 0.3
    if kind == "decode":
      case["batch"] = _log_int(rng, 1, 64)
      case["length"] = _log_int(rng, 64, 2048)
    else:
      case["batch"] = rng.randint(1, 12)
      case["length"] = _log_int(rng, 100, 2048)
      case["padded"] = rng.random() < 0.4
  case["group"] = max(256, case["length"])
  case["d_ff"] = case["d_model"] * rng.choice([2, 3, 4])
  return case


def draw(rng):
  """One more case of the same ranges, without a name; never more work than
  the largest of the listed ones."""
  most = max(work(c)["flops"] for c in listed())
  while True:
    case = _draw(rng)
    if work(case)["flops"] <= most:
      return case


# ---------------------------------------------------------------------------
# the program around the pass
# ---------------------------------------------------------------------------
def _torch_dtype(case):
  return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _normal(gen, sizes, std, dtype):
  """N(0, std), drawn a leading index at a time: the largest variable never
  needs a float32 temporary of its full size."""
  out = torch.empty(sizes, dtype=dtype, device="cuda")
  flat = out.reshape(sizes[0], -1) if len(sizes) > 2 else out.reshape(1, -1)
  for i in range(flat.shape[0]):
    flat[i] = torch.randn(flat.shape[1], generator=gen, device="cuda") * std
  return out


def _initial_values(case, graph, gen):
  """Values for every variable: kernels N(0, 1 / fan_in), queries with the
  1 / sqrt(d_kv) scaling folded in, norm scales near 1."""
  init = {}
  for v in graph.all_variables:
    sizes = v.shape.to_integer_list
    if v.name.endswith("/scale"):
      value = 1.0 + _normal(gen, sizes, 0.1, torch.float32)
    elif v.name.endswith("relative_attention_bias"):
      value = _normal(gen, sizes, 0.5, torch.float32)
    else:
      std = sizes[-2] ** -0.5
      if v.name.endswith("/q"):
        std *= case["d_kv"] ** -0.5
      value = _normal(gen, sizes, std, _torch_dtype(case))
    if case.get("skewed") and v.name.endswith("_gating/kernel"):
      # row 0 multiplies a feature that is 1 in every token
      ranks = torch.randperm(sizes[-1], generator=gen, device="cuda") + 1
      value[0] = (3.0 * ranks.double() ** -1.2).to(value.dtype)
    init[v.name] = value
  return init


def _sequence_lengths(case, gen):
  """Between half and all of the positions are filled."""
  least = max(1, case["length"] // 2)
  return torch.randint(least, case["length"] + 1, (case["batch"], 1),
                       generator=gen, device="cuda")


def _sequence_ids(case, gen):
  """Two sequences packed into a row, then padding (id 0)."""
  total = _sequence_lengths(case, gen)
  first = (total * torch.rand((case["batch"], 1), generator=gen,
                              device="cuda")).long()
  at = torch.arange(case["length"], device="cuda")[None]
  return ((at < total).int() + ((at >= first) & (at < total)).int()).contiguous()


def _hparams(case):
  experts = case["experts"]
  if case["kind"] == "hierarchical":
    experts = [case["experts_outer"], experts // case["experts_outer"]]
  hp = moe.HParams()
  moe.set_default_moe_hparams(hp)
  for key, value in dict(
      num_experts=experts, gating=case["gating"], hidden_size=case["d_ff"],
      group_size=case["group"], min_expert_capacity=4,
      capacity_factor_train=case["capacity_factor"],
      capacity_factor_eval=case["capacity_factor"],
      capacity_factor_second_level=case["capacity_factor"],
      second_policy_train="all", second_policy_eval="all", dropout_rate=0.0,
      use_experts_attention=False, ntlb_top_k=4, z_loss=None,
      switch_policy_train="argmax", switch_policy_eval="argmax").items():
    setattr(hp, "moe_" + key, value)
  return hp


def _stack(case):
  """Attention, experts, attention, dense layers.  In training the experts
  come first: what their router sees then does not hang on the order of sums
  in a layer before it, so every correct implementation routes alike."""
  attention = (transformer_layers.SelfAttention, dict(
      num_heads=case["d_model"] // case["d_kv"], key_value_size=case["d_kv"],
      relative_attention_type="bias_shared" if case["relative"] else None))
  experts = (moe.MoE1D, dict(
      num_experts=case["experts"], hidden_size=case["d_ff"],
      group_size=case["group"], capacity_factor_train=case["capacity_factor"],
      capacity_factor_eval=case["capacity_factor"],
      second_policy_train="all", second_policy_eval="all"))
  dense = (transformer_layers.DenseReluDense, dict(hidden_size=case["d_ff"]))
  layers = ([experts, attention, dense] if case["train"]
            else [attention, experts, attention, dense])
  stack = transformer.make_layer_stack(layers, num_layers=1, block_scope=False)
  return transformer.Unitransformer(stack, d_model=case["d_model"],
                                    name="decoder", autoregressive=True)


class _Program(object):
  """A graph on the GPU and the tensors that one pass feeds to it."""

  def __init__(self):
    self.graph = mtf.Graph()
    self.mesh = mtf.Mesh(self.graph, "mesh")
    self.feeds = {}
    self.outputs = []
    self.lowering = None
    self.step = None

  def feed(self, value, dims):
    tensor = mtf.import_tf_tensor(self.mesh, value, mtf.Shape(dims))
    self.feeds[tensor] = value
    return tensor


def prepare(case, seed):
  dt = _torch_dtype(case)
  gen = torch.Generator(device="cuda")
  gen.manual_seed(seed)
  b, l, m = case["batch"], case["length"], case["d_model"]
  program = _Program()
  batch, length, model = (mtf.Dimension("batch", b), mtf.Dimension("length", l),
                          mtf.Dimension("d_model", m))
  vdt = mtf.VariableDType(dt, dt, dt)
  decode = case["kind"] == "decode"
  in_stack = case["kind"] in ("block", "decode")
  value = _normal(gen, [b, m] if decode else [b, l, m],
                  STREAM_RMS if in_stack else 1.0, dt)
  if case.get("skewed"):
    value[..., 0] = 1.0
  x = program.feed(value, [batch, model] if decode else [batch, length, model])
  if in_stack:
    network = _stack(case)
    if decode:
      heads = mtf.Dimension("heads", m // case["d_kv"] * case["d_kv"])
      memory = mtf.Dimension("memory_length", l)
      states = [program.feed(_normal(gen, [b, l, heads.size], 1.0, dt),
                             [batch, memory, heads]) for _ in range(4)]
      position = torch.randint(l // 2, l, (b,), generator=gen, device="cuda",
                               dtype=torch.int32)
      position = program.feed(position, [batch])
      new_states = []
      # (the variables are created here: no earlier call of the network)
      y, losses = network.call_layers(
          x, vdt, mode="incremental", position=position, states=states,
          new_states=new_states, length_dim=length, reuse=False)
      program.outputs = [y] + new_states
    else:
      ids = None
      if case["padded"]:
        ids = program.feed(_sequence_ids(case, gen), [batch, length])
      y, losses = network.call_layers(
          x, vdt, mode="train" if case["train"] else "eval", sequence_id=ids)
      program.outputs = [y] + losses
  else:
    nonpadding = None
    if case["padded"]:
      at = torch.arange(l, device="cuda")[None]
      nonpadding = program.feed((at < _sequence_lengths(case, gen)).to(dt),
                                [batch, length])
    layer = (moe.transformer_moe_layer_v2 if case["kind"] == "hierarchical"
             else moe.transformer_moe_layer_v1)
    with mtf.variable_scope("moe"):
      y, loss = layer(x, model, _hparams(case), case["train"], vdt,
                      nonpadding=nonpadding, num_microbatches=1)
    losses = [loss]
    program.outputs = [y, loss]
  if case["train"]:
    dy = program.feed(_normal(gen, [b, l, m], 1.0, dt), [batch, length, model])
    wrt = [x] + [v.outputs[0] for v in program.graph.trainable_variables]
    program.outputs = program.outputs + mtf.gradients(
        [y] + losses, wrt, grad_ys=[dy] + [None] * len(losses))
  program.lowering = mtf.Lowering(
      program.graph, {program.mesh: mtf.HipMeshImpl()},
      initial_values=_initial_values(case, program.graph, gen))
  if case["graph"]:
    program.step = program.lowering.capture()
  return program


def run(program):
  if program.step is not None:
    program.step.replay(program.feeds)
  else:
    program.lowering.run(program.feeds)
  return [program.lowering.export_to_tf_tensor(t) for t in program.outputs]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _experts_work(case, tokens, size):
  """(weights read, flops forward) of one Mixture-of-Experts layer."""
  m, h = case["d_model"], case["d_ff"]
  choices = {"top_2": 2, "expert_selection": case["capacity_factor"]}.get(
      case["gating"], 1)
  # slots of the layer: capacity per expert and group, and no fewer than 4
  groups = max(1, tokens // case["group"])
  slots = max(tokens * case["capacity_factor"], 4 * case["experts"] * groups)
  rows = min(choices * tokens, slots)
  if case["kind"] == "hierarchical":
    # one choice in the second-choice group, two in the first
    rows = min(3 * tokens, slots * case["capacity_factor"])
  # an expert that no token chose need not be read
  used = case["experts"] * (1 - (1 - 1 / case["experts"]) ** rows)
  routers = m * case["experts"]
  return (size * (2 * used * m * h + routers),
          4 * rows * m * h + 2 * tokens * routers)


def work(case):
  size = 2 if case["dtype"] == "bf16" else 4
  m, h = case["d_model"], case["d_ff"]
  b, l = case["batch"], case["length"]
  decode = case["kind"] == "decode"
  tokens = b if decode else b * l
  weights, flops = _experts_work(case, tokens, size)
  data = 2 * size * tokens * m
  if case["kind"] in ("block", "decode"):
    width = m // case["d_kv"] * case["d_kv"]
    attentions = 1 if case["train"] else 2
    weights += size * (attentions * 4 * m * width + 2 * m * h)
    flops += 2 * tokens * (attentions * 4 * m * width + 2 * m * h)
    # q . k and weights . v over the positions that are seen
    seen = 3 * l / 4 if decode else l / 2
    scores = 4 * tokens * seen * width * attentions
    if decode:
      # the states come in and go out whole
      data += 2 * attentions * 2 * size * b * l * width
  else:
    scores = 0
  if case["train"]:
    # gradients of both operands of every product; the attention backward
    # has five products to the forward's two
    return {"bytes": 2 * weights + 2 * data, "flops": 3 * flops + 3.5 * scores}
  return {"bytes": weights + data, "flops": flops + scores}


def tolerance(case):
  """About four times what the outputs moved, over the listed cases and a
  hundred drawn ones, when every sum over features was taken in another order
  (the features of inputs and variables permuted).  The largest single
  differences in training are weight gradients at a hidden unit whose
  pre-activation is 0 up to rounding: the unit is on in one order and off in
  the other."""
  if case["dtype"] == "f32":          # seen: 1.4e-6, largest 2.9e-5
    return {"rel": 5e-6, "max": 1.2e-4}
  stack = case["kind"] in ("block", "decode")
  if case["train"]:                   # seen: 1.5e-2 and 1.1e-3, largest 0.62
    return {"rel": 3e-2 if stack else 4.5e-3, "max": 0.99}
  if stack:                           # seen: 1.4e-3, largest 0.16
    return {"rel": 6e-3, "max": 0.6}
  return {"rel": 1.5e-3, "max": 0.1}  # seen: 3.5e-4, largest 2.4e-2
