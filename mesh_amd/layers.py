"""Dense layers as the Mixture-of-Experts layers and the transformer block
around them use them.

Mirrors the part of mesh_tensorflow/layers.py those paths touch:
get_dense_kernel_weights (layers.py:211-253: variable `<name>/kernel` of shape
expert_dims + reduced_dims + new_dims), VarianceScalingInitializer
(layers.py:310-369: truncated normal with stddev sqrt(scale / fan_in)), and
dense / dense_product without bias (layers.py:112-160, :256-295).  The MoE
operations consume their variables directly.
"""

import torch

from mesh_amd import ops as mtf


class DenseInitializer(object):
  """Initializer that is told (reduced_dims, new_dims) first."""

  def __call__(self, reduced_dims, new_dims):
    raise NotImplementedError("not implemented")


def truncated_normal_initializer(stddev=1.0, seed=None):
  """Normal(0, stddev) redrawn outside two standard deviations, like
  tf.truncated_normal_initializer.  Returns f(sizes, dtype, device)."""
  def init(sizes, dtype, device):
    gen = None
    if seed is not None:
      gen = torch.Generator(device=device)
      gen.manual_seed(seed)
    t = torch.empty(sizes, dtype=torch.float32, device=device)
    torch.nn.init.trunc_normal_(t, mean=0.0, std=stddev, a=-2 * stddev,
                                b=2 * stddev, generator=gen)
    return t.to(dtype)
  return init


def random_normal_initializer(stddev=1.0, seed=None):
  """Normal(0, stddev), like tf.random_normal_initializer.  Returns
  f(sizes, dtype, device)."""
  def init(sizes, dtype, device):
    gen = None
    if seed is not None:
      gen = torch.Generator(device=device)
      gen.manual_seed(seed)
    t = torch.empty(sizes, dtype=torch.float32, device=device)
    t.normal_(0.0, stddev, generator=gen)
    return t.to(dtype)
  return init


def ones_initializer():
  """tf.ones_initializer.  Returns f(sizes, dtype, device)."""
  return lambda sizes, dtype, device: torch.ones(sizes, dtype=dtype,
                                                 device=device)


def random_uniform_initializer(minval, maxval, seed=None):
  def init(sizes, dtype, device):
    gen = None
    if seed is not None:
      gen = torch.Generator(device=device)
      gen.manual_seed(seed)
    t = torch.rand(sizes, dtype=torch.float32, device=device, generator=gen)
    return (t * (maxval - minval) + minval).to(dtype)
  return init


class VarianceScalingInitializer(DenseInitializer):
  """stddev = sqrt(scale / n) with n = fan_in, fan_out or their average."""

  def __init__(self, scale=1.0, mode="fan_in", distribution="normal"):
    self.scale = scale
    self.mode = mode.lower()
    self.distribution = distribution.lower()

  def __call__(self, reduced_dims, new_dims):
    fan_in = mtf.list_product(d.size for d in reduced_dims)
    fan_out = mtf.list_product(d.size for d in new_dims)
    scale = self.scale
    if self.mode == "fan_in":
      scale /= max(1., fan_in)
    elif self.mode == "fan_out":
      scale /= max(1., fan_out)
    elif self.mode == "fan_avg":
      scale /= max(1., float(fan_in + fan_out) / 2)
    else:
      raise ValueError(
          "Invalid `mode` argument: "
          "expected on of {\"fan_in\", \"fan_out\", \"fan_avg\"} "
          "but got %s" % (self.mode,))
    stddev = scale ** 0.5
    if self.distribution == "normal":
      return truncated_normal_initializer(stddev=stddev)
    elif self.distribution == "uniform":
      limit = stddev * 3. ** 0.5
      return random_uniform_initializer(minval=-limit, maxval=limit)
    raise ValueError("Invalid `distribution` argument: "
                     "expected one of {\"normal\", \"uniform\"} "
                     "but got %s" % (self.distribution,))


def get_dense_kernel_weights(x, new_dims, reduced_dims, expert_dims,
                             kernel_initializer, name=None,
                             variable_dtype=None, master_dtype=mtf.float32,
                             slice_dtype=mtf.float32):
  """Creates the variable `<name>/kernel` with shape
  expert_dims + reduced_dims + new_dims and returns its Tensor (in the
  activation dtype)."""
  if variable_dtype is None:
    variable_dtype = mtf.VariableDType(master_dtype, slice_dtype, x.dtype)
  w_shape = mtf.Shape(list(expert_dims) + list(reduced_dims) + list(new_dims))
  with mtf.variable_scope(name or "dense"):
    if kernel_initializer is None:
      kernel_initializer = VarianceScalingInitializer()
    if isinstance(kernel_initializer, DenseInitializer):
      kernel_initializer = kernel_initializer(reduced_dims, new_dims)
    return mtf.get_variable(x.mesh, "kernel", w_shape,
                            initializer=kernel_initializer,
                            dtype=variable_dtype)


class SharedInput(object):
  """Dense layers without activation, of one input and of kernels of one shape:
  their products, the gradients of their kernels, and that of their input are made in
  one launch each."""

  def __init__(self, layers):
    x, kernel = layers[0].inputs
    self.layers = list(layers)
    self.gradients = {}        # {layer: its DenseGradOperation}
    self._ahead = {}           # {all of them: every dy is there when the last runs}
    if all(op.inputs[0] is x and op.inputs[1].shape.to_integer_list ==
           kernel.shape.to_integer_list and op.inputs[1].dtype == kernel.dtype and
           op._activation is None and op.siblings is None   # pylint: disable=protected-access
           for op in layers):
      for op in layers:
        op.siblings = self

  def _joint_gradients(self, lowering, first):
    """Called by the first of the gradient operations: the gradients of all layers'
    outputs as one tensor [layers, ...], if every one is there and they lie one after
    the other in memory (as the attention's gradient leaves them), else None."""
    grads = tuple(self.gradients.get(op) for op in self.layers)
    operations = first.graph.operations
    if grads not in self._ahead:
      at = operations.index(first)
      self._ahead[grads] = None not in grads and all(
          operations.index(g.inputs[0].operation) < at for g in grads)
    if not self._ahead[grads]:
      return None
    dys = [_rows_of(lowering, g.inputs[0]) for g in grads]
    d = dys[0]
    step = d.numel()
    if not all(
        t.is_contiguous() and t.dtype == d.dtype and t.shape == d.shape and
        t.untyped_storage().data_ptr() == d.untyped_storage().data_ptr() and
        t.storage_offset() == d.storage_offset() + i * step
        for i, t in enumerate(dys)):
      return None
    return d.as_strided((len(dys),) + tuple(d.shape), (step,) + d.stride())

  def make_gradients(self, lowering, first):
    """Called by the first of the gradient operations: {layer: its kernel gradient}
    and, under the operation whose dx is the sum over all layers, that sum; without the
    sum, or {}, where there is no kernel for it."""
    from mesh_amd import moe_hip
    joint = self._joint_gradients(lowering, first)
    if joint is None:
      return {}
    x = _rows_of(lowering, first.inputs[1])
    if not (x.dtype == joint.dtype and joint.data_ptr() % 16 == 0 and
            moe_hip.shared_linear_backward_supported(x, joint.shape[-1])):
      return {}
    mesh_impl = lowering.mesh_impl(first)
    made = dict(zip(self.layers, mesh_impl.slicewise(
        lambda rows: tuple(moe_hip.shared_linear_backward(rows, joint).unbind(0)),
        lowering.tensors[first.inputs[1]])))
    last = first.sums_up_in(self.layers)
    if last is not None:
      n = joint.shape[-1]
      kernels = [
          _rows_of(lowering, self.gradients[op].inputs[2]).to(joint.dtype).reshape(
              -1, n).contiguous() for op in self.layers]
      if moe_hip.shared_linear_backward_input_supported(joint, kernels):
        made[last] = mesh_impl.slicewise(
            lambda _: moe_hip.shared_linear_backward_input(joint, kernels),
            lowering.tensors[first.inputs[0]])
    return made


def _rows_of(lowering, tensor):
  return lowering.tensors[tensor].to_laid_out_tensor().tensor_list[0]


class DenseOperation(mtf.Operation):
  """y = activation(x . kernel) over the last dim of x: the einsum (+ relu) of
  mtf.layers.dense without bias (mesh_tensorflow/layers.py:112-160) as one
  operation on the matrix cores.  The kernel is read from the variable's
  K-contiguous packed copy."""

  def __init__(self, x, kernel, new_dims, activation, name=None):
    super(DenseOperation, self).__init__([x, kernel], name=name or "dense")
    self._activation = activation
    shape = mtf.Shape(x.shape.dims[:-1] + list(new_dims))
    self._outputs = [mtf.Tensor(self, shape, x.dtype)]
    self.siblings = None       # a SharedInput

  def _lower_siblings(self, lowering):
    """All layers of one input in one launch, by the first of them.  False where
    there is no kernel for that."""
    from mesh_amd import moe_hip
    layers = self.siblings.layers
    if layers[0] is not self:
      return False
    mesh_impl = lowering.mesh_impl(self)
    x = lowering.tensors[self.inputs[0]].to_laid_out_tensor().tensor_list[0]
    n = self.outputs[0].shape.dims[-1].size
    if not moe_hip.shared_linear_supported(x, n):
      return False
    variables = [lowering.variables[op.inputs[1].operation] for op in layers]
    packed = variables[0].packed_together(variables, x.dtype)
    if packed is None:
      return False
    outs = mesh_impl.slicewise(
        lambda rows: tuple(moe_hip.shared_linear(rows, packed).unbind(0)),
        lowering.tensors[self.inputs[0]])
    for op, out in zip(layers, outs):
      lowering.set_tensor_lowering(op.outputs[0], out)
      lowering.done_ahead.add(op)
    return True

  def lower(self, lowering):
    from mesh_amd import moe_hip
    if self in lowering.done_ahead or (
        self.siblings is not None and self._lower_siblings(lowering)):
      return
    x, kernel = self.inputs
    mesh_impl = lowering.mesh_impl(self)
    packed = lowering.variables[kernel.operation].packed(x.dtype)
    act = self._activation

    def fn(xs):
      return moe_hip.dense(xs.contiguous(), packed, act)
    lowering.set_tensor_lowering(
        self.outputs[0], mesh_impl.slicewise(fn, lowering.tensors[x]))

  def gradient(self, grad_ys):
    return list(DenseGradOperation(self, grad_ys[0]).outputs)


class DenseGradOperation(mtf.Operation):
  """(dx, dkernel) of a DenseOperation: what mtf.gradients derives from the
  einsum (mesh_tensorflow/ops.py:2846-2854) and the relu of layers.dense, as
  dpre = dy * (y > 0), dx = dpre . kernel^T, dkernel = x^T . dpre on the
  grouped GEMM with one group."""

  def __init__(self, forward, dy, name=None):
    x, kernel = forward.inputs
    super(DenseGradOperation, self).__init__(
        [dy, x, kernel, forward.outputs[0]], name=name or "dense_grad")
    self._relu = forward._activation == "relu"   # pylint: disable=protected-access
    # When x = relu(dense(...)) feeds nothing but `forward` and nobody asked
    # for d/dx itself, the only reader of dx is the producer's backward, whose
    # first step is the ReLU mask: dx then leaves this operation already
    # multiplied by (x > 0) -- the mask applied on the stores of the GEMM, so
    # dx is d/d(pre-activation) -- and the producer's backward skips its own
    # pass over it (_dy_is_masked below).  Decided here, at gradient time,
    # when every consumer of x is known.
    producer_x = x.operation
    consumers = [op for op in x.graph.operations
                 if x in op.inputs and not isinstance(op, DenseGradOperation)]
    self._masks_dx = (
        isinstance(producer_x, DenseOperation)
        and producer_x._activation == "relu"      # pylint: disable=protected-access
        and x is producer_x.outputs[0]
        and consumers == [forward]
        and not mtf.gradient_is_returned(x))
    # dy already carries this layer's ReLU mask when it is the input gradient
    # of the one operation that consumes the output and that operation masks
    producer = dy.operation
    self._dy_is_masked = (
        self._relu and isinstance(producer, DenseGradOperation)
        and producer._masks_dx and dy is producer.outputs[0]
        and producer.inputs[1] is forward.outputs[0])
    if forward._activation not in (None, "relu"):  # pylint: disable=protected-access
      raise NotImplementedError("gradient of dense with activation %r"
                                % (forward._activation,))  # pylint: disable=protected-access
    self._outputs = [mtf.Tensor(self, x.shape, x.dtype, index=0),
                     mtf.Tensor(self, kernel.shape, kernel.dtype, index=1)]
    self._dx, self._dw = self._outputs
    self._forward = forward
    self._adds = self.added_by = None    # layers of the same input (add_to_output)
    siblings = forward.siblings
    if siblings is not None and not self._masks_dx:
      siblings.gradients[forward] = self

  def add_to_output(self, output, addend):
    """Makes dx the sum of what it was and addend, the dx of another layer of the same
    input, before anything reads it; False where this operation cannot.  Nothing else
    reads addend: it leaves the graph."""
    other, siblings = addend.operation, self._forward.siblings
    # pylint: disable=protected-access
    if (output is not self._dx or self._adds is not None or siblings is None or
        siblings.gradients.get(self._forward) is not self or
        not isinstance(other, DenseGradOperation) or addend is not other._dx or
        other.added_by is not None or
        siblings.gradients.get(other._forward) is not other):
      return False
    self._adds, other.added_by = other, self
    other._outputs.remove(addend)
    return True

  def sums_up_in(self, layers):
    """The operation whose dx is the sum of those of all `layers`, or None.  None too
    where a later mtf.gradients has made another gradient operation of one of the
    layers: what is made ahead is made for, and from the dy of, that one."""
    last = self
    while last.added_by is not None:
      last = last.added_by
    known, summed, op = self._forward.siblings.gradients, {}, last
    while op is not None:
      summed[op._forward] = op           # pylint: disable=protected-access
      op = op._adds                      # pylint: disable=protected-access
    return last if summed == {layer: known.get(layer) for layer in layers} else None

  def _made_ahead(self, lowering):
    """What the first gradient operation of layers with one input made for all."""
    siblings = self._forward.siblings
    if siblings is None or siblings.gradients.get(self._forward) is not self:
      return {}
    if self._forward is siblings.layers[-1]:
      # (the backward walk meets the last layer first)
      lowering.run_values[siblings] = siblings.make_gradients(lowering, self)
    return lowering.run_values.get(siblings, {})

  def _set_dx(self, lowering, value):
    """Lowers dx: `value` is what this layer gives to it."""
    if self._adds is not None:
      value = lowering.mesh_impl(self).slicewise(
          lambda one, dx: one + dx, lowering.run_values.pop(self._adds), value)
    if self.added_by is not None:
      lowering.run_values[self] = value
    else:
      lowering.set_tensor_lowering(self._dx, value)

  def lower(self, lowering):
    from mesh_amd import moe_hip
    mesh_impl = lowering.mesh_impl(self)
    made = self._made_ahead(lowering)
    last = self._forward.siblings and self.sums_up_in(self._forward.siblings.layers)
    whole = last is not None and last in made
    dw = made.pop(self._forward, None)
    if dw is not None:
      k = self.inputs[1].shape.dims[-1].size
      kernel_sizes = self.inputs[2].shape.to_integer_list
      if not whole:
        self._set_dx(lowering, mesh_impl.slicewise(
            lambda dy, x, w: moe_hip.dense(
                dy, w.to(x.dtype).reshape(1, k, -1).contiguous()),
            *[lowering.tensors[t] for t in self.inputs[:3]]))
      elif last is self:
        lowering.set_tensor_lowering(self._dx, made.pop(self))
      lowering.set_tensor_lowering(self._dw, mesh_impl.slicewise(
          lambda dw, w: dw.reshape(kernel_sizes).to(w.dtype), dw,
          lowering.tensors[self.inputs[2]]))
      return
    relu = self._relu and not self._dy_is_masked
    masks_dx = self._masks_dx
    k = self.inputs[1].shape.dims[-1].size
    kernel_sizes = self.inputs[2].shape.to_integer_list

    def fn(dy, x, w, y):
      w2 = w.to(x.dtype).reshape(k, -1)
      dx, dw = moe_hip.dense_backward(x.contiguous(), w2, dy.contiguous(),
                                      y if relu else None,
                                      dx_relu_mask=masks_dx)
      return dx, dw.reshape(kernel_sizes).to(w.dtype)
    dx, dw = mesh_impl.slicewise(
        fn, *[lowering.tensors[t] for t in self.inputs])
    self._set_dx(lowering, dx)
    lowering.set_tensor_lowering(self._dw, dw)


def _activation_name(activation):
  if activation is None or activation == "linear":
    return None
  name = activation if isinstance(activation, str) else getattr(
      activation, "__name__", None)
  if name != "relu":
    raise NotImplementedError("dense activation %r is not implemented"
                              % (activation,))
  return name


def dense(x, new_dims, reduced_dims=None, expert_dims=None, use_bias=True,
          activation=None, master_dtype=mtf.float32, slice_dtype=mtf.float32,
          variable_dtype=None, kernel_initializer=None, kernel_weights=None,
          name=None):
  """mtf.layers.dense (mesh_tensorflow/layers.py:112-160) for the case the
  transformer layers use: no bias, no expert dims, the reduced dims being the
  trailing dims of x; activation None / "linear" / relu.  The variable is
  `<name>/kernel` with shape reduced_dims + new_dims."""
  if isinstance(new_dims, mtf.Dimension) or not isinstance(new_dims,
                                                           (list, tuple)):
    new_dims = [new_dims]
  new_dims = [mtf.convert_to_dimension(d) for d in new_dims]
  if reduced_dims is None:
    reduced_dims = x.shape.dims[-1:]
  reduced_dims = list(reduced_dims)
  if use_bias:
    raise NotImplementedError("dense with a bias is not implemented")
  if expert_dims:
    raise NotImplementedError("dense with expert (ensemble) dims is not "
                              "implemented; the MoE layers have their own op")
  if kernel_weights is not None:
    raise NotImplementedError("dense with external kernel_weights")
  if len(reduced_dims) != 1 or len(new_dims) != 1:
    raise NotImplementedError("dense over several reduced or new dims")
  if x.shape.dims[-1] != reduced_dims[0]:
    raise NotImplementedError("the reduced dim must be the last dim of x")
  act = _activation_name(activation)
  w = get_dense_kernel_weights(x, new_dims, reduced_dims, [],
                               kernel_initializer, name, variable_dtype,
                               master_dtype, slice_dtype)
  return DenseOperation(x, w, new_dims, act, name=name).outputs[0]


def dense_product(x, reduced_dims, new_dims, activation_functions=None,
                  name="dense_product", **kwargs):
  """mtf.layers.dense_product (mesh_tensorflow/layers.py:256-295) with one
  factor; gated (list) activations are not implemented."""
  if isinstance(activation_functions, list):
    if len(activation_functions) != 1:
      raise NotImplementedError("gated (list) activations are not implemented")
    activation_functions = activation_functions[0]
  return dense(x, new_dims=new_dims, reduced_dims=reduced_dims,
               activation=activation_functions, name=name, **kwargs)
