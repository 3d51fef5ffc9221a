"""SGD training-step executor.

Counterpart of the reference ``pycode/tinyflow/TrainExecute.py``: given a loss
node it collects the trainable variables, differentiates, appends one ``sgd_op``
per variable, orders everything topologically and moves each update behind the
last reader of its parameter (``swapsgd``).  The first ``run`` infers shapes
(which creates the C-side descriptors) and allocates one device array per node;
later runs copy the feeds in and recompute every node in place.

A step only enqueues work: nothing waits for the GPU except the read-back of a
(1,)-shaped operand inside Add/Mul (the upstream-gradient scalar), a feed for the last but
one before it, and whatever
the caller reads afterwards with ``asnumpy``.
"""
import numpy as np

from . import autodiff as ad
from . import gpu_op, ndarray
from ._base import c_array


class TrainExecutor(object):
    """Runs forward + backward + SGD update for one loss node."""

    _update_op = ad.SgdOp   # the update nodes that one multi-tensor call can apply together

    def __init__(self, targetloss, learning_rate, ctx=ndarray.gpu(0), fuse_bn_relu=False, fused_update=True):
        """``fuse_bn_relu`` (no counterpart in the reference): evaluate every batch
        norm whose only reader is a ReLU together with that ReLU, forward and
        backward, through the fused entry points.  Results are bit-identical; the
        batch-norm output and the ReLU's input gradient are then never materialised
        (``value_of`` does not know them).

        ``fused_update``: apply all updates of a step with one call of the
        multi-tensor entry point (``sgd_compute_o``, reference gpu_op.py:939-945, or its
        Adam counterpart) behind the last node of the step instead of calls per variable.  Every
        update still comes after the last reader of its parameter, which is all
        ``swapsgd`` asks for, and the arithmetic per element is the same.  2**31
        parameters or more, which the entry point's tables cannot address, and a device
        without room for the tables get the calls per variable."""
        self.fuse_bn_relu = fuse_bn_relu
        self.fused_update = fused_update
        self._fused_sgd = None   # the step's one-call update, of whichever optimizer
        self.fused_pairs = 0
        self.targetloss = targetloss
        self.learning_rate = learning_rate
        self.Variable_node_list = ad.get_Variable_node_list(targetloss)
        self.Variable_node_list.reverse()
        self.Variable_node_grad_list = ad.gradients(targetloss, self.Variable_node_list)
        self.eval_node_list = self._update_nodes()
        self.ctx = ctx
        self.topo_order = swapsgd(ad.find_topo_sort(self.eval_node_list))
        self.node_to_shape_map = None
        self.node_to_arr_map = {}
        self.Variable_node_np_value = None
        self.cudaStream = gpu_op.create_cudaStream()
        self.cudnnHandle = gpu_op.create_cudnnHandle(self.cudaStream)
        self.cublasHandle = gpu_op.create_cublasHandle(self.cudaStream)
        self.isfirstrun = 0
        self._plan = None

    def _update_nodes(self):
        """One in-place update node per variable, in ``Variable_node_list`` order."""
        return getcomputelist(self.Variable_node_list, self.Variable_node_grad_list, self.learning_rate)

    def _fuse_updates(self, updates):
        return _FusedSgd(updates)

    def infer_shape(self, feed_shapes):
        """Shapes of every node from the shapes of the fed nodes."""
        self.node_to_shape_map = dict(feed_shapes)
        slices = keeps_rounding_small(self.topo_order, self._update_op is ad.SgdOp)
        for node in self.topo_order:
            if node in self.node_to_shape_map:
                continue
            input_shapes = [self.node_to_shape_map[i] for i in node.inputs]
            assert None not in input_shapes
            self.node_to_shape_map[node] = tuple(node.op.infer_shape(node, input_shapes, self.cudnnHandle))
            if slices and isinstance(node.op, ad.Convolution2DForwardOp):
                gpu_op.convolution_allow_slices(node.cudnnlist[0])

    def init_Variable(self, feed_dict):
        """Initial values (numpy) of the trainable variables, used by the first run."""
        self.Variable_node_np_value = feed_dict

    def _alloc(self, shape):
        arr = ndarray.empty(shape, ctx=self.ctx)
        if isinstance(arr, int):
            raise MemoryError("device out of memory: %d more bytes wanted" % arr)
        return arr

    def _first_run(self, feed_dict):
        feed_dict = dict(feed_dict)
        feed_dict.update(self.Variable_node_np_value or {})
        self.infer_shape({node: np.shape(value) for node, value in feed_dict.items()})
        plan = []
        fused = {}
        fused_updates = []   # (update node, its input arrays) of the updates applied in one call
        if self.fuse_bn_relu:
            fused.update(find_bn_relu_pairs(self.topo_order, {self.targetloss}))
            fused.update(find_add_relu_pairs(self.topo_order, {self.targetloss}, self.node_to_shape_map))
        self.fused_pairs = sum(1 for v in fused.values() if v[0] in ("forward", "add_relu"))
        unread_zeros = _zeros_only_added(self.topo_order, self.node_to_shape_map,
                                         set(self.eval_node_list) | {self.targetloss})
        for role in fused.values():   # a fused call reads its sources as arrays
            if len(role) == 3:
                unread_zeros -= set(role[2])
        joined = find_joins(self.topo_order, self.node_to_shape_map, set(feed_dict) | unread_zeros, fused)
        groups = find_groups(self.topo_order, self.node_to_shape_map, set(feed_dict) | unread_zeros, fused, joined)
        in_group = {n for members in groups.values() for n in members}
        joined = {n: r for n, r in joined.items() if n not in in_group}
        by_join = set(joined.values())
        for node in self.topo_order:
            if node in groups:
                for n in groups[node]:
                    self.node_to_arr_map[n] = self._alloc(self.node_to_shape_map[n])
                plan.append((_group_compute(groups[node], self.node_to_shape_map, self.node_to_arr_map), node, None, None))
            if node in by_join or node in in_group:
                continue   # computed with its first operand, or with the first of its group
            if node in joined:
                reader = joined[node]
                outputs = [self._alloc(self.node_to_shape_map[n]) for n in (node, reader)]
                self.node_to_arr_map[node], self.node_to_arr_map[reader] = outputs
                sources = fused[reader][2] if reader in fused else reader.inputs
                plan.append((_join_compute(node, reader), reader,
                             [self.node_to_arr_map[i] for i in list(node.inputs) + list(sources)], outputs))
                continue
            if node in unread_zeros:
                continue   # every reader adds it as the constant 0.0: never materialised
            role = fused.get(node)
            if role is not None and role[0] == "skip":
                continue   # its value is folded into the fused call of its reader
            if role is not None:
                kind, bn, sources = role
                inputs = [self.node_to_arr_map[i] for i in sources]
                node_val = self._alloc(self.node_to_shape_map[node])
                self.node_to_arr_map[node] = node_val
                plan.append((_fused_compute(kind, bn), node, inputs, node_val))
                continue
            if node in feed_dict:
                arr = ndarray.array(feed_dict[node], ctx=self.ctx)
                if isinstance(arr, int):
                    raise MemoryError("device out of memory: %d more bytes wanted" % arr)
                self.node_to_arr_map[node] = arr
                continue
            assert node.isw not in (1, 2), "no value fed for %s" % node.name
            input_vals = [self.node_to_arr_map.get(i) if i in unread_zeros else self.node_to_arr_map[i]
                          for i in node.inputs]
            if node.issgd and self.fused_update and isinstance(node.op, self._update_op):
                fused_updates.append((node, input_vals))
                continue
            if node.issgd:
                node_val = None  # updates its parameter in place
            else:
                node_val = self._alloc(self.node_to_shape_map[node])
                self.node_to_arr_map[node] = node_val
            plan.append((_known_scalar_compute(node, self.node_to_shape_map)
                         or _known_zeros_compute(node, self.node_to_shape_map) or node.op.compute, node, input_vals,
                         node_val))
        self._plan = plan
        if self._fused_sgd is not None:
            self._fused_sgd.close()
            self._fused_sgd = None
        if fused_updates:
            try:
                self._fused_sgd = self._fuse_updates(fused_updates) if FusedUpdate.fits(fused_updates) else None
            except RuntimeError:   # no device memory for the tables: the calls per variable need none
                self._fused_sgd = None
            if self._fused_sgd is None:
                plan += [(node.op.compute, node, input_vals, None) for node, input_vals in fused_updates]
        if ndarray.is_gpu_ctx(self.ctx):   # the second step's feed finds its room made
            ndarray.reserve_feed([self.node_to_arr_map[node] for node in feed_dict
                                  if node.isw != 1 and node in self.node_to_arr_map], self.cudaStream)
        self.isfirstrun = 1

    def _feed(self, pairs):
        """The batch of a step, in front of it on the executor's stream; the step before may still run."""
        if ndarray.is_gpu_ctx(self.ctx):
            ndarray.feed(pairs, self.cudaStream)
            return
        for array, value in pairs:
            array._sync_copyfrom(value)

    def run(self, feed_dict, Accuracy_node=None, convert_to_numpy_ret_vals=False):
        """One step.  Returns [loss, variables in network order (, accuracy node)]."""
        if self.isfirstrun == 0:
            self._first_run(feed_dict)
        else:
            # variables live on the device; only data is re-fed
            self._feed([(self.node_to_arr_map[node], value) for node, value in feed_dict.items() if node.isw != 1])
        handles = (self.cudnnHandle, self.cublasHandle, self.cudaStream)
        for compute, node, input_vals, node_val in self._plan:
            wanted = compute(node, input_vals, node_val, *handles)
            if wanted:
                raise MemoryError("%s: %d bytes of device scratch could not be allocated" % (node.name, wanted))
        if self._fused_sgd is not None:
            self._fused_sgd.apply(*handles)
        result = [self.node_to_arr_map[self.targetloss]]
        result += [self.node_to_arr_map[v] for v in reversed(self.Variable_node_list)]
        if Accuracy_node is not None:
            result.append(self.node_to_arr_map[Accuracy_node])
        if convert_to_numpy_ret_vals:
            return [r.asnumpy() for r in result]
        return result

    def value_of(self, node):
        """Device array currently holding ``node`` (any node of the step graph)."""
        return self.node_to_arr_map[node]

    def close(self):
        """Gives the stream and the two handles back to the library (waits for the
        stream first).  The library orders copies and storage reuse against every
        stream that has run kernels, so an executor that is done should not leave
        its stream registered; the fused update's device tables go back to the pool.
        Arrays already returned stay valid."""
        if self.cudaStream is None:
            return
        stream, self.cudaStream = self.cudaStream, None
        self._plan = None
        if self._fused_sgd is not None:
            self._fused_sgd.close()
            self._fused_sgd = None
        gpu_op.destroy_cudnnHandle(self.cudnnHandle)
        gpu_op.destroy_cublasHandle(self.cublasHandle)
        gpu_op.destroy_cudaStream(stream)

    def __del__(self):
        try:
            self.close()
        except Exception:   # interpreter shutdown: the library may already be gone
            pass


def keeps_rounding_small(topo_order, is_sgd):
    """Whether a step passes another rounding of its convolutions on about as small as it is: an SGD update scales it, where Adam's may
    take its sign for a direction; and no batch norm divides by a spread that may itself be rounding.  With batch norms two
    roundings of a ResNet-50 step differ by up to a tenth in single parameters' gradients."""
    return is_sgd and not any(isinstance(n.op, ad.BNForwardOp) for n in topo_order)


class FusedUpdate(object):
    """All parameter updates of a step as one launch: the pointer tables and the index ->
    (tensor, offset) tables of ``sgd_compute_o`` / ``adam_compute_o`` (reference
    gpu_op.py:887-945), built once for the step's arrays, which keep their storage from
    step to step.

    ``updates``: pairs of an update node and its input arrays, parameter first."""

    max_parameters = 2 ** 31 - 1   # the tables count in 32 bits

    def __init__(self, updates):
        self.arrays = [arrays for _, arrays in updates]   # keeps the storage alive
        sizes = [int(np.prod(arrays[0].shape)) for arrays in self.arrays]
        for arrays, n in zip(self.arrays, sizes):
            assert all(int(np.prod(a.shape)) == n for a in arrays), "gradient and parameter sizes differ"
        # whole tensors end to end: the tables are built from the sizes, not from
        # per-parameter (tensor, offset) arrays
        self.tables, self.count = gpu_op.get_tensor_runs_cuda_pointer(sizes)
        columns = [[a.handle.contents.data for a in column] for column in zip(*self.arrays)]
        self.n_tables = len(columns)
        try:
            self.pointers = self._pointer_tables(columns, len(sizes))
        except RuntimeError:
            gpu_op.free_index_cuda_pointer(self.tables)
            raise

    @classmethod
    def fits(cls, updates):
        """Whether the tables can address the parameters of these updates."""
        return sum(int(np.prod(arrays[0].shape)) for _, arrays in updates) <= cls.max_parameters

    def close(self):
        """Gives the device tables back (waits for the last update that reads them)."""
        if self.tables is not None:
            gpu_op.free_index_cuda_pointer(self.tables)
            gpu_op.free_n_cuda_pointer(self.pointers, self.n_tables)
            self.tables = self.pointers = None
            self.arrays = []


class _FusedSgd(FusedUpdate):
    def __init__(self, updates):
        rates = set(node.learning_rate for node, _ in updates)
        assert len(rates) == 1, "one learning rate per step"
        self.learning_rate = rates.pop()
        FusedUpdate.__init__(self, updates)
        self.written = c_array(ndarray.DLArrayHandle, [arrays[0].handle for arrays in self.arrays])

    @staticmethod
    def _pointer_tables(columns, n):
        return gpu_op.get_n2_cuda_pointer(*columns, n)

    def apply(self, cudnnHandle, cublasHandle, cudaStream):
        gpu_op.sgd_compute_o_on_stream(self.pointers, self.tables, self.count, self.learning_rate, self.written,
                                       cudaStream)


def find_bn_relu_pairs(topo_order, outputs):
    """Batch norms that can be evaluated together with the ReLU that follows them.

    A per-activation batch-norm node B qualifies when its only readers are a ReLU
    activation R and that activation's backward node A (which reads B as the ReLU
    input), and A's only reader is B's own backward node D.  Returns a dict:
    B and A -> ("skip",); R -> ("forward", B, [x]); D -> ("backward", B, [x, dR])."""
    readers = {}
    for n in topo_order:
        for inp in n.inputs:
            readers.setdefault(inp, []).append(n)
    roles = {}
    for r in topo_order:
        if not (isinstance(r.op, ad.ActivationForwardOp) and r.activationMode == "relu"):
            continue
        b = r.inputs[0]
        if not isinstance(b.op, ad.BNForwardOp) or b.batchNormMode != "pre_activation" or b in outputs:
            continue
        others = [n for n in readers.get(b, []) if n is not r]
        if len(others) != 1:
            continue
        a = others[0]
        if not (isinstance(a.op, ad.ActivationBackwardOp) and a.inputs[0] is b and a.inputs[2] is r) or a in outputs:
            continue
        a_readers = readers.get(a, [])
        if len(a_readers) != 1:
            continue
        d = a_readers[0]
        if not (isinstance(d.op, ad.BNBackwardOp) and d.inputs[1] is a and d.inputs[0] is b.inputs[0]
                and d.Save_p is b.Save_p):
            continue
        roles[b] = ("skip",)
        roles[a] = ("skip",)
        roles[r] = ("forward", b, [b.inputs[0]])
        roles[d] = ("backward", b, [b.inputs[0], a.inputs[1]])
    return roles


def find_add_relu_pairs(topo_order, outputs, shapes):
    """Elementwise sums that can be evaluated together with the ReLU that follows them
    (the join of a residual block).  A sum S of two equally shaped values qualifies
    when its only readers are a ReLU activation R and R's backward node A, which
    reads S only to rebuild the mask S > 0 -- and R > 0 is the same mask.  Returns
    S -> ("skip",); R -> ("add_relu", S, [a, b]); A -> ("mask_from_output", S, [R, dR, R])."""
    readers = {}
    for n in topo_order:
        for inp in n.inputs:
            readers.setdefault(inp, []).append(n)
    roles = {}
    for r in topo_order:
        if not (isinstance(r.op, ad.ActivationForwardOp) and r.activationMode == "relu"):
            continue
        s = r.inputs[0]
        if not isinstance(s.op, ad.AddOp) or s in outputs or len(s.inputs) != 2:
            continue
        if not (shapes[s.inputs[0]] == shapes[s.inputs[1]] == shapes[s]):
            continue   # a (1,)-shaped operand is applied as a constant, not added elementwise
        others = [n for n in readers.get(s, []) if n is not r]
        if len(others) != 1:
            continue
        a = others[0]
        if not (isinstance(a.op, ad.ActivationBackwardOp) and a.inputs[0] is s and a.inputs[2] is r):
            continue
        roles[s] = ("skip",)
        roles[r] = ("add_relu", s, list(s.inputs))
        roles[a] = ("mask_from_output", s, [r, a.inputs[1], r])
    return roles


def find_joins(topo_order, shapes, unavailable, roles):
    """Nodes S that are computed together with a reader: one pass that writes both, where the second of two passes would
    read S again (64 images of 256 channels of 56 x 56, sum and ReLU: 20 bytes per element become 16).  S is

    - an elementwise sum or a batch norm, its reader a ReLU (a batch norm that no one pass takes with it keeps its two calls);
    - an elementwise sum, its reader a ReLU backward whose upstream gradient it is;
    - the ReLU backward behind such a batch norm, its reader that batch norm's backward.

    Returns S -> reader.  Both run at S's place: the reader's other operands have to precede S.  Other readers of either
    do not matter, both arrays hold what they would.  ``unavailable`` nodes are fed or never materialised; ``roles`` are
    the fused roles, of which only a backward that takes its mask from the ReLU's output can join."""
    at = {n: i for i, n in enumerate(topo_order)}
    joins, taken = {}, unavailable | {n for n, role in roles.items() if role[0] != "mask_from_output"}

    def is_sum(s):
        return (isinstance(s.op, ad.AddOp) and len(s.inputs) == 2   # a (1,)-shaped operand is applied as a constant
                and shapes[s.inputs[0]] == shapes[s.inputs[1]] == shapes[s])

    def is_norm(s):
        return isinstance(s.op, ad.BNForwardOp)

    for r in topo_order:
        if r in taken:
            continue
        if isinstance(r.op, ad.ActivationForwardOp) and r.activationMode == "relu":
            s, others = r.inputs[0], []
            fits = is_sum(s) or is_norm(s)
        elif isinstance(r.op, ad.ActivationBackwardOp) and r.activationMode == "relu":
            s, others = r.inputs[1], roles[r][2] if r in roles else r.inputs
            others = [n for n in others if n is not s]
            fits = is_sum(s)
        elif isinstance(r.op, ad.BNBackwardOp):
            s, others = r.inputs[1], r.inputs[:1]
            fits = (isinstance(s.op, ad.ActivationBackwardOp) and s.activationMode == "relu" and s not in roles
                    and is_norm(s.inputs[0]) and s.inputs[0].Save_p is r.Save_p and s.inputs[0].inputs[0] is r.inputs[0])
        else:
            continue
        if not fits or s in taken or unavailable & set(s.inputs) or any(at[n] >= at[s] for n in others):
            continue
        joins[s] = r
        taken |= {r, s}
    return joins


def _join_compute(first, reader):
    """Plan entry (same signature as ``Op.compute``) of a join: ``input_vals`` are what ``first`` reads and then what
    ``reader`` reads, ``output_val`` the arrays of both."""
    if isinstance(first.op, ad.BNForwardOp):
        def compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream):
            wanted = gpu_op.bn_and_relu_forward(input_vals[0], output_val[0], output_val[1], first.batchNormMode, first.n,
                                                first.Save_p[0], first.Save_p[1], first.cudnnlist[0],
                                                reader.cudnnlist[0], cudnnHandle, cudaStream)
            first.n += 1
            return wanted
    elif isinstance(first.op, ad.ActivationBackwardOp):
        def compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream):
            bn_out, dy, relu_out, x = input_vals[:4]
            return gpu_op.bn_and_relu_backward(x, bn_out, relu_out, dy, output_val[0], output_val[1],
                                               reader.batchNormMode, reader.Save_p[0], reader.Save_p[1],
                                               reader.cudnnlist[0], first.cudnnlist[0], cudnnHandle, cudaStream)
    elif isinstance(reader.op, ad.ActivationForwardOp):
        def compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream):
            a, b = input_vals[:2]
            gpu_op.add_activation_forward(a, b, output_val[0], output_val[1], reader.cudnnlist[0], cudnnHandle,
                                          cudaStream)
            return 0
    else:
        def compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream):
            a, b, x, _, y = input_vals
            gpu_op.add_activation_backward(a, b, output_val[0], x, output_val[1], y, reader.cudnnlist[0], cudnnHandle,
                                           cudaStream)
            return 0
    return compute


# Longer arrays gain nothing from fewer launches: their joins move as many bytes and keep the ReLU's sign bits.
MAX_GROUP_ELEMENTS = 1 << 23


def _group_step(node, shapes):
    """How one step of ``elementwise_group`` computes ``node``: (kind, constant, operands), or None.  Operands of another shape are
    left to the node's own call, which takes or refuses them."""
    step = _step_of(node, shapes)
    if step is not None and step[0] != gpu_op.GROUP_BROADCAST and any(shapes[i] != shapes[node] for i in step[2]):
        return None
    return step


def _step_of(node, shapes):
    op, inputs = node.op, node.inputs
    if isinstance(op, (ad.AddOp, ad.MulOp)) and len(inputs) == 2:
        which = _added_zeros_operand(node, shapes)
        if which is not None:
            return gpu_op.GROUP_ADD_CONST, 0.0, [inputs[1 - which]]
        add = isinstance(op, ad.AddOp)
        if shapes[inputs[0]] == shapes[inputs[1]]:
            return gpu_op.GROUP_ADD if add else gpu_op.GROUP_MUL, 0.0, list(inputs)
        known = _known_scalar_operand(node, shapes)
        if known is not None:
            return gpu_op.GROUP_ADD_CONST if add else gpu_op.GROUP_MUL_CONST, known[1], [inputs[1 - known[0]]]
    elif isinstance(op, (ad.AddByConstOp, ad.MulByConstOp)):
        kind = gpu_op.GROUP_ADD_CONST if isinstance(op, ad.AddByConstOp) else gpu_op.GROUP_MUL_CONST
        return kind, node.const_attr, list(inputs)
    elif isinstance(op, (ad.OnesLikeOp, ad.ZerosLikeOp)):
        return gpu_op.GROUP_SET, 1.0 if isinstance(op, ad.OnesLikeOp) else 0.0, []
    elif isinstance(op, ad.BroadcastToOp):
        # a bias: one value for each channel, or for each column
        if node.type == "NCHW" or len(shapes[inputs[0]]) == 1 and shapes[node][-1:] == shapes[inputs[0]]:
            return gpu_op.GROUP_BROADCAST, 0.0, [inputs[0]]
    elif isinstance(op, ad.ReluOp):
        return gpu_op.GROUP_RELU, 0.0, list(inputs)
    elif isinstance(op, ad.ReluGradientOp):
        return gpu_op.GROUP_RELU_GRADIENT, 0.0, list(inputs)
    elif isinstance(op, ad.ActivationForwardOp) and node.activationMode == "relu":
        return gpu_op.GROUP_RELU, 0.0, list(inputs)
    elif isinstance(op, ad.ActivationBackwardOp) and node.activationMode == "relu":
        return gpu_op.GROUP_RELU_GRADIENT, 0.0, [inputs[0], inputs[1]]
    return None


def find_groups(topo_order, shapes, unavailable, roles, joins):
    """Elementwise nodes of one length that are computed by one launch (``gpu_op.elementwise_group``): a fully connected
    layer's bias broadcast, sum and ReLU, the ReLU's gradient and the sum with zeros behind it.  Returns first node -> the nodes in
    order.  They run at the first one's place, so what the others read has to precede it or be in the group; every array
    holds what it would.  A join of a sum and its ReLU comes apart only where the group brings the sum's operand with it."""
    at = {n: i for i, n in enumerate(topo_order)}
    by_join = {r: n for n, r in joins.items()}
    steps, groups, taken = {}, {}, set()
    for n in topo_order:
        if n in unavailable or n in roles or n.issgd or n.isw or int(np.prod(shapes[n])) > MAX_GROUP_ELEMENTS:
            continue
        if not all(isinstance(s.op, ad.AddOp) and isinstance(r.op, ad.ActivationForwardOp)
                   for s, r in joins.items() if n in (s, r)):
            continue   # joins of a batch norm, or of two adjoints
        step = _group_step(n, shapes)
        if step is not None:
            steps[n] = step
    for first in topo_order:
        if first not in steps or first in taken or first in joins or first in by_join or shapes[first] == (1,):
            continue
        size = int(np.prod(shapes[first]))
        members = [first]
        for n in topo_order[at[first] + 1:]:
            if len(members) == gpu_op.GROUP_MAX_STEPS:
                break
            if n not in steps or n in taken or not (shapes[n] == (1,) and steps[n][0] == gpu_op.GROUP_SET
                                                    or int(np.prod(shapes[n])) == size):
                continue
            kind, _, operands = steps[n]
            spread = kind == gpu_op.GROUP_BROADCAST
            if not all(at[i] < at[first] or (i in members and not spread) for i in operands):
                continue
            if n in joins and not any(i in members for i in operands):
                continue   # the sum keeps its ReLU
            if n in by_join and by_join[n] not in members:
                continue
            members.append(n)
        # a sum whose ReLU found no room stays with it, and with it what reads the two
        while True:
            kept = [n for n in members if not (n in joins and joins[n] not in members)
                    and all(at[i] < at[first] or i in members for i in steps[n][2])]
            if kept == members:
                break
            members = kept
        if sum(shapes[n] != (1,) for n in members) > 1:   # a single element to set is no reason for a group
            groups[first] = members
            taken |= set(members)
    return groups


def _group_compute(members, shapes, arrays):
    """Plan entry (same signature as ``Op.compute``) of a group."""
    steps = (gpu_op.GroupStep * len(members))()
    held = []   # a handle alone does not keep its storage
    for entry, n in zip(steps, members):
        entry.kind, entry.value, operands = _group_step(n, shapes)
        held += [arrays[i] for i in [n] + operands]
        entry.per_channel = isinstance(n.op, ad.BroadcastToOp) and n.type == "NCHW"
        entry.out = arrays[n].handle
        for field, operand in zip(("a", "b"), operands):
            setattr(entry, field, arrays[operand].handle)
    # a constant is the node's at the time of the step
    constants = [(entry, n) for entry, n in zip(steps, members) if isinstance(n.op, (ad.AddByConstOp, ad.MulByConstOp))]
    # the calls without a stream argument in the reference are ordered against every stream
    ordered = int(any(isinstance(n.op, (ad.ReluOp, ad.ReluGradientOp)) for n in members))

    def compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream):
        for entry, n in constants:
            entry.value = n.const_attr
        gpu_op.elementwise_group(steps, ordered, cudaStream)
        return 0
    compute.arrays = held
    return compute


def _known_scalar_operand(node, shapes):
    """(index, value) of the (1,)-shaped operand of an Add / Mul node that is a ``oneslike`` / ``zeroslike``, or None."""
    a, b = node.inputs
    which = 1 if shapes[b] == (1,) else 0 if shapes[a] == (1,) else None
    if which is None or shapes[a] == shapes[b]:
        return None
    producer = node.inputs[which]
    if isinstance(producer.op, ad.OnesLikeOp):
        return which, 1.0
    if isinstance(producer.op, ad.ZerosLikeOp):
        return which, 0.0
    return None


def _known_scalar_compute(node, shapes):
    """Plan entry for an Add / Mul node one of whose operands is a (1,)-shaped
    ``oneslike`` / ``zeroslike`` value, or None.  The op itself reads a (1,) operand
    back to the host every step and applies it as a constant (reference
    autodiff.py:302-348, 376-413), which makes the host wait for the whole forward pass
    at the upstream-gradient scalar of the loss; the value of such a producer is 1.0 or
    0.0 whatever its input holds, so the constant is known without reading it."""
    if not isinstance(node.op, (ad.AddOp, ad.MulOp)) or len(node.inputs) != 2:
        return None
    known = _known_scalar_operand(node, shapes)
    if known is None:
        return None
    which, constant = known
    by_const = (gpu_op.matrix_elementwise_add_by_const if isinstance(node.op, ad.AddOp)
                else gpu_op.matrix_elementwise_multiply_by_const)

    def compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream):
        by_const(input_vals[1 - which], constant, output_val, cudaStream)
        return 0
    return compute


def _added_zeros_operand(node, shapes):
    """Index of the operand of an Add node that is a ``zeroslike`` of the other
    operand's shape, or None."""
    if not isinstance(node.op, ad.AddOp) or len(node.inputs) != 2:
        return None
    for which in (0, 1):
        z, other = node.inputs[which], node.inputs[1 - which]
        if isinstance(z.op, ad.ZerosLikeOp) and shapes[z] == shapes[other] and not isinstance(other.op, ad.ZerosLikeOp):
            return which
    return None


def _known_zeros_compute(node, shapes):
    """Plan entry for ``x + zeroslike(.)`` of equal shapes, or None.  The reference's
    broadcast gradient hands a zeros tensor to its second input (autodiff.py, the
    ``broadcastto`` gradient), which the accumulation of adjoints then adds to the real
    gradient: a fill and a two-operand add per bias.  Adding the constant 0.0 gives the
    same bits (x + 0.0 is the same IEEE sum) with one read less and no fill."""
    which = _added_zeros_operand(node, shapes)
    if which is None:
        return None

    def compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream):
        gpu_op.matrix_elementwise_add_by_const(input_vals[1 - which], 0.0, output_val, cudaStream)
        return 0
    return compute


def _zeros_only_added(topo_order, shapes, outputs):
    """``zeroslike`` nodes all of whose readers are such additions (and that nobody
    asks for): their value is never needed as an array."""
    readers = {}
    for n in topo_order:
        for inp in n.inputs:
            readers.setdefault(inp, []).append(n)
    unread = set()
    for z in topo_order:
        if not isinstance(z.op, ad.ZerosLikeOp) or z in outputs or not readers.get(z):
            continue
        if all((_added_zeros_operand(r, shapes) is not None and r.inputs[_added_zeros_operand(r, shapes)] is z)
               for r in readers[z]):
            unread.add(z)
    return unread


def _fused_compute(kind, bn):
    """Plan entry (same signature as ``Op.compute``) for a fused node: batch norm
    ``bn`` with its ReLU (forward / backward), a sum with its ReLU, or a ReLU backward
    that takes its mask from the ReLU output."""
    if kind == "add_relu":
        def compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream):
            assert input_vals[0].shape == input_vals[1].shape == output_val.shape
            gpu_op.matrix_elementwise_add_relu(input_vals[0], input_vals[1], output_val, cudaStream)
            return 0
        return compute
    if kind == "mask_from_output":
        def compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream):
            return node.op.compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream)
        return compute
    if kind == "forward":
        def compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream):
            wanted = gpu_op.bn_relu_forward(input_vals[0], output_val, bn.batchNormMode, bn.n, bn.Save_p[0],
                                            bn.Save_p[1], bn.cudnnlist[0], cudnnHandle, cudaStream)
            bn.n += 1
            return wanted
    else:
        def compute(node, input_vals, output_val, cudnnHandle, cublasHandle, cudaStream):
            return gpu_op.bn_relu_backward(input_vals[0], input_vals[1], output_val, bn.batchNormMode, bn.Save_p[0],
                                           bn.Save_p[1], bn.cudnnlist[0], cudnnHandle, cudaStream)
    return compute


def getcomputelist(Variable_node_list, Variable_node_grad_list, learning_rate):
    """One in-place SGD node per variable (reference TrainExecute.py:315-324)."""
    computelist = []
    for var, grad in zip(Variable_node_list, Variable_node_grad_list):
        node = ad.sgd_op(var, grad, learning_rate)
        node.issgd = 1
        computelist.append(node)
    return computelist


def swapsgd(topoorder):
    """Move every update node to just behind the last non-update node that reads
    its parameter, so that e.g. the grad-data convolution of a layer still sees
    the weights the forward pass used (reference TrainExecute.py:329-349)."""
    topoorder = list(topoorder)
    i = 0
    while i < len(topoorder):
        node = topoorder[i]
        if node.issgd == 1 and node.isw == 0:
            node.isw = 3
            param = node.inputs[0]
            j = len(topoorder) - 1
            while j > i:
                other = topoorder[j]
                if other.issgd != 1 and param in other.inputs:
                    break
                j -= 1
            if j > i:
                topoorder.pop(i)
                topoorder.insert(j, node)
                continue  # position i now holds the next node
        i += 1
    return topoorder
