"""Adam training-step executor.

Counterpart of the reference ``pycode/tinyflow/TrainExecuteAdam.py``: the step
graph of ``TrainExecute.TrainExecutor`` with one ``adam_op`` per variable in place
of the SGD node.  Every variable gets two moment variables, ``<name>m`` and
``<name>v``, that start at zero (reference TrainExecuteAdam.py:80-86) and live on
the device next to the parameter.  The bias-correction powers start at b1 and b2
and are multiplied by b1 and b2 after every step (reference :16-21, :196-198), so
step t (counted from 1) corrects with 1 - b1^t and 1 - b2^t.
"""
import numpy as np

from . import autodiff as ad
from . import _base, gpu_op, ndarray
from . import TrainExecute as _sgd


class TrainExecutor(_sgd.TrainExecutor):
    """Runs forward + backward + Adam update for one loss node."""

    _update_op = ad.AdamOp

    def __init__(self, targetloss, learning_rate=0.001, ctx=ndarray.gpu(0), fuse_bn_relu=False,
                 fused_update=True):
        self.b1 = 0.9
        self.b2 = 0.999
        self.e = 0.00000001
        self.b1t = [0.9]
        self.b2t = [0.999]
        self.mv = []
        self.Variable_node_to_mv = {}
        _sgd.TrainExecutor.__init__(self, targetloss, learning_rate, ctx, fuse_bn_relu, fused_update)

    def _update_nodes(self):
        nodes, self.mv, self.Variable_node_to_mv = getcomputelist(
            self.Variable_node_list, self.Variable_node_grad_list, self.b1, self.b2, self.b1t, self.b2t, self.e,
            self.learning_rate)
        return nodes

    def _fuse_updates(self, updates):
        return _FusedAdam(updates)

    def init_Variable(self, feed_dict):
        """Initial values (numpy) of the trainable variables; the moments start at zero."""
        values = dict(feed_dict)
        for node in self.Variable_node_list:
            m, v = self.Variable_node_to_mv[node]
            values[m] = np.zeros(np.shape(feed_dict[node]), dtype=np.float32)
            values[v] = np.zeros(np.shape(feed_dict[node]), dtype=np.float32)
        self.Variable_node_np_value = values

    def run(self, feed_dict, Accuracy_node=None, convert_to_numpy_ret_vals=False):
        """One step.  Returns [loss, variables in network order (, accuracy node)]."""
        result = _sgd.TrainExecutor.run(self, feed_dict, Accuracy_node, convert_to_numpy_ret_vals)
        self.b1t[0] = self.b1t[0] * self.b1
        self.b2t[0] = self.b2t[0] * self.b2
        return result

    def moments_of(self, variable):
        """Device arrays (m, v) of a trainable variable."""
        m, v = self.Variable_node_to_mv[variable]
        return self.node_to_arr_map[m], self.node_to_arr_map[v]


class _FusedAdam(_sgd.FusedUpdate):
    """One launch that reads and writes each parameter and moment once (28 bytes per
    parameter), where the two calls of an ``adam_op`` move 36 and every variable costs two
    launches: VGG-16 at batch 6, 96 pixels 0.40 ms in 38 launches.  The same arithmetic per
    element."""

    def __init__(self, updates):
        _sgd.FusedUpdate.__init__(self, updates)
        self.nodes = [node for node, _ in updates]
        self.written = _base.c_array(ndarray.DLArrayHandle, [a.handle for arrays in self.arrays for a in arrays[:3]])

    @staticmethod
    def _pointer_tables(columns, n):
        return gpu_op.get_n4_cuda_pointer(*columns, n)

    def apply(self, cudnnHandle, cublasHandle, cudaStream):
        node = self.nodes[0]
        # the executor gives every node the same numbers, but they are the nodes' and a caller may change them
        # between steps
        if len(set((n.b1, n.b2, n.b1t[0], n.b2t[0], n.e, n.learning_rate) for n in self.nodes)) != 1:
            for n, arrays in zip(self.nodes, self.arrays):
                n.op.compute(n, arrays, None, cudnnHandle, cublasHandle, cudaStream)
            return
        gpu_op.adam_compute_o_on_stream(self.pointers, self.tables, self.count, node.b1, node.b2, node.b1t[0],
                                        node.b2t[0], node.e, node.learning_rate, self.written, cudaStream)


def getcomputelist(Variable_node_list, Variable_node_grad_list, b1, b2, b1t, b2t, e, learning_rate):
    """One in-place Adam node and two moment variables per variable
    (reference TrainExecuteAdam.py:347-362)."""
    computelist, mv, var_to_mv = [], [], {}
    for var, grad in zip(Variable_node_list, Variable_node_grad_list):
        m = ad.Variable(var.name + "m")
        v = ad.Variable(var.name + "v")
        mv += [m, v]
        var_to_mv[var] = (m, v)
        node = ad.adam_op(var, m, v, grad, b1, b2, b1t, b2t, e, learning_rate)
        node.issgd = 1
        computelist.append(node)
    return computelist, mv, var_to_mv


# an update node moves behind the last reader of its parameter exactly as for SGD
# (reference TrainExecuteAdam.py:367-388)
swapadam = _sgd.swapsgd
