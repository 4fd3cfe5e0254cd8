"""Many uneven trajectories in one captured launch sequence.

The discretization of a whole data set -- lagged moments of every trajectory
(LaggedCovariance over RunningCovar.add, coordinates/estimation/
covariance.py:219-244) and the assignment of every frame to a center set
(AbstractClustering._transform_array, clustering/interface.py:157-167) -- is
one fixed sequence of kernel launches over device-resident inputs:

  emma_moments_lagged: k_prep -> moments (one launch over all trajectories and
                       pair slices) -> FP64 reductions
  emma_assign:         center mean / pack -> MFMA distances -> exact recheck

BatchedDiscretizer runs that sequence eagerly once (which also lets the
autotuner pick the first pass for these sizes), then captures it into a HIP
graph; replay() re-issues the whole sequence with one call.  The graph reads
the input buffers in place, so new frames of the same shape can be copied
into `X` between replays.  Nothing inside the sequence allocates memory, uses
a memset node or synchronizes the host.  The scratch buffers belong to the
plan: the graph holds their addresses, so they stay in place however much the
calls made between replays need.
"""
import numpy as np

from . import _native, autotune

__all__ = ["BatchedDiscretizer"]


class BatchedDiscretizer(object):
    """Lagged moments + assignment of all trajectories, captured as one graph.

    X          (n_rows, d) float32 device tensor, trajectories concatenated
    offsets    int64 trajectory offsets (ntraj + 1)
    lag        TICA lag time
    centers    (k, d) float32 cluster centers
    precision  moment tile arithmetic ('bf16x4-acc', 'bf16x4', 'fp32', 'fp64')
    """

    def __init__(self, X, offsets, lag, centers, precision="bf16x4-acc", reversible=True,
                 assign_mode=_native.EMMA_ASSIGN_BF16X3_RECHECK):
        from .coordinates.covariance import PRECISIONS

        t = _native.torch()
        dev = _native.device()
        self.X = _native.as_device_f32(X)
        self.offsets = t.as_tensor(np.asarray(offsets, dtype=np.int64), device=dev)
        self.C = _native.as_device_f32(centers)
        if self.C.shape[1] != self.X.shape[1]:
            raise ValueError("cluster centers have wrong dimension. Have dim=%i, but input has %i"
                             % (self.C.shape[1], self.X.shape[1]))
        self.lag = int(lag)
        self.reversible = bool(reversible)
        self.precision = PRECISIONS[precision]
        self.assign_mode = int(assign_mode)
        n, d = self.X.shape
        self.labels = t.empty(n, dtype=t.int32, device=dev)
        self.n_rechecked = t.zeros(1, dtype=t.int64, device=dev)
        self.graph = None
        self.out = None
        self._workspaces = _native.Workspaces()

    def _sequence(self):
        """The moments as device tensors; the labels go to self.labels."""
        out = _native.moments_lagged(self.X, self.offsets, self.lag, reversible=self.reversible,
                                     remove_mean=True, c0t=True, precision=self.precision,
                                     workspaces=self._workspaces)
        _native.assign(self.X, self.C, mode=self.assign_mode, labels=self.labels, n_rechecked=self.n_rechecked,
                       workspaces=self._workspaces)
        return out

    def run_eager(self):
        """One uncaptured pass (tunes the first pass on first use); returns host results."""
        autotune.tune_assign(self.X, self.C, self.assign_mode)
        self.out = self._sequence()
        return self.results()

    def capture(self):
        """Eager warm-up, then capture the launch sequence into a HIP graph."""
        t = _native.torch()
        self.run_eager()
        t.cuda.synchronize()
        g = t.cuda.CUDAGraph()
        with t.cuda.graph(g):
            out = self._sequence()
        self.graph = g
        for a, b in zip(out, self.out):  # the capture has not run them: the warm-up's values
            if a is not None:
                a.copy_(b)
        self.out = self._graph_out = out
        # everything whose address the graph holds
        self._captured = (self.X, self.offsets, self.C, self.labels, self.n_rechecked,
                          tuple(self._workspaces.buffers.values()))
        return self

    def replay(self):
        if self.graph is None:
            raise RuntimeError("capture() first")
        self.graph.replay()
        self.out = self._graph_out

    def results(self):
        """(w, mean, C00, C0t, labels) on the host (synchronizes)."""
        w, sx, sy, Mxx, Mxy, _ = self.out
        wh = float(w.item())
        return (wh, sx.cpu().numpy() / wh, Mxx.cpu().numpy() / wh, Mxy.cpu().numpy() / wh,
                self.labels.cpu().numpy())
