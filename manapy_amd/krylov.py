"""Arena of block-diagonal sparse systems solved on the GPU (``mfv_krylov_fused_tick``).

An ``EllBatch`` owns one ELL matrix of ``max_slices`` 64-row slices and the vectors
of the mixed-precision solver. Independent systems ``(sigma I + tau A) x = b``
occupy contiguous slice ranges; ``alloc`` / ``release`` manage those ranges (first
fit) and ``publish`` uploads the live lists (slices, instances, chunks of slices) that
the kernels walk. Because every device pointer and grid size stays fixed,
one tick is valid for any set of instances at any stage of their solve, and each
instance's arithmetic is independent of the others (see mfv_krylov.hip).

The solver replaces the factorisation of ``ScipySolver`` / ``MUMPSSolver``
(``solvers/ls/system.py:236-379, 624-744``): FP32 BiCGStab with Jacobi scaling
inside FP64 iterative refinement, stopped at ``||b - A x|| <= tol ||b||``. The inner
solves stop on the Jacobi-scaled residual (``tol_in``).
"""
import collections
import ctypes

import numpy as np

from . import _lib
from .device import require_gpu, stream_ptr


def _pow2(n):
    return 1 << max(0, int(n) - 1).bit_length()


class RangeAllocator(object):
    """First-fit allocator of contiguous ranges of ``[0, size)`` with coalescing frees."""

    def __init__(self, size):
        self.size = int(size)
        self.free = [(0, self.size)]

    def alloc(self, n):
        for k, (s0, m) in enumerate(self.free):
            if m >= n:
                if m == n:
                    self.free.pop(k)
                else:
                    self.free[k] = (s0 + n, m - n)
                return s0
        return None

    def release(self, s0, n):
        self.free.append((s0, n))
        self.free.sort()
        merged = []
        for s, m in self.free:
            if merged and merged[-1][0] + merged[-1][1] == s:
                merged[-1] = (merged[-1][0], merged[-1][1] + m)
            else:
                merged.append((s, m))
        self.free = merged

    def available(self):
        return sum(m for _, m in self.free)

    def largest(self):
        return max((m for _, m in self.free), default=0)


def chunk_list(ranges):
    """Chunks [n][4] int32 (mfv_krylov_fused in include/mfv.h) of live instances given as
    (instance, first slice, slices), in the order given."""
    out = []
    for inst, s0, ns in ranges:
        span = 4 * ((ns + 4 * _lib.KRYLOV_MAX_CHUNKS - 1) // (4 * _lib.KRYLOV_MAX_CHUNKS))
        n = (ns + span - 1) // span
        c = np.empty((n, 4), dtype=np.int32)
        c[:, 0], c[:, 1], c[:, 3] = inst, s0, ns
        c[:, 2] = np.arange(n) | (n << 16)
        out.append(c)
    return np.concatenate(out) if out else np.zeros((0, 4), np.int32)


class EllBatch(object):
    def __init__(self, max_slices, max_inst=64, width=32, device=None):
        torch = require_gpu()
        if width < 1 or width > 128:  # the diamond assembly holds 32 columns per row in 2D, 128 in 3D
            raise ValueError("ELL width must be in [1, 128]")
        self.S, self.I, self.W = int(max_slices), int(max_inst), int(width)
        self.device = torch.device(device if device is not None else 'cuda')
        S, I, W = self.S, self.I, self.W
        dev = self.device
        i32, f32, f64 = torch.int32, torch.float32, torch.float64
        self.slice_inst = torch.full((S,), -1, dtype=i32, device=dev)
        self.slice_w = torch.zeros(S, dtype=i32, device=dev)
        self.cols = torch.zeros(S * W * 64, dtype=i32, device=dev)
        self.cols16 = torch.zeros(S * W * 64, dtype=torch.int16, device=dev)
        self.slice_narrow = torch.zeros(S, dtype=torch.uint8, device=dev)
        self.vals = torch.zeros(S * W * 64, dtype=f64, device=dev)
        self.vals32 = torch.zeros(S * W * 64, dtype=f32, device=dev)
        self.diag = torch.zeros(S * 64, dtype=f64, device=dev)
        self.inst_slice0 = torch.zeros(I, dtype=i32, device=dev)
        self.inst_nslices = torch.zeros(I, dtype=i32, device=dev)
        self.live_slices = torch.zeros(S, dtype=i32, device=dev)
        self.n_live_slices = torch.zeros(1, dtype=i32, device=dev)
        self.live_inst = torch.zeros(I, dtype=i32, device=dev)
        self.n_live_inst = torch.zeros(1, dtype=i32, device=dev)
        R = S * 64
        self.x = torch.zeros(R, dtype=f64, device=dev)
        self.b = torch.zeros(R, dtype=f64, device=dev)
        self.f32 = {k: torch.zeros(R, dtype=f32, device=dev) for k in ('d', 'rh', 'dinv', 'p')}
        self.f32.update({k: torch.zeros((R, n), dtype=f32, device=dev) for k, n in (('u', 4), ('w', 2))})
        self.partial = {k: torch.zeros(S * n, dtype=f64, device=dev) for k, n in (('pa', 1), ('pb', 5))}
        self.chunks = torch.zeros((S, 4), dtype=i32, device=dev)
        self.n_chunks = torch.zeros(1, dtype=i32, device=dev)
        self.scal = torch.zeros(I * _lib.KS_NSCAL, dtype=f64, device=dev)
        self._state = torch.zeros((2, I), dtype=i32, device=dev)  # read by the host in one copy
        self.status, self.steps_left = self._state[0], self._state[1]
        self.status_t = torch.zeros(I, dtype=i32, device=dev)
        self._posts, self._spare = collections.deque(), []

        e = _lib.MfvEllBatch()
        e.nb_slices, e.width, e.nb_inst = S, W, I
        for k in ('slice_inst', 'slice_w', 'cols', 'vals', 'vals32', 'diag', 'inst_slice0', 'inst_nslices',
                  'live_slices', 'n_live_slices', 'live_inst', 'n_live_inst', 'cols16', 'slice_narrow'):
            setattr(e, k, getattr(self, k).data_ptr())
        w = _lib.MfvKrylovFused()
        for k, t in dict(self.f32, **self.partial).items():
            setattr(w, k, t.data_ptr())
        for k in ('x', 'b', 'scal', 'status', 'status_t', 'chunks', 'n_chunks'):
            setattr(w, k, getattr(self, k).data_ptr())
        self._e, self._w = e, w
        self._ranges = RangeAllocator(S)
        self._inst = {}                # inst -> (slice0, nslices, nrows)
        self._free_ids = list(range(I - 1, -1, -1))
        self._slice_bytes = self._count_slice_bytes()

    def enable_advection(self, slots):
        """Time steps on the device (mfv_krylov_fused_tick with steps_left): tables of ``slots``
        (a multiple of four) faces a row. Before the first graph tick."""
        import torch
        R = self.S * 64
        self.adv_up = torch.full((slots, R), -1, dtype=torch.int32, device=self.device)
        self.adv_coef = torch.zeros((slots, R), dtype=torch.float64, device=self.device)
        self.adv_vol = torch.ones(R, dtype=torch.float64, device=self.device)
        for k in ('steps_left', 'adv_up', 'adv_coef', 'adv_vol'):
            setattr(self._w, k, getattr(self, k).data_ptr())
        self._w.adv_slots = int(slots)
        self._slice_bytes = self._count_slice_bytes()

    # -- arena ----------------------------------------------------------------------------------
    @property
    def eptr(self):
        return ctypes.byref(self._e)

    @property
    def wptr(self):
        return ctypes.byref(self._w)

    def bytes_per_slice(self):
        """HBM bytes one slice of an instance occupies: matrix slots, vectors, chunk sums and lists, and the
        advection tables once they are enabled."""
        return self._slice_bytes

    def _count_slice_bytes(self):
        own = [self.slice_inst, self.slice_w, self.slice_narrow, self.cols, self.cols16, self.vals, self.vals32,
               self.diag, self.live_slices, self.chunks, self.x, self.b]
        own += list(self.f32.values()) + list(self.partial.values())
        own += [getattr(self, k) for k in ('adv_up', 'adv_coef', 'adv_vol') if hasattr(self, k)]
        return sum(t.numel() * t.element_size() for t in own) // max(1, self.S)

    def free_slices(self):
        return self._ranges.available()

    def alloc(self, nrows):
        """Reserve ceil(nrows/64) contiguous slices; returns the instance id or None."""
        ns = (int(nrows) + 63) // 64
        if ns == 0 or not self._free_ids:
            return None
        s0 = self._ranges.alloc(ns)
        if s0 is None:
            return None
        inst = self._free_ids.pop()
        self._inst[inst] = (s0, ns, int(nrows))
        self.slice_inst[s0:s0 + ns] = inst
        self.slice_w[s0:s0 + ns] = 0
        self.slice_narrow[s0:s0 + ns] = 0  # int32 columns until narrow_columns has checked this matrix
        self.status[inst] = _lib.KS_IDLE
        return inst

    def release(self, inst):
        s0, ns, _ = self._inst.pop(inst)
        self.slice_inst[s0:s0 + ns] = -1
        self.status[inst] = _lib.KS_IDLE
        self._free_ids.append(inst)
        self._ranges.release(s0, ns)

    def rows(self, inst):
        s0, ns, n = self._inst[inst]
        return s0 * 64, n, ns

    def publish(self):
        """Upload the live lists (ascending slice order; instances by id)."""
        import torch
        insts = sorted(self._inst)
        slices = [np.arange(self._inst[i][0], self._inst[i][0] + self._inst[i][1], dtype=np.int32) for i in insts]
        sl = np.concatenate(slices) if slices else np.zeros(0, np.int32)
        sl.sort()
        if len(sl):
            self.live_slices[:len(sl)] = torch.from_numpy(sl).to(self.device)
        self.n_live_slices.fill_(len(sl))
        if insts:
            self.live_inst[:len(insts)] = torch.tensor(insts, dtype=torch.int32, device=self.device)
            s0 = torch.tensor([self._inst[i][0] for i in insts], dtype=torch.int32, device=self.device)
            ns = torch.tensor([self._inst[i][1] for i in insts], dtype=torch.int32, device=self.device)
            idx = torch.tensor(insts, dtype=torch.long, device=self.device)
            self.inst_slice0[idx] = s0
            self.inst_nslices[idx] = ns
        self.n_live_inst.fill_(len(insts))
        ch = chunk_list([(i,) + self._inst[i][:2] for i in insts])
        if len(ch):
            self.chunks[:len(ch)] = torch.from_numpy(ch).to(self.device)
        self.n_chunks.fill_(len(ch))
        self._n_live = (len(sl), len(insts), len(ch))

    # -- matrix and system ------------------------------------------------------------------------
    def assemble_diamond(self, inst, ddia, node_dir, face_dir_rank):
        """Writes the diamond matrix of a DeviceDiamond into the instance's slices
        (get_triplet_2d, ast/functions2d.py:328-580; get_triplet_3d, ast/functions3d.py:498-782)."""
        import torch
        row0, n, ns = self.rows(inst)
        if n != ddia.dmesh.C:
            raise ValueError("instance has %d rows, mesh %d cells" % (n, ddia.dmesh.C))
        s0 = row0 // 64
        info = torch.zeros(2, dtype=torch.int32, device=self.device)
        st = stream_ptr()
        sw = self.slice_w[s0:s0 + ns]
        _lib.call('mfv_diamond_widths', ddia.ptr, node_dir.data_ptr(), face_dir_rank.data_ptr(), sw.data_ptr(),
                  info.data_ptr(), st)
        ov, wmax = info.tolist()
        if ov or wmax > self.W:
            raise _lib.MfvError("diamond matrix rows need %d slots, the ELL arena has %d" % (wmax, self.W))
        off = s0 * self.W * 64
        _lib.call('mfv_diamond_assemble', ddia.ptr, node_dir.data_ptr(), face_dir_rank.data_ptr(), row0, self.W,
                  sw.data_ptr(), self.cols[off:].data_ptr(), self.vals[off:].data_ptr(), self.vals32[off:].data_ptr(),
                  self.diag[row0:].data_ptr(), st)
        self.narrow_columns(inst)
        return wmax

    def narrow_columns(self, inst, enable=True):
        """16-bit column offsets for the instance's slices whose columns stay within +-32767 of
        their rows (mfv_ell_narrow_columns); enable=False makes every slice read the int32
        columns (same results)."""
        row0, _, ns = self.rows(inst)
        s0 = row0 // 64
        if enable:
            _lib.call('mfv_ell_narrow_columns', self.eptr, s0, ns, self.cols16.data_ptr(), self.slice_narrow.data_ptr(),
                      stream_ptr())
        else:
            self.slice_narrow[s0:s0 + ns].zero_()

    def configure(self, inst, sigma, tau, tol=1e-10, tol_in=1e-4, maxit_in=400, maxit_out=60, dt=0.):
        """Operator coefficients, stopping parameters and time step of one instance (counters
        zeroed)."""
        import torch
        sc = np.zeros(_lib.KS_NSCAL)
        sc[_lib.KS_DT] = dt
        sc[_lib.KS_SIGMA], sc[_lib.KS_TAU] = sigma, tau
        sc[_lib.KS_TOL_OUT], sc[_lib.KS_TOL_IN] = tol, tol_in
        sc[_lib.KS_MAXIT_IN], sc[_lib.KS_MAXIT_OUT] = maxit_in, maxit_out
        k = inst * _lib.KS_NSCAL
        self.scal[k:k + _lib.KS_NSCAL] = torch.from_numpy(sc).to(self.device)

    def set_system(self, inst, sigma, tau, b, x0=None, tol=1e-10, tol_in=1e-4, maxit_in=400, maxit_out=60):
        """Right-hand side, initial guess and parameters of one instance; status -> START."""
        row0, n, ns = self.rows(inst)
        seg = slice(row0, row0 + ns * 64)
        self.b[seg].zero_()
        self.x[seg].zero_()
        self.b[row0:row0 + n] = b
        if x0 is not None:
            self.x[row0:row0 + n] = x0
        self.configure(inst, sigma, tau, tol, tol_in, maxit_in, maxit_out)
        self.status[inst] = _lib.KS_START

    def solution(self, inst):
        row0, n, _ = self.rows(inst)
        return self.x[row0:row0 + n]

    def scalars(self, inst):
        k = inst * _lib.KS_NSCAL
        return self.scal[k:k + _lib.KS_NSCAL].cpu().numpy()

    # -- execution ----------------------------------------------------------------------------
    def grids(self):
        """Blocks of the per-slice (spmv) and per-instance kernels."""
        nsl, ni, _ = getattr(self, '_n_live', (0, 0, 0))
        return max(1, min(4096, (nsl + 3) // 4)), max(1, ni)

    def tick(self, n_iter=8, grid_slices=None, grid_inst=None, stream=None, graph=False):
        """One tick of every live instance (``grid_slices``: blocks of its kernels; ``grid_inst`` is
        taken and not used, no kernel runs per instance). With ``graph=True`` the tick's launches are
        replayed from a HIP graph captured once per (n_iter, grid size rounded up to a power of
        two): the kernels read the live lists from device memory, so a graph stays valid as
        instances come and go, and the result is the same bits as the eager tick."""
        gs = int(grid_slices or max(1, min(16384, getattr(self, '_n_live', (0, 0, 0))[2])))
        n_iter = int(n_iter) or 1
        if not graph:
            _lib.call('mfv_krylov_fused_tick', self.eptr, self.wptr, n_iter, gs, stream_ptr(stream))
            return
        key = (n_iter, min(16384, _pow2(gs)))
        graphs = self.__dict__.setdefault('_graphs', {})
        g = graphs.get(key)
        if g is None:
            out = ctypes.c_void_p()
            _lib.call('mfv_krylov_fused_graph', self.eptr, self.wptr, key[0], key[1], ctypes.byref(out))
            g = graphs[key] = out.value
        _lib.call('mfv_graph_launch', g, stream_ptr(stream))

    def post_state(self, tag=None):
        """Asks for a host copy of (status, steps_left) as they are at this point of the current
        stream; ``take_state`` returns the copies in the order they were asked for, with ``tag``."""
        import torch
        buf, ev = self._spare.pop() if self._spare else \
            (torch.empty((2, self.I), dtype=torch.int32, pin_memory=True), torch.cuda.Event())
        buf.copy_(self._state, non_blocking=True)
        ev.record()
        self._posts.append((buf, ev, tag))

    def posted(self):
        return len(self._posts)

    def take_state(self):
        buf, ev, tag = self._posts.popleft()
        ev.synchronize()
        st = buf.numpy().copy()
        self._spare.append((buf, ev))
        return st[0], st[1], tag

    def drop_states(self):
        """Forgets the copies still on their way (waits for them: their buffers are used again)."""
        while self._posts:
            self.take_state()

    def close_graphs(self):
        """Release the captured ticks (after the device has finished any replay of them)."""
        graphs = self.__dict__.pop('_graphs', {})
        if graphs:
            import torch
            torch.cuda.synchronize(self.device)
        for g in graphs.values():
            _lib.call('mfv_graph_destroy', g)

    def __del__(self):
        try:
            self.close_graphs()
        except Exception:
            pass

    def spmv(self, x, y):
        gs, _ = self.grids()
        _lib.call('mfv_ell_spmv', self.eptr, x.data_ptr(), y.data_ptr(), gs, stream_ptr())

    def run(self, insts, n_iter=8, max_ticks=20000, graph=False):
        """Tick until every listed instance is DONE or FAILED; returns their statuses."""
        idx = np.asarray(list(insts), dtype=np.int64)
        # the next tick is on its way while the state after the last one is looked at; a finished
        # instance stays as it is
        try:
            for k in range(max_ticks + 1):
                if k < max_ticks:
                    self.tick(n_iter, graph=graph)
                    self.post_state()
                if self.posted() > 1 or (k == max_ticks and self.posted()):
                    st = self.take_state()[0][idx]
                    if np.all((st == _lib.KS_DONE) | (st == _lib.KS_FAILED)):
                        return st
        finally:
            self.drop_states()
        raise _lib.MfvError("Krylov solve did not finish in %d ticks" % max_ticks)
