"""Batched wave scaling: structure-of-arrays kernel records in HBM, one HIP
launch per (origin, up to 8 destinations).

This is the entry the scalar strategies (roofline.py, resimplified.py,
unified.py in this package) are thin wrappers of.  It stands in for the
reference's per-kernel loop (analyzer/habitat/analysis/predictor.py:116-124).
torch is used only to own device memory and to name the stream.
"""
import ctypes

import numpy as np
import torch

from habitat_amd import _lib

INT_COLUMNS = ("num_blocks", "block_size", "dynamic_smem", "static_smem", "regs_per_thread")
F64_COLUMNS = ("run_time_ns", "flop_sp_efficiency", "dram_read_bytes", "dram_write_bytes")


class KernelRecords:
    """Kernel records as columns on one GPU.

    Columns (length n): the launch geometry and resource use of
    cpp/src/cuda/kernel.h:64-151 as int32 (`num_blocks` = grid x*y*z), the
    measured time and the three metrics of wave_scaling/roofline.py:69-71 as
    float64.  Optional: `dest_regs` (int32, < 0 = no entry in the register
    table for the destination architecture) and `has_metrics` (uint8).
    """

    def __init__(self, columns, dest_regs=None, has_metrics=None):
        n = None
        self.columns = {}
        for name in INT_COLUMNS + F64_COLUMNS:
            t = columns[name]
            want = torch.int32 if name in INT_COLUMNS else torch.float64
            if not isinstance(t, torch.Tensor) or t.dtype != want or t.dim() != 1:
                raise TypeError("column %s must be a 1-D %s tensor" % (name, want))
            if not t.is_cuda:
                raise ValueError("column %s must live on the GPU" % name)
            t = t.contiguous()
            n = t.shape[0] if n is None else n
            if t.shape[0] != n:
                raise ValueError("column %s has length %d, expected %d" % (name, t.shape[0], n))
            self.columns[name] = t
        self.n = int(n)
        self.device = self.columns["num_blocks"].device
        self.dest_regs = self._optional(dest_regs, torch.int32, "dest_regs")
        self.has_metrics = self._optional(has_metrics, torch.uint8, "has_metrics")

    def _optional(self, t, dtype, name):
        if t is None:
            return None
        if t.dtype != dtype or t.dim() != 1 or t.shape[0] != self.n or not t.is_cuda:
            raise TypeError("%s must be a 1-D %s GPU tensor of length %d" % (name, dtype, self.n))
        return t.contiguous()

    def __len__(self):
        return self.n

    @classmethod
    def from_numpy(cls, rec, device="cuda"):
        """Upload a dict of numpy columns (synchronous copy)."""
        cols = {}
        for name in INT_COLUMNS:
            cols[name] = torch.from_numpy(np.ascontiguousarray(rec[name], np.int32)).to(device)
        for name in F64_COLUMNS:
            cols[name] = torch.from_numpy(np.ascontiguousarray(rec[name], np.float64)).to(device)
        dr = rec.get("dest_regs")
        hm = rec.get("has_metrics")
        if dr is not None:
            dr = torch.from_numpy(np.ascontiguousarray(dr, np.int32)).to(device)
        if hm is not None:
            hm = torch.from_numpy(np.ascontiguousarray(hm, np.uint8)).to(device)
        return cls(cols, dr, hm)


class WaveScaleOutput:
    """Preallocated outputs of one `wave_scale` call (all on the GPU).

    time_ns, occ_dest, wave_dest, status: [n_dest, n]; occ_origin, wave_origin: [n].
    """

    def __init__(self, n, n_dest, device, waves=True, status=True):
        self.n, self.n_dest = n, n_dest
        self.time_ns = torch.empty((n_dest, n), dtype=torch.float64, device=device)
        self.occ_origin = occ = torch.empty((n,), dtype=torch.int32, device=device)
        # (a tensor like one that is there takes three quarters of torch.empty's time)
        self.occ_dest = occ.new_empty((n_dest, n))
        self.wave_origin = torch.empty_like(occ) if waves else None
        self.wave_dest = torch.empty_like(self.occ_dest) if waves else None
        self.status = torch.empty((n_dest, n), dtype=torch.uint8, device=device) if status else None

    def wave_counts(self, num_blocks):
        """(origin [n], destination [n_dest, n]) int64 tensors of
        `num_blocks // wave_size`, the quotient the reference compares with zero
        to tell a kernel that fits one wave (wave_scaling/roofline.py:29-30),
        with Python's floor semantics; -1 where the wave size is 0 (the
        reference raises ZeroDivisionError there).  Needs the wave-size outputs."""
        if self.wave_origin is None:
            raise ValueError("allocate the output with waves=True")
        nb = num_blocks.to(torch.int64)

        def quotient(wave):
            wave = wave.to(torch.int64)
            safe = torch.where(wave == 0, torch.ones_like(wave), wave)
            q = torch.div(nb.expand_as(wave), safe, rounding_mode="floor")
            return torch.where(wave == 0, torch.full_like(q, -1), q)

        return quotient(self.wave_origin), quotient(self.wave_dest)


def _ptr(t):
    return t.data_ptr() if t is not None else None


try:
    # the current stream's handle without an object around it
    from torch._C import _cuda_getCurrentRawStream as _raw_stream
except ImportError:
    def _raw_stream(index):
        return torch.cuda.current_stream(index).cuda_stream


def wave_scale(records, origin, dests, out=None, stream=None, waves=True, status=True):
    """Scale every record from `origin` to each device in `dests`.

    `origin` and the items of `dests` are DeviceProperties.  Returns a
    WaveScaleOutput (the one passed in `out`, if any); the work is enqueued on
    `stream` (default: torch's current stream) and not synchronised.
    """
    if not isinstance(dests, (list, tuple)):
        dests = [dests]
    n_dest = len(dests)
    if out is None:
        out = WaveScaleOutput(records.n, n_dest, records.device, waves=waves, status=status)
    elif out.n != records.n or out.n_dest != n_dest:
        raise ValueError("output buffers were allocated for another shape")
    specs = (ctypes.byref(dests[0].spec) if n_dest == 1 else
             (_lib.DeviceSpec * max(n_dest, 1))(*[d.spec for d in dests]))
    index = records.device.index
    handle = _raw_stream(index) if stream is None else stream.cuda_stream
    # A call for the kernels of one trace is what the host does for it: 4.4 us in
    # hbt_wave_scale with its launch, and half of the rest was wrapping 18 pointers, asking
    # for the stream and entering the device that is the current one already.
    if torch.cuda.current_device() == index:
        rc = _enqueue_wave_scale(records, origin, specs, n_dest, out, handle)
    else:
        with torch.cuda.device(index):
            rc = _enqueue_wave_scale(records, origin, specs, n_dest, out, handle)
    _lib.check(rc, "hbt_wave_scale")
    return out


def _enqueue_wave_scale(records, origin, specs, n_dest, out, stream):
    c, regs, metrics = records.columns, records.dest_regs, records.has_metrics
    return _lib.lib().hbt_wave_scale(
        ctypes.byref(origin.spec), specs, n_dest, records.n,
        c["num_blocks"].data_ptr(), c["block_size"].data_ptr(), c["dynamic_smem"].data_ptr(),
        c["static_smem"].data_ptr(), c["regs_per_thread"].data_ptr(),
        None if regs is None else regs.data_ptr(),
        c["run_time_ns"].data_ptr(), c["flop_sp_efficiency"].data_ptr(),
        c["dram_read_bytes"].data_ptr(), c["dram_write_bytes"].data_ptr(),
        None if metrics is None else metrics.data_ptr(),
        _ptr(out.time_ns), _ptr(out.occ_origin), _ptr(out.occ_dest), _ptr(out.wave_origin),
        _ptr(out.wave_dest), _ptr(out.status), stream)


class DeviceTable:
    """A sweep of destination devices resident on the GPU (`hbt_device_table`)."""

    def __init__(self, origin, dests):
        self.origin = origin
        self.dests = list(dests)
        if not self.dests:
            raise ValueError("a device table needs at least one destination")
        specs = (_lib.DeviceSpec * len(self.dests))(*[d.spec for d in self.dests])
        err = ctypes.c_int(0)
        self.torch_device = torch.device("cuda", torch.cuda.current_device())
        self.handle = _lib.lib().hbt_device_table_create(
            ctypes.byref(origin.spec), specs, len(self.dests), ctypes.byref(err))
        if not self.handle:
            raise _lib.HabitatLibraryError(err.value, "hbt_device_table_create")

    def __len__(self):
        return len(self.dests)

    def __del__(self):
        try:
            if getattr(self, "handle", None):
                _lib.lib().hbt_device_table_destroy(self.handle)
                self.handle = None
        except Exception:
            pass


def wave_scale_sum(records, table, segment=None, n_segments=1, stream=None, segment_start=None,
                   workspace=None):
    """Per destination of `table` and per segment, the sum of the scaled times
    of `records` (see hbt_wave_scale_sum).  `segment`: int32 GPU tensor [n] or
    None.  Or `segment_start`: int64 GPU tensor [n_segments + 1] when segment s
    is the run of records [segment_start[s], segment_start[s + 1]): the times
    are then added in the records' order, as the reference adds a pass's
    kernels, without floating-point atomics (hbt_wave_scale_sum_ordered; the
    scaled times pass through `workspace`, a float64 GPU tensor of n_dest x n
    elements, allocated here when not given).
    Returns (sums [n_dest, n_segments] float64, bad [n_dest] int32), both GPU
    tensors, not synchronised."""
    if records.device != table.torch_device:
        raise ValueError("records and device table live on different GPUs")
    if segment_start is not None:
        if segment is not None:
            raise ValueError("give segment or segment_start, not both")
        if (segment_start.dtype != torch.int64 or segment_start.shape != (n_segments + 1,)
                or segment_start.device != records.device):
            raise TypeError("segment_start must be an int64 GPU tensor of length %d"
                            % (n_segments + 1))
        n_dest = len(table)
        sums = torch.empty((n_dest, n_segments), dtype=torch.float64, device=records.device)
        bad = torch.empty((n_dest,), dtype=torch.int32, device=records.device)
        if workspace is None:
            workspace = torch.empty((n_dest, max(records.n, 1)), dtype=torch.float64,
                                    device=records.device)
        elif (workspace.dtype != torch.float64 or workspace.numel() < n_dest * records.n
              or workspace.device != records.device or not workspace.is_contiguous()):
            raise TypeError("workspace must be a contiguous float64 GPU tensor of at least "
                            "%d elements" % (n_dest * records.n))
        if stream is None:
            stream = torch.cuda.current_stream(records.device)
        c = records.columns
        with torch.cuda.device(records.device):
            rc = _lib.lib().hbt_wave_scale_sum_ordered(
                table.handle, records.n,
                _ptr(c["num_blocks"]), _ptr(c["block_size"]), _ptr(c["dynamic_smem"]),
                _ptr(c["static_smem"]), _ptr(c["regs_per_thread"]), _ptr(records.dest_regs),
                _ptr(c["run_time_ns"]), _ptr(c["flop_sp_efficiency"]),
                _ptr(c["dram_read_bytes"]), _ptr(c["dram_write_bytes"]),
                _ptr(records.has_metrics), _ptr(segment_start.contiguous()), n_segments,
                _ptr(workspace), _ptr(sums), _ptr(bad), ctypes.c_void_p(stream.cuda_stream))
        _lib.check(rc, "hbt_wave_scale_sum_ordered")
        return sums, bad
    if segment is not None and (segment.dtype != torch.int32 or segment.shape != (records.n,)
                                or segment.device != records.device):
        raise TypeError("segment must be an int32 GPU tensor of length %d" % records.n)
    n_dest = len(table)
    sums = torch.empty((n_dest, n_segments), dtype=torch.float64, device=records.device)
    bad = torch.empty((n_dest,), dtype=torch.int32, device=records.device)
    if stream is None:
        stream = torch.cuda.current_stream(records.device)
    c = records.columns
    with torch.cuda.device(records.device):
        rc = _lib.lib().hbt_wave_scale_sum(
            table.handle, records.n,
            _ptr(c["num_blocks"]), _ptr(c["block_size"]), _ptr(c["dynamic_smem"]),
            _ptr(c["static_smem"]), _ptr(c["regs_per_thread"]), _ptr(records.dest_regs),
            _ptr(c["run_time_ns"]), _ptr(c["flop_sp_efficiency"]), _ptr(c["dram_read_bytes"]),
            _ptr(c["dram_write_bytes"]), _ptr(records.has_metrics),
            _ptr(segment.contiguous() if segment is not None else None), n_segments,
            _ptr(sums), _ptr(bad), ctypes.c_void_p(stream.cuda_stream))
    _lib.check(rc, "hbt_wave_scale_sum")
    return sums, bad


def _is_buffer(t, dtype, shape, device):
    """Whether a kernel can write (or read) `t` as [shape] of dtype from its first element."""
    return t.dtype == dtype and t.shape == shape and t.device == device and t.is_contiguous()


class TotalsCall:
    """hbt_wave_scale_sum_totals for records and destinations that stay the same: what the
    call is made of is looked over and laid out once.  `rows`: int32 GPU tensor naming each
    destination's row of the outputs (None: row d)."""

    def __init__(self, records, table, segment_start, n_segments, workspace, rows, n_rows,
                 constant_ms):
        if records.device != table.torch_device:
            raise ValueError("records and device table live on different GPUs")
        if (segment_start.dtype != torch.int64 or segment_start.shape != (n_segments + 1,)
                or workspace.dtype != torch.float64
                or workspace.numel() < len(table) * records.n
                or (rows is not None and (rows.dtype != torch.int32 or len(rows) != len(table)))
                or any(t.device != records.device or not t.is_contiguous()
                       for t in (segment_start, workspace) + (() if rows is None else (rows,)))):
            raise TypeError("segment_start must be int64 [%d], workspace float64 [%d] and rows "
                            "int32 [%d], on the records' GPU"
                            % (n_segments + 1, len(table) * records.n, len(table)))
        self.shape = (n_rows, n_segments)
        self._device = records.device
        c = dict(records.columns)
        # what the pointers point into, whatever becomes of the objects they came in
        self._keep = (c, records.dest_regs, records.has_metrics, table, segment_start, workspace, rows)
        self._args = (
            table.handle, records.n,
            _ptr(c["num_blocks"]), _ptr(c["block_size"]), _ptr(c["dynamic_smem"]),
            _ptr(c["static_smem"]), _ptr(c["regs_per_thread"]), _ptr(records.dest_regs),
            _ptr(c["run_time_ns"]), _ptr(c["flop_sp_efficiency"]),
            _ptr(c["dram_read_bytes"]), _ptr(c["dram_write_bytes"]),
            _ptr(records.has_metrics), _ptr(segment_start), n_segments, _ptr(workspace),
            _ptr(rows), n_rows, constant_ms)

    def __call__(self, sums, bad, totals, stream):
        """sums float64 [n_rows, n_segments], bad int32 [n_rows], totals float64 [n_rows]:
        contiguous GPU tensors; only the rows of this call are written."""
        if not (_is_buffer(sums, torch.float64, self.shape, self._device)
                and _is_buffer(bad, torch.int32, self.shape[:1], self._device)
                and _is_buffer(totals, torch.float64, self.shape[:1], self._device)):
            raise TypeError("sums must be float64 %s, bad int32 and totals float64 of its rows, "
                            "contiguous on the records' GPU" % (list(self.shape),))
        with torch.cuda.device(self._device):
            rc = _lib.lib().hbt_wave_scale_sum_totals(
                *self._args, sums.data_ptr(), bad.data_ptr(), totals.data_ptr(),
                stream.cuda_stream)
        _lib.check(rc, "hbt_wave_scale_sum_totals")


def ratio_scale_kinds(kinds, n_dest, totals, stream):
    """ratio_scale for several kinds of operation in one launch.  kinds: (name, pred,
    run_time_ms, op_row) each, as there.  Adds to `totals`; returns ({name: ms [n_dest,
    n_ops]}, clamped int32 [n_dest]).  All tensors are on one GPU, `totals` is contiguous."""
    device = totals.device
    if not totals.is_cuda or not _is_buffer(totals, torch.float64, (n_dest,), device):
        raise TypeError("totals must be a contiguous float64 GPU tensor [%d]" % n_dest)
    clamped = torch.empty((n_dest,), dtype=torch.int32, device=totals.device)
    array = (_lib.RatioKind * max(len(kinds), 1))()
    out, keep = {}, []
    for entry, (name, pred, run_time_ms, op_row) in zip(array, kinds):
        n_ops = run_time_ms.shape[0]
        if pred.dtype != torch.float32 or pred.dim() != 2 or pred.shape[0] != n_dest + 1:
            raise TypeError("pred must be float32 [%d, rows]" % (n_dest + 1))
        if (run_time_ms.dtype != torch.float64 or op_row.dtype != torch.int32
                or op_row.shape != (n_ops,)):
            raise TypeError("run_time_ms must be float64 and op_row int32, both [%d]" % n_ops)
        if any(t.device != device for t in (pred, run_time_ms, op_row)):
            raise ValueError("pred, run_time_ms and op_row must live on the totals' GPU")
        pred, run_time_ms, op_row = pred.contiguous(), run_time_ms.contiguous(), op_row.contiguous()
        out[name] = torch.empty((n_dest, n_ops), dtype=torch.float64, device=pred.device)
        keep.append((pred, run_time_ms, op_row))
        entry.pred, entry.op_row = pred.data_ptr(), op_row.data_ptr()
        entry.run_time_ms, entry.out_ms = run_time_ms.data_ptr(), out[name].data_ptr()
        entry.n_rows, entry.n_ops = pred.shape[1], n_ops
    with torch.cuda.device(totals.device):
        rc = _lib.lib().hbt_ratio_scale_kinds(array, len(kinds), n_dest, totals.data_ptr(),
                                              clamped.data_ptr(), stream.cuda_stream)
    _lib.check(rc, "hbt_ratio_scale_kinds")
    return out, clamped


def ratio_scale(pred, run_time_ms, n_dest, totals=None, want_ms=True, stream=None, op_row=None,
                clamped=None):
    """MLP-predicted operations on a sweep (see hbt_ratio_scale).  pred: float32
    GPU tensor [(n_dest + 1), n_rows] whose last row is the origin; run_time_ms:
    float64 GPU tensor [n_ops]; op_row: int32 GPU tensor [n_ops] naming each
    operation's column of pred (None: column o, n_rows == n_ops).  Returns ms
    [n_dest, n_ops] (or None), adds the per-destination sums to `totals`
    ([n_dest] float64) and the number of negative predictions replaced by 0 to
    `clamped` ([n_dest] int32) if given."""
    n_ops = run_time_ms.shape[0]
    n_rows = pred.shape[1] if pred.dim() == 2 else -1
    if pred.dtype != torch.float32 or pred.dim() != 2 or pred.shape[0] != n_dest + 1 or (
            op_row is None and n_rows != n_ops):
        raise TypeError("pred must be float32 [%d, %d]" % (n_dest + 1, n_ops))
    if op_row is not None and (op_row.dtype != torch.int32 or op_row.shape != (n_ops,)):
        raise TypeError("op_row must be int32 [%d]" % n_ops)
    if run_time_ms.dtype != torch.float64 or (totals is not None and (
            totals.dtype != torch.float64 or totals.shape != (n_dest,))):
        raise TypeError("run_time_ms and totals must be float64")
    if clamped is not None and (clamped.dtype != torch.int32 or clamped.shape != (n_dest,)):
        raise TypeError("clamped must be int32 [%d]" % n_dest)
    if any(t is not None and (t.device != pred.device or not t.is_contiguous())
           for t in (totals, clamped)):
        raise TypeError("totals and clamped must be contiguous, on the predictions' GPU")
    pred = pred.contiguous()
    out = (torch.empty((n_dest, n_ops), dtype=torch.float64, device=pred.device)
           if want_ms else None)
    if stream is None:
        stream = torch.cuda.current_stream(pred.device)
    with torch.cuda.device(pred.device):
        rc = _lib.lib().hbt_ratio_scale(
            _ptr(pred), n_dest, n_rows, _ptr(op_row.contiguous() if op_row is not None else None),
            n_ops, _ptr(run_time_ms.contiguous()), _ptr(out), _ptr(totals), _ptr(clamped),
            ctypes.c_void_p(stream.cuda_stream))
    _lib.check(rc, "hbt_ratio_scale")
    return out


def roofline_gamma(records, origin, dest, stream=None):
    """The roofline exponent of every record (see hbt_roofline_gamma): a float64
    GPU tensor [n], NaN where the reference's assertion on gamma fails.  Every
    record is taken to have its metrics."""
    out = torch.empty((records.n,), dtype=torch.float64, device=records.device)
    if stream is None:
        stream = torch.cuda.current_stream(records.device)
    c = records.columns
    with torch.cuda.device(records.device):
        rc = _lib.lib().hbt_roofline_gamma(
            ctypes.byref(origin.spec), ctypes.byref(dest.spec), records.n,
            _ptr(c["run_time_ns"]), _ptr(c["flop_sp_efficiency"]), _ptr(c["dram_read_bytes"]),
            _ptr(c["dram_write_bytes"]), _ptr(out), ctypes.c_void_p(stream.cuda_stream))
    _lib.check(rc, "hbt_roofline_gamma")
    return out
