"""Series plan: the series -> chunk -> tile decomposition of the chunked scan.

Wraps bn_plan_create (include/bn_hip.h).  The reference handles one series per
model and sorts it in input_admin (bayesnewton/utils.py:234-265); a plan holds
any number of already-sorted series as CSR offsets and owns the device tables
and the workspace the chunked kernels need.
"""
import ctypes

import numpy as np
import torch

from . import _native as nat


def default_chunk_len(lengths, parallel=True):
    """Chunk length: the sequential filter (one chunk per series) when
    parallel=False, else a length that keeps every lane busy for a handful of
    steps while bounding each series to 128 x 128 chunks."""
    lengths = np.asarray(lengths, dtype=np.int64)
    nmax = int(lengths.max()) if lengths.size else 1
    if not parallel:
        return max(nmax, 1)
    c = 32
    while -(-nmax // c) > 128 * 128:
        c *= 2
    return c


def model_chunk_len(lengths, parallel=True, state_dim=1):
    """Chunk length of a model's (or a single operation's) own plan.

    The lane-per-chunk kernels take about 1 us a step of the longest chunk and a few
    wavefronts leave the chip idle, while the scans over the chunks' elements grow with the
    logarithm of their number.  Measured on MI355X (fused pass, chunk 32 -> this rule):
    10,000 steps 115 -> 66 us (Matern52) and 213 -> 147 us (Matern52 + Matern32), flat
    between 2 and 8; 200,000 steps 246 -> 206 us; 256 series with 276,000 steps
    204 -> 163 us; past about 60,000 chunks the chip is full, and short chunks only add
    scan work.
    Longer chunks than the default 32 save scan work but leave the site kernels, which take
    four lanes a chunk, fewer wavefronts: site update and pass of 4 M steps at 32 and 70 steps
    a chunk 406 and 484 us (state dimension 1), 531 and 587 (3), 589 and 627 (4), 703 and 728
    (5); of 8 M steps at 32 and 128 950 and 1005 (3), 1084 and 1060 (4), 1273 and 1216 (5); of
    15.7 M 1754 and 1838 (3), 2015 and 1918 (4), 2397 and 2145 (5).  (The gradient alone would
    take the longer ones a little sooner: 6016 and 5617 us at 4 M steps, state dimension 5.)
    Below 4096 steps in all the length stays 32, though 300 steps would take 47 us instead
    of 100: the float32 rows of the smoother are rounded from the chunk's end onwards, and in
    the energy of so few steps another length moves that rounding by as much as its whole
    error.  Series of at most 32 steps stay in one chunk each: no scan at all."""
    if not parallel:
        return default_chunk_len(lengths, parallel)
    lengths = np.asarray(lengths, dtype=np.int64)
    nmax = max(int(lengths.max()) if lengths.size else 1, 1)
    total = int(lengths.sum())
    if nmax <= 32:
        return nmax
    if total < 4096:
        return 32
    if state_dim > 3 and total >= 128 * 57344:
        return max(128, -(-nmax // (128 * 128)))
    return max(8, -(-nmax // (128 * 128)), min(32, -(-total // 57344)))


class SeriesPlan:
    """Device-side decomposition of B sorted series (CSR offsets) into chunks.

    offsets: int64 [B+1] with offsets[0] = 0.  chunk_len: steps per lane.
    """

    def __init__(self, offsets, chunk_len=None, parallel=True, device=None):
        off = np.ascontiguousarray(np.asarray(offsets, dtype=np.int64))
        if off.ndim != 1 or off.size < 2 or off[0] != 0 or np.any(np.diff(off) < 0):
            raise ValueError("offsets must be a non-decreasing int64 vector starting at 0")
        self.offsets = off
        self.lengths = np.diff(off)
        self.n_series = off.size - 1
        self.n_steps = int(off[-1])
        if chunk_len is None:
            chunk_len = default_chunk_len(self.lengths, parallel)
        self.device = torch.device(device) if device is not None else torch.device("cuda", torch.cuda.current_device())
        h = ctypes.c_void_p()
        with torch.cuda.device(self.device):
            nat.check(nat.lib().bn_plan_create(off.ctypes.data_as(ctypes.c_void_p), self.n_series, int(chunk_len),
                                               ctypes.byref(h)))
        self._adopt(h, chunk_len)

    @classmethod
    def for_call(cls, n, chunk_len, device):
        """Plan of one series that is used and dropped on the current stream of the current
        device: its tables are made and given back in the stream's order, so that neither
        waits for the device.  Not under graph capture, where a plan has to exist before."""
        off = np.array([0, n], dtype=np.int64)
        if torch.cuda.is_current_stream_capturing():
            return cls(off, chunk_len=chunk_len, device=device)
        L = nat.lib()
        nbytes = int(L.bn_plan_single_bytes(n, chunk_len))
        nat.check(0 if nbytes > 0 else -1)
        self = cls.__new__(cls)
        self.offsets, self.lengths, self.n_series, self.n_steps = off, np.diff(off), 1, int(n)
        self.device = device
        self._tables = torch.empty(nbytes, dtype=torch.uint8, device=device)
        h = ctypes.c_void_p()
        nat.check(L.bn_plan_create_single(n, chunk_len, nat.ptr(self._tables), nbytes, nat.stream_ptr(),
                                          ctypes.byref(h)))
        self._adopt(h, chunk_len)
        return self

    def _adopt(self, h, chunk_len):
        L = nat.lib()
        self.chunk_len = int(chunk_len)
        self._h = h
        self.n_slots = int(L.bn_plan_num_slots(h))
        self.n_chunks = int(L.bn_plan_num_chunks(h))
        self.n_tiles = int(L.bn_plan_num_tiles(h))
        self._ws = {}

    @property
    def handle(self):
        return self._h

    def __del__(self):
        h = getattr(self, "_h", None)
        if h is not None and h.value:
            try:
                nat.lib().bn_plan_destroy(h)
            except Exception:
                pass
            self._h = None

    def workspace(self, desc):
        """Workspace tensor for a kernel descriptor (cached per state dimension)."""
        key = (desc.n_comp, desc.kind[0], desc.kind[1])
        ws = self._ws.get(key)
        if ws is None:
            nbytes = int(nat.lib().bn_workspace_bytes(self._h, ctypes.byref(desc)))
            if nbytes < 0:
                raise nat.NativeError("bn_workspace_bytes failed")
            ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device=self.device)
            self._ws[key] = ws
        return ws

    # ---- layout conversion -----------------------------------------------------
    def gather(self, x, pad=0.0):
        """[N] or [N, w] (float32/float64, on the device) -> tiled [w, n_slots]."""
        if x.dim() == 1:
            x = x[:, None]
        x = x.contiguous()
        if x.shape[0] != self.n_steps:
            raise ValueError(f"expected {self.n_steps} rows, got {x.shape[0]}")
        w = x.shape[1]
        out = torch.empty((w, self.n_slots), dtype=x.dtype, device=self.device)
        L = nat.lib()
        if x.dtype == torch.float32:
            nat.check(L.bn_plan_gather_f32(self._h, nat.ptr(x), nat.ptr(out), w, float(pad), nat.stream_ptr()))
        elif x.dtype == torch.float64:
            nat.check(L.bn_plan_gather_f64(self._h, nat.ptr(x), nat.ptr(out), w, float(pad), nat.stream_ptr()))
        else:
            raise TypeError(f"gather supports float32/float64, got {x.dtype}")
        return out

    def gather_mask(self, mask):
        """bool/uint8 [N] -> tiled uint8 [n_slots] (padding = 1, i.e. missing)."""
        m = mask.reshape(-1).to(torch.uint8).contiguous()
        out = torch.empty(self.n_slots, dtype=torch.uint8, device=self.device)
        nat.check(nat.lib().bn_plan_gather_u8(self._h, nat.ptr(m), nat.ptr(out), 1, nat.stream_ptr()))
        return out

    def scatter_planes(self, t):
        """tiled float32 [w, n_slots] -> float64 [w, N]."""
        if t.dtype != torch.float32:
            raise TypeError(f"scatter_planes supports float32, got {t.dtype}")
        t = t.contiguous()
        out = torch.empty((t.shape[0], self.n_steps), dtype=torch.float64, device=self.device)
        nat.check(nat.lib().bn_plan_scatter_planes(self._h, nat.ptr(t), nat.ptr(out), t.shape[0], nat.stream_ptr()))
        return out

    def scatter(self, t):
        """tiled [w, n_slots] -> [N, w]."""
        if t.dim() == 1:
            t = t[None, :]
        t = t.contiguous()
        w = t.shape[0]
        out = torch.empty((self.n_steps, w), dtype=t.dtype, device=self.device)
        L = nat.lib()
        if t.dtype == torch.float32:
            nat.check(L.bn_plan_scatter_f32(self._h, nat.ptr(t), nat.ptr(out), w, nat.stream_ptr()))
        elif t.dtype == torch.float64:
            nat.check(L.bn_plan_scatter_f64(self._h, nat.ptr(t), nat.ptr(out), w, nat.stream_ptr()))
        else:
            raise TypeError(f"scatter supports float32/float64, got {t.dtype}")
        return out
