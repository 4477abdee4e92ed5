"""Seeded device draws, regenerated by libnoise_amd instead of materialised.

`DeviceGenerator` follows torch.Generator('cuda').manual_seed(seed): every draw takes the generator's
current philox offset and advances it by torch's increment for that draw's size
(torch: ATen/native/hip/DistributionTemplates.h:52-65, 126-131). A `Draw` names one such draw, and any
slice of it can be produced on the device without the rest (noise_normal_fill, noise_gather_slices).
"""
from dataclasses import dataclass

import ctypes

import torch

from . import _lib

GATHER_ROWS = 65535  # rows of one gather launch (a grid's second dimension)


def draw_layout(numel, device=None):
    """(threads, offset increment) of a torch draw of `numel` values on `device`."""
    dev = torch.device('cuda', torch.cuda.current_device()) if device is None else torch.device(device)
    threads, inc = ctypes.c_int64(), ctypes.c_int64()
    _lib.call('noise_draw_layout', dev.index or 0, int(numel), ctypes.byref(threads), ctypes.byref(inc))
    return threads.value, inc.value


@dataclass(frozen=True)
class Draw:
    """One draw of `numel` values by a device generator at (seed, offset), laid out over `threads`."""
    seed: int
    offset: int
    threads: int
    numel: int
    device: torch.device

    def normal(self, first=0, n=None, mean=0.0, std=1.0, out=None):
        """Elements [first, first + n) of torch.randn(numel) * std + mean from this draw (fp32)."""
        n = self.numel - first if n is None else n
        if first < 0 or n < 0 or first + n > self.numel:
            raise ValueError(f'slice [{first}, {first + n}) outside a draw of {self.numel}')
        out = torch.empty(n, device=self.device, dtype=torch.float32) if out is None else out
        if out.dtype != torch.float32 or not out.is_contiguous() or out.numel() != n:
            raise ValueError('out must be a contiguous float32 tensor of n elements')
        _lib.call('noise_normal_fill', _lib.ptr(out), n, first, self.seed, self.offset, self.threads,
                  float(mean), float(std), _lib.stream_ptr(self.device))
        return out

    def gather(self, offsets, width, rows=None):
        """[len(rows), width] with out[r, j] = element offsets[rows[r]] + j (rows None: all offsets)."""
        offsets = offsets.to(device=self.device, dtype=torch.int64).contiguous()
        if rows is not None:
            rows = rows.to(device=self.device, dtype=torch.int64).contiguous()
        nrows = offsets.numel() if rows is None else rows.numel()
        out = torch.empty(nrows, width, device=self.device, dtype=torch.float32)
        for start in range(0, nrows, GATHER_ROWS):
            n = min(GATHER_ROWS, nrows - start)
            sub_rows = None if rows is None else rows[start:start + n]
            sub_offsets = offsets[start:start + n] if rows is None else offsets
            _lib.call('noise_gather_slices', _lib.ptr(out[start:start + n]), n, width, _lib.ptr(sub_offsets),
                      _lib.ptr(sub_rows), self.numel, self.seed, self.offset, self.threads,
                      _lib.stream_ptr(self.device))
        return out

    def gather_many(self, offsets, widths, rows):
        """The slices of several parameters at the same rows in one launch per 64 parameters:
        [len(rows), sum(widths)] with columns c_k .. c_k + widths[k] holding gather(offsets[k], widths[k], rows)
        (c_k the running sum of the widths), so each parameter's slice is a column view. Widths must be multiples
        of 256."""
        rows = rows.to(device=self.device, dtype=torch.int64).contiguous()
        nrows = rows.numel()
        if nrows > GATHER_ROWS:
            raise ValueError(f'gather_many: at most {GATHER_ROWS} rows per call')
        offsets = [o if o.dtype == torch.int64 and o.device == self.device and o.is_contiguous() else
                   o.to(device=self.device, dtype=torch.int64).contiguous() for o in offsets]
        total = int(sum(widths))
        out = torch.empty(nrows, total, device=self.device, dtype=torch.float32)
        col = 0
        for g0 in range(0, len(widths), _lib.SLICE_GROUPS_MAX):
            part = list(range(g0, min(len(widths), g0 + _lib.SLICE_GROUPS_MAX)))
            desc = _lib.SliceGroups()
            desc.count = len(part)
            start = col
            for i, k in enumerate(part):
                desc.offsets[i] = offsets[k].data_ptr()
                desc.width[i] = int(widths[k])
                desc.col[i] = col - start
                col += int(widths[k])
            _lib.call('noise_gather_slice_groups', out.data_ptr() + 4 * start, nrows, total, ctypes.byref(desc),
                      rows.data_ptr(), self.numel, self.seed, self.offset, self.threads, _lib.stream_ptr(self.device))
        return out


class DeviceGenerator:
    """Offset bookkeeping of torch.Generator('cuda').manual_seed(seed) for randn/randint draws."""

    def __init__(self, seed, device=None):
        self.seed = int(seed)
        self.device = torch.device('cuda', torch.cuda.current_device()) if device is None else torch.device(device)
        self.offset = 0

    def manual_seed(self, seed):
        self.seed, self.offset = int(seed), 0
        return self

    def take(self, numel):
        """Reserve the next draw of `numel` values (advances the offset as torch does)."""
        threads, inc = draw_layout(numel, self.device)
        draw = Draw(self.seed, self.offset, threads, int(numel), self.device)
        self.offset += inc
        return draw

    def randn(self, numel):
        """torch.randn(numel, generator=this) as fp32, bit for bit."""
        return self.take(numel).normal()

    def randint(self, low, high, size):
        """torch.randint(low, high, size, generator=this) as int64, bit for bit (high - low < 2^28)."""
        size = (size,) if isinstance(size, int) else tuple(size)
        numel = 1
        for s in size:
            numel *= s
        rng = int(high) - int(low)
        if not 1 <= rng < 2 ** 28:
            raise ValueError(f'randint range must be in [1, 2^28) (torch 32-bit path), got {rng}')
        out = torch.empty(size, device=self.device, dtype=torch.int64)
        if numel == 0:
            return out
        draw = self.take(numel)
        _lib.call('noise_randint', _lib.ptr(out), numel, draw.seed, draw.offset, draw.threads, rng, int(low),
                  _lib.stream_ptr(self.device))
        return out


    def randint_many(self, highs, n):
        """[randint(0, high, n) for high in highs], bit for bit and in that order, in one launch per 64 draws: rows
        of one int64 tensor [len(highs), n]."""
        out = torch.empty(len(highs), n, device=self.device, dtype=torch.int64)
        for high in highs:
            if not 1 <= int(high) < 2 ** 28:
                raise ValueError(f'randint range must be in [1, 2^28) (torch 32-bit path), got {int(high)}')
        if n == 0 or not len(highs):
            return out
        threads, inc = draw_layout(n, self.device)
        for first in range(0, len(highs), _lib.RANDINT_SETS_MAX):
            part = highs[first:first + _lib.RANDINT_SETS_MAX]
            desc = _lib.RandintSet()
            desc.count = len(part)
            for i, high in enumerate(part):
                desc.offset[i] = self.offset
                desc.range[i] = int(high)
                self.offset += inc
            _lib.call('noise_randint_many', out.data_ptr() + 8 * n * first, n, ctypes.byref(desc), self.seed, threads,
                      _lib.stream_ptr(self.device))
        return out


class OrthogonalDraws:
    """DUST.orthogonal_noise (run.py:223-238) on the device, bit for bit.

    Two generators as run.py:168-169 makes them: `generator` (seed + 3 + 7777 * rank) for each draw's own
    sign, `shared` (seed + 5, the same on every GPU) for each site's frame, drawn when the site is first
    used: the cycle sign patterns randint(0, 2, (cycles, d)), then the frame's row offsets
    randint(0, d, (b, t)). Draw i of a call is row (offset + index) mod d of the Sylvester Hadamard
    matrix (run.py:143-152) times the pattern of cycle index // d times its sign, with
    index = rank * draws + chunk * n + i (run.py:235)."""

    def __init__(self, seed=0, rank=0, world=1, device=None):
        self.rank, self.world = int(rank), int(world)
        self.generator = DeviceGenerator(int(seed) + 3 + 7777 * self.rank, device)
        self.shared = DeviceGenerator(int(seed) + 5, device)
        self.device = self.generator.device
        self.frames = {}

    def __call__(self, site, draws, chunk, n, b, t, d, dtype=torch.float32):
        """[n, b, t, d] +-1 in `dtype` (float32 or bfloat16): draws chunk*n .. chunk*n + n of this rank's
        `draws` at `site`."""
        if d < 1 or d & (d - 1):
            raise ValueError(f'Orthogonal draws need a power-of-two width, not {d}.')
        if dtype not in (torch.float32, torch.bfloat16):
            raise ValueError(f'orthogonal draws are produced as float32 or bfloat16, not {dtype}')
        if chunk < 0 or n < 0 or chunk * n + n > draws:
            raise ValueError(f'draws {chunk * n}..{chunk * n + n} of chunk {chunk} lie beyond the {draws} draws per rank')
        if site not in self.frames:
            cycles = -(-self.world * draws // d)
            self.frames[site] = (self.shared.randint(0, 2, (cycles, d)), self.shared.randint(0, d, (b, t)), cycles)
        pattern, offset, cycles = self.frames[site]
        if offset.shape != (b, t):
            raise ValueError(f'site {site!r} was framed for (b, t) = {tuple(offset.shape)}, not {(b, t)}')
        sign = self.generator.randint(0, 2, (n, b, t, 1))
        out = torch.empty(n, b, t, d, dtype=dtype, device=self.device)
        _lib.call('noise_orthogonal_draws', _lib.ptr(out), 1 if dtype == torch.bfloat16 else 0, n, b * t, d,
                  self.rank * draws + chunk * n, _lib.ptr(offset), _lib.ptr(pattern), cycles, _lib.ptr(sign),
                  _lib.stream_ptr(self.device))
        return out
