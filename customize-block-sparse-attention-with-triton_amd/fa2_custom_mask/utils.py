"""Mask preprocessing on the GPU and small helpers.

`is_hip` / `keep` keep the names exported by the reference (fa2_custom_mask/utils.py:3-14).
"""
import collections
import weakref

import torch

from . import _ext

_host = _ext.host()

TILE = 64


def is_hip():
    """The reference hard-wires False (fa2_custom_mask/utils.py:3-4); this build only runs on HIP."""
    return True


def keep(conf):
    """Autotune filter of the reference (fa2_custom_mask/utils.py:9-14).  There is no autotuner
    here; every configuration is kept."""
    return True


# Device-resident kept-tile lists of a block mask (csrc/host.cpp)
TileLists = _host.TileLists


def _check_mask(mask):
    if not isinstance(mask, torch.Tensor) or mask.dtype != torch.bool:
        raise TypeError("mask must be a torch.bool tensor")       # fa2_custom_mask.py:20
    if mask.dim() != 4:
        raise ValueError("mask must have 4 dimensions [B, H, rows, cols]")
    if not mask.is_cuda:
        raise RuntimeError("mask must live on the GPU")


def reduce_dense_mask(mask):
    """Elementwise mask [Bm,Hm,N,N] -> block mask [Bm,Hm,N/64,N/64] (tile kept iff any element
    set; exact inverse of the expansion at kernel-test.py:18 for tile-constant masks)."""
    _check_mask(mask)
    Bm, Hm, N, N2 = mask.shape
    if N != N2 or N % TILE != 0:
        raise ValueError("dense mask must be [.., N, N] with N a multiple of 64")
    if mask.stride(3) != 1 or any(s % 16 for s in mask.stride()[:3]) or mask.data_ptr() % 16:
        mask = mask.contiguous()
    nb = N // TILE
    block = torch.empty((Bm, Hm, nb, nb), dtype=torch.bool, device=mask.device)
    rc = _ext.lib().bsattn_reduce_dense_mask(mask.data_ptr(), Bm, Hm, N, mask.stride(0), mask.stride(1),
                                             mask.stride(2), block.data_ptr(),
                                             _ext.current_stream(mask.device))
    _ext.check(rc, "bsattn_reduce_dense_mask")
    return block


def block_mask_to_lists(block, transpose=False, want_groups=False):
    """Block mask -> TileLists.  transpose=True lists, for every column block, the kept row
    blocks (what the dK/dV pass walks)."""
    _check_mask(block)
    Bm, Hm, nb, nb2 = block.shape
    if nb != nb2:
        raise ValueError("block mask must be square")
    return _host.block_mask_to_lists(block, transpose, want_groups)


def pack_mask_tiles(mask, lists, transpose=False):
    """Elementwise mask [Bm,Hm,N,N] + the TileLists of its reduced form -> (tile_partial uint8
    [cap], tile_bits int64 [cap, 64]) with one slot per kept tile: is the tile only partly set,
    and its 64 x 64 bools as 64 words (word r, bit c = element (r, c) of the tile; with
    transpose=True, matching transposed lists, element (c, r))."""
    _check_mask(mask)
    Bm, Hm, N, N2 = mask.shape
    if N != N2 or N % TILE != 0 or N // TILE != lists.nb or (Bm, Hm) != (lists.Bm, lists.Hm):
        raise ValueError("mask and lists do not belong together")
    sb, sh, sm, sn = mask.stride()
    if min(sm, sn) != 1 or any(s % 4 for s in (sb, sh, max(sm, sn))) or mask.data_ptr() % 4:
        mask = mask.contiguous()
        sb, sh, sm, sn = mask.stride()
    if transpose:
        sm, sn = sn, sm
    cap = Bm * Hm * lists.nb * lists.nb
    partial = torch.empty(cap, dtype=torch.uint8, device=mask.device)
    bits = torch.empty((cap, 64), dtype=torch.int64, device=mask.device)
    rc = _ext.lib().bsattn_pack_mask_tiles(mask.data_ptr(), Bm, Hm, N, sb, sh, sm, sn, lists.row_ptr_ptr,
                                           lists.col_idx_ptr, partial.data_ptr(), bits.data_ptr(),
                                           _ext.current_stream(mask.device))
    _ext.check(rc, "bsattn_pack_mask_tiles")
    return partial, bits


def reduce_pack_dense_mask(mask):
    """Elementwise mask [Bm,Hm,N,N] -> (block mask [Bm,Hm,nb,nb], grid_partial uint8 [Bm*Hm*nb*nb], grid_bits int64
    [Bm*Hm*nb*nb, 64]) in one pass over the mask: the reduced mask, and the "partly set" flag and packed words of
    every tile that has a set element, at the tile's position in the grid (gather_mask_tiles brings them into
    list order)."""
    _check_mask(mask)
    Bm, Hm, N, N2 = mask.shape
    if N != N2 or N % TILE != 0:
        raise ValueError("dense mask must be [.., N, N] with N a multiple of 64")
    if mask.stride(3) != 1 or any(s % 16 for s in mask.stride()[:3]) or mask.data_ptr() % 16:
        mask = mask.contiguous()
    nb = N // TILE
    tiles = Bm * Hm * nb * nb
    block = torch.empty((Bm, Hm, nb, nb), dtype=torch.bool, device=mask.device)
    grid_partial = torch.empty(tiles, dtype=torch.uint8, device=mask.device)
    grid_bits = torch.empty((tiles, 64), dtype=torch.int64, device=mask.device)
    rc = _ext.lib().bsattn_reduce_pack_dense_mask(mask.data_ptr(), Bm, Hm, N, mask.stride(0), mask.stride(1),
                                                  mask.stride(2), block.data_ptr(), grid_partial.data_ptr(),
                                                  grid_bits.data_ptr(), _ext.current_stream(mask.device))
    _ext.check(rc, "bsattn_reduce_pack_dense_mask")
    return block, grid_partial, grid_bits


def gather_mask_tiles(grid_partial, grid_bits, lists, transpose=False):
    """(tile_partial, tile_bits) in the format of pack_mask_tiles for `lists` (the row lists, or with
    transpose=True the column lists: words per key, bits per query) from the grid-ordered result of
    reduce_pack_dense_mask."""
    dev = lists.row_ptr.device
    cap = lists.Bm * lists.Hm * lists.nb * lists.nb
    partial = torch.empty(cap, dtype=torch.uint8, device=dev)
    bits = torch.empty((cap, 64), dtype=torch.int64, device=dev)
    rc = _ext.lib().bsattn_gather_mask_tiles(grid_partial.data_ptr(), grid_bits.data_ptr(), lists.Bm, lists.Hm, lists.nb,
                                             1 if transpose else 0, lists.row_ptr_ptr, lists.col_idx_ptr,
                                             partial.data_ptr(), bits.data_ptr(), _ext.current_stream(dev))
    _ext.check(rc, "bsattn_gather_mask_tiles")
    return partial, bits


def tail_mask_tiles(lists, valid_last, transpose=False):
    """Words of the kept tiles of a block mask whose last column block holds only `valid_last`
    real keys (sequence length not a multiple of 64): (tile_partial, tile_bits) in the format of
    pack_mask_tiles, every tile completely set except for the padding keys."""
    dev = lists.row_ptr.device
    cap = lists.Bm * lists.Hm * lists.nb * lists.nb
    partial = torch.empty(cap, dtype=torch.uint8, device=dev)
    bits = torch.empty((cap, 64), dtype=torch.int64, device=dev)
    rc = _ext.lib().bsattn_tail_mask_tiles(lists.Bm, lists.Hm, lists.nb, valid_last, 1 if transpose else 0,
                                           lists.row_ptr_ptr, lists.col_idx_ptr, partial.data_ptr(),
                                           bits.data_ptr(), _ext.current_stream(dev))
    _ext.check(rc, "bsattn_tail_mask_tiles")
    return partial, bits


def num_tiles(N):
    """Row (and column) blocks of a sequence of N tokens; the last one may be partly filled."""
    return -(-N // TILE)


def is_block_form(mask, N):
    """True for the reference's block form [.,.,nb,nb], False for an elementwise [.,.,N,N] mask."""
    nb = num_tiles(N)
    if mask.shape[2] == nb and mask.shape[3] == nb and N != nb:
        return True
    if mask.shape[2] == N and mask.shape[3] == N:
        return False
    raise ValueError("mask shape %s matches neither [.., %d, %d] nor [.., %d, %d]"
                     % (tuple(mask.shape), nb, nb, N, N))


def to_block_mask(mask, N):
    """Accepts the reference's block form [.,.,N/64,N/64] or an elementwise [.,.,N,N] mask
    (N a multiple of 64)."""
    _check_mask(mask)
    return mask if is_block_form(mask, N) else reduce_dense_mask(mask)


# In place of the lists of a block mask that forwards so far have done without (they took its rows from the mask itself): they are made
# when they are asked for, from the copy of the mask that the first of these forwards has left.
UNMADE = object()


class _Captured:
    """What captured graphs read of the caches' entries (lists, copies of masks, words by grid position), kept as long as the mask
    tensor: an entry goes when its mask is written to or many others are used, and a graph's replays would read freed memory."""

    def __init__(self):
        self._held = {}        # id of mask -> (weakref to mask, [objects])

    def hold(self, mask, *objects):
        key = id(mask)
        entry = self._held.get(key)
        if entry is None or entry[0]() is not mask:
            held = self._held
            def drop(ref):
                if key in held and held[key][0] is ref:
                    del held[key]
            entry = self._held[key] = (weakref.ref(mask, drop), [])
        entry[1].extend(x for x in objects if all(x is not y for y in entry[1]))


captured = _Captured()
_capturing = torch.cuda.is_current_stream_capturing


class _ListsCache:
    """Kept-tile lists of the most recently used masks.  A static mask (the usual case: one mask
    for every layer and step) is indexed once instead of once per call.  An entry is only used
    for the very tensor object it was built from, and only while that tensor has not been
    written to (autograd's version counter)."""

    def __init__(self, capacity=8):
        self.capacity = capacity
        # (id of mask, N, transpose) -> (weakref to mask, version, lists, stream the lists were built on, copy of the mask if the
        # lists are UNMADE), most recent last
        self._entries = collections.OrderedDict()

    @staticmethod
    def _version(mask):
        """The tensor's write counter, or None for a tensor that keeps none (one created under
        torch.inference_mode()): writes to such a tensor cannot be seen, so it is never cached."""
        try:
            return mask._version
        except RuntimeError:
            return None

    def _entry(self, mask, key):
        entry = self._entries.get(key)
        if entry is None or entry[0]() is not mask or self._version(mask) != entry[1]:
            return None
        return entry

    def seen(self, mask, N):
        """Is there an entry for the row lists of the mask as it is: its lists, UNMADE, or None."""
        entry = self._entry(mask, (id(mask), N, False))
        return None if entry is None else entry[2]

    def _use(self, mask, key, entry):
        """The lists of an entry (or the copy of the mask, where they are UNMADE) for a call on the current stream."""
        try:
            self._entries.move_to_end(key)
        except KeyError:           # (another thread has dropped it)
            pass
        _, _, lists, stream, block = entry
        current = _ext.raw_stream(mask.device)
        if current and _capturing():                 # (the default stream cannot be captured)
            captured.hold(mask, block if lists is UNMADE else lists)
        # they were filled by kernels on `stream` (a raw handle): work on another stream waits
        # for what that stream has been given so far (no event is recorded when the lists are made: a mask
        # that changes with every call would pay for it every time)
        if current != stream:
            torch.cuda.current_stream(mask.device).wait_stream(
                torch.cuda.ExternalStream(stream, device=mask.device) if stream else torch.cuda.default_stream(mask.device))
            if lists is UNMADE and not _capturing():
                block.record_stream(torch.cuda.current_stream(mask.device))
        return block if lists is UNMADE else lists

    def get(self, mask, N, transpose):
        key = (id(mask), N, transpose)
        entry = self._entry(mask, key)
        if entry is None:
            return None
        lists = self._use(mask, key, entry)
        if entry[2] is UNMADE:
            lists = block_mask_to_lists(lists, transpose=transpose)
            self.put(mask, N, transpose, lists)
        return lists

    def copy_of(self, mask, N):
        """Of a mask whose row lists are UNMADE: the copy of it that they will be made from, else None.  Forwards that need no lists
        take the copy, not the mask: a graph that captures one keeps seeing the mask as it was, as it would with lists."""
        key = (id(mask), N, False)
        entry = self._entry(mask, key)
        return self._use(mask, key, entry) if entry is not None and entry[2] is UNMADE else None

    def keeps(self, mask):
        """(version of the mask, current stream) if `put` would keep something for this mask, else None.  (Lists made while a graph is
        being captured are filled by its replays only, in memory that is the graph's.)"""
        version = self._version(mask)
        if version is None:
            return None
        stream = _ext.raw_stream(mask.device)
        return None if stream and _capturing() else (version, stream)       # (the default stream cannot be captured)

    def put(self, mask, N, transpose, lists, copy=None, kept=None):
        """kept: what `keeps` said in front of the call that made the lists, or None to ask it now."""
        kept = kept or self.keeps(mask)
        if kept is None:
            return
        version, stream = kept
        key = (id(mask), N, transpose)
        self._entries.pop(key, None)
        if len(self._entries) >= self.capacity:
            for dead in [k for k, e in self._entries.items() if e[0]() is None]:
                del self._entries[dead]
            while len(self._entries) >= self.capacity:
                self._entries.popitem(last=False)
        self._entries[key] = (weakref.ref(mask), version, lists, stream, copy)

    def clear(self):
        self._entries.clear()
        if "grid_cache" in globals():
            grid_cache.clear()


lists_cache = _ListsCache()


class _GridCache:
    """The grid-ordered words of the most recently used elementwise masks (reduce_pack_dense_mask), so that the
    second form of the lists (the column lists a backward asks for after the forward asked for the row lists)
    does not read the mask again.  Same identity rule as the lists cache; two entries, since one holds as
    many bytes as an eighth of its mask."""

    def __init__(self, capacity=2):
        self.capacity = capacity
        self._entries = []     # (weakref to mask, version, N, (block, grid_partial, grid_bits), stream, event)

    def get(self, mask, N):
        version = _ListsCache._version(mask)
        if version is None:
            return None
        for ref, ver, n, grid, stream, ready in self._entries:
            if ref() is mask and ver == version and n == N:
                current = torch.cuda.current_stream(mask.device)
                if current != stream:
                    current.wait_event(ready)
                if _capturing():
                    captured.hold(mask, *grid)
                return grid
        return None

    def put(self, mask, N, grid):
        version = _ListsCache._version(mask)
        if version is None or _capturing():
            return
        stream = torch.cuda.current_stream(mask.device)
        ready = torch.cuda.Event()
        ready.record(stream)
        self._entries = [e for e in self._entries if e[0]() is not None]
        self._entries.append((weakref.ref(mask), version, N, grid, stream, ready))
        del self._entries[:-self.capacity]

    def clear(self):
        self._entries = []


grid_cache = _GridCache()


def mask_to_lists(mask, N, transpose=False, both=False):
    """TileLists of a block or elementwise mask for sequence length N, through the cache.  both: the caller will
    also ask for the other orientation (a backward follows): an elementwise mask is then read once for both
    (one pass that packs every tile of the grid, 63 us at N = 17536, against 49 us for the reduction plus 34-78 us
    per orientation for packing the kept tiles from the mask: the one pass wins when both forms are needed or
    most tiles are kept, the two passes when a sparse mask is only used forward)."""
    lists = lists_cache.get(mask, N, transpose)
    if lists is None:
        _check_mask(mask)
        pad = num_tiles(N) * TILE - N          # keys of the last tile that do not exist: their bits stay clear
        if is_block_form(mask, N):
            lists = block_mask_to_lists(mask, transpose=transpose)
        else:                                  # elementwise form: exact inside tiles
            grid = grid_cache.get(mask, N)
            if grid is None and not (both or transpose):
                dense = torch.nn.functional.pad(mask, (0, pad, 0, pad)) if pad else mask
                lists = block_mask_to_lists(reduce_dense_mask(dense), transpose=transpose)
                lists.partial, lists.bits = pack_mask_tiles(dense, lists, transpose=transpose)
            else:
                if grid is None:
                    dense = torch.nn.functional.pad(mask, (0, pad, 0, pad)) if pad else mask
                    grid = reduce_pack_dense_mask(dense)
                    grid_cache.put(mask, N, grid)
                block, grid_partial, grid_bits = grid
                lists = block_mask_to_lists(block, transpose=transpose)
                lists.partial, lists.bits = gather_mask_tiles(grid_partial, grid_bits, lists, transpose=transpose)
        lists_cache.put(mask, N, transpose, lists)
    return lists
