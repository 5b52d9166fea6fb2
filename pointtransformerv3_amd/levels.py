"""The index of a whole forward from one batched pass (ptv3_index_*): every table that follows from the coordinates
alone, for every encoder level, in about 24 launches and three waits (model.py:81-174, :382-453, :652-703)."""
import ctypes
import math

import torch

from . import _lib, hostslot, ops

MAX_LEVELS = MAX_ORDERS = 8
_STATE_BYTES = 16384
_SLOT_DATA = hostslot.DATA
_SLOT_ENDS = _SLOT_DATA + 4 + MAX_LEVELS + 2 * MAX_LEVELS
PAIRS, TILES, PAIRS5, PAIR_OUT, PAIR_OUT5 = 1, 2, 4, 8, 32

_i32, _i64, _ptr = ctypes.c_int32, ctypes.c_int64, ctypes.c_void_p


class Cfg(ctypes.Structure):
    """ptv3_index_cfg"""
    _fields_ = [("n", _i64), ("n_levels", _i32), ("n_orders", _i32), ("n_scenes", _i32), ("stem5", _i32), ("pads_all", _i32),
                ("reserved", _i32), ("pool_depth", _i32 * MAX_LEVELS), ("patch", _i32 * MAX_LEVELS),
                ("only128", _i32 * MAX_LEVELS), ("slot_orders", ctypes.c_uint32 * MAX_LEVELS)]


class Level(ctypes.Structure):
    """ptv3_level"""
    _fields_ = ([(f, _i64) for f in ("n", "n_pad", "n_seq", "n_pairs", "n_pairs5")]
                + [(f, _ptr) for f in ("code", "order", "inverse", "grid", "batch", "offset", "indices", "cluster", "idx_ptr",
                                       "pad", "unpad", "cu")]
                + [("slot_src", _ptr * MAX_ORDERS), ("slot_dst", _ptr * MAX_ORDERS)]
                + [(f, _ptr) for f in ("tap_ptr", "row_ptr", "pair_in", "pair_slot", "tile_tap", "tile_pair", "vox_taps",
                                       "tap_ptr5", "row_ptr5", "pair_in5", "pair_slot5", "pair_out", "pair_out5")]
                + [("tile_voxels", _i32), ("depth", _i32)])


class SceneFacts:
    """Grid extent and scene ends of (n, 3) int32 coordinates, on their way to the host behind the work queued so far."""

    def __init__(self, grid_coord, offset):
        lib = _lib.load()
        self.nb = offset.shape[0]
        self.slot, self.seq, self.stream = hostslot.take(_SLOT_ENDS + self.nb), hostslot.next_seq(), ops._stream()
        nbytes = lib.ptv3_scene_facts_bytes(grid_coord.shape[0])
        self.scratch = torch.empty(nbytes, dtype=torch.uint8, device=grid_coord.device)
        _lib.check(lib.ptv3_scene_facts(grid_coord.data_ptr(), grid_coord.shape[0], offset.data_ptr(), self.nb,
                                        self.scratch.data_ptr(), nbytes, self.slot.ptr, self.seq, self.stream), "ptv3_scene_facts")

    def get(self):
        """(per-axis maxima, scene ends) as lists."""
        if self.slot.words[0] != self.seq:
            ops.refresh_derived_copies()   # as Readback.get: work for the wait
        _lib.check(_lib.load().ptv3_index_wait(self.slot.ptr, 0, self.seq, self.stream), "ptv3_index_wait")
        out = self.slot.words[_SLOT_DATA:_SLOT_DATA + 3], self.slot.words[_SLOT_ENDS:_SLOT_ENDS + self.nb]
        hostslot.give(self.slot)
        return out


class Layout:
    """What the index of a model needs to know of its modules, worked out once: per level the pooling in front of it, the
    patch size, the attention rows in use and the convolutions that share the level's lists."""

    def __init__(self, n_orders, strides, patches, slot_rows, convs, stem5, shuffles, only_pads0=True):
        self.cfg = c = Cfg()
        c.n_levels, c.n_orders, c.stem5, c.pads_all = len(patches), n_orders, int(stem5), int(not only_pads0)
        self.convs = convs           # per level: [(channels in, channels out)] of its 3x3x3 convolutions
        self.shuffles = shuffles     # per pooling module: whether it draws a row shuffle
        for level, patch in enumerate(patches):
            c.patch[level] = patch
            c.pool_depth[level] = (math.ceil(strides[level - 1]) - 1).bit_length() if level else 0
            c.slot_orders[level] = sum(1 << r for r in set(slot_rows[level]))
            tiled = {ci for ci, co in convs[level] if ci == co and ci in ops.CONV_TILE_CHANNELS + ops.CONV_SPARSE_CHANNELS}
            c.only128[level] = int(tiled == {128})

    def copy_cfg(self):
        c = Cfg()
        ctypes.memmove(ctypes.byref(c), ctypes.byref(self.cfg), ctypes.sizeof(Cfg))
        return c


class Index:
    """One forward's index: `levels` (an array of Level), the tensors of level 0 and the buffers everything else lies in."""

    def tensor(self, ptr, shape, dtype, which="tables"):
        """The table at `ptr` as a tensor (a view of the buffer it lies in)."""
        buf = self.buffers[which]
        size = dtype.itemsize
        for s in shape:
            size *= s
        at = ptr - buf.data_ptr()
        return buf[at:at + size].view(dtype).view(shape)


def build(layout, grid_coord, offset, batch, orders, shuffle, want, between=None, sized=None):
    """Queues the whole index on the current stream and waits for what the host has to know. grid_coord (n, 3) int32 and
    offset (scenes,) int64 contiguous, batch (n,) int64 or None; orders: names of the curves, shuffled with torch's CPU
    generator when `shuffle` (and per pooling module as layout.shuffles says, in the order the modules would draw);
    want(level number, Level) -> PTV3_LISTS_* flags of the level once its pair count is known;
    between() is called behind the first stage's launches, while the host would wait for them, sized(levels) behind the
    third's, when every level's number of points is known."""
    lib = _lib.load()
    stream = ops._stream()
    dev = grid_coord.device
    cfg = layout.copy_cfg()
    n, nb, k = grid_coord.shape[0], offset.shape[0], cfg.n_orders
    cfg.n, cfg.n_scenes = n, nb
    check = _lib.check
    out = Index()
    u8 = dict(dtype=torch.uint8, device=dev)
    state = ctypes.create_string_buffer(_STATE_BYTES)
    slot = hostslot.take(lib.ptv3_index_slot_words(cfg.n_levels, nb))
    words, seq = slot.words, hostslot.next_seq()
    sizes = (ctypes.c_size_t * 2)()
    check(lib.ptv3_index_begin_bytes(ctypes.byref(cfg), ctypes.byref(sizes, 0), ctypes.byref(sizes, 8)), "ptv3_index_begin_bytes")
    # the scratch of this stage and of the pooling goes when this function returns: later work on the stream may have it
    first, scratch0 = torch.empty(sizes[0], **u8), torch.empty(sizes[1], **u8)
    out.batch = batch if batch is not None else torch.empty(n, dtype=torch.int64, device=dev)
    check(lib.ptv3_index_begin(state, ctypes.byref(cfg), grid_coord.data_ptr(), None if batch is None else batch.data_ptr(),
                               offset.data_ptr(), out.batch.data_ptr(), first.data_ptr(), sizes[0], scratch0.data_ptr(), sizes[1],
                               slot.ptr, seq, stream), "ptv3_index_begin")
    if between is not None:
        between()
    check(lib.ptv3_index_wait(slot.ptr, 0, seq, stream), "ptv3_index_wait")
    out.grid_max = words[_SLOT_DATA:_SLOT_DATA + 3]
    out.offset_host = words[_SLOT_ENDS:_SLOT_ENDS + nb]
    if out.offset_host[-1] != n or any(b < a for a, b in zip(out.offset_host, out.offset_host[1:])):
        hostslot.give(slot)
        raise _lib.Ptv3Error(f"offset {out.offset_host[-4:]} does not end the scenes of {n} points in ascending order")
    depth = max(out.grid_max).bit_length()            # model.py:98-101
    assert depth * 3 + nb.bit_length() <= 63          # model.py:103
    assert depth <= 16                                # model.py:108
    if shuffle:
        perm = torch.randperm(k).tolist()             # CPU generator, as model.py:129
        orders = [orders[i] for i in perm]
    perms = (ctypes.c_int32 * (max(cfg.n_levels - 1, 1) * k))()
    for j, shuffled in enumerate(layout.shuffles):    # model.py:675-679, in module order
        perms[j * k:(j + 1) * k] = torch.randperm(k).tolist() if shuffled else list(range(k))
    ids = (ctypes.c_int32 * k)(*[ops.ORDER_IDS[o] for o in orders])
    out.code, out.order, out.inverse = torch.empty((3, k, n), dtype=torch.int64, device=dev).unbind(0)
    nbytes = lib.ptv3_index_sort_bytes(state)
    ws = torch.empty(nbytes, **u8)
    key_bits = 3 * depth + max(1, (nb - 1).bit_length())
    check(lib.ptv3_index_sort(state, depth, key_bits, ids, out.code.data_ptr(), out.order.data_ptr(), out.inverse.data_ptr(),
                              ws.data_ptr(), nbytes, stream), "ptv3_index_sort")
    check(lib.ptv3_index_wait(slot.ptr, 1, seq, stream), "ptv3_index_wait")
    check(lib.ptv3_index_pool_bytes(state, ctypes.byref(sizes, 0), ctypes.byref(sizes, 8)), "ptv3_index_pool_bytes")
    tables, scratch = torch.empty(sizes[0], **u8), torch.empty(sizes[1], **u8)
    check(lib.ptv3_index_pool(state, perms, tables.data_ptr(), sizes[0], scratch.data_ptr(), sizes[1], stream),
          "ptv3_index_pool")
    out.levels = levels = (Level * cfg.n_levels).from_address(lib.ptv3_index_levels(state))
    if sized is not None:
        sized(levels)
    check(lib.ptv3_index_wait(slot.ptr, 2, seq, stream), "ptv3_index_wait")
    out.level_offsets = [words[_SLOT_ENDS + level * nb:_SLOT_ENDS + (level + 1) * nb] for level in range(cfg.n_levels)]
    wanted = (ctypes.c_int32 * cfg.n_levels)()
    # the pair counts enter `levels` with the size query; the flags decide what is sized, so the query runs twice
    check(lib.ptv3_index_lists_bytes(state, wanted, sizes), "ptv3_index_lists_bytes")
    for level in range(cfg.n_levels):
        wanted[level] = want(level, levels[level])
    check(lib.ptv3_index_lists_bytes(state, wanted, sizes), "ptv3_index_lists_bytes")
    lists = torch.empty(sizes[0], **u8)
    check(lib.ptv3_index_lists(state, wanted, lists.data_ptr(), sizes[0], stream), "ptv3_index_lists")
    hostslot.give(slot)
    out.state = state                # `levels` lies in it
    out.offset, out.grid_coord, out.depth, out.n_orders = offset, grid_coord, depth, k
    # `first` holds level 0's sparse indices, the pooled scene ends and level 0's tap_ptr
    out.buffers = dict(first=first, tables=tables, lists=lists)
    out.buffers["scratch"] = tables   # where the pooled tap_ptr lie, under the name of the buffer that used to hold them
    out.lists = list(wanted)
    return out
