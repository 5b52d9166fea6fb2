"""A training step's description over addresses that are no memory: for host code alone (tests/hip_stub.py)."""
import ctypes

from pointtransformerv3_amd import levels, native_train as t

AT = 1 << 20   # 256-byte aligned, like every buffer


def _linear(i, o):
    return t._Linear(AT, AT, AT, i, o, 0, 0)


def _block(c):
    norm, bn = t._Norm(AT, AT, 1e-5, 0, 0, 0), None
    return t._Block(channels=c, heads=c // 16, row=0, scale=0.25, conv_w=AT, conv_b=AT, conv_mirror=AT, conv_packed=AT,
                    conv_mirror_packed=AT, cpe=_linear(c, c), qkv=_linear(c, 3 * c), proj=_linear(c, c), fc1=_linear(c, 4 * c),
                    fc2=_linear(4 * c, c), ln_cpe=norm, ln1=norm, ln2=norm)


class Step:
    """net and levels of an encoder of two blocks a stage and a decoder of one, on `points` voxels a level."""

    def __init__(self, points=(60_000, 40_000, 12_000), widths=(32, 64, 128)):
        bn = t._Bn(AT, AT, AT, AT, AT, AT, 1e-3, 0.1, 0)
        self.net = net = t._Net(dtype=1, n_stages=len(points), max_pair_density=16.0, zero=AT, n_zero=1, zero_blocks=1, has_side=1,
                                stem=t._Stem(AT, 6, 16, 0, bn))
        self.levels = (levels.Level * len(points))()
        self.keep, self.blocks = [], 0
        for s, (n, c) in enumerate(zip(points, widths)):
            d, last = net.stage[s], s == len(points) - 1
            d.channels, d.n_enc, d.dec_channels, d.n_dec = c, 2, 0 if last else c, 0 if last else 1
            enc, dec = (t._Block * 2)(*[_block(c) for _ in range(2)]), (t._Block * 1)(_block(c))
            self.keep += [enc, dec]
            d.enc, d.dec = ctypes.addressof(enc), 0 if last else ctypes.addressof(dec)
            self.blocks += d.n_enc + d.n_dec
            d.pool, d.up, d.up_skip = _linear(widths[s - 1], c), _linear(widths[min(s + 1, len(points) - 1)], c), _linear(c, c)
            d.pool_bn = d.up_bn = d.up_skip_bn = bn
            net.patch[s] = 1024
            v = self.levels[s]
            for name, kind in levels.Level._fields_:
                if kind is ctypes.c_void_p:
                    setattr(v, name, AT)
            v.slot_src[0] = v.slot_dst[0] = AT
            v.n, v.n_pad, v.n_seq, v.n_pairs, v.n_pairs5, v.tile_voxels, v.depth = n, -(-n // 1024) * 1024, -(-n // 1024), 8 * n, 5 * n, 128, 9

    def sizes(self, lib):
        out = (ctypes.c_size_t * 3)()
        at = ctypes.addressof(out)
        assert lib.ptv3_train_bytes(ctypes.byref(self.net), self.levels, at, at + 8, at + 16) == 0
        return list(out)

    def backward(self, lib, stream, scratch_bytes, net=None):
        masks = (ctypes.c_void_p * (2 * self.blocks))()
        return lib.ptv3_train_bwd(ctypes.byref(self.net) if net is None else net, self.levels, AT, 0, masks, AT, AT, scratch_bytes, AT, stream)
