"""Rules of the library that go by the part: over a stand-in for the runtime that claims other numbers of CUs than this part has
(tests/hip_stub.py)."""
import hip_stub


def test_a_workspace_of_the_attention_backward_serves_every_device(tmp_path):
    """Its size is asked for on one device and used on another: it is the same for both, and no launch asks for more."""
    hip_stub.run(r'''
AT = 1 << 20
for n_seq, length, heads in ((15, 1024, 4), (23, 1024, 4), (32, 1024, 2), (38, 900, 8), (16, 500, 8), (40, 200, 5), (198, 1024, 4)):
    n, c = n_seq * length, heads * 16
    for dtype in (0, 1, 2):
        sizes = set()
        for cus in (32, 256, 304):
            clear(cus=cus)
            sizes.add(lib.ptv3_patch_attn_bwd_workspace_bytes(dtype, n, c, heads))
        assert len(sizes) == 1, (n_seq, length, heads, dtype, sizes)
        for cus in (32, 256, 304):
            clear(cus=cus)
            rc = lib.ptv3_patch_attn_bwd(AT, AT, AT, dtype, n, c, heads, AT, AT, AT, n_seq, 1024, n, 0.25, AT if dtype else None,
                                         0.0, 0, AT, AT, min(sizes), None)
            assert rc == 0 and calls(), (n_seq, length, heads, dtype, cus, rc)
''', tmp_path)
