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


def test_attention_backward_takes_the_two_kernels_where_sequences_are_short(tmp_path):
    """Launches on both sides of every line of the rule: the both-sides kernel and the one behind it are two, with a part that is
    shared three, the two kernels three, behind full rounds of the both-sides kernel four."""
    hip_stub.run(r'''
AT = 1 << 20
def launches(items, mean, longest, cus=256):
    clear(cus=cus)
    n, c = items * mean, 16
    size = lib.ptv3_patch_attn_bwd_workspace_bytes(1, n, c, 1)
    assert lib.ptv3_patch_attn_bwd(AT, AT, AT, 1, n, c, 1, AT, AT, AT, items, longest, n, 0.25, AT, 0.0, 0, AT, AT, size, None) == 0
    return [c[2] for c in calls()]
for longest, items, mean, count in (
        (1024, 32, 704, 3), (1024, 32, 705, 2), (1024, 33, 704, 2), (1024, 64, 576, 3), (1024, 64, 577, 2), (1024, 65, 577, 3), (1024, 85, 768, 3), (1024, 85, 769, 2), (1024, 86, 768, 2),
        (1024, 128, 160, 3), (1024, 128, 161, 2), (1024, 128, 256, 2), (1024, 128, 257, 3), (1024, 128, 384, 3), (1024, 128, 385, 2),
        (1024, 129, 100, 2), (1024, 256, 100, 2), (1024, 512, 320, 2), (1024, 288, 320, 4), (1024, 288, 1000, 3), (1024, 400, 320, 2),
        (512, 64, 256, 2), (512, 64, 257, 3), (512, 64, 384, 3), (512, 64, 385, 2), (512, 65, 300, 2), (512, 256, 300, 2),
        (512, 320, 320, 3), (512, 320, 400, 3), (512, 320, 200, 2), (512, 576, 300, 3), (256, 64, 200, 2), (256, 300, 20, 2)):
    got = launches(items, mean, longest)
    assert len(got) == count, (longest, items, mean, got)
# one launch for 320 items of 512 slots whose mean is 320 is the query kernel, at 400 the both-sides kernel, and a shared part
assert launches(320, 320, 512)[:2] == launches(64, 300, 512)[:2] and launches(320, 400, 512)[0] == launches(256, 400, 512)[0]
assert len(launches(32, 300, 1024, cus=128)) == 3 and len(launches(43, 577, 1024, cus=128)) == 2   # a quarter and a third of 128
''', tmp_path)


def test_rules_of_the_256_channel_layers_and_of_product_rows_go_by_the_device(tmp_path):
    """The first half of a block in one kernel up to five rounds of 32 rows a CU; product rows that the L2s (4 MB for 32 CUs) do
    not hold are read past them, by another instantiation of the kernel that sums them."""
    hip_stub.run(r'''
AT = 1 << 20
for cus in (256, 128, 32, 304):
    clear(cus=cus)
    rounds = 5 * 32 * cus
    assert [lib.ptv3_block_head_wide_pays(n, 256) for n in (256, 257, rounds, rounds + 1)] == [0, 1, 1, 0], cus
    assert lib.ptv3_block_head_wide_pays(10 * rounds, 128) == 1 and lib.ptv3_block_head_wide_pays(300, 64) == 0
    held = (cus // 32 << 22) // (256 * 2)   # pairs whose 256 half-precision products the L2s hold
    sums = []
    for pairs in (1000, held, held + 1, 10 * held):
        clear(cus=cus)
        assert lib.ptv3_subm_conv_pairs_fwd(AT, 1, 900, 256, 27, pairs, AT, AT, AT, AT, AT, AT, 256, AT, AT, None) == 0
        sums.append(calls()[-1][2])
    assert sums[0] == sums[1] != sums[2] == sums[3], cus
''', tmp_path)
