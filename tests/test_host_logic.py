"""CPU: host-side logic of the operator mirror that needs no GPU - argument parsing of the overloaded
`fused_experts_compute`, `fused_moe` argument errors, launch-parameter guards, workspace sizing."""
import os

import pytest
import torch

from muxi_native_layout_kernels_amd import ops, arg_selector, _lib
from muxi_native_layout_kernels_amd.moe_planC import fused_moe


def test_gemm_guard_accepts_both_kernels_and_rejects_bad_rows():
    assert ops._gemm_guard((1, 4, 4, 1), 11008) == (1, 4, 4, 1)
    assert ops._gemm_guard((2, 2, 1, 2), 11008) == (2, 2, 1, 2)
    assert ops._gemm_guard((14, 4, 2, 1), 11008) == (14, 4, 2, 1)    # kernel 1 with an explicit ring depth
    assert ops._gemm_guard((13, 4, 2, 1), 11008) == (1, 1, 4, 1)
    assert ops._gemm_guard((4, 1, 2, 1), 11008) == (4, 1, 2, 1)      # one workgroup per CU
    assert ops._gemm_guard((18, 8, 4, 1), 28672) == (18, 8, 4, 1)    # eight row groups per wave
    assert ops._gemm_guard((3, 1, 1, 2), 11008) == (3, 1, 1, 2)      # panel kernel
    assert ops._gemm_guard((3, 2, 4, 2), 272) == (3, 2, 4, 2)        # its row groups per wave need not divide N/16
    assert ops._gemm_guard((5, 4, 1, 2), 11008) == (5, 4, 1, 2)      # panel kernel, last round sliced
    assert ops._gemm_guard((5, 2, 4, 3), 272) == (5, 2, 4, 3)
    assert ops._gemm_guard((6, 1, 1, 1), 11008) == (1, 1, 4, 1)      # unknown kernel id
    assert ops._gemm_guard((1, 3, 4, 1), 11008) == (1, 1, 4, 1)      # row groups per wave not in {1,2,4}
    assert ops._gemm_guard((1, 4, 4, 1), 16 * 6) == (1, 1, 4, 1)     # 6 row groups are not a multiple of 4
    assert ops._gemm_guard((1, 1, 5, 1), 4096) == (1, 1, 4, 1)       # waves per workgroup not a power of two


def test_default_heuristics_are_valid_launch_parameters():
    for n, k in ((16, 32), (4096, 4096), (152064, 3584)):
        block, kid, p1, p2 = arg_selector._gemv_default(n, k)
        assert kid == 1 and 64 <= block <= 1024 and block % 64 == 0 and p1 == 1 and p2 in (1, 2, 4, 6, 8)
    for n, m, k in ((128, 1, 128), (11008, 64, 4096), (4096, 16, 14336)):
        kid, p1, p2, p3 = arg_selector._gemm_default(n, m, k)
        assert ops._gemm_guard((kid, p1, p2, p3), n) == (kid, p1, p2, p3)


def test_fused_moe_argument_errors_before_any_gpu_work():
    h = torch.zeros(2, 128, dtype=torch.bfloat16)
    g = torch.zeros(2, 8, dtype=torch.bfloat16)
    w1 = torch.zeros(8, 256, 128, dtype=torch.bfloat16)
    w2 = torch.zeros(8, 128, 128, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="num_expert_group must be 1"):
        fused_moe(h, w1, w2, g, 2, True, use_grouped_topk=False, num_expert_group=2)
    with pytest.raises(ValueError, match="Unsupported scoring function"):
        fused_moe(h, w1, w2, g, 2, True, score_func="tanh")
    with pytest.raises(AssertionError, match="Number of tokens mismatch"):
        fused_moe(h, w1, w2, g[:1], 2, True)
    with pytest.raises(RuntimeError, match="CUDA"):
        fused_moe(h, w1, w2, g, 2, True)


def test_fused_experts_compute_overload_resolution_errors():
    t = torch.zeros(1)
    args = [t] * 3 + [1, 8, 2] + [t] * 8
    with pytest.raises(RuntimeError, match="too many positional"):
        ops.fused_experts_compute(*args, 2, 3, 128, 16, 128, 256, 16, None, 99)
    with pytest.raises(RuntimeError, match="unexpected argument"):
        ops.fused_experts_compute(*args, bogus=1)
    with pytest.raises(RuntimeError, match="unexpected argument"):
        ops.fused_experts_compute(*args, 2, APerWarp=4)      # given twice


def test_workspace_sizes_from_the_library():
    lib = _lib.load()
    small = lib.mlk_moe_workspace_bytes(1, 8, 2, 4096, 14336)
    big = lib.mlk_moe_workspace_bytes(256, 8, 2, 4096, 14336)
    huge = lib.mlk_moe_workspace_bytes(4096, 8, 2, 4096, 14336)
    assert 0 < small < big == huge          # tokens are processed in passes of 256
    assert lib.mlk_gemm_counter_bytes() == 65536


def test_workspace_of_an_empty_batch():
    """No tokens need no scratch (the calls themselves return at once); the queries ended the process with a division by zero.
    Asked in a process of its own."""
    import subprocess
    import sys
    code = ("from muxi_native_layout_kernels_amd import _lib\nlib = _lib.load()\n"
            "print(lib.mlk_moe_workspace_bytes(0, 8, 2, 4096, 14336), lib.mlk_moe_wide_workspace_bytes(0, 8, 2, 4096, 14336))")
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300,
                         cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert out.returncode == 0 and out.stdout.split() == ["0", "0"], out.stderr


def test_beta_must_be_zero():
    with pytest.raises(RuntimeError, match="beta"):
        ops._check_beta(0.5)
    ops._check_beta(0)


def test_panel_kernel_default_shape():
    """Unscanned row-major shapes: the panel kernel above 64 tokens; 128-row panels while there
    are few of them, and as many K slices as keep panels x slices within the CU count."""
    from muxi_native_layout_kernels_amd import arg_selector as sel
    assert sel.panel_shape(11008, 128, 4096) == (2, 2)         # 43 panels of 256 rows -> 86 of 128 rows
    assert sel.panel_shape(11008, 256, 4096) == (2, 1)         # 86 -> 172
    assert sel.panel_shape(11008, 512, 4096) == (4, 1)         # 172 panels
    assert sel.panel_shape(8192, 128, 8192) == (2, 4)          # 32 -> 64
    assert sel.panel_shape(8192, 512, 8192) == (4, 2)          # 128 panels
    assert sel.panel_shape(28672, 128, 8192) == (4, 2)         # 112 panels
    assert sel.panel_shape(1024, 128, 1024) == (2, 2)          # 8 windows: at least four per slice
    assert sel.panel_shape(1024, 128, 384) == (2, 1)
    assert sel._gemm_default_rowmajor(11008, 512, 4096) == (3, 4, 4, 1)
    assert sel._gemm_default_rowmajor(11008, 72, 4096) == (3, 2, 4, 2)
    assert sel._gemm_default_rowmajor(11008, 64, 4096)[0] == 1      # the narrow kernels up to 64 tokens
    assert sel._gemm_default_rowmajor(11008, 512, 4096 + 64)[0] == 2  # K is no multiple of 128
    assert sel._gemm_default(11008, 512, 4096)[0] == 2              # native operands never get the panel kernel


def test_workspace_pool_never_frees_what_it_handed_out():
    """A larger request gets a new buffer; the earlier one stays owned (a captured graph may still use its
    address).  Streams do not share buffers, repeated requests on one stream do."""
    pool = ops.WorkspacePool(1024, zero_prefix=True)
    cpu = torch.device("cpu")
    a = pool.get(cpu, 0, 1000, 64)
    ptr_a = a.data_ptr()
    assert a.numel() >= 1024 and not a[:64].any()
    assert pool.get(cpu, 0, 512, 64) is a                     # fits: same buffer
    b = pool.get(cpu, 0, 1 << 16, 64)
    assert b is not a and b.numel() >= 1 << 16 and not b[:64].any()
    assert pool.get(cpu, 0, 1000, 64) is b                    # new calls use the larger one
    c = pool.get(cpu, 7, 1000, 64)                            # another stream: its own buffer
    assert c is not a and c is not b
    owned = {t.data_ptr() for t in pool.owned()}
    assert {ptr_a, b.data_ptr(), c.data_ptr()} <= owned
    a.fill_(3)                                                # still valid memory of ours
    assert int(a[5]) == 3
    # growth is geometric, so a slowly growing series of shapes retires few buffers
    for n in range(1 << 16, 1 << 18, 4096):
        pool.get(cpu, 0, n, 64)
    assert len(pool.owned()) <= 8


def test_workspace_pool_release():
    """release() drops the retired buffers (and the live ones unless asked not to) and says how much that was;
    the next request simply gets a new buffer."""
    pool = ops.WorkspacePool(1024)
    cpu = torch.device("cpu")
    a = pool.get(cpu, 0, 1000)
    b = pool.get(cpu, 0, 1 << 16)                             # retires a
    assert pool.held_bytes() == a.numel() + b.numel()
    assert pool.release(retired_only=True) == a.numel() and pool.held_bytes() == b.numel()
    assert pool.get(cpu, 0, 100) is b                         # the live buffer is still the one in use
    assert pool.release() == b.numel() and pool.held_bytes() == 0
    c = pool.get(cpu, 0, 100)
    assert c is not b and c.numel() >= 1024


def test_moe_scratch_falls_back_to_passes_of_256_tokens(monkeypatch):
    """Where the card has no room for the scratch of the wide kernels the call gets that of 256-token passes; the pool keeps
    what it had and counts it once.  Up to 256 tokens there is nothing smaller to fall back to."""
    lib, layer = _lib.load(), (8, 2, 4096, 14336)
    pool = ops.WorkspacePool(1024)
    cpu = torch.device("cpu")
    monkeypatch.setattr(ops, "_moe_workspace", lambda device, nbytes: pool.get(device, 0, nbytes))
    small = pool.get(cpu, 0, 1 << 20)
    narrow = lib.mlk_moe_workspace_bytes(4096, *layer)
    real = torch.empty

    def empty(size, **kw):
        if size > room:
            raise torch.OutOfMemoryError("no room for %d bytes" % size)
        return real(size, **kw)
    monkeypatch.setattr(torch, "empty", empty)
    room = 2 * narrow
    got = ops._moe_scratch(cpu, 4096, *layer)
    assert got.numel() >= narrow and got.numel() < lib.mlk_moe_wide_workspace_bytes(4096, *layer)
    assert pool.held_bytes() == small.numel() + got.numel() and any(b is small for b in pool.owned())
    pool.release()
    room = 1 << 20
    with pytest.raises(torch.OutOfMemoryError):
        ops._moe_scratch(cpu, 256, *layer)
    assert pool.held_bytes() == 0


def test_moe_workspace_follows_the_plan():
    """The fp32 buffer of the K-sliced down projections is sized for the slices the plan uses (not for the most
    the kernels could take), a call of several passes covers its shorter last pass, and the query grows with the
    token count within a pass."""
    lib = _lib.load()
    E, K, H, I = 256, 8, 7168, 2048
    sizes = [lib.mlk_moe_workspace_bytes(t, E, K, H, I) for t in (1, 16, 64, 256)]
    assert sizes == sorted(sizes)
    # 256 tokens: 2048 pairs; eight slices of fp32 rows would be 470 MB, the plan uses far fewer
    slices = max(_plan(256, E, K, H, I, kind)["down_slices"] for kind in (1, 2))
    assert sizes[-1] < 2048 * H * 4 * (slices + 1) + (64 << 20)
    for n in (257, 300, 500, 511, 1024):
        last = n % 256
        need = lib.mlk_moe_workspace_bytes(n, E, K, H, I)
        assert need >= lib.mlk_moe_workspace_bytes(256, E, K, H, I)
        if last:
            assert need >= lib.mlk_moe_workspace_bytes(last, E, K, H, I)


def _first_pass(T, E, K, H, I, kind, workspace=None):
    """(tokens, wide) of the first pass with a workspace of the wide kernels, or of the size given."""
    import ctypes
    lib, out = _lib.load(), (ctypes.c_int32 * 2)()
    need = lib.mlk_moe_wide_workspace_bytes(T, E, K, H, I) if workspace is None else workspace
    assert lib.mlk_moe_first_pass(T, E, K, H, I, kind, need, ctypes.addressof(out)) == 0
    return out[0], bool(out[1])


@pytest.mark.parametrize("E,K,H,I,kind,two_passes,wide", [
    # measured (256 CUs): tokens whose pass of 256 and remainder are the faster, more tokens whose wide pass is (two passes and wide, us:
    # the third and the next row at 268 tokens 2513 / 2196 and 932 / 795, (256, 1, 2048, 512) at 264 tokens 139 / 154)
    (8, 2, 4096, 14336, 2, 256, 260), (256, 8, 7168, 256, 2, 259, 264), (256, 8, 7168, 2048, 2, 259, 268),
    (128, 8, 2048, 768, 2, 257, 264), (160, 6, 5120, 1536, 2, 257, 264), (256, 2, 4096, 1024, 2, 264, 288),
    (64, 1, 4096, 2048, 2, 257, 268), (128, 2, 4096, 2048, 1, 257, 268), (256, 8, 7168, 256, 1, 257, 264),
    (8, 2, 4096, 14336, 1, 256, 257), (16, 4, 4096, 2048, 2, 256, 257), (64, 6, 2048, 1024, 1, 256, 257),
    (256, 1, 2048, 512, 2, 264, 304), (256, 6, 5120, 1024, 1, 257, 264), (8, 2, 1024, 512, 2, 256, 257),
])
def test_moe_pass_above_256_tokens_is_the_cheaper_one(E, K, H, I, kind, two_passes, wide):
    assert _first_pass(two_passes, E, K, H, I, kind) == (256, False)
    assert _first_pass(wide, E, K, H, I, kind) == (wide, True)
    most = min(4096, 16384 // K)
    assert _first_pass(most + two_passes, E, K, H, I, kind) == (most, True)
    # once wide, wide for every larger count; without the scratch in passes of 256
    was = False
    for T in range(257, 600):
        tokens, now = _first_pass(T, E, K, H, I, kind)
        assert now or not was, T
        assert tokens == (T if now else 256)
        was = now
    assert _first_pass(600, E, K, H, I, kind, 1) == (256, False)


@pytest.mark.parametrize("E,K,H,I", [(8, 2, 4096, 14336), (256, 8, 7168, 256), (1, 1, 4096, 14336), (4, 1, 4224, 2048),
                                     (60, 5, 768, 5376), (16, 16, 1024, 2048)])
def test_moe_wide_workspace_holds_for_every_shorter_call(E, K, H, I):
    """Above 256 tokens the query never falls, covers every call of up to 256 tokens, and leaves room for the fp32 products of
    at least one K slice."""
    lib = _lib.load()
    most = max(lib.mlk_moe_workspace_bytes(t, E, K, H, I) for t in range(1, 257))
    before = 0
    for t in range(257, 4400):
        need = lib.mlk_moe_wide_workspace_bytes(t, E, K, H, I)
        assert need >= before and need >= most and need >= min(t, 4096, 16384 // K) * K * H * 4, t
        before = need
    for t in range(257, 4400, 7):
        for kind in (1, 2):
            assert _first_pass(t, E, K, H, I, kind, before) == _first_pass(t, E, K, H, I, kind), t
    for t in (1, 16, 171, 256):
        assert lib.mlk_moe_wide_workspace_bytes(t, E, K, H, I) == lib.mlk_moe_workspace_bytes(t, E, K, H, I)


def test_routing_buffers_are_kept_for_every_shape_and_stream():
    from muxi_native_layout_kernels_amd import moe_planC
    cpu = torch.device("cpu")
    first = moe_planC._routing_buffers(3, 2, torch.bfloat16, cpu, stream=0)
    ptr = first[0].data_ptr()
    for t in range(4, 140):                                   # many other shapes must not evict it
        moe_planC._routing_buffers(t, 2, torch.bfloat16, cpu, stream=0)
    again = moe_planC._routing_buffers(3, 2, torch.bfloat16, cpu, stream=0)
    assert again[0].data_ptr() == ptr and again[1] is first[1]
    other = moe_planC._routing_buffers(3, 2, torch.bfloat16, cpu, stream=5)
    assert other[0].data_ptr() != ptr


def _plan(T, E, K, H, I, kind):
    import ctypes
    out = (ctypes.c_int32 * 8)()
    rc = _lib.load().mlk_moe_plan(T, E, K, H, I, kind, ctypes.addressof(out))
    assert rc == 0
    return dict(path=out[0], cb=out[1], max_tasks=out[2], down_r=out[3], down_slices=out[4], down_wk=out[5],
                down_lds=out[6], static_lds=out[7])


@pytest.mark.parametrize("kind", [1, 2])
@pytest.mark.parametrize("E,K,H,I", [(256, 8, 7168, 256), (256, 8, 256, 128), (128, 8, 2048, 768), (8, 2, 4096, 14336),
                                     (64, 6, 1024, 512)])
def test_moe_plan_fits_the_workgroup_lds_for_every_token_count(E, K, H, I, kind):
    """Every pass of 1..256 tokens (also the remainder passes of longer inputs) must get a down-projection
    shape whose LDS fits the 64 KiB a workgroup gets by default, with at least four waves whenever more
    than one row group per wave was chosen."""
    for T in range(1, 257):
        p = _plan(T, E, K, H, I, kind)
        assert p["path"] in (0, 1, 2, 3, 4) and p["cb"] in (1, 2, 3, 4, 6, 8)
        if p["path"] in (1, 2):
            assert p["down_lds"] + p["static_lds"] <= 64 * 1024, (T, p)
            assert p["down_wk"] >= 1 and p["down_lds"] == p["down_wk"] * p["down_r"] * p["cb"] * 1024 + T * 16 * p["down_r"] * 4
            if p["down_r"] > 1:
                assert p["down_wk"] >= 4 and p["cb"] == 1 and p["down_slices"] == p["down_r"], (T, p)
                assert (H // 16) % p["down_r"] == 0 and (I // 32) % p["down_r"] == 0
        if p["path"] == 3:
            assert p["cb"] >= 2 and (I // 32) % (p["down_slices"] * (2 if p["cb"] > 4 else 4)) == 0
        if p["path"] == 4:          # panel kernels: output rows in tiles of 256, at least four k windows per slice
            assert kind == 2 and p["cb"] >= 5 and H % 256 == 0 and 1 <= p["down_slices"] <= 8
            assert p["down_slices"] == 1 or (I // 128) // p["down_slices"] >= 4
            assert p["down_wk"] in (1, 2)       # workgroups per CU the down kernel is built for
            if p["down_wk"] == 2:               # two per CU only where the expected grid fills them (256 CUs assumed)
                assert (H // 256) * min(E, T * K) * p["down_slices"] >= 512, (T, p)
        assert p["path"] != 0 or T == 1


def test_moe_plan_known_cases():
    # soft-FP8, 256 experts, top-8 (the DeepSeek configuration): 4 row groups per wave while the output tile
    # fits, 2 from 172 tokens up (the tile of 4 row groups would leave fewer than four waves)
    assert _plan(16, 256, 8, 7168, 256, 2)["down_r"] == 4
    assert _plan(171, 256, 8, 7168, 256, 2)["down_r"] == 4
    assert _plan(172, 256, 8, 7168, 256, 2)["down_r"] == 2
    assert _plan(244, 256, 8, 7168, 256, 2)["down_r"] == 2
    assert _plan(244, 256, 8, 7168, 256, 2)["path"] == 2
    # Mixtral shape: one token -> GeMV kernels; 16 tokens -> in-kernel alignment; 64 and 256 -> row-shared kernels
    assert _plan(1, 8, 2, 4096, 14336, 1)["path"] == 0
    assert _plan(16, 8, 2, 4096, 14336, 1)["path"] == 1
    assert _plan(64, 8, 2, 4096, 14336, 1)["path"] == 3
    assert _plan(256, 8, 2, 4096, 14336, 1)["path"] == 3
    # soft-FP8 with more than 64 tokens per pass over an expert: panel kernels, if the output rows tile in 256
    assert _plan(64, 8, 2, 4096, 14336, 2)["path"] == 3
    assert _plan(256, 8, 2, 4096, 14336, 2)["path"] == 4
    # its down projection: 16 row tiles x 8 experts x 4 K slices = two workgroups on each of 256 CUs
    mixtral = _plan(256, 8, 2, 4096, 14336, 2)
    assert (mixtral["down_slices"], mixtral["down_wk"]) == (4, 2)
    # a grid that cannot reach two per CU keeps one per CU: 4 row tiles x 8 experts x 8 slices = 256
    small = _plan(256, 8, 2, 1024, 14336, 2)
    assert small["path"] == 4 and small["down_wk"] == 1
    assert _plan(256, 8, 2, 4096 + 128, 14336, 2)["path"] == 3
    # above 256 tokens: the plan of the passes of 256 that a call without the scratch of the wide kernels runs in
    assert _plan(500, 256, 8, 7168, 256, 2) == _plan(256, 256, 8, 7168, 256, 2)


def test_panel_plan_is_a_shape_the_kernel_takes():
    """The eight-wave panels' plan over odd and ordinary shapes: launch parameters that the guard passes, K slices of at least two k
    windows, a workspace exactly where panels are split, and table rows of the very shape in front of it."""
    import ctypes
    import random
    from muxi_native_layout_kernels_amd import _lib, arg_selector
    lib = _lib.load()
    rng = random.Random(7)
    for _ in range(300):
        n, k, m = 128 * rng.randint(1, 250), 128 * rng.randint(1, 140), rng.choice([1, 33, 64, 65, 100, 256, 257, 777, 4096])
        out = (ctypes.c_int32 * 4)()
        assert lib.mlk_gemm_plan(m, n, k, rng.choice([0, 2]), out) == 0
        kid, p1, p2, p3 = out
        assert ops._gemm_guard(tuple(out), n) == tuple(out)
        if kid != 8:
            assert m <= 64 and kid in (1, 4) and p2 in (1, 2, 4, 8, 16) and (kid == 1 or n // 16 > 256)
            continue
        panels = -(-n // (64 * p1)) * -(-m // (64 * p2))
        assert p3 == 1 or (p3 == 64 and panels > 256) or (panels * p3 <= 256 and k // 64 // p3 >= 2)
        assert (lib.mlk_gemm_panel_workspace_bytes(m, n, k, p1, p2, p3) > 0) == (p3 > 1)
    assert lib.mlk_gemm_plan(100, 128, 96, 0, out) != 0          # K % 128
    assert lib.mlk_gemm_plan(1 << 24, 128, 128, 0, out) != 0     # activations beyond 32-bit offsets
    assert ops._gemm_args("layoutA_gemm", 4224, 300, 1024, 1)[0] == 8
    assert ops._gemm_args("layout_gemm", 4224, 304, 1024, 1)[0] == 8
    assert ops._gemm_args("layoutA_gemm", 4224, 300, 1088, 1)[0] == 2  # K % 128
    assert ops._gemm_args("layoutA_gemm", 11008, 50, 4096, 1) == \
        arg_selector.selector("layoutA_gemm").table()[(11008, 64, 4096)]   # borrowed, not planned
    table = arg_selector.selector("layoutA_gemm").table()
    table[(4224, 300, 1024)] = (3, 4, 1, 1)
    try:
        assert ops._gemm_args("layoutA_gemm", 4224, 300, 1024, 1) == (3, 4, 1, 1)
    finally:
        del table[(4224, 300, 1024)]


@pytest.mark.parametrize("a_kind,n,k,m,want", [
    (1, 11008, 4096, 1302, lambda p1, p2, p3: p3 == 64 or p1 * p2 < 16),      # 36 panels of 256 x 256 on the fullest XCD, two of the last four full
    (1, 27648, 5120, 578, lambda p1, p2, p3: (p1, p2, p3) != (4, 4, 1)),      # 14 rows of panels of 256, 256 and 66 tokens
    (1, 11008, 4096, 128, lambda p1, p2, p3: p3 == 1),                        # few weights per CU: no second launch
    (1, 11008, 4096, 256, lambda p1, p2, p3: p3 == 1),
    (2, 512, 1408, 86, lambda p1, p2, p3: p3 > 1),
])
def test_gemm_plan_choices(a_kind, n, k, m, want):
    """Choices that cost 10 to 40 % the other way round: a last round that holds full panels is as long as a full panel, a split has
    to pay for its fold, and a small grid is cut."""
    import ctypes
    from muxi_native_layout_kernels_amd import _lib
    out = (ctypes.c_int32 * 4)()
    assert _lib.load().mlk_gemm_plan(m, n, k, a_kind, out) == 0
    assert out[0] == 8 and want(*out[1:]), list(out)


def test_shipped_panel_rows_fit_the_documented_workspace():
    """A C caller sizes the K split of a table row with mlk_gemm_workspace_bytes(): enough for the rows of kernel id 8 too, at their own
    token count and at every smaller one that borrows them."""
    from muxi_native_layout_kernels_amd import _lib, arg_selector
    lib = _lib.load()
    rows = 0
    for name in ("layout_gemm", "continuous_gemm", "layoutA_gemm", "layoutA_soft_fp8_gemm"):
        for (n, m, k), (kid, p1, p2, p3) in arg_selector.selector(name).table().items():
            if kid == 8:
                rows += 1
                for tokens in range(max(1, m - 31), m + 1):
                    assert lib.mlk_gemm_panel_workspace_bytes(tokens, n, k, p1, p2, p3) <= lib.mlk_gemm_workspace_bytes(tokens, n, p1, p3), \
                        (name, n, tokens, k)
    assert rows > 0


def test_rows_above_64_tokens_are_borrowed_and_misses_are_named(capsys, tmp_path, monkeypatch):
    """Rows that a user has scanned above 64 tokens serve nearby counts above 64, in front of the library's plan and never below; a shape
    without any gets the plan.  Either is named on stderr once."""
    from muxi_native_layout_kernels_amd import arg_selector
    p = tmp_path / "t.csv"
    p.write_text("m,n,k,kernelId,kernelParam1,kernelParam2,kernelParam3\n"
                 "4224,32,1024,1,2,4,1\n4224,256,1024,3,4,1,2\n4224,1024,1024,5,4,2,2\n4352,32,1024,1,2,4,1\n")
    sel = arg_selector._Selector(str(p), 3, arg_selector.GEMM_FALLBACK, "tmp", lambda n, m, k: (1, 1, 8, 1), True)
    sel.path = lambda: str(p)
    monkeypatch.setattr(arg_selector, "selector", lambda name: sel)
    for _ in range(2):
        assert ops._gemm_args("layoutA_gemm", 4224, 256, 1024, 1) == (3, 4, 1, 2)
        assert ops._gemm_args("layoutA_gemm", 4224, 65, 1024, 1) == (3, 4, 1, 2)
        assert ops._gemm_args("layoutA_gemm", 4224, 300, 1024, 1) == (5, 4, 2, 2)
        assert ops._gemm_args("layoutA_gemm", 4224, 4096, 1024, 1) == (5, 4, 2, 2)
        assert ops._gemm_args("layoutA_gemm", 4224, 64, 1024, 1) == (1, 2, 4, 1)
        assert ops._gemm_args("layoutA_gemm", 4352, 300, 1024, 1)[0] == 8          # no row above 64 tokens: planned
        assert ops._gemm_args("layoutA_gemm", 4224, 300, 1088, 1) == (1, 1, 8, 1)  # K % 128: no plan
    err = capsys.readouterr().err
    assert err.count("Borrowing the args of") == 4 and err.count("Fallback args to") == 2


def test_plan_of_native_activations_names_kernels_that_take_them():
    """Layout-B activations of one token block have no kernel id 4: the plan leaves it out there (a launch that asks for it runs kernel id 1
    with the least of everything), offers it from 17 tokens on, and is the row-major one wherever that names another kernel."""
    import ctypes
    from muxi_native_layout_kernels_amd import _lib
    lib = _lib.load()
    met = 0
    for n in range(128, 32768, 384):
        for k in (512, 2688, 4096, 7168, 14336):
            for m in (16, 32, 64):
                row, nat = (ctypes.c_int32 * 4)(), (ctypes.c_int32 * 4)()
                assert lib.mlk_gemm_plan_placed(m, n, k, 1, 0, row) == 0 and lib.mlk_gemm_plan_placed(m, n, k, 1, 1, nat) == 0
                if m == 16 and row[0] == 4:
                    met += 1
                    assert nat[0] in (1, 8) and (n // 16) % nat[1] == 0
                else:
                    assert list(nat) == list(row)
    assert met > 0
    assert lib.mlk_gemm_plan_placed(16, 128, 128, 1, 2, nat) != 0
    assert ops._gemm_args("layout_gemm", 9344, 16, 2688, 1, 1)[0] != 4


def test_launches_off_16_bytes_are_planned():
    """What kernel id 8 stands for with operands off 16 bytes: kernel 3 on row-major operands above 64 tokens, with as many K slices as
    put a workgroup on every CU, else kernels 1 and 4; never the panels, and always parameters the library takes."""
    import random
    rng = random.Random(9)
    for _ in range(300):
        m, k, n = 128 * rng.randint(1, 250), 128 * rng.randint(1, 140), rng.choice([1, 16, 33, 64, 65, 100, 256, 777, 4096])
        kind, native = rng.choice([0, 2]), rng.randint(0, 2)
        if native and (kind == 2 or n % 16):
            continue
        kid, p1, p2, p3, ws = ops._off16_plan(m, n, k, kind, int(native > 0), int(native == 2))
        assert ops._gemm_guard((kid, p1, p2, p3), m) == (kid, p1, p2, p3) and (ws > 0) == (p3 > 1)
        assert kid == 3 if n > 64 and not native else kid in (1, 4)
        if kid == 3:
            panels = -(-m // (64 * p1)) * -(-n // 128)
            assert p2 == 1 and (p3 == 1 or panels * p3 <= 256)
    assert ops._off16_plan(4096, 100, 4096, 1, 0, 0)[:4] == (3, 2, 1, 4)
    assert ops._off_panels(8, 0x1002) and not ops._off_panels(8, 0x1010) and not ops._off_panels(3, 0x1002)


def test_moe_pass_plan_names_what_runs():
    """One token block per task: with all the scratch it asks for a pass above 48 experts in reach (soft-FP8 weights: and three workgroups
    on two CUs) is the row-shared kernels, two blocks per task, else the decode kernels; on the scratch of the decode kernels, and
    everywhere else, it is what mlk_moe_plan() says."""
    import ctypes
    lib, out = _lib.load(), (ctypes.c_int32 * 8)()

    def pass_plan(T, E, K, H, I, kind, size):
        assert lib.mlk_moe_pass_plan(T, E, K, H, I, kind, size, out) == 0
        return list(out)

    def plan(T, E, K, H, I, kind):
        assert lib.mlk_moe_plan(T, E, K, H, I, kind, out) == 0
        return list(out)
    for T, E, K, H, I, kind, shared in [(7, 64, 7, 256, 384, 1, True), (8, 64, 6, 256, 384, 1, False), (17, 48, 4, 256, 384, 0, False),
                                        (17, 49, 4, 1152, 256, 0, True), (12, 64, 8, 256, 384, 2, True), (12, 63, 8, 256, 384, 2, False),
                                        (16, 256, 8, 7168, 256, 2, True), (244, 256, 8, 7168, 256, 2, True), (1, 256, 8, 7168, 256, 1, False),
                                        (64, 8, 2, 4096, 14336, 1, False), (256, 8, 2, 4096, 14336, 2, False)]:
        full = lib.mlk_moe_workspace_bytes(T, E, K, H, I)
        got, decode = pass_plan(T, E, K, H, I, kind, full), plan(T, E, K, H, I, kind)
        if shared:
            assert decode[0] in (1, 2) and got[:3] == [3, 2, min(E, T * K) + T * K // 32]
            assert pass_plan(T, E, K, H, I, kind, full // 2) == decode
        else:
            assert got == decode
    assert lib.mlk_moe_pass_plan(16, 8, 2, 4096, 100, 1, 0, out) != 0


def test_scan_grid_holds_what_the_plan_chooses_from():
    """A scan tries every launch of the eight-wave panels that the library's plan can answer and that the packaged tables hold, so that a
    scanned row in front of the plan is no slower for want of having been tried."""
    import ctypes
    import random
    from muxi_native_layout_kernels_amd import arg_selector
    from muxi_native_layout_kernels_amd.kernel_args_scan import scan
    lib, out, rng, met = _lib.load(), (ctypes.c_int32 * 4)(), random.Random(11), 0
    for _ in range(300):
        n, k, m = 128 * rng.randint(1, 250), 128 * rng.randint(1, 140), rng.choice([1, 33, 64, 65, 100, 256, 300, 777, 4096])
        assert lib.mlk_gemm_plan(m, n, k, rng.choice([0, 2]), out) == 0
        if out[0] == 8:
            met += 1
            assert tuple(out) in scan.panel_grid(n, m, k)
    assert met > 100
    for name in ("layout_gemm", "continuous_gemm", "layoutA_gemm", "layoutA_soft_fp8_gemm"):
        for (n, m, k), args in arg_selector.selector(name).table().items():
            assert args[0] != 8 or args in scan.panel_grid(n, m, k)


def test_panels_off_16_bytes_have_a_counter_each_or_run_whole():
    """Kernel ids 3 and 5 asked for 256 x 256 panels in K slices with operands off 16 bytes run twice as many panels of 128 tokens: where those are
    more than there are counters for, the call runs whole panels and is not refused (here it gets as far as the launch, which has no GPU)."""
    import torch
    from muxi_native_layout_kernels_amd import _lib
    if torch.cuda.is_available():
        pytest.skip("the operands are addresses of nothing")
    lib = _lib.load()
    n, m, k, at = 131072, 8192, 256, 1 << 40                  # 512 x 32 panels of 256 x 256: as many as there are counters
    size = lib.mlk_gemm_workspace_bytes(m, n, 4, 2)
    for kid in (3, 5):
        for shift in (0, 2):
            rc = lib.mlk_gemm_layout_a(at, at + shift, at, m, n, k, 1, 1, 0, 0, 1.0, None, None, kid, 4, 2, 2, at, size, None)
            assert rc != 0 and b"counter region" not in lib.mlk_last_error() and b"workspace" not in lib.mlk_last_error()
