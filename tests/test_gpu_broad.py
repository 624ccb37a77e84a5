"""The broad product kernel (tiles of 256 x 288 to 192 x 256 outputs, four waves) at the edges of its tiles, rings and cuts."""
import pytest
import torch

import torch_ops as ref
from test_gpu_kernels import check, gated, rand

TILES = [256288, 256256, 192288, 192256]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (191, 256, 128), (193, 264, 192), (257, 296, 320), (255, 1000, 448), (300, 584, 1088),
                                   (513, 2304, 2304)])
def test_gemm_broad(gpu_lib, M, N, K):
    """Against the 32-bit reference, one bfloat16 step (gated: three, its two products are rounded first); uncut to the bit what the
    wide kernel gives, whose sums run along K in the same order; strided rows in and out; fewer slabs than the rings hold."""
    from simply_amd.kernels import ops
    from simply_amd.kernels.lib import KernelError
    from simply_amd.kernels.packing import pack_gate_up, pack_tiles
    a, w, w2 = rand((M, K), torch.bfloat16, 1), rand((N, K), torch.bfloat16, 2, 0.05), rand((N, K), torch.bfloat16, 3, 0.05)
    tw, tw2 = pack_tiles(w), pack_gate_up(w, w2)
    t = dict(bf16_steps=1.0)
    big = rand((M, K + 16), torch.bfloat16, 4)
    for tile in TILES:
        kw = dict(algo=ops.ALGO_WIDE, shape=1000000 + tile)
        check(ops.gemm(a, tw, **kw), ref.gemm(a, w), **t)
        assert torch.equal(ops.gemm(a, tw, **kw), ops.gemm(a, tw, algo=ops.ALGO_WIDE, shape=3128128))
        assert torch.equal(ops.gemm(a, tw2, **kw), ops.gemm(a, tw2, algo=ops.ALGO_WIDE, shape=3128128))
        for act in range(5):
            opt = {"activation": act, **({"limit": 0.9} if act == 4 else {})}
            check(ops.gemm(a, tw2, **kw, **opt), ref.gemm(a, w, w2=w2, **opt), bf16_steps=4.0 if act == 2 else 3.0)
            if act < 4:
                assert torch.equal(ops.gemm(a, tw, activate=act, **kw), ops.gemm(a, tw, activate=act, algo=ops.ALGO_WIDE, shape=3128128))
        out = torch.full((M, N + 16), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.gemm(big[:, 8:8 + K], tw, out=out[:, 8:8 + N], **kw)
        check(out[:, 8:8 + N], ref.gemm(big[:, 8:8 + K], w), **t)
        assert (out[:, :8] == 7.0).all() and (out[:, 8 + N:] == 7.0).all()
        for cuts in (2, 3):   # (more than K has slabs shrinks to what it has)
            check(ops.gemm(a, tw, algo=ops.ALGO_WIDE, shape=cuts * 10000000 + 1000000 + tile), ref.gemm(a, w), **t)
        # rows that are not of whole 16-byte pieces are refused where the tile is asked for, and go another way by themselves
        odd = torch.empty((M, N + 4), dtype=torch.bfloat16, device="cuda")
        with pytest.raises(KernelError, match="broad"):
            ops.gemm(a, tw, out=odd[:, :N], **kw)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,is_gated", [(1024, 9216, 2304, True), (2048, 8192, 2048, False), (1056, 4096, 14336, False)])
def test_gemm_takes_broad_tiles_by_itself(gpu_lib, M, N, K, is_gated):
    """The dispatcher's choice with the broad kernel, and beside it what that kernel does not take: rows 8 bytes off."""
    from simply_amd.kernels import ops
    from simply_amd.kernels.packing import pack_gate_up, pack_tiles
    assert gpu_lib.load().sa_gemm_broad_tile(M, N, K, int(is_gated), 256 << 20) > 0
    a, w, w2 = rand((M, K), torch.bfloat16, 5), rand((N, K), torch.bfloat16, 6, 0.03), rand((N, K), torch.bfloat16, 7, 0.03)
    tw, want = (pack_gate_up(w, w2), ref.gemm(a, w, w2=w2)) if is_gated else (pack_tiles(w), ref.gemm(a, w))
    t = gated(dict(bf16_steps=1.0)) if is_gated else dict(bf16_steps=1.0)
    check(ops.gemm(a, tw), want, **t)
    off = torch.empty((M, N + 8), dtype=torch.bfloat16, device="cuda")
    check(ops.gemm(a, tw, out=off[:, 4:4 + N]), want, **t)


def test_broad_tiles_where_they_are_ahead():
    """(M, N, K, gated): cuts * 1000000 + rows * 1000 + weight rows, or 0 where the wide kernel's tiles are taken."""
    from simply_amd.kernels import lib
    tile = lambda *at: lib.load().sa_gemm_broad_tile(*at, 256 << 20)
    assert tile(2048, 9216, 2304, 1) == 1256288 and tile(2048, 8192, 2048, 0) == 1256256 and tile(1056, 36864, 4608, 1) == 1192288
    assert tile(2048, 4096, 2304, 0) == tile(2048, 2048, 2048, 0) == tile(512, 2304, 9216, 0) == tile(64, 9216, 2304, 1) == 0
    assert tile(1056, 4608, 36864, 0) // 1000000 > 1 and lib.load().sa_gemm_broad_tile(1056, 4608, 36864, 0, 0) // 1000000 <= 1


@pytest.mark.gpu
@pytest.mark.parametrize("M,n,last,K", [(4096, 1024, 64, 1024), (1031, 2048, 2048, 1088), (2047, 2048, 16, 2048)])
def test_sections_on_broad_tiles(gpu_lib, M, n, last, K):
    """Several products at once of many rows, with a last section that is shorter (on the wide kernel) or whole (on the broad one)."""
    from simply_amd.kernels import ops
    ws = [rand((last if s == 3 else n, K), torch.bfloat16, 20 + s, 0.05) for s in range(4)]
    a = rand((M, 4 * K), torch.bfloat16, 30)
    got = ops.gemm_sections(a, ops.SectionedWeight(ws))
    for s, w in enumerate(ws):
        check(got[:, s * n:s * n + w.shape[0]], ref.gemm(a[:, s * K:(s + 1) * K], w), bf16_steps=1.0)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1537, 4, 512), (2047, 64, 2048), (2048, 512, 4096), (4096, 132, 1088), (1600, 640, 2304)])
def test_many_rows_against_few_outputs(gpu_lib, M, N, K):
    """Beyond 1,536 rows: tiles and a cut of K as for fewer rows, up to 64 tiles of 128 x 128 (and the first size with more)."""
    from simply_amd.kernels import ops
    from simply_amd.kernels.packing import pack_tiles
    a, w = rand((M, K), torch.bfloat16, 40), rand((N, K), torch.bfloat16, 41, 0.05)
    check(ops.gemm(a, pack_tiles(w)), ref.gemm(a, w), bf16_steps=1.0)
    check(ops.gemm(a, pack_tiles(w), out_dtype=torch.float32), ref.gemm(a, w, out_dtype=torch.float32), rtol=2e-3, atol=2e-3)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [8, 1028, 2304, 3588, 4608, 5120])
def test_norm_of_any_number_of_planes(gpu_lib, D):
    """A product's planes added up in the norm behind it: to the bit what the sum kernel and the norm of its result give."""
    from simply_amd.kernels import ops
    T = 70
    kw = dict(post_weight=rand((D,), torch.bfloat16, 50, 0.3), post_eps=1e-6, post_plus_one=True, next_weight=rand((D,), torch.bfloat16, 51, 0.3),
              next_eps=1e-6, next_plus_one=True, out_dtype=torch.bfloat16)
    for count in (1, 2, 3, 4, 5, 6, 7, 8, 11):
        planes, h = rand((count, T, D), torch.float32, 60 + count), rand((T, D), torch.float32, 52)
        h2 = h.clone()
        y = torch.empty((T, D), dtype=torch.bfloat16, device="cuda")
        whole = ops.PartialSums(planes, y.clone()).materialize()
        got, want = ops.add_rmsnorm(ops.PartialSums(planes, y), h, **kw), ops.add_rmsnorm(whole, h2, **kw)
        assert torch.equal(got, want) and torch.equal(h, h2)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 1, 32), (64, 16, 64), (100, 20, 96), (129, 33, 1056), (257, 48, 2080), (2047, 64, 2048), (1000, 64, 4096)])
def test_many_rows_against_a_handful_of_outputs(gpu_lib, M, N, K):
    """A workgroup for 16 rows and all outputs: fewer chunks of K than waves, remainders, one to four tiles, both types of result; and a
    row's bits do not depend on the rows beside it."""
    from simply_amd.kernels import ops
    from simply_amd.kernels.packing import pack_tiles
    big, w = rand((M, K + 16), torch.bfloat16, 70), rand((N, K), torch.bfloat16, 71, 0.05)
    a, tw = big[:, 8:8 + K], pack_tiles(w)
    assert ops.gemm_plan(M, N, K)[0] == ops.ALGO_TILED
    check(ops.gemm(a, tw), ref.gemm(a, w), bf16_steps=1.0)
    got = ops.gemm(a, tw, out_dtype=torch.float32)
    torch.testing.assert_close(got, (a.double() @ w.double().T).float(), rtol=1e-5, atol=2e-6 * K ** 0.5)
    assert torch.equal(got[-33:], ops.gemm(a[-33:], tw, out_dtype=torch.float32))
    out = torch.full((M, N + 3), 7.0, device="cuda")
    ops.gemm(a, tw, out=out[:, 2:2 + N])
    assert torch.equal(out[:, 2:2 + N], got) and (out[:, :2] == 7.0).all() and (out[:, 2 + N:] == 7.0).all()


@pytest.mark.parametrize("M", [1, 96, 512, 4096])
def test_plan_of_a_lone_section_shorter_than_a_step(M):
    """No whole section: nothing for the broad kernel (its plan of no outputs divided by their tiles)."""
    from simply_amd.kernels import lib
    for N in (16, 1024, 2047):
        assert lib.load().sa_gemm_sections_tile(M, N, 2048, 2048, 256 << 20) == 0


@pytest.mark.gpu
def test_a_lone_section_shorter_than_a_step(gpu_lib):
    from simply_amd.kernels import ops
    from simply_amd.kernels.packing import pack_tiles
    M, N, K = 512, 1024, 2048
    a, w = rand((M, K), torch.bfloat16, 80), rand((N, K), torch.bfloat16, 81, 0.05)
    tw, out, ws = pack_tiles(w), torch.empty((M, N), dtype=torch.bfloat16, device="cuda"), ops._workspace(a.device)
    gpu_lib.call("sa_gemm_sections", a.data_ptr(), K, tw.data.data_ptr(), out.data_ptr(), 1, N, M, N, K, 2048, K, ws.data_ptr(), ws.numel(),
                 ops._stream())
    check(out, ref.gemm(a, w), bf16_steps=1.0)


@pytest.mark.gpu
@pytest.mark.parametrize("M,n,sections,last,K", [(2047, 2048, 4, 64, 2048), (2047, 2048, 4, 16, 2048), (700, 4096, 4, 64, 4096), (3000, 1024, 4, 64, 1024),
                                                 (1500, 2048, 4, 304, 2048)])
def test_whole_sections_on_broad_tiles_and_a_shorter_last_one(gpu_lib, M, n, sections, last, K):
    """The whole sections in the broad kernel's launch, the last one by itself from where they end: its rows of W, its columns of A and C."""
    from simply_amd.kernels import ops
    assert gpu_lib.load().sa_gemm_sections_tile(M, sections * n + last, K, n, ops.WORKSPACE_BYTES) > 0
    ws = [rand((last if s == sections else n, K), torch.bfloat16, 90 + s, 0.05) for s in range(sections + 1)]
    big = rand((M, (sections + 1) * K + 16), torch.bfloat16, 99)
    a = big[:, 8:8 + (sections + 1) * K]
    got = ops.gemm_sections(a, ops.SectionedWeight(ws))
    for s, w in enumerate(ws):
        check(got[:, s * n:s * n + w.shape[0]], ref.gemm(a[:, s * K:(s + 1) * K], w), bf16_steps=1.0)


def test_sections_where_the_broad_tiles_are_ahead():
    """(M, outputs, K, n_step): by the rounds of the wide kernel's tiles against those of the broad one's, for prompts and shorter portions."""
    from simply_amd.kernels import lib
    tile = lambda *at: lib.load().sa_gemm_sections_tile(*at, 256 << 20)
    assert tile(2047, 8256, 2048, 2048) == 256256 and tile(1024, 16384, 4096, 4096) == 256256 and tile(3000, 4160, 1024, 1024) == 192256
    assert tile(512, 16384, 4096, 4096) == tile(2047, 4096, 1024, 1024) == tile(774, 8256, 2048, 2048) == tile(64, 8256, 2048, 2048) == 0


def test_broad_tiles_with_a_cut_of_their_own():
    """Beside tiles whose K is cut too: a cut for the broad tiles' size well ahead, the other tiles' cut where it serves both, else the others."""
    from simply_amd.kernels import lib
    tile = lambda *at: lib.load().sa_gemm_broad_tile(*at, 0, 256 << 20)
    assert tile(544, 4608, 36864) == 5192288 and tile(320, 6144, 14336) == 5192256 and tile(1024, 4608, 36864) == 4256288
    assert tile(1056, 4608, 36864) == 3256288
    assert tile(160, 2304, 9216) == tile(896, 2304, 9216) == tile(129, 2048, 8192) == tile(129, 12288, 4096) == 0
    # a workspace that holds two of the five planes, or none
    two = 2 * 544 * 4608 * 4
    assert lib.load().sa_gemm_broad_tile(544, 4608, 36864, 0, two) // 1000000 <= 2
    assert lib.load().sa_gemm_broad_tile(544, 4608, 36864, 0, 0) // 1000000 <= 1


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(544, 4096, 14336), (320, 6144, 14336)])
def test_gemm_takes_broad_tiles_with_a_cut_of_their_own(gpu_lib, M, N, K):
    from simply_amd.kernels import ops
    from simply_amd.kernels.packing import pack_tiles
    assert gpu_lib.load().sa_gemm_broad_tile(M, N, K, 0, ops.WORKSPACE_BYTES) // 1000000 > 1
    a, w = rand((M, K), torch.bfloat16, 110), rand((N, K), torch.bfloat16, 111, 0.02)
    tw, want = pack_tiles(w), ref.gemm(a, w)
    check(ops.gemm(a, tw), want, bf16_steps=1.0)
    left = ops.gemm(a, tw, defer_sum=True)
    assert isinstance(left, ops.PartialSums)
    check(left.materialize(), want, bf16_steps=1.0)


def test_cuts_where_the_sum_is_a_kernel_of_its_own():
    """Beyond 1,536 rows: cuts that pay where a norm adds the planes up are not taken where a kernel has to."""
    from simply_amd.kernels import lib
    planes = lambda *at: lib.load().sa_gemm_planes_broad_tile(*at, 256 << 20)
    summed = lambda *at: lib.load().sa_gemm_broad_tile(*at, 0, 256 << 20)
    assert planes(2047, 2304, 9216) == 4256288 and planes(4096, 2048, 16384) == 2256256 and planes(1056, 4608, 36864) == 3256288
    assert summed(2047, 2304, 9216) == summed(4096, 2048, 16384) == summed(1600, 1024, 4096) == summed(1600, 640, 4608) == 0
    assert summed(4096, 2304, 9216) == 2256288 and summed(1056, 4608, 36864) == 3256288


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,shape", [(300, 584, 1088, 31192256), (257, 296, 320, 21256288), (544, 4096, 14336, 0)])
def test_activated_products_with_a_cut_on_broad_tiles(gpu_lib, M, N, K, shape):
    """The activation of the summed product rounded to bfloat16, by a pass behind the sum: within one step of it on what the product gives."""
    from simply_amd.kernels import ops
    from simply_amd.kernels.packing import pack_tiles
    if shape == 0:
        assert gpu_lib.load().sa_gemm_broad_tile(M, N, K, 0, ops.WORKSPACE_BYTES) // 1000000 > 1
    a, w = rand((M, K), torch.bfloat16, 120), rand((N, K), torch.bfloat16, 121, 0.03)
    tw, kw = pack_tiles(w), dict(algo=ops.ALGO_WIDE, shape=shape) if shape else {}
    plain = ops.gemm(a, tw, **kw)
    check(plain, ref.gemm(a, w), bf16_steps=1.0)
    for act in range(4):
        check(ops.gemm(a, tw, activate=act, **kw), ref.ACTIVATIONS[act](plain.float()).to(torch.bfloat16), bf16_steps=1.0)


def test_few_outputs_of_a_long_k_keep_their_cuts():
    """(rows, outputs, K): up to K = 4,096 the narrow kernel whatever the rows; beyond only with rows for many workgroups."""
    from simply_amd.kernels import lib, ops
    takes = lib.load().sa_gemm_narrow_takes
    assert all(takes(M, N, K) for M in (33, 100, 2047, 8192) for N in (1, 16, 64) for K in (32, 2048, 4096))
    assert takes(200, 16, 8192) and takes(2047, 64, 8192) and takes(1031, 16, 16384) and takes(4096, 64, 16384) and takes(2047, 16, 36864)
    assert not any(takes(*at) for at in ((33, 16, 8192), (200, 64, 8192), (200, 16, 16384), (1031, 64, 16384), (33, 16, 36864), (2047, 64, 36864),
                                         (32, 16, 2048), (100, 65, 2048), (100, 16, 2056)))
    assert ops.gemm_plan(33, 16, 36864)[1]["tiled"] < 16   # (not the 41 us of 16 rows' workgroups that walk it all)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 16, 8192), (200, 16, 8192), (40, 64, 16416), (100, 48, 36864)])
def test_few_outputs_on_both_sides_of_the_line(gpu_lib, M, N, K):
    from simply_amd.kernels import ops
    from simply_amd.kernels.packing import pack_tiles
    a, w = rand((M, K), torch.bfloat16, 130), rand((N, K), torch.bfloat16, 131, 0.05)
    tw = pack_tiles(w)
    check(ops.gemm(a, tw), ref.gemm(a, w), bf16_steps=1.0)
    torch.testing.assert_close(ops.gemm(a, tw, out_dtype=torch.float32), (a.double() @ w.double().T).float(), rtol=1e-5, atol=2e-6 * K ** 0.5)
