"""The no-allocation attention entry point (ae_attention_varlen_noalloc, static device scratch)
against the allocating operator ae_attention_varlen, through the C ABI."""
import ctypes

import numpy as np
import pytest

import arctic_embed_amd as ae

pytestmark = pytest.mark.gpu


def _call(lib, qkv, cu, n, t, max_len, ctx):
    return lib.ae_attention_varlen_noalloc(ctypes.c_void_p(qkv), ctypes.c_void_p(cu), n, t, max_len,
                                           ctypes.c_void_p(ctx), None)


@pytest.fixture(params=[0, 1], ids=["by_shape", "tiles32"])
def form(request, torch_gpu):
    """By their shapes all but the last set take kernels without a plan; forced, the 32-query tiles."""
    ae.set_attention_form(request.param)
    yield request.param
    ae.set_attention_form(0)


def test_noalloc_attention_matches_allocating_operator(torch_gpu, form):
    """Bit-identical to ae_attention_varlen on consecutive calls through every kernel form.  The
    static plan keeps the last call's records, so each call must rewrite what it reads: with the
    tiles forced, after the first (split into two lists) set come the short-row kernels, then
    smaller tiled sets with fewer segments and tiles, a split set and a non-split set after it."""
    torch = torch_gpu
    lib = ae.lib()
    rng = np.random.default_rng(7)
    for lens in ([130, 512, 7, 64, 1, 300, 33, 257],  # tiled, split (max > 400, mean <= 448): 46 tiles
                 [100, 3, 70, 9],  # 8 tiles
                 [40, 2, 17],  # max_len <= 64: short-row kernel
                 [200, 90, 150, 77, 120],  # tiled, one list: 22 tiles
                 [450, 20, 66],  # tiled, split: 19 tiles
                 [300, 250, 100],  # tiled, one list after a split call
                 [96] * 3 + [15] * 14):  # 17 segments: the plan for 16-query tiles too
        cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        T = int(cu[-1])
        print("noalloc attention lens", lens, flush=True)
        qkv = torch.from_numpy(rng.normal(0, 1.0, (T, 1152)).astype(np.float32)).cuda()
        cu_d = torch.from_numpy(cu).cuda()
        ref = torch.full((T, 384), float("nan"), dtype=torch.float32, device="cuda")
        out = torch.full((T, 384), float("nan"), dtype=torch.float32, device="cuda")
        ae.attention_varlen(qkv.data_ptr(), cu_d.data_ptr(), len(lens), T, ref.data_ptr())
        torch.cuda.synchronize()
        assert _call(lib, qkv.data_ptr(), cu_d.data_ptr(), len(lens), T, max(lens), out.data_ptr()) == ae.AE_OK
        torch.cuda.synchronize()
        r, o = ref.cpu().numpy(), out.cpu().numpy()
        assert np.all(np.isfinite(r))
        assert np.array_equal(r.view(np.uint32), o.view(np.uint32)), lens
