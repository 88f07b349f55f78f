"""bfloat16 activations and outputs inside the kernels' loads and stores (the op
orcasaq2::shards_linear behind Exl3LinearMethod.apply): bit for bit what converting x to fp16, the
fp16 ops, and converting the concatenated outputs back give, on every route -- one to four rows,
five to sixteen, the K-split GEMM, the stream-K GEMM (one shard and grouped) and the reconstruct
branch into its columns -- with values that round to fp16 infinity and outputs that are NaN."""
import pytest
import torch

from orcasaq2 import _native
from orcasaq2 import ops as O
from orcasaq2 import synthetic as syn

pytestmark = pytest.mark.gpu
D = torch.device("cuda", 0)


def _bits(t):
    return torch.where(t.isnan(), torch.full_like(t, 7.0), t).view(torch.int16)


@pytest.mark.parametrize("rows,ic,spec", [
    (1, 384, [(256, 4)]), (1, 17408, [(128, 3)]),       # a whole segment; split into accumulator words
    (4, 640, [(256, 3), (128, 5)]),
    (9, 384, [(256, 4), (128, 2)]),
    (33, 640, [(256, 3), (128, 6)]), (129, 384, [(128, 4)]),
    (600, 8192, [(128, 4)]), (2000, 4096, [(8192, 2), (8192, 3)]),   # stream-K: one shard, grouped
    (600, 640, [(256, 4), (128, 5)]),                    # above 512 rows: the K split at 600,
    (2500, 5120, [(6144, 4), (128, 5), (256, 3)]),       # the narrow shards beside a reconstruct branch,
    (1100, 5120, [(5120, 2)]),                           # the reconstruct branch alone
    (515, 8192, [(128, 4), (256, 3)]),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_typed_io_is_conversion_around_fp16(native, rows, ic, spec, dtype):
    print(f"typed io rows={rows} ic={ic} {spec} {dtype}", flush=True)
    g = torch.Generator(device=D).manual_seed(rows)
    lins = [syn.linear_gpu(ic, oc, K, g, D) for oc, K in spec]
    x = (torch.randn(rows, ic, generator=g, device=D) * 3).to(dtype)
    if dtype == torch.bfloat16:
        x[rows // 2, 5] = 1e6            # infinity in fp16
    a = ([l["trellis"] for l in lins], [l["suh"] for l in lins], [l["svh"] for l in lins], [oc for oc, _ in spec],
         [float(K) for _, K in spec], [False] * len(spec), [False] * len(spec))
    got = torch.ops.orcasaq2.shards_linear(x, *a)
    assert got.dtype == dtype and got.shape == (rows, sum(oc for oc, _ in spec))
    assert torch.equal(_bits(torch.ops.orcasaq2.shards_linear_eager(x, *a)), _bits(got))
    xh = x.half()
    shards = [dict(l, codebook=0) for l in lins]
    split = O._ksplit_shards(rows, ic, tuple(oc for oc, _ in spec)) if rows > O.SPLIT_MAX_ROWS else ()
    if rows <= 16:
        want = _native.gemv_grouped(xh, shards)
    elif not split and all(O._op_route(rows, ic, oc) for oc, _ in spec):
        want = _native.gemm_grouped(xh, shards)
    else:
        want = torch.empty(rows, sum(a[3]), dtype=torch.half, device=D)
        cols = [sum(a[3][:i]) for i in range(len(spec))]
        if split:
            _native.linear_io(xh, want, [cols[i] for i in split], *([v[i] for i in split] for v in a[:5]), [0] * len(split),
                              True)
        for i in set(range(len(spec))) - set(split):
            want[:, cols[i]:cols[i] + a[3][i]] = O._shard_gemm_impl(xh, *(v[i] for v in a))
    assert torch.equal(_bits(got), _bits(want.to(dtype)))


def test_gradient_of_the_layer_is_still_refused(native):
    """An x that requires a gradient takes the op whose backward raises, not the eager form."""
    from orcasaq2.config import Exl3Config, Exl3LinearMethod
    layer, method = torch.nn.Module(), Exl3LinearMethod(Exl3Config.from_config({}), "p")
    method.create_weights(layer, 256, [128], 256, 128, torch.half)
    lin = syn.linear(256, 128, 4, seed=1)
    for name in ("trellis", "suh", "svh"):
        getattr(layer, name).weight_loader(getattr(layer, name), lin[name].to(D))
    method.process_weights_after_loading(layer)
    x = torch.randn(2, 256, device=D).half()
    y = method.apply(layer, x.clone().requires_grad_())
    with pytest.raises(RuntimeError):
        y.float().sum().backward()
    assert torch.equal(method.apply(layer, x), y.detach())
    for v in (x, x.bfloat16()):
        got = torch.compile(lambda t: method.apply(layer, t * 1.0), backend="eager", fullgraph=True)(v)
        assert torch.equal(got, method.apply(layer, v))
    # bf16 at an odd element offset: as good as an aligned copy
    flat = torch.cat([x.flatten()[:1], x.flatten()]).bfloat16()
    assert torch.equal(method.apply(layer, flat[1:].view(2, 256)), method.apply(layer, x.bfloat16()))
