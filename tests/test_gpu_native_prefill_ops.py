"""The prefill path's ops in the C++ extension against the ctypes ops of the same names: same results on every form they take
(no rows, one weight matrix or four, outputs given, prologues), and the same refusals."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def both():
    from flh_amd import _ext_ops, _ops
    return _ext_ops, _ops


def same(a, b):
    if isinstance(a, torch.Tensor):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)
    else:
        assert len(a) == len(b)
        for x, y in zip(a, b):
            same(x, y)


def codes(rows, k, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + rows)
    return torch.randint(0, 256, (rows, k // 2), dtype=torch.uint8, device="cuda", generator=g)


def halves(*shape, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + shape[0])
    return (torch.randn(*shape, device="cuda", generator=g) * 0.05).half()


@pytest.mark.parametrize("m", [0, 1, 130])
@pytest.mark.parametrize("a_groups,b_groups", [(False, False), (False, True), (True, True)])
def test_six_bit_products(m, a_groups, b_groups):
    ext, ctypes_ops = both()
    k, n, ng = 512, 256, 4
    a6, w = ctypes_ops.encode_f6(codes(m, k)), [codes(r, k, 7) for r in (n, 128, 128, 0)]
    sa = halves(m, ng if a_groups else 1).abs() if m else torch.empty(0, ng if a_groups else 1, device="cuda", dtype=torch.half)
    cols = ng if b_groups else 1
    sw = [halves(r, cols, seed=3).abs() if r else torch.empty(0, cols, device="cuda", dtype=torch.half) for r in (n, 128, 128, 0)]
    res = halves(m, n) if m else torch.empty(0, n, device="cuda", dtype=torch.half)
    w6 = [ext.encode_f6_many([x])[0] for x in w]
    same(ext.encode_f6_many(w[:4]), [ctypes_ops.encode_f6(x) for x in w])
    out = []
    for ops in (ext, ctypes_ops):
        r = [ops.gemm_f6_dequant_multi(a6, w6[:3], sa, sw[:3]), ops.gemm_f6_dequant_multi(a6, w6, sa, sw),
             ops.gemm_f6_dequant_add(a6, w6[0], sa, sw[0], res), ops.gemm_f6_swiglu(a6, w6[0], w6[0].clone(), sa, sw[0], sw[0].clone())]
        r.append(ops.gemm_f6_dequant_o16_gs(a6, w6[0], sa, sw[0]) if b_groups else ops.gemm_f6_dequant_o16(a6, w6[0], sa, sw[0]))
        kept = res.clone()
        assert ops.gemm_f6_dequant_add(a6, w6[0], sa, sw[0], kept, out=kept).data_ptr() == kept.data_ptr()
        r.append(kept)
        if m:
            cos, sin = halves(m, 128, seed=5), halves(m, 128, seed=6)
            caches = [torch.zeros(1, 1, m + 2, 128, device="cuda", dtype=torch.half) for _ in range(4)]
            pos = torch.arange(2, m + 2, device="cuda")
            r += [ops.gemm_f6_qkv_rope(a6, sa, w6[:3], sw[:3], cos, sin, pos, caches[0], caches[1], 1),
                  ops.gemm_i4_qkv_rope(codes(m, k), sa, w[:3], sw[:3], cos, sin, pos, caches[2], caches[3], 1, 128), caches]
        out.append(r)
    same(*out)


@pytest.mark.parametrize("m", [0, 3, 257])
def test_producers(m):
    ext, ctypes_ops = both()
    k = 1024
    x, y = (halves(m, k, seed=i) if m else torch.empty(0, k, device="cuda", dtype=torch.half) for i in (1, 2))
    weight = halves(k)
    out = []
    for ops in (ext, ctypes_ops):
        out.append([ops.group_quantize_f6(x, False), ops.group_quantize_f6(x, scale_mul=0.5), ops.rmsnorm_group_quantize_f6(x, weight, 1e-5),
                    ops.rmsnorm_group_quantize_f6(x, None, 1e-6), ops.silu_mul_group_quantize_f6(x, y),
                    ops.add_rmsnorm_rotate_and_quantize_i4(x, y, weight, 1e-5), ops.add_rmsnorm_rotate_and_quantize_i4(x, y, None, 1e-5, False, 0.9),
                    ops.rotate_and_quantize_f6(x), ops.rotate_and_quantize_f6(x, "exact", 0.9), ops.rotate_and_quantize_f6(x, False),
                    ops.rotate_and_quantize_f6(x, norm_weight=weight, eps=1e-5), ops.rotate_and_quantize_f6(x, norm_weight=weight, eps=1e-5, add=y),
                    ops.rotate_and_quantize_f6(halves(2, 11008))])
    same(*out)


def test_refusals():
    ext, ctypes_ops = both()
    k = 512
    a, w, x = codes(4, k), codes(128, k, 1), halves(4, 1024)
    a6, w6 = ctypes_ops.encode_f6(a), ctypes_ops.encode_f6(w)
    sa, sw, sg = halves(4, 1).abs(), halves(128, 1).abs(), halves(128, 4).abs()
    cos, cache, pos = halves(4, 128), torch.zeros(1, 1, 4, 128, device="cuda", dtype=torch.half), torch.arange(4, device="cuda")
    calls = [lambda o: o.encode_f6_many([]), lambda o: o.encode_f6_many([w, codes(2, 256)]), lambda o: o.encode_f6_many([w.cpu()]),
             lambda o: o.encode_f6_many([w[:, :32]]), lambda o: o.encode_f6_many([w] * 5),
             lambda o: o.group_quantize_f6(x[:, :100]), lambda o: o.group_quantize_f6(x.float()), lambda o: o.group_quantize_f6(x[0]),
             lambda o: o.rmsnorm_group_quantize_f6(x, cos, 1e-5), lambda o: o.silu_mul_group_quantize_f6(x, x[:2]),
             lambda o: o.gemm_f6_dequant_o16(a6, w6, sa, sg), lambda o: o.gemm_f6_dequant_o16(a6, w6[:, :96], sa, sw),
             lambda o: o.gemm_f6_dequant_o16(a6.cpu(), w6, sa, sw), lambda o: o.gemm_f6_dequant_o16_gs(a6, w6, sa, sw),
             lambda o: o.gemm_f6_dequant_o16_gs(a6, w6, halves(4, 2), sg), lambda o: o.gemm_f6_dequant_add(a6, w6, sa, sw, halves(4, 64)),
             lambda o: o.gemm_f6_dequant_add(a6, w6, halves(4, 4), sw, halves(4, 128)),
             lambda o: o.gemm_f6_dequant_add(a6, w6, sa, sw, halves(4, 128), out=halves(2, 128)),
             lambda o: o.gemm_f6_swiglu(a6, w6, w6[:64], sa, sw, sw), lambda o: o.gemm_f6_swiglu(a6, w6, w6, sa, sw, sg),
             lambda o: o.gemm_f6_dequant_multi(a6, [], sa, []), lambda o: o.gemm_f6_dequant_multi(a6, [w6, w6], sa, [sw, sg]),
             lambda o: o.gemm_f6_dequant_multi(a6, [w6], sa.float(), [sw]),
             lambda o: o.gemm_f6_qkv_rope(a6, sa, [w6] * 2, [sw] * 2, cos, cos, pos, cache, cache, 1),
             lambda o: o.gemm_f6_qkv_rope(a6, sa, [w6] * 3, [sw] * 3, cos, cos, pos, cache, cache, 3),
             lambda o: o.gemm_f6_qkv_rope(a6, sa, [w6] * 3, [sw] * 3, cos, cos, pos.int(), cache, cache, 1),
             lambda o: o.gemm_i4_qkv_rope(a, sa, [w] * 3, [sw, sw, sg], cos, cos, pos, cache, cache, 1),
             lambda o: o.gemm_i4_qkv_rope(a, sa, [w] * 3, [sw] * 3, cos[:2], cos, pos, cache, cache, 1),
             lambda o: o.gemm_i4_qkv_rope(a, sa, [w] * 3, [sw] * 3, cos, cos, pos, cache.float(), cache, 1),
             lambda o: o.add_rmsnorm_rotate_and_quantize_i4(x, x[:2], None, 1e-5), lambda o: o.add_rmsnorm_rotate_and_quantize_i4(x, x, cos, 1e-5),
             lambda o: o.add_rmsnorm_rotate_and_quantize_i4(x, x, None, 1e-5, "other"), lambda o: o.rotate_and_quantize_f6(x, add=x),
             lambda o: o.rotate_and_quantize_f6(x, "fast"), lambda o: o.rotate_and_quantize_f6(x[0]), lambda o: o.rotate_and_quantize_f6(x[:, :384].contiguous()),
             lambda o: o.rotate_and_quantize_f6(x, norm_weight=halves(1024)), lambda o: o.rotate_and_quantize_f6(halves(2, 11008), "exact")]
    for ops in both():
        for i, call in enumerate(calls):
            with pytest.raises(RuntimeError):
                call(ops)
                print("accepted", ops.__name__, i)
