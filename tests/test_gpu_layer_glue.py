"""The launches around a layer's attention: rotated heads, open-page buffers,
sequence reset, against the elementwise forms, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu
F16 = torch.float16


@pytest.fixture(autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")


def _cfg(care_kv, Hq, Hkv, D, **kw):
    args = dict(num_layers=2, num_heads=Hq, num_kv_heads=Hkv, head_dim=D, page_size=16, max_pages=8, base_bits=3,
                group_size=32, k_channel_group=32, v_token_block=4, sketch_dim=32, packed_base=True, scale_quant="int8",
                store_budget_mode="absolute", store_abs_k=1, store_abs_v=1)
    args.update(kw)
    return care_kv.CacheConfig(**args)


@pytest.mark.parametrize("tables", ["shared", "batch", "sliced", "fp32", "misaligned", "none"])
@pytest.mark.parametrize("B,T,Hq,Hkv,D", [(3, 5, 8, 2, 64), (1, 1, 4, 4, 128), (2, 33, 5, 1, 64)])
def test_heads_match_elementwise(tables, B, T, Hq, Hkv, D):
    """Every form of the tables: those carekv_rope_heads reads and those that
    take the elementwise operations."""
    import care_kv
    from care_kv.layer import _rope
    print(f"rotated heads {tables} B={B} T={T} Hq={Hq} Hkv={Hkv} D={D}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    dim = Hq * D
    w = [torch.randn(o, dim, generator=g, device="cuda").half() * 0.05 for o in (dim, Hkv * D, Hkv * D, dim)]
    lay = care_kv.CAREKVLayer(_cfg(care_kv, Hq, Hkv, D), 0, *w)
    x = torch.randn(B, T, dim, generator=g, device="cuda").half()
    cos, sin = (torch.randn(B if tables == "batch" else 1, T + 9, D, generator=g, device="cuda") for _ in range(2))
    if tables != "fp32":
        cos, sin = cos.half(), sin.half()
    pe = (cos[:, 4:T + 4], sin[:, 4:T + 4]) if tables in ("sliced", "batch") else (cos[:, :T].contiguous(), sin[:, :T].contiguous())
    if tables == "misaligned":
        pe = tuple(torch.cat((t.flatten()[:1], t.flatten()))[1:].view(t.shape) for t in pe)
    Q, K, V = lay._project(x)
    if tables == "none":
        pe = None
    else:
        Q, K = _rope(Q, K, pe[0].to(F16), pe[1].to(F16))
    for got, ref in zip(lay._heads(x, pe), (Q, K, V)):
        assert got.is_contiguous() and torch.equal(got.view(torch.int16), ref.contiguous().view(torch.int16))


@pytest.mark.parametrize("T", [16, 35, 47, 1])
@pytest.mark.parametrize("base,bits,D", [("uniform", 3, 64), ("uniform", 4, 128), ("kivi_style", 2, 64)])
def test_open_rows_and_append(base, bits, D, T):
    """The open-page buffers after a prompt hold its last page's rows (zeros
    when it is full) and the rows' fp16 group scales; an append adds its row
    at its offset; other sequences' buffers stay."""
    import care_kv
    print(f"open rows {base} INT{bits} D={D} T={T}", flush=True)
    Hkv = 2
    cache = care_kv.CAREKVCache(_cfg(care_kv, 4, Hkv, D, base_bits=bits, base_quantizer=base), n_seq=3)
    g = torch.Generator(device="cuda").manual_seed(T + D)
    cache.open_k.fill_(7.0)
    cache.open_v.fill_(7.0)
    K, V = (torch.randn(2, Hkv, T, D, generator=g, device="cuda").half() for _ in range(2))
    cache.write_prefill(1, K, V, seqs=[2, 0])
    last = (T - 1) % 16 + 1
    want_k, want_v = (torch.full_like(cache.open_k, 7.0) for _ in range(2))
    for b, s in enumerate((2, 0)):
        want_k[1, s], want_v[1, s] = 0, 0
        if last < 16:
            want_k[1, s, :, :last], want_v[1, s, :, :last] = K[b, :, T - last:], V[b, :, T - last:]
    assert torch.equal(cache.open_k, want_k) and torch.equal(cache.open_v, want_v)
    if cache.rescale_open and last < 16:
        for X, op in ((K, cache.open_ks), (V, cache.open_vs)):
            _, sc = care_kv.quantize_rows(X[:, :, T - last:], bits)
            for b, s in enumerate((2, 0)):
                assert torch.equal(op[1, :, s, :last], sc[b])
    k, v = (torch.randn(2, Hkv, D, generator=g, device="cuda").half() for _ in range(2))
    cache.append(1, k, v, seqs=[2, 0])
    off = last % 16
    for b, s in enumerate((2, 0)):
        if off + 1 < 16:  # a filled page's buffers are cleared behind its store
            want_k[1, s, :, off], want_v[1, s, :, off] = k[b], v[b]
        else:
            want_k[1, s], want_v[1, s] = 0, 0
    assert torch.equal(cache.open_k, want_k) and torch.equal(cache.open_v, want_v)


def test_reset_sequence():
    import care_kv
    print("reset sequence", flush=True)
    cache = care_kv.CAREKVCache(_cfg(care_kv, 4, 2, 64), n_seq=3)
    g = torch.Generator(device="cuda").manual_seed(1)
    for layer in range(2):
        cache.write_prefill(layer, *(torch.randn(3, 2, 40, 64, generator=g, device="cuda").half() for _ in range(2)),
                            seqs=[0, 1, 2])
    names = ("valid", "has_meta", "k_slot", "v_slot", "next_slot")
    want = {n: getattr(cache, n).clone() for n in names}
    for n, fill in zip(names, (0, 0, -1, -1, 0)):
        (want[n] if n == "next_slot" else want[n].transpose(0, 2))[2] = fill
    cache.reset_sequence(-1)
    assert all(torch.equal(getattr(cache, n), want[n]) for n in names)
    assert cache.num_pages(0, 0, 2) == 0 and cache.num_pages(1, 1, 1) == 3
    with pytest.raises(IndexError):
        cache.reset_sequence(3)
