"""Which kernels the library's calls launch, what they allocate and what they do when a call of the
HIP runtime fails, on the CPU: the runtime is host_hip.c, which runs no kernel."""
import pytest

import host_hip


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    return host_hip.build(tmp_path_factory)


def test_narrow_dense_matrices_take_the_general_kernel(runtime):
    # on both sides of each part of the rule, and the matrices the shared body cannot take
    host_hip.run(runtime, """
    def general(nrows, ncols):
        m = W.GpuQuantMatrix(gpu, W.F32, nrows, ncols, np.zeros(4 * nrows * ncols, np.uint8))
        out, x = W.GpuVector.uninit(gpu, nrows), W.GpuVector.uninit(gpu, ncols)
        names = launched(lambda: W.GemvQuant(gpu).dispatch(out, m, x))
        assert len(names) == 1
        return "gemv_f32_kernel" in names[0]

    for shape in ((1, 16), (4096, 64), (50257, 128), (300001, 128), (515, 512), (8192, 512), (32768, 256),
                  (262145, 256), (17, 20), (50257, 772)):
        assert general(*shape), shape
    for shape in ((1, 528), (768, 768), (17, 4096), (8193, 272), (8193, 512), (32769, 256), (262144, 256), (262145, 272)):
        assert not general(*shape), shape

    # folded norms (fusion level 2: Q, K, V, gate, up, output): the general kernel up to 128 columns
    for dim, hidden, n_general in ((128, 352, 8), (288, 768, 1)):
        m = llama(gpu, Llama2Config(dim, hidden, 1, 4, 4, 331, 64), W.F32)
        m.set_fusion(2)
        assert count(launched(lambda: m.forward(0, 0)), "gemv_f32_kernel") == n_general, dim
    """)


def test_sampled_generation_follows_the_fusion_level(runtime):
    # level 0 is one launch per operation of the reference, in the prompt too
    host_hip.run(runtime, """
    m = llama(gpu, Llama2Config(256, 512, 2, 4, 2, 331, 64))
    prompt = np.zeros(20, np.uint32)
    for level, batched in ((0, False), (1, True), (2, True), (3, True)):
        m.set_fusion(level)
        one = launched(lambda: m.forward(0, 0))
        names = launched(lambda: m.generate_sampled(prompt, 23, 0.7, 0.9, 1))
        assert (count(names, "gemm_lds_kernel") > 0) == batched, level
        assert batched or names == one * 23
    """)


def test_sampled_generation_refuses_a_temperature_before_it_starts(runtime):
    # (refused by the first sample, it left a copy of logits under way to memory that the call frees
    # where there is no pinned memory)
    host_hip.run(runtime, """
    m = llama(gpu, Llama2Config(256, 512, 2, 4, 2, 331, 64))
    for n_prompt, temperature in ((1, -1.0), (3, -1.0), (20, -0.5), (3, float("nan"))):
        def call():
            try:
                m.generate_sampled(np.zeros(n_prompt, np.uint32), 23, temperature, 0.9, 1)
            except W.WgmlError as e:
                assert e.code == _lib.E_INVALID and "temperature" in str(e)
            else:
                assert False
        assert launched(call) == []
    m.generate_sampled(np.zeros(3, np.uint32), 0, -1.0, 0.9, 1)  # nothing to do: accepted as before
    """)


def test_rows_whose_long_runs_the_products_cannot_address_go_in_short_ones(runtime):
    # 2^20 columns: the low halves of 1024 packed tokens would lie 2^31 bytes behind the high ones
    host_hip.run(runtime, """
    m = llama(gpu, Llama2Config(256, 1 << 20, 1, 4, 4, 331, 400))
    names = launched(lambda: m.prefill(np.zeros(300, np.uint32)))
    assert count(names, "gemm_tile") == 0 and count(names, "gemm_lds") > 0
    m = llama(gpu, Llama2Config(256, 1 << 19, 1, 4, 4, 331, 400))
    assert count(launched(lambda: m.prefill(np.zeros(300, np.uint32))), "gemm_tile") > 0
    """)


def test_partial_sums_take_a_launch_only_where_it_pays(runtime):
    # nothing adds a product's partial sums on its way: two parts of 512 columns were slower than one for a few vectors
    host_hip.run(runtime, """
    def reductions(nrows, ncols, n, qtype=W.Q8_0):
        m = W.GpuQuantMatrix(gpu, qtype, nrows, ncols, np.zeros(W.quant_bytes(qtype, nrows * ncols), np.uint8))
        out, x = W.GpuVector.uninit(gpu, n * nrows), W.GpuVector.uninit(gpu, n * ncols)
        names = launched(lambda: W.GemmQuant.from_device(gpu).dispatch(out, m, x, n))
        assert count(names, "gemm_lds_kernel") == 1 and len(names) == 2 + count(names, "gemm_reduce_kernel")
        return count(names, "gemm_reduce_kernel")

    for shape in ((64, 256, 128), (64, 288, 1), (64, 512, 16), (4096, 512, 16), (1024, 768, 1), (32000, 1024, 48)):
        assert reductions(*shape) == 0, shape
    for shape in ((64, 512, 128), (64, 1024, 128), (64, 4096, 1), (4096, 4096, 1), (256, 16384, 16)):
        assert reductions(*shape) == 1, shape
    assert reductions(1024, 768, 1, W.Q4_0) == 1  # a unit takes longer there
    """)


def test_matrices_that_the_products_address(runtime):
    # rows of a tile at 32-bit offsets from its first one: below 2^32 weights as before, also where they take more bytes
    # (Q8_K, 292 per 256), unless one tile alone does
    host_hip.run(runtime, """
    def product(nrows, ncols):
        m = W.GpuQuantMatrix(gpu, W.Q8_K, nrows, ncols, np.zeros(W.quant_bytes(W.Q8_K, nrows * ncols), np.uint8))
        out, x = W.GpuVector.uninit(gpu, nrows), W.GpuVector.uninit(gpu, ncols)
        try:
            return count(launched(lambda: W.GemmQuant.from_device(gpu).dispatch(out, m, x, 1)), "gemm_lds_kernel")
        except W.WgmlError as e:
            assert e.code == _lib.E_UNSUPPORTED
            return 0

    assert product(58000, 1 << 16) == 1
    assert product(112, 1 << 22) == 1 and product(1000, 1 << 21) == 1
    assert product(1 << 16, 1 << 16) == 0
    gpu.set_gemm_precision(0)
    assert product(112, 1 << 25) == 1 and product(114, 1 << 25) == 0
    """)


def test_only_missing_memory_sends_a_prompt_down_the_slower_path(runtime):
    # runs of 1024 tokens, then of 128, then (where a loop has them) steps; any other failure of the
    # faster path is the caller's to see
    host_hip.run(runtime, """
    def failure(call):
        try:
            call()
        except W.WgmlError as e:
            return e.code
    prompt, long_prompt = np.zeros(20, np.uint32), np.zeros(300, np.uint32)
    cfg = Llama2Config(256, 512, 2, 4, 2, 331, 400)
    p = Gpt2Params(n_vocab=331, n_seq=64, n_embd=128, n_head=4, n_layer=2, ff_len=512, attn_b=384)
    sampled = lambda m: m.generate_sampled(prompt, 23, 0.7, 0.9, 1)

    # no memory for the larger workspaces, or for any
    m = llama(gpu, cfg)
    fake.host_hip_malloc_limit(1 << 20)
    names = launched(lambda: m.prefill(long_prompt))
    assert count(names, "gemm_tile") == 0 and count(names, "gemm_lds") > 0
    fake.host_hip_malloc_limit(NO_LIMIT)
    assert count(launched(lambda: m.prefill(long_prompt)), "gemm_tile") > 0
    m, g = llama(gpu, cfg), gpt2(gpu, p)
    one = launched(lambda: m.forward(0, 0))
    g.record_steps(23)
    fake.host_hip_malloc_limit(1 << 10)
    assert launched(lambda: sampled(m)) == one * 23
    assert count(launched(lambda: g.generate_greedy(prompt, 23)), "gemm_") == 0
    fake.host_hip_malloc_limit(NO_LIMIT)
    assert count(launched(lambda: sampled(m)), "gemm_lds") > 0
    assert count(launched(lambda: g.generate_greedy(prompt, 23)), "gemm_lds") > 0

    # no memory for the partial sums of a product, in the middle of a run
    wide = llama(W.GpuInstance(0), Llama2Config(1024, 2816, 2, 8, 8, 331, 400))
    one = launched(lambda: wide.forward(0, 0))
    fake.host_hip_malloc_limit(6 << 20)
    names = launched(lambda: sampled(wide))
    assert count(names, "prep_x") == 1 and names[-23 * len(one):] == one * 23
    assert failure(lambda: wide.prefill(long_prompt)) == _lib.E_OOM
    fake.host_hip_malloc_limit(NO_LIMIT)

    # a launch that fails
    fake.host_hip_fail_kernel(b"gemm_tile_kernel")
    assert failure(lambda: m.prefill(long_prompt)) == _lib.E_HIP
    fake.host_hip_fail_kernel(b"gemm_lds_kernel")
    assert failure(lambda: sampled(m)) == _lib.E_HIP
    assert failure(lambda: g.generate_greedy(prompt, 23)) == _lib.E_HIP
    """)


def test_partial_sums_of_growing_prompts_keep_little_memory(runtime):
    # buffers that were outgrown stay with the context; a buffer holds at most 136 MiB here
    host_hip.run(runtime, """
    def kept(lengths):
        m = llama(W.GpuInstance(0), Llama2Config(4096, 11008, 1, 32, 32, 331, 1100))
        before = fake.host_hip_allocated()
        for n in lengths:
            m.prefill(np.zeros(n, np.uint32))
        return fake.host_hip_allocated() - before

    assert kept(range(1, 1025, 3)) - kept((1, 1024)) <= 2 * 136 << 20
    assert kept(range(1, 129)) - kept((1,)) <= 2 * 136 << 20
    """)


def test_longer_prompts_pin_no_new_memory(runtime):
    host_hip.run(runtime, """
    m = llama(gpu, Llama2Config(256, 512, 2, 4, 2, 331, 400))
    before = fake.host_hip_pinned()
    for n in (1, 6, 7, 12, 40, 128, 129, 5):
        assert m.generate_sampled(np.zeros(n, np.uint32), n + 9, 0.7, 0.9, 1).size == n + 9
    assert fake.host_hip_pinned() == before + 1
    """)


def test_short_contexts_share_the_compute_units_out(runtime):
    # two slices per head while all have a compute unit (256), then one workgroup per head, or per two that share rows
    host_hip.run(runtime, """
    def attention(n_heads, kv_mul, hs):
        kv_dim = n_heads // kv_mul * hs
        q, out = W.GpuVector.uninit(gpu, n_heads * hs), W.GpuVector.uninit(gpu, n_heads * hs)
        k, v = (W.GpuMatrix.init(gpu, np.zeros((256, kv_dim), np.float32)) for _ in range(2))
        p = W.BatchedMultiqueryAttentionParams(256, kv_dim, kv_mul, n_heads, hs, 40)
        run = lambda: W.BatchedMultiqueryAttention.from_device(gpu).dispatch_multi(p, q, k, v, out)
        assert count(launched(run), "attn_fast_kernel") == 1
        return workgroups(run)[0]

    for n_heads, kv_mul, hs, want in ((32, 1, 128, 64), (128, 8, 128, 256), (129, 3, 128, 129), (130, 1, 68, 130), (132, 4, 68, 66),
                                      (160, 8, 128, 80), (129, 3, 68, 129), (192, 6, 96, 96), (192, 3, 128, 192), (256, 8, 128, 128), (12, 1, 64, 12),
                                      (252, 4, 64, 252), (256, 4, 64, 128), (255, 5, 64, 255), (300, 1, 64, 300)):
        assert attention(n_heads, kv_mul, hs) == want, (n_heads, kv_mul, hs)
    """)


def test_short_runs_pack_their_tokens_in_order(runtime):
    # (nothing of the longer runs' order in their kernel)
    host_hip.run(runtime, """
    def packing(qtype, n):
        m = W.GpuQuantMatrix(gpu, qtype, 64, 256, np.zeros(W.quant_bytes(qtype, 64 * 256), np.uint8))
        out, x = W.GpuVector.uninit(gpu, n * 64), W.GpuVector.uninit(gpu, n * 256)
        run = lambda: W.GemmQuant.from_device(gpu).dispatch(out, m, x, n)
        return "prep_x_kernelILi0ELb1E" in launched(run)[0], workgroups(run)[0]

    for n in (1, 17, 63, 64):
        assert packing(W.Q8_0, n) == packing(W.Q4_K, n) == (True, n)
    for n in (65, 100, 128):
        assert packing(W.Q8_0, n) == packing(W.Q4_K, n) == (False, 128)
    """)


def test_f16_beside_f32_takes_no_more_launches(runtime):
    # a layer that mixes them in Q/K/V or gate/up, at widths where F16 stays 16 bits wide
    host_hip.run(runtime, """
    cfg = Llama2Config(768, 2048, 2, 12, 12, 331, 64)
    def launches(f16):
        m = llama(gpu, cfg, W.F32)
        for l in range(cfg.n_layers):
            for name, (r, k) in {"attn_q": (768, 768), "attn_k": (768, 768), "ffn_gate": (2048, 768), "ffn_up": (2048, 768)}.items():
                if name in f16:
                    m.set_matrix(name, l, HostMatrix(W.F16, r, k, np.zeros(2 * r * k, np.uint8)))
        return launched(lambda: m.forward(0, 0))

    plain = launches(())
    for f16 in (("attn_q",), ("ffn_up",), ("attn_k", "ffn_gate"), ("attn_q", "attn_k", "ffn_gate", "ffn_up")):
        assert len(launches(f16)) == len(plain), f16
    """)


def test_bytes_of_f16_matrices(runtime):
    # what a product streams; the rule that shares fused launches out goes by it (64 MB: one workgroup per compute unit)
    host_hip.run(runtime, """
    for qtype, cols, per in ((W.F16, 768, 2), (W.F16, 32768, 2), (W.F16, 512, 4), (W.F16, 772, 4), (W.F16, 32784, 4), (W.F32, 768, 4)):
        m = W.GpuQuantMatrix(gpu, qtype, 5, cols, np.zeros((2 if qtype == W.F16 else 4) * 5 * cols, np.uint8))
        assert m.gguf_bytes() == per * 5 * cols and m.shape() == (W.F32, 5, cols), (qtype, cols)
    """)


def test_workgroups_of_products_with_fp32_activations(runtime):
    host_hip.run(runtime, """
    fake.host_hip_blocks_per_cu(2)
    def grid(qtype, nrows, ncols):
        m = W.GpuQuantMatrix(gpu, qtype, nrows, ncols, np.zeros(4 * nrows * ncols if qtype == W.F32 else W.quant_bytes(qtype, nrows * ncols), np.uint8))
        out, x = W.GpuVector.uninit(gpu, nrows), W.GpuVector.uninit(gpu, ncols)
        return workgroups(lambda: W.GemvQuant(gpu).dispatch(out, m, x))

    for shape in ((6000, 1024), (10239, 1024), (20000, 528), (20000, 1040), (6000, 2048)):
        assert grid(W.F32, *shape)[0] <= 256, shape
    for shape in ((10240, 1024), (20000, 896), (12000, 1808), (12000, 2048)):
        assert grid(W.F32, *shape)[0] > 256, shape
    gpu.set_tuning(gpu.TUNE_GEMV_F32_ACTIVATIONS, 1)
    for shape in ((6144, 1024), (5000, 4096), (10239, 256), (20000, 4096)):
        assert grid(W.Q6_K, *shape)[0] <= 256, shape
    for shape in ((10240, 256), (20000, 2048)):
        assert grid(W.Q6_K, *shape)[0] > 256, shape
    """)


def test_workgroups_of_large_q5_1_matrices(runtime):
    host_hip.run(runtime, """
    fake.host_hip_blocks_per_cu(2)
    def grid(qtype, nrows, ncols):
        m = W.GpuQuantMatrix(gpu, qtype, nrows, ncols, np.zeros(W.quant_bytes(qtype, nrows * ncols), np.uint8))
        out, x = W.GpuVector.uninit(gpu, nrows), W.GpuVector.uninit(gpu, ncols)
        return workgroups(lambda: W.GemvQuant(gpu).dispatch(out, m, x))[0]

    for ncols, limit in ((8192, 43690), (2048, 174762), (3072, 116508)):  # rows of 256 MB
        assert grid(W.Q5_1, limit, ncols) > 256 and grid(W.Q5_1, limit + 1, ncols) == 256, ncols
    assert grid(W.Q5_1, 200000, 2112) > 256 and grid(W.Q5_0, 45000, 8192) > 256  # lanes without a tile; another format
    """, timeout=300)


def test_launch_shapes_do_not_bound_the_folded_layernorm(runtime):
    # its kernels have workgroups of 1024 threads whatever the overrides say (they refused rows of more than 12 columns per thread
    # of a smaller workgroup that never ran)
    host_hip.run(runtime, """
    n = 6400
    p = Gpt2Params(n_vocab=64, n_seq=8, n_embd=n, n_head=50, n_layer=1, ff_len=64, attn_b=3 * n)
    w = Gpt2HostWeights(params=p)
    w.layers.append({"attn_w": zeros(W.Q8_0, 3 * n, n), "attn_proj_w": zeros(W.Q8_0, n, n), "mlp_fc_w": zeros(W.Q8_0, 64, n),
                     "mlp_proj_w": zeros(W.Q8_0, n, 64)} | {k: np.zeros(c, np.float32) for k, c in
                    dict(attn_b=3 * n, attn_proj_b=n, mlp_fc_b=64, mlp_proj_b=n, ln_1_g=n, ln_1_b=n, ln_2_g=n, ln_2_b=n).items()})
    w.wte, w.wpe, w.lm_head = np.zeros((64, n), np.float32), np.zeros((8, n), np.float32), zeros(W.Q8_0, 64, n)
    w.ln_f_g = w.ln_f_b = np.zeros(n, np.float32)
    m = Gpt2(gpu, p).load(w)
    plain = launched(lambda: m.forward(0, 0))
    for waves in (4, 8, 16, 12):
        gpu.set_tuning(gpu.TUNE_GEMV_WAVES_PER_WG, waves)
        names = launched(lambda: m.forward(0, 0))
        assert len(names) == len(plain) and names[-1] == plain[-1], waves
    """)


def test_maxima_of_more_waves_than_there_is_room_for(runtime):
    # a wave parks 64 results: 1048576 rows are 16384 waves
    host_hip.run(runtime, """
    def arg_max(vocab):
        names = launched(lambda: llama(gpu, Llama2Config(64, 64, 1, 1, 1, vocab, 16)).decode_greedy(1, 0, 1))
        return [n for n in names if "next_embed" in n][0]

    assert "maxima_next_embed" in arg_max(331) and "maxima_next_embed" in arg_max(1048576)
    assert "argmax_next_embed" in arg_max(1048578)
    """)
