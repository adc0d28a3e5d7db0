"""GPU parity of MUL_MAT_ID (MoE expert routing) against the oracle and the reference CPU backend."""
import numpy as np
import pytest

import orc

pytestmark = pytest.mark.gpu


def routed(t, n_used, T, K):
    """mi355_mul_mat_id sorts the slots by expert and uses the K-quant tile kernel (ggml-cpu's Q8_K arithmetic)"""
    return T * n_used >= 32 and ((t in (orc.Q4_K, orc.Q5_K) and K % 256 == 0) or (t == orc.Q6_K and K % 2048 == 0) or (t == orc.IQ4_XS and K % 512 == 0))


def expected_per_expert(kind, t, Wq, b, ids_full, n_expert, n_used, nb1, N):
    """every expert's product over the rows routed to it (ggml.c:2723-2759), one mul_mat per expert"""
    T = b.shape[0]
    want = np.zeros((T, n_used, N), dtype=np.float32)
    for ex in range(n_expert):
        where = [(tt, e) for tt in range(T) for e in range(n_used) if ids_full[tt, e] == ex]
        if not where:
            continue
        rows = np.stack([b[tt, e % nb1] for tt, e in where])
        out = orc.mul_mat(kind, t, Wq[ex * N:(ex + 1) * N], rows)
        for (tt, e), o in zip(where, out):
            want[tt, e] = o
    return want


@pytest.mark.parametrize("name,t", list(orc.WEIGHT_TYPES.items()))
@pytest.mark.parametrize("n_expert,n_used,nb1_bcast,T,N,K", [(8, 2, True, 1, 512, 4096), (8, 2, False, 5, 256, 2048),
                                                              (4, 4, True, 32, 128, 2048), (8, 1, False, 3, 64, 4096),
                                                              (8, 2, True, 512, 192, 2048), (8, 2, False, 300, 64, 4096)])
def test_mul_mat_id(dev, name, t, n_expert, n_used, nb1_bcast, T, N, K):
    import torch
    import mi355
    rng = np.random.default_rng(n_expert + T + N)
    nb1 = 1 if nb1_bcast else n_used
    Wf = (rng.standard_normal((n_expert * N, K)) * 0.02).astype(np.float32)
    Wq = orc.quantize("ref" if orc.ref is not None else "oracle", t, Wf)
    b = rng.standard_normal((T, nb1, K)).astype(np.float32)
    ids_full = np.stack([rng.permutation(n_expert) for _ in range(T)]).astype(np.int32)
    Wd = mi355.upload_weights(t, torch.from_numpy(Wq).to(dev)).reshape(n_expert, N, -1)
    idd = torch.from_numpy(ids_full).to(dev)[:, :n_used]          # strided view, as ggml_view of the argsort result
    got = mi355.mul_mat_id(t, Wd, torch.from_numpy(b).to(dev), idd, n_used).cpu().numpy()
    if routed(t, n_used, T, K):
        want = expected_per_expert("cpu", t, Wq, b, ids_full, n_expert, n_used, nb1, N)
    else:
        want = np.zeros((T, n_used, N), dtype=np.float32)
        assert orc.oracle.orc_mul_mat_id_q8_1(t, orc._ptr(Wq), orc._ptr(b), orc._ptr(ids_full), n_expert, orc._ptr(want), N, K,
                                              n_expert, n_used, nb1, T) == 0
    assert orc.nmse(got, want) < 1e-11      # exact block dots, f32 sums over at most 128 blocks (an f16 block minimum would leave 1e-7)
    if orc.ref is not None:
        cpu = np.zeros_like(want)
        assert orc.ref.ref_mul_mat_id(t, orc._ptr(Wq), orc._ptr(b), orc._ptr(ids_full), orc._ptr(cpu), N, K, n_expert, n_used,
                                      nb1, T, 4, 0) >= 0
        assert orc.nmse(got, cpu) <= 5e-4      # tests/test-backend-ops.cpp:2001


@pytest.mark.parametrize("name,t", [("q4_k", orc.Q4_K), ("q6_k", orc.Q6_K), ("q5_k", orc.Q5_K), ("iq4_xs", orc.IQ4_XS), ("q4_0", orc.Q4_0), ("q8_0", orc.Q8_0),
                                    ("q5_1", orc.Q5_1)])
@pytest.mark.parametrize("pattern", ["one_expert", "two_of_eight", "out_of_range"])
def test_mul_mat_id_skewed_routing(dev, name, t, pattern):
    """experts with no slots, one expert with more slots than a column tile, ids outside [0, n_expert) clamped like the GEMV path"""
    import torch
    import mi355
    n_expert, n_used, T, N, K = 8, 2, 200, 128, 2048
    rng = np.random.default_rng(5)
    Wf = (rng.standard_normal((n_expert * N, K)) * 0.02).astype(np.float32)
    Wq = orc.quantize("ref" if orc.ref is not None else "oracle", t, Wf)
    b = rng.standard_normal((T, 1, K)).astype(np.float32)
    if pattern == "one_expert":
        ids = np.full((T, n_expert), 3, dtype=np.int32)
    elif pattern == "two_of_eight":
        ids = np.tile(np.array([[6, 1, 0, 0, 0, 0, 0, 0]], dtype=np.int32), (T, 1))
    else:
        ids = rng.integers(-2, n_expert + 2, size=(T, n_expert)).astype(np.int32)
    Wd = mi355.upload_weights(t, torch.from_numpy(Wq).to(dev)).reshape(n_expert, N, -1)
    idd = torch.from_numpy(ids).to(dev)[:, :n_used]
    got = mi355.mul_mat_id(t, Wd, torch.from_numpy(b).to(dev), idd, n_used).cpu().numpy()
    kind = "cpu" if t in (orc.Q4_K, orc.Q6_K, orc.Q5_K, orc.IQ4_XS) else "q8_1"   # the activation format of the type's routed tile kernel
    want = expected_per_expert(kind, t, Wq, b, np.clip(ids, 0, n_expert - 1), n_expert, n_used, 1, N)
    assert orc.nmse(got, want) < 1e-11


@pytest.mark.parametrize("name,t", list(orc.WEIGHT_TYPES.items()))
@pytest.mark.parametrize("K", [1280, 2048])
def test_mul_mat_id_last_column_tiles(dev, name, t, K):
    """experts whose second 128-column tile holds 1, 64 and 65 slots (up to 64 it runs with half the columns per wave)"""
    import torch
    import mi355
    counts, N = (129, 192, 193, 64), 70
    T = sum(counts)
    rng = np.random.default_rng(K)
    Wq = orc.quantize("oracle", t, (rng.standard_normal((len(counts) * N, K)) * 0.02).astype(np.float32))
    b = rng.standard_normal((T, 1, K)).astype(np.float32)
    ids = rng.permutation(np.repeat(np.arange(len(counts)), counts)).astype(np.int32).reshape(T, 1)
    Wd = mi355.upload_weights(t, torch.from_numpy(Wq).to(dev)).reshape(len(counts), N, -1)
    got = mi355.mul_mat_id(t, Wd, torch.from_numpy(b).to(dev), torch.from_numpy(ids).to(dev), 1).cpu().numpy()
    want = expected_per_expert("cpu" if routed(t, 1, T, K) else "q8_1", t, Wq, b, ids, len(counts), 1, 1, N)
    assert orc.nmse(got, want) < 1e-11   # exact integer sums, f32 sums over at most 64 blocks


@pytest.mark.parametrize("name,t", [("q4_k", orc.Q4_K), ("q5_k", orc.Q5_K), ("q6_k", orc.Q6_K)])
@pytest.mark.parametrize("n_expert,n_used,nb1_bcast,T,N,K", [(8, 2, True, 512, 192, 2048), (8, 2, False, 300, 64, 4096), (4, 4, True, 70, 256, 2048),
                                                              (8, 1, False, 3, 130, 2048)])   # Q6_K rows are 16-byte aligned from K = 2048 on
def test_mul_mat_id_on_tile_images(dev, name, t, n_expert, n_used, nb1_bcast, T, N, K):
    """the routed form of the wide-tile kernel: slots sorted by expert, activations gathered into one tile image, rows
    scattered to their slots; against ggml-cpu's arithmetic per expert (Q8_K activations) and the reference's MUL_MAT_ID"""
    import torch
    import mi355
    rng = np.random.default_rng(n_expert + T + N + K)
    nb1 = 1 if nb1_bcast else n_used
    Wf = (rng.standard_normal((n_expert * N, K)) * 0.02).astype(np.float32)
    Wq = orc.quantize("ref" if orc.ref is not None else "oracle", t, Wf)
    b = rng.standard_normal((T, nb1, K)).astype(np.float32)
    ids_full = np.stack([rng.permutation(n_expert) for _ in range(T)]).astype(np.int32)
    Wd = mi355.upload_weights(t, torch.from_numpy(Wq).to(dev)).reshape(n_expert, N, -1)
    tiles = mi355.kq_unpack_expert_tiles(t, Wd)
    idd = torch.from_numpy(ids_full).to(dev)[:, :n_used]
    got = mi355.mul_mat_id_tiled(t, tiles, N, torch.from_numpy(b).to(dev), idd, n_used).cpu().numpy()
    want = expected_per_expert("cpu", t, Wq, b, ids_full, n_expert, n_used, nb1, N)
    assert orc.nmse(got, want) < 1e-9
    if orc.ref is not None:
        cpu = np.zeros_like(want)
        assert orc.ref.ref_mul_mat_id(t, orc._ptr(Wq), orc._ptr(b), orc._ptr(ids_full), orc._ptr(cpu), N, K, n_expert, n_used,
                                      nb1, T, 4, 0) >= 0
        assert orc.nmse(got, cpu) <= 5e-4      # tests/test-backend-ops.cpp:2001


@pytest.mark.parametrize("pattern", ["one_expert", "two_of_eight", "out_of_range"])
def test_mul_mat_id_on_tile_images_skewed_routing(dev, pattern):
    """experts without slots, one expert with more slots than a column tile, ids outside [0, n_expert) clamped"""
    import torch
    import mi355
    t = orc.Q4_K
    n_expert, n_used, T, N, K = 8, 2, 200, 128, 2048
    rng = np.random.default_rng(6)
    Wf = (rng.standard_normal((n_expert * N, K)) * 0.02).astype(np.float32)
    Wq = orc.quantize("ref" if orc.ref is not None else "oracle", t, Wf)
    b = rng.standard_normal((T, 1, K)).astype(np.float32)
    if pattern == "one_expert":
        ids = np.full((T, n_expert), 3, dtype=np.int32)
    elif pattern == "two_of_eight":
        ids = np.tile(np.array([[6, 1, 0, 0, 0, 0, 0, 0]], dtype=np.int32), (T, 1))
    else:
        ids = rng.integers(-2, n_expert + 2, size=(T, n_expert)).astype(np.int32)
    Wd = mi355.upload_weights(t, torch.from_numpy(Wq).to(dev)).reshape(n_expert, N, -1)
    tiles = mi355.kq_unpack_expert_tiles(t, Wd)
    idd = torch.from_numpy(ids).to(dev)[:, :n_used]
    got = mi355.mul_mat_id_tiled(t, tiles, N, torch.from_numpy(b).to(dev), idd, n_used).cpu().numpy()
    want = expected_per_expert("cpu", t, Wq, b, np.clip(ids, 0, n_expert - 1), n_expert, n_used, 1, N)
    assert orc.nmse(got, want) < 1e-9


@pytest.mark.parametrize("name,t,blocks", [("q6_k", orc.Q6_K, 3), ("iq4_xs", orc.IQ4_XS, 5), ("q4_0", orc.Q4_0, 3), ("q8_0", orc.Q8_0, 9), ("q5_1", orc.Q5_1, 7)])
@pytest.mark.parametrize("T", [3, 16, 60, 130])
def test_mul_mat_id_ragged_rows(dev, name, t, blocks, T):
    """expert rows that start at any even address, K no whole number of the tile kernel's stages: per-slot GEMV and routed tiles"""
    import torch
    import mi355
    n_expert, n_used, N, K = 5, 2, 70, orc.BLOCK[t][0] * blocks
    rng = np.random.default_rng(T)
    Wq = orc.quantize("oracle", t, (rng.standard_normal((n_expert * N, K)) * 0.02).astype(np.float32))
    b = rng.standard_normal((T, 1, K)).astype(np.float32)
    ids = np.stack([rng.permutation(n_expert) for _ in range(T)]).astype(np.int32)
    Wd = mi355.upload_weights(t, torch.from_numpy(Wq).to(dev)).reshape(n_expert, N, -1)
    got = mi355.mul_mat_id(t, Wd, torch.from_numpy(b).to(dev), torch.from_numpy(ids).to(dev)[:, :n_used], n_used).cpu().numpy()
    assert orc.nmse(got, expected_per_expert("q8_1", t, Wq, b, ids, n_expert, n_used, 1, N)) < 1e-11


@pytest.mark.parametrize("name,t", list(orc.WEIGHT_TYPES.items()))
@pytest.mark.parametrize("n_expert,n_used,bcast,T,pattern", [(8, 2, True, 7, "spread"), (4, 3, False, 33, "spread"), (6, 2, True, 150, "spread"), (8, 2, True, 90, "one_expert"),
                                                             (3, 2, True, 20, "out_of_range")])
def test_mul_mat_id_skinny(dev, name, t, n_expert, n_used, bcast, T, pattern):
    """the weight-streaming kernel over experts: none, one and several passes over an expert's columns, a ragged last row tile, ids outside
    [0, n_expert) clamped; against exact integer block dots (f32 sums: NMSE of some 1e-14)"""
    import torch
    import mi355
    lib = mi355.load()
    N, K = 70, 1024
    nb1 = 1 if bcast else n_used
    rng = np.random.default_rng(T)
    Wq = orc.quantize("oracle", t, (rng.standard_normal((n_expert * N, K)) * 0.02).astype(np.float32))
    b = rng.standard_normal((T, nb1, K)).astype(np.float32)
    ids = np.stack([rng.permutation(max(n_expert, n_used))[:n_used] for _ in range(T)]).astype(np.int32)
    if pattern == "one_expert":
        ids[:] = 5
    elif pattern == "out_of_range":
        ids = rng.integers(-2, n_expert + 2, size=ids.shape).astype(np.int32)
    Wd = mi355.upload_weights(t, torch.from_numpy(Wq).to(dev))
    act = mi355.quantize_act(torch.from_numpy(b.reshape(T * nb1, K)).to(dev))
    idd = torch.from_numpy(ids).to(dev)
    got = torch.full((T, n_used, N), float("nan"), device=dev)
    mi355.check(lib.mi355_mul_mat_id_skinny(None, t, Wd.data_ptr(), act.data_ptr(), idd.data_ptr(), idd.stride(0), got.data_ptr(), N, K, n_expert, n_used, nb1, T))
    torch.cuda.synchronize()
    want = expected_per_expert("q8_1", t, Wq, b, np.clip(ids, 0, n_expert - 1), n_expert, n_used, nb1, N)
    assert orc.nmse(got.cpu().numpy(), want) < 1e-11
    if t in (orc.Q4_K, orc.Q5_K, orc.Q6_K, orc.IQ4_XS):   # the form on Q8_K activations: the CPU path's integer sums
        act = mi355.quantize_act_q8k(torch.from_numpy(b.reshape(T * nb1, K)).to(dev))
        got.fill_(float("nan"))
        mi355.check(lib.mi355_mul_mat_id_skinny_q8k(None, t, Wd.data_ptr(), act.data_ptr(), idd.data_ptr(), idd.stride(0), got.data_ptr(), N, K, n_expert, n_used, nb1, T))
        torch.cuda.synchronize()
        want = expected_per_expert("cpu", t, Wq, b, np.clip(ids, 0, n_expert - 1), n_expert, n_used, nb1, N)
        assert orc.nmse(got.cpu().numpy(), want) < 1e-11


@pytest.mark.parametrize("name,t", [("q4_0", orc.Q4_0), ("q4_k", orc.Q4_K), ("q5_k", orc.Q5_K), ("q6_k", orc.Q6_K), ("iq4_xs", orc.IQ4_XS)])
@pytest.mark.parametrize("n_expert,n_used,T,N", [(16, 2, 128, 2048), (16, 2, 65, 2080), (256, 4, 66, 128), (256, 4, 66, 129), (5, 3, 300, 33), (5, 3, 64, 33)])
def test_mul_mat_id_skinny_same_experts_for_all_tokens(dev, name, t, n_expert, n_used, T, N):
    """every token chooses the same experts, and spread-out routing, where one or two groups share an expert's passes (32-row tiles times
    experts on both sides of 1024, tokens on both sides of 64): every slot exactly once; exact integer dots, f32 sums over 32 blocks"""
    import torch
    import mi355
    lib = mi355.load()
    K = 1024
    rng = np.random.default_rng(N + T)
    Wq = orc.quantize("oracle", t, (rng.standard_normal((64, K)) * 0.02).astype(np.float32))
    pick = rng.integers(0, 64, n_expert * N)          # the experts' rows are drawn from 64
    Wd = mi355.upload_weights(t, torch.from_numpy(Wq[pick]).to(dev))
    x = rng.standard_normal((T, K)).astype(np.float32)
    same = np.tile(rng.permutation(n_expert)[:n_used].astype(np.int32), (T, 1))
    spread = np.stack([rng.permutation(n_expert)[:n_used] for _ in range(T)]).astype(np.int32)
    forms = [("q8_1", mi355.quantize_act, lib.mi355_mul_mat_id_skinny)]
    if t != orc.Q4_0:
        forms.append(("cpu", mi355.quantize_act_q8k, lib.mi355_mul_mat_id_skinny_q8k))
    for kind, quantize, product in forms:
        act = quantize(torch.from_numpy(x).to(dev))
        rows = orc.mul_mat(kind, t, Wq, x)
        for ids in (same, spread):
            idd = torch.from_numpy(ids).to(dev)
            got = torch.full((T, n_used, N), float("nan"), device=dev)
            mi355.check(product(None, t, Wd.data_ptr(), act.data_ptr(), idd.data_ptr(), n_used, got.data_ptr(), N, K, n_expert, n_used, 1, T))
            torch.cuda.synchronize()
            want = rows[np.arange(T)[:, None, None], pick.reshape(n_expert, N)[ids]]
            assert orc.nmse(got.cpu().numpy(), want) < 1e-11


def test_routed_tiles_over_more_than_2_32_activation_blocks(dev):
    """the last of 2^24 - 1 tokens lie beyond 2^32 blocks: zeros but for the first and last 64, whose levels are all 1"""
    import torch
    import mi355
    lib = mi355.load()
    t, K, T, N, E = orc.Q8_0, 8320, (1 << 24) - 1, 1, 2
    if torch.cuda.mem_get_info()[0] < 200 << 30:
        pytest.skip("needs 174 GB of activations")
    W = torch.ones((E, K), device=dev) * torch.tensor([[127.0], [254.0]], device=dev)         # levels 127, scales 1 and 2
    Wd = mi355.upload_weights(t, mi355.quantize_weights(t, W))
    act = torch.zeros(int(lib.mi355_act_bytes(K, T)), dtype=torch.uint8, device=dev)
    ends = torch.cat([torch.arange(64), torch.arange(T - 64, T)]).to(dev)
    act[:T * K].view(T, K)[ends] = 1
    ds = act[T * K:T * K + T * (K // 32) * 8].view(torch.int32).view(T, K // 32, 2)
    ds[ends, :, 0] = 0x3F800000                                                                 # scale 1.0f
    ds[ends, :, 1] = 32
    ids = torch.arange(T, dtype=torch.int32, device=dev) % E
    got = torch.full((T,), float("nan"), device=dev)
    route = torch.empty(int(lib.mi355_mul_mat_id_q8k_route_bytes(E, 1, T)), dtype=torch.uint8, device=dev)
    mi355.check(lib.mi355_mul_mat_id_q(None, t, Wd.data_ptr(), act.data_ptr(), ids.data_ptr(), 1, got.data_ptr(), N, K, E, 1, 1, T, route.data_ptr(), route.numel()))
    torch.cuda.synchronize()
    want = torch.zeros(T, device=dev)
    want[ends] = 127.0 * K * (1 + ids[ends].float())
    assert torch.equal(got, want)                                                               # whole numbers below 2^24
    del act, ds
    torch.cuda.empty_cache()


@pytest.mark.parametrize("name,t", [(n, t) for n, t in orc.WEIGHT_TYPES.items() if t not in (orc.Q4_K, orc.Q5_K)])
@pytest.mark.parametrize("n_expert,n_used,T,N", [(4, 1, 32, 130), (4, 4, 32, 64), (8, 2, 128, 70), (16, 2, 128, 33), (16, 3, 65, 129)])
def test_routed_tiles_with_few_slots_per_expert(dev, name, t, n_expert, n_used, T, N):
    """mi355_mul_mat_id_q called directly where mi355_mul_mat_id prefers the weight-streaming kernel; and the stack at an odd address, where
    mi355_mul_mat_id falls back to byte loads"""
    import torch
    import mi355
    lib = mi355.load()
    K = 1280
    rng = np.random.default_rng(T + N)
    Wq = orc.quantize("oracle", t, (rng.standard_normal((n_expert * N, K)) * 0.02).astype(np.float32))
    b = rng.standard_normal((T, 1, K)).astype(np.float32)
    ids = np.stack([rng.permutation(n_expert)[:n_used] for _ in range(T)]).astype(np.int32)
    Wd = mi355.upload_weights(t, torch.from_numpy(Wq).to(dev))
    act, idd = mi355.quantize_act(torch.from_numpy(b[:, 0]).to(dev)), torch.from_numpy(ids).to(dev)
    got = torch.full((T, n_used, N), float("nan"), device=dev)
    route = torch.empty(int(lib.mi355_mul_mat_id_q8k_route_bytes(n_expert, n_used, T)), dtype=torch.uint8, device=dev)
    mi355.check(lib.mi355_mul_mat_id_q(None, t, Wd.data_ptr(), act.data_ptr(), idd.data_ptr(), n_used, got.data_ptr(), N, K, n_expert, n_used, 1, T,
                                       route.data_ptr(), route.numel()))
    torch.cuda.synchronize()
    want = expected_per_expert("q8_1", t, Wq, b, ids, n_expert, n_used, 1, N)
    assert orc.nmse(got.cpu().numpy(), want) < 1e-11
    odd = torch.empty(Wd.numel() + 1, dtype=torch.uint8, device=dev)[1:].reshape(n_expert, N, -1)
    odd.copy_(Wd.reshape(odd.shape))
    assert odd.data_ptr() % 2 == 1
    got = mi355.mul_mat_id(t, odd, torch.from_numpy(b).to(dev), idd, n_used).cpu().numpy()
    assert orc.nmse(got, want) < 1e-11
