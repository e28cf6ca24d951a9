"""The GPU edge-MLP kernels (BF16 MFMA GEMMs, fused edge gather/scatter,
forward and backward) against the FP64 network oracle on the same graph.

Two references: the oracle with its matrix-product operands rounded to
bfloat16 where the GPU stores them so (outputs and every gradient tensor
within 3e-3 normwise relative: the FP32 accumulation order and the edge
aggregation's split-BF16 products, ~2^-16, differ), and the plain FP64
oracle (outputs within 3e-2, gradients within 5e-2: the error that BF16
operands cost, reported)."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import mlp_oracle as M
from pysph_amd.solver import generators as gen
from pysph_amd.surrogate.graph import ParticleGraph, combined_array
from pysph_amd.surrogate.model import EdgeMLP, init_params

pytestmark = pytest.mark.gpu


def _graph(width=0.2, height=0.3, dx=0.01, hdx=1.3, max_per=48):
    f, b, info = gen.dam_break_2d(width=width, height=height, dx=dx, hdx=hdx,
                                  precision="single", jitter=0.1, seed=4)
    rng = np.random.Generator(np.random.PCG64(2))
    nf = f.get_number_of_particles()
    f.set(u=rng.normal(0, 0.5, nf), v=rng.normal(0, 0.5, nf))
    g = ParticleGraph(combined_array(f, b), info, domain=info["domain"], max_per=max_per)
    g.build()
    return g, info


def _host(g):
    sc = g.pa.__dict__["_pack_scratch"]
    n = g.n
    pos4 = sc["pos4"][:n].double().cpu().numpy()
    vel4 = sc["vel4"][:n].double().cpu().numpy()
    rho = g.pa.get_carray("rho").double().cpu().numpy()
    bt = g.pa.get_carray("btype").cpu().numpy()
    off = g.off.cpu().numpy()
    nbr = g.nbr[:g.nedges_exact()].cpu().numpy()
    s = g.struct
    c = dict(rho0=s.rho0, co=s.co, gamma=s.gamma, u_scale=s.u_scale, g=s.g,
             rho_scale=s.rho_scale, alpha=s.alpha, eta=s.eta, dim=2)
    return pos4, vel4, rho, bt, off, nbr, c


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) /
                 max(np.linalg.norm(np.asarray(b)), 1e-30))


def _params(seed):
    theta = init_params(seed).astype(np.float64)
    rng = np.random.Generator(np.random.PCG64(seed + 7))
    p = M.unflatten(theta)
    for k in p:
        if p[k].ndim == 1:
            p[k] = rng.normal(0, 0.1, p[k].shape)
    # the trained decoder starts at zero; give it weights so that every
    # layer receives gradient
    p["w_out"] = rng.normal(0, 0.1, p["w_out"].shape)
    return M.flatten(p).astype(np.float32)


def test_graph_is_symmetric_with_self_edges():
    g, _ = _graph()
    off = g.off.cpu().numpy()
    nbr = g.nbr[:g.nedges_exact()].cpu().numpy()
    dst = np.repeat(np.arange(g.n), np.diff(off))
    pairs = set(zip(dst.tolist(), nbr.tolist()))
    assert all((b, a) in pairs for a, b in pairs)
    assert all((k, k) in pairs for k in range(g.n))


@pytest.mark.parametrize("hdx", [1.3, 1.8])
def test_forward_matches_oracle(hdx):
    # h = 1.8 dx: ~40 edges per interior node, so the aggregation takes
    # nodes of one and of two 32-edge blocks (fewer at the free surface)
    g, _ = _graph(hdx=hdx, max_per=96)
    g.check_overflow()
    deg = np.diff(g.off.cpu().numpy())
    if hdx > 1.5:
        assert deg.max() > 32 and deg.min() <= 32
    theta = _params(1)
    model = EdgeMLP(params=theta)
    y = model.forward(g)[:g.n].double().cpu().numpy()
    pos4, vel4, rho, bt, off, nbr, c = _host(g)
    X, E, dst, src = M.features(pos4, vel4, rho, bt, off, nbr, c)
    p = M.unflatten(theta.astype(np.float64))
    Y, _ = M.forward(p, X, E, dst, src, g.n)
    Yb, _ = M.forward(p, X, E, dst, src, g.n, round_bf16=True)
    err, errb = _rel(y, Y), _rel(y, Yb)
    print("forward normwise rel err: %.3e vs FP64, %.3e vs BF16-rounded oracle" % (err, errb))
    # measured 3.8e-4 against the BF16-rounded oracle (FP32 summation
    # order, split-BF16 edge products) and ~4e-3 against plain FP64
    assert errb < 3e-3
    assert err < 3e-2
    assert np.abs(Y).max() > 1e-3


def test_fp32_edge_aggregation_matches_matrix_core():
    """The FP32 vector-unit edge aggregation (the path that graphs of 2^22
    nodes or more take) against the matrix-core one on the same graph, and
    against the BF16-rounded oracle."""
    g, _ = _graph(hdx=1.8, max_per=96)
    theta = _params(1)
    model = EdgeMLP(params=theta)
    y_mc = model.forward(g)[:g.n].double().cpu().numpy()
    y_32 = model.forward(g, edge_fp32=True)[:g.n].double().cpu().numpy()
    pos4, vel4, rho, bt, off, nbr, c = _host(g)
    X, E, dst, src = M.features(pos4, vel4, rho, bt, off, nbr, c)
    p = M.unflatten(theta.astype(np.float64))
    Yb, _ = M.forward(p, X, E, dst, src, g.n, round_bf16=True)
    d, errb = _rel(y_32, y_mc), _rel(y_32, Yb)
    print("FP32 vs matrix-core aggregation: %.3e; FP32 path vs BF16-rounded oracle: %.3e"
          % (d, errb))
    # the split-BF16 products differ from FP32 FMAs by ~2^-16, and the BF16
    # copy of the aggregate can round the other way
    assert 0 < d < 1e-3
    assert errb < 3e-3


def test_inference_forward_same_output_and_no_backward():
    """A forward pass for inference (SPH_MLP_INFER: the activations of the
    backward pass are not stored) gives the same bits as a training forward
    pass, and a backward pass after it is refused until a training forward
    pass runs again."""
    from pysph_amd import _abi
    g, _ = _graph()
    model = EdgeMLP(params=_params(3))
    y_train = model.forward(g)[:g.n].cpu().numpy()
    y_infer = model.forward(g, infer=True)[:g.n].cpu().numpy()
    assert np.array_equal(y_train, y_infer)
    dout = torch.zeros((max(g.n, 1), 2), dtype=torch.float32, device=g.device)
    with pytest.raises(_abi.SphError):
        _abi.call("sph_mlp_backward", model.handle, torch.cuda.current_stream().cuda_stream,
                  ctypes.byref(g.struct), dout.data_ptr())
    tgt = torch.zeros_like(dout)
    loss = model.loss_backward(g, tgt)
    assert torch.isfinite(loss).all()


def test_backward_matches_oracle():
    g, _ = _graph()
    theta = _params(2)
    model = EdgeMLP(params=theta)
    rng = np.random.Generator(np.random.PCG64(5))
    T = rng.normal(0, 1, (g.n, 2))
    tgt = torch.tensor(T, dtype=torch.float32, device=g.device)
    stream = torch.cuda.current_stream().cuda_stream
    model.zero_grad(stream)
    loss = float(model.loss_backward(g, tgt).item())
    grads = model.grads()
    pos4, vel4, rho, bt, off, nbr, c = _host(g)
    X, E, dst, src = M.features(pos4, vel4, rho, bt, off, nbr, c)
    p = M.unflatten(theta.astype(np.float64))
    gg = M.unflatten(grads.astype(np.float64))
    # measured <= 3e-4 against the BF16-rounded oracle and 1.6e-2 to 2.7e-2
    # against plain FP64 (the BF16 rounding of activations and weights)
    for round_bf16, tol in ((True, 3e-3), (False, 5e-2)):
        Y, cache = M.forward(p, X, E, dst, src, g.n, round_bf16=round_bf16)
        L, dY = M.loss(Y, T, bt)
        gref = M.backward(p, cache, dY)
        assert abs(loss - L) < 1e-2 * L
        worst = {}
        for k in gref:
            if k == "b_out":
                a, b = gg[k][:2], gref[k][:2]
            else:
                a, b = gg[k], gref[k]
            worst[k] = _rel(a, b)
        print("gradient normwise rel errors (%s):" % ("BF16-rounded oracle" if round_bf16
                                                      else "FP64 oracle"),
              {k: "%.2e" % v for k, v in worst.items()})
        assert max(worst.values()) < tol, worst


def test_adam_steps_reduce_the_loss():
    g, _ = _graph()
    model = EdgeMLP(seed=3)
    rng = np.random.Generator(np.random.PCG64(6))
    tgt = torch.tensor(rng.normal(0, 1, (g.n, 2)) * 0.3, dtype=torch.float32, device=g.device)
    stream = torch.cuda.current_stream().cuda_stream
    losses = []
    for _ in range(60):
        model.zero_grad(stream)
        losses.append(float(model.loss_backward(g, tgt).item()))
        model.adam(stream, lr=3e-3)
    print("loss %.3e -> %.3e" % (losses[0], losses[-1]))
    assert losses[-1] < 0.7 * losses[0]


@pytest.mark.parametrize("width,height", [(0.01, 0.01), (0.02, 0.03), (0.05, 0.07), (0.3, 0.43)])
def test_gradients_at_chunk_remainders(width, height):
    """Weight and bias gradients where the node count leaves remainders of
    the 32-row steps, the 64-row bias blocks and the chunks of up to 256 rows (one
    chunk of a few rows up to several chunks), each tensor against the
    BF16-rounded oracle.  Biases and non-negative H x H weights keep every ReLU
    active, so that no unit near zero is masked on one side only (one such unit of one node is worth
    up to 1/nodes of a gradient).  What is left: FP32 sums of at most 2e3
    terms in another order (2e3 * 2^-24 = 1e-4), the aggregation's split
    products (2^-16) and BF16 copies of H, A and dZ that round the other way
    (2^-8 of a value, on a small share of them): below 1e-3."""
    g, _ = _graph(width=width, height=height)
    p = M.unflatten(_params(2).astype(np.float64))
    for k in p:
        if k.startswith(("b_in", "b_e", "c_u")):
            p[k] = np.full(p[k].shape, 200.0)
        elif k.startswith(("w_ab", "w_u")):
            p[k] = np.abs(p[k])
    theta = M.flatten(p).astype(np.float32)
    p = M.unflatten(theta.astype(np.float64))
    model = EdgeMLP(params=theta)
    pos4, vel4, rho, bt, off, nbr, c = _host(g)
    rng = np.random.Generator(np.random.PCG64(9))
    T = rng.normal(0, 1, (g.n, 2)).astype(np.float32)
    X, E, dst, src = M.features(pos4, vel4, rho, bt, off, nbr, c)
    Y, cache = M.forward(p, X, E, dst, src, g.n, round_bf16=True)
    assert cache["H0"].min() > 0
    for r in range(M.ROUNDS):
        assert cache["r%d" % r]["S"].min() > 0 and cache["r%d" % r]["U"].min() > 0
    ref = M.backward(p, cache, M.loss(Y, T, bt)[1])
    model.zero_grad(torch.cuda.current_stream().cuda_stream)
    model.loss_backward(g, torch.from_numpy(T).cuda())
    got = M.unflatten(model.grads().astype(np.float64))
    for k in ref:
        assert _rel(got[k], ref[k]) < 3e-3, (k, g.n)


DEGREES = [[0], [1], [0, 0, 0, 0, 0], [32], [0, 33, 0], [1, 0, 31, 32, 33, 0, 64, 65, 2, 96, 0],
           [21] * 9, [65, 1] * 20, [40] * 3 + [0] + [7] * 4099]
# more than two nodes for each of the forward kernel's 4096 waves (the backward
# kernel's 2048), counts mixed so that waves pass from every kind of node to
# every other
DEGREES.append(np.random.Generator(np.random.PCG64(8)).choice(
    [0, 1, 2, 31, 32, 33, 64, 65], 9500).tolist())


def _graph_for(degrees):
    """A graph with at least as many nodes as there are degrees."""
    return _graph(*((0.2, 0.3) if len(degrees) < 1000 else (0.8, 1.2)))[0]


def _set_edges(g, degrees):
    """Give the graph's first nodes these edge counts, with nearby nodes as
    neighbours (repeated ones are edges of their own)."""
    n = len(degrees)
    assert n <= g.n
    rng = np.random.Generator(np.random.PCG64(n))
    dst = np.repeat(np.arange(n), degrees)
    nbr = np.clip(dst + rng.integers(-9, 10, len(dst)), 0, n - 1)
    off = torch.tensor(np.concatenate([[0], np.cumsum(degrees)]), dtype=torch.int64,
                       device=g.device)
    nbr = torch.tensor(nbr if len(nbr) else [0], dtype=torch.int64, device=g.device)
    g.n = g.struct.n = n
    g.struct.off, g.struct.nbr, g.struct.nedges = off.data_ptr(), nbr.data_ptr(), len(dst)
    return off, nbr


@pytest.mark.parametrize("degrees", DEGREES)
def test_edge_blocks_and_node_runs(degrees):
    """The matrix-core edge aggregation on given edge counts (none, whole and
    partial blocks of 32, several blocks; fewer nodes than waves up to several
    nodes per wave, which a wave passes between in every combination) against the FP32 vector-unit one on the same graph.  What
    differs is the split-BF16 products (2^-16) and BF16 copies of the
    aggregate that round the other way (2^-8 of a value, on a share of about
    2^-7 of them): below 1e-3, as in the test above."""
    g = _graph_for(degrees)
    keep = _set_edges(g, degrees)
    model = EdgeMLP(params=_params(5))
    y = model.forward(g)[:g.n].double().cpu().numpy()
    ref = model.forward(g, edge_fp32=True)[:g.n].double().cpu().numpy()
    assert np.isfinite(y).all()
    assert _rel(y, ref) < 1e-3
    del keep


@pytest.mark.parametrize("degrees", DEGREES)
def test_edge_backward_blocks_and_node_runs(degrees):
    """The matrix-core edge backward pass against the FP32 vector-unit one
    after the same forward pass.  The masks of edges whose pre-activation is
    within 2^-16 of its terms of zero can differ (a share of about 1e-5 of
    them, each a term of the sums of the size of the others), then the BF16
    copies of dP and dQ round the other way; feature and mask products are
    exact: below 1e-3."""
    from pysph_amd import _abi
    g = _graph_for(degrees)
    keep = _set_edges(g, degrees)
    model = EdgeMLP(params=_params(6))
    rng = np.random.Generator(np.random.PCG64(len(degrees)))
    dout = torch.tensor(rng.normal(0, 1, (g.n, 2)), dtype=torch.float32, device=g.device)
    stream = torch.cuda.current_stream().cuda_stream
    model.forward(g)
    grads = []
    for flags in (0, _abi.SPH_MLP_EDGE_FP32):
        model.zero_grad(stream)
        g.struct.flags = flags
        _abi.call("sph_mlp_backward", model.handle, stream, ctypes.byref(g.struct),
                  dout.data_ptr())
        grads.append(M.unflatten(model.grads().astype(np.float64)))
    for k in grads[0]:
        assert np.isfinite(grads[0][k]).all()
        assert _rel(grads[0][k], grads[1][k]) < 1e-3 or np.abs(grads[1][k]).max() == 0, k
        if np.abs(grads[1][k]).max() == 0:
            assert np.abs(grads[0][k]).max() == 0, k
    del keep


def _aggregate_order(x, b, q):
    """The edge aggregation's roundings, z = (x + b) + q per edge and FP32
    sums in the order of the matrix cores' rows: edges are taken 32 at a time,
    half-wave h sums rows 4h + 8k .. 4h + 8k + 3 for k = 0 .. 3 one after
    another, and the halves are added at the end."""
    half = [np.float32(0), np.float32(0)]
    z = np.maximum((x + np.float32(b)) + np.float32(q), np.float32(0))
    for e, v in enumerate(z):
        h = (e >> 2) & 1
        half[h] = np.float32(half[h] + v)
    return half[0] + half[1]


def test_edge_aggregation_rounds_in_a_fixed_order():
    """Outputs of the matrix-core aggregation bit for bit against its
    roundings on the host: P + b is added to the edge product first, Q_j
    second, and the rows one after another.  Every product is exact here: the
    network passes one edge feature, a velocity difference of at most 16
    bits, through two units of one round to the output.  Unit 0 sums 1 + 2^-8
    (halfway between two bfloat16 values) and terms below half its last bit,
    so that the order of the sum decides how it rounds; unit 1 has b = 2^14
    and Q = -2^14, so that the order of the additions decides which bits of
    the feature are kept."""
    g, _ = _graph()
    rng = np.random.Generator(np.random.PCG64(21))
    n = 600
    vals = np.zeros(n, dtype=np.float32)
    vals[0] = 1 + 2.0 ** -8
    vals[1:10] = 3 * 2.0 ** -26
    vals[10:40] = rng.integers(1, 2 ** 12, 30) * 2.0 ** -12
    lists = [rng.permutation([0] + [1 + k % 9 for k in range(d)]) for d in range(1, 70)]
    lists += [rng.integers(10, 40, d) for d in rng.integers(0, 70, 200)]
    lists = [np.zeros(0, np.int64)] * 40 + lists
    lists += [rng.integers(1, 40, 3)] * (n - len(lists))
    off = np.concatenate([[0], np.cumsum([len(v) for v in lists])])
    nbr = np.concatenate(lists)
    dev = [torch.from_numpy(a).to(g.device) for a in
           (off.astype(np.int64), nbr.astype(np.int64),
            np.stack([-vals, 0 * vals, 0 * vals, 0 * vals + 1], 1), 0 * vals + 1)]
    s = g.struct
    s.off, s.nbr, s.vel4, s.rho = (t.data_ptr() for t in dev)
    g.n = s.n = n
    s.nedges = len(nbr)
    s.rho0 = s.u_scale = 1.0
    s.alpha = 0.0  # with rho = rho0: no pressure or viscous terms in the output
    B, c = 2.0 ** 14, (3, 77)
    p = {k: 0 * v for k, v in M.unflatten(_params(0).astype(np.float64)).items()}
    p["b_in"][5] = 1.0
    p["w_ab0"][5, M.H + c[1]] = -B
    p["b_e0"][c[1]] = B
    for k in range(2):
        p["w_c0"][3, c[k]] = 1.0
        p["w_u0"][M.H + c[k], c[k]] = 1.0
        p["w_out"][c[k], k] = 1.0
    y = EdgeMLP(params=M.flatten(p).astype(np.float32)).forward(g)[:n].cpu().numpy()
    own = vals.copy()
    for i in range(n):
        x = vals[lists[i]] - own[i]
        for k, (b, q) in enumerate(((0.0, 0.0), (B, -B))):
            want = M.bf16(_aggregate_order(x, b, q))
            assert y[i, k] == want, (i, k, len(x), y[i, k], want)


@pytest.mark.parametrize("edge_fp32", [False, True])
def test_edge_backward_masks_in_fp32(edge_fp32):
    """The ReLU masks of the edge backward pass where the pre-activations of
    both directions differ from zero by a few last bits of an FP32 product:
    features of 24 bits times 1, and weights of 24 bits times a feature of 1,
    against biases next to them.  With a gradient of 1 at every aggregate,
    the bias's gradient and the two halves of dW_ab count the masks, whole
    numbers that FP32 (and BF16, up to 256 a node) holds exactly."""
    from pysph_amd import _abi
    g, _ = _graph()
    rng = np.random.Generator(np.random.PCG64(31))
    n, nd = 600, 400  # nodes; the first nd have edges, the others are their sources
    thr = np.float32(1.2345678)
    units = list(range(4, 4 + 48, 3))
    w = np.ones(len(units), dtype=np.float32)
    w[1:] = rng.uniform(1.0, 2.0, len(units) - 1)
    b = -w * np.float32(1)
    b[0] = -thr
    for k in range(1, len(units)):  # a few last bits to either side of w
        for _ in range(1 + k % 3):
            b[k] = np.nextafter(b[k], np.float32(-9 if k & 1 else 0))
    vals = np.zeros(n, dtype=np.float32)
    k = rng.integers(1, 9, n - nd) * rng.choice([-1, 1], n - nd)
    vals[nd:] = rng.choice([-1, 1], n - nd) * np.where(
        rng.random(n - nd) < 0.3, np.float32(1), thr + (k * 2.0 ** -23).astype(np.float32))
    deg = rng.integers(0, 80, n)
    deg[nd:] = 0
    off = np.concatenate([[0], np.cumsum(deg)])
    nbr = rng.integers(nd, n, off[-1])
    dev = [torch.from_numpy(a).to(g.device) for a in
           (off.astype(np.int64), nbr.astype(np.int64),
            np.stack([-vals, 0 * vals, 0 * vals, 0 * vals + 1], 1), 0 * vals + 1)]
    s = g.struct
    s.off, s.nbr, s.vel4, s.rho = (t.data_ptr() for t in dev)
    g.n = s.n = n
    s.nedges = len(nbr)
    s.rho0 = s.u_scale = 1.0
    s.alpha = 0.0
    p = {key: 0 * v for key, v in M.unflatten(_params(0).astype(np.float64)).items()}
    p["b_in"][5] = 1.0
    for q, c in enumerate(units):
        p["w_c1"][3, c], p["b_e1"][c] = w[q], b[q]
        p["w_u1"][M.H + c, c] = p["c_u1"][c] = p["w_out"][c, 0] = 1.0
    model = EdgeMLP(params=M.flatten(p).astype(np.float32))
    model.forward(g)
    stream = torch.cuda.current_stream().cuda_stream
    dout = torch.zeros((n, 2), dtype=torch.float32, device=g.device)
    dout[:, 0] = 1.0
    s.flags = _abi.SPH_MLP_EDGE_FP32 if edge_fp32 else 0
    model.zero_grad(stream)
    _abi.call("sph_mlp_backward", model.handle, stream, ctypes.byref(s), dout.data_ptr())
    got = M.unflatten(model.grads().astype(np.float64))
    x = vals[nbr].astype(np.float64)
    for q, c in enumerate(units):
        fwd = x * w[q] + b[q].astype(np.float64)
        rev = -x * w[q] + b[q].astype(np.float64)
        assert (fwd != 0).all() and (rev != 0).all()
        want = int((fwd > 0).sum()), int((fwd > 0).sum()), int((rev > 0).sum())
        assert (got["b_e1"][c], got["w_ab1"][5, c], got["w_ab1"][5, M.H + c]) == want, q


@pytest.mark.parametrize("edge_fp32", [False, True])
def test_edges_past_the_capacity_are_left_out(edge_fp32):
    """A graph with more edges than its room: the offsets of the rows that did
    not fit point past the neighbour array, and the network's passes end
    every row at the room's end (the same bits as with clamped offsets).  The
    array read here has spare entries behind the room, so that a pass that
    read on would differ, not fault."""
    from pysph_amd import _abi
    g, _ = _graph(max_per=8)
    total, cap = g.nedges_exact(), g.cap
    assert total > cap and int(g.overflow.item()) == 1
    with pytest.raises(RuntimeError, match="more than 8 neighbours"):
        g.check_overflow()
    s = g.struct
    nbr = torch.cat([g.nbr, torch.zeros(total - cap, dtype=torch.int64, device=g.device)])
    clamped = g.off.clamp(max=cap)
    s.nbr = nbr.data_ptr()
    model = EdgeMLP(params=_params(5))
    rng = np.random.Generator(np.random.PCG64(4))
    dout = torch.tensor(rng.normal(0, 1, (g.n, 2)), dtype=torch.float32, device=g.device)
    stream = torch.cuda.current_stream().cuda_stream
    res = []
    for off in (clamped, g.off):
        s.off = off.data_ptr()
        y = model.forward(g, edge_fp32=edge_fp32)
        model.zero_grad(stream)
        _abi.call("sph_mlp_backward", model.handle, stream, ctypes.byref(s), dout.data_ptr())
        res.append((y.cpu().numpy(), model.grads()))
    assert np.isfinite(res[0][0]).all()
    for a, b in zip(*res):
        assert np.array_equal(a, b)
