"""The work that programs have this package do, as timed cases.

Three kinds of whole calls (an energy + forces step of the uma-s-1 architecture on a molecule, on
a crystal with its stress and on a 2048-atom cluster; a batch of Orb molecules) and the single
layers, blocks and per-op calls that programs run one by one: Orb's attention layer and MLP blocks
with their reverse passes, the isolated edgewise map with its VJP, the rotation and segment-sum
calls, and the device neighbour list.  ``listed`` names the standing cases, ``draw`` gives others
of the same ranges, ``exact`` is each path in 64-bit torch.
"""
from __future__ import annotations

import math
import pathlib
import sys

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parents[1] / "tt-atom_amd"))

DEV = "cuda"
UMA_CUTOFF, UMA_CAP = 6.0, 30
ORB_CUTOFF, ORB_CAP = 6.0, 20
ORB_C, ORB_H = 256, 1024
FCC_A = 3.61
PERM_M = (0, 2, 6, 3, 7, 1, 5, 8, 4)      # m-primed order of the nine coefficients


# ---------------------------------------------------------------------------------- the cases
def listed():
    return [
        # an MD loop on one small molecule: every launch is latency
        dict(name="uma_molecule", kind="uma", atoms=24, reps=0, stress=False),
        # a relaxation or NPT step of a small supercell (4 x 4 x 4 FCC Cu), with the stress
        dict(name="uma_crystal_stress", kind="uma", atoms=256, reps=4, stress=True),
        # the large end of single-system MD: 2048 atoms, about 61,000 edges
        dict(name="uma_cluster", kind="uma", atoms=2048, reps=0, stress=False),
        # screening throughput: 256 molecules of 20 to 60 atoms in one disjoint union
        dict(name="orb_batch", kind="orb", systems=256),
        # one message-passing layer and its reverse pass on eight small molecules
        dict(name="orb_layer_small", kind="orb_layer", nodes=72, edges=576, fast=False),
        # the same on a few thousand atoms, sizes that no tile divides
        dict(name="orb_layer_large", kind="orb_layer", nodes=4003, edges=78_909, fast=False),
        # a node MLP block ([n | recv | sent] -> n) of a mid-size batch, forward and reverse
        dict(name="orb_node_mlp", kind="mlp", rows=1237, n_in=768, fast=False),
        # the edge encoder with reduced-precision operands (fast=True), forward and reverse
        dict(name="orb_edge_encoder_fast", kind="mlp", rows=30_011, n_in=128, fast=True),
        # the isolated edgewise map with its VJP: a molecule-sized graph with ragged degrees ...
        dict(name="edgewise_small", kind="edgewise", nodes=150, edges=1937, precision="f32"),
        # ... and 8192 nodes of degree 25
        dict(name="edgewise_large", kind="edgewise", nodes=8192, edges=204_800, precision="f32"),
        # callers of the single rotation / segment-sum operations, forward and adjoint
        dict(name="rotation_ops", kind="rotation", nodes=1000, edges=20_011, width=128),
        # a fresh neighbour list of a ten-thousand-atom system
        dict(name="neighbors", kind="neighbors", atoms=10_007, cap=30),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["uma", "uma", "orb", "orb_layer", "orb_layer", "mlp", "mlp", "edgewise",
                       "edgewise", "rotation", "neighbors"])
    if kind == "uma":
        if rng.random() < 0.35:
            reps = rng.randint(3, 6)
            return dict(kind=kind, atoms=4 * reps ** 3, reps=reps, stress=rng.random() < 0.7)
        return dict(kind=kind, atoms=_log_int(rng, 20, 2040), reps=0, stress=rng.random() < 0.2)
    if kind == "orb":
        return dict(kind=kind, systems=_log_int(rng, 2, 240))
    if kind == "orb_layer":
        nodes = _log_int(rng, 40, 6000)
        return dict(kind=kind, nodes=nodes, edges=int(nodes * rng.uniform(8, 20)),
                    fast=rng.random() < 0.25)
    if kind == "mlp":
        return dict(kind=kind, rows=_log_int(rng, 50, 60_000), n_in=rng.choice([128, 256, 768]),
                    fast=rng.random() < 0.3)
    if kind == "edgewise":
        nodes = _log_int(rng, 60, 8000)
        return dict(kind=kind, nodes=nodes, edges=int(nodes * rng.uniform(6, 25)),
                    precision=rng.choice(["f32", "f32", "bf16"]))
    if kind == "rotation":
        nodes = _log_int(rng, 60, 4000)
        return dict(kind=kind, nodes=nodes, edges=int(nodes * rng.uniform(6, 25)),
                    width=rng.choice([16, 64, 128, 256]))
    return dict(kind=kind, atoms=_log_int(rng, 500, 16_000), cap=rng.choice([0, 20, 30]))


# ------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _cluster(rng, n, spacing=2.2):
    """n atoms of a jittered cubic lattice inside a ball, in random order (about 75 neighbours
    within 6 A in the bulk)."""
    m = int(math.ceil((3.0 * n / (4.0 * math.pi)) ** (1.0 / 3.0))) + 1
    site = np.stack(np.meshgrid(*[np.arange(-m, m + 1)] * 3, indexing="ij"), -1).reshape(-1, 3)
    site = site[np.argsort((site * site).sum(1), kind="stable")[:n]] * spacing
    pos = site + rng.normal(0.0, 0.15 * spacing, site.shape)
    return pos[rng.permutation(n)].astype(np.float32)


def _fcc(rng, reps):
    from tt_atom import synthetic
    pos, Z, cell = synthetic.c4_system(seed=int(rng.integers(1 << 30)), reps=reps, a=FCC_A)
    return pos, Z, cell


def _nearest(pos, cutoff, cap, cell=None):
    """[2, E] (source, target) and [E, 3] image shifts: each target's ``cap`` nearest sources
    within the cutoff."""
    if cell is None:
        shifts = torch.zeros(1, 3, device=pos.device)
    else:
        r = torch.arange(-1.0, 2.0, device=pos.device)
        shifts = torch.cartesian_prod(r, r, r) @ cell
    image = (pos[None] + shifts[:, None]).reshape(-1, 3)          # [S * N, 3]
    d = (image[None] - pos[:, None]).norm(dim=-1)                 # [N, S * N]
    d = torch.where((d < cutoff) & (d > 1e-4), d, torch.inf)
    d, j = d.topk(min(cap, d.shape[1]), dim=1, largest=False)
    ok = torch.isfinite(d)
    tgt = torch.arange(pos.shape[0], device=pos.device)[:, None].expand_as(j)[ok]
    j = j[ok]
    return torch.stack([j % pos.shape[0], tgt]), shifts[j // pos.shape[0]]


def _uma_inputs(case, seed):
    from tt_atom import synthetic
    rng = np.random.default_rng(seed)
    cfg = dict(synthetic.CFG_UMA_S, task="omat" if case["reps"] else "omol")
    if case["reps"]:
        pos, Z, cell = _fcc(rng, case["reps"])
        cell = torch.from_numpy(cell).to(DEV)
    else:
        pos, cell = _cluster(rng, case["atoms"]), None
        Z = rng.choice(synthetic.ELEMENTS, size=case["atoms"], p=synthetic.ELEMENT_P)
    weights, host = synthetic.random_uma_bundle(cfg, seed)
    pos = torch.from_numpy(pos).to(DEV)
    edges, shift = _nearest(pos, UMA_CUTOFF, UMA_CAP, cell)
    # one charge / spin / dataset embedding row, the same for every node
    sys_emb = (torch.from_numpy(rng.standard_normal((1, cfg["sphere_channels"]))).float()
               .to(DEV).expand(len(Z), -1).contiguous())
    return dict(cfg=cfg, w=weights, host=host, pos=pos, Z=torch.from_numpy(np.asarray(Z)),
                edges=edges, shift=shift if case["reps"] else None, sys_emb=sys_emb)


def _orb_inputs(case, seed):
    """Molecules of 20 to 60 atoms on jittered sites of a 7 A cube; each sender's 20 nearest."""
    from tt_atom import synthetic
    rng = np.random.default_rng(seed)
    K = case["systems"]
    cfg = dict(synthetic.CFG_ORB_C5)
    weights = synthetic.random_orb_weights(cfg, seed)
    natoms = np.random.default_rng(K).integers(20, 61, K)   # the sizes belong to the case
    site = np.stack(np.meshgrid(*[np.arange(6)] * 3, indexing="ij"), -1).reshape(-1, 3) * 1.2
    pick = np.argsort(rng.random((K, len(site))), axis=1)[:, :60]
    pos = torch.from_numpy((site[pick] + rng.uniform(-0.12, 0.12, (K, 60, 3))).astype(np.float32))
    pos, n = pos.to(DEV), torch.from_numpy(natoms).to(DEV)
    own = torch.arange(60, device=DEV)[None] < n[:, None]          # [K, 60] real atoms
    d = torch.cdist(pos, pos, compute_mode="donot_use_mm_for_euclid_dist")
    d = torch.where((d < ORB_CUTOFF) & (d > 1e-4) & own[:, None, :] & own[:, :, None], d, torch.inf)
    d, j = d.topk(ORB_CAP, dim=2, largest=False)
    ok = torch.isfinite(d)
    off = torch.cumsum(n, 0) - n
    send = (off[:, None, None] + torch.arange(60, device=DEV)[None, :, None]).expand_as(j)[ok]
    recv = (off[:, None, None] + j)[ok]
    Z = rng.choice(synthetic.ELEMENTS, size=int(natoms.sum()), p=synthetic.ELEMENT_P)
    return dict(cfg=cfg, w=weights, pos=pos[own], Z=torch.from_numpy(Z), send=send, recv=recv,
                natoms=[int(v) for v in natoms])


def _linear(g, w, name, n_in, n_out):
    b = 1.0 / math.sqrt(n_in)
    w[f"{name}.weight"] = (torch.rand(n_out, n_in, generator=g, device=DEV) * 2 - 1) * b
    w[f"{name}.bias"] = (torch.rand(n_out, generator=g, device=DEV) * 2 - 1) * b


def _mlp_norm(g, w, name, n_in):
    for i, (a, b) in enumerate(((n_in, ORB_H), (ORB_H, ORB_H), (ORB_H, ORB_C))):
        _linear(g, w, f"{name}.mlp.NN-{i}", a, b)
    w[f"{name}.layer_norm.weight"] = 1.0 + 0.1 * _randn(g, ORB_C)


def _layer_inputs(case, seed):
    g = _gen(seed)
    N, E = case["nodes"], case["edges"]
    w = {}
    _mlp_norm(g, w, "l._edge_mlp", 3 * ORB_C)
    _mlp_norm(g, w, "l._node_mlp", 3 * ORB_C)
    _linear(g, w, "l._receive_attn", ORB_C, 1)
    _linear(g, w, "l._send_attn", ORB_C, 1)
    # edges in the order of a neighbour list (by sender), receivers a few nodes away
    send = torch.randint(N, (E,), generator=g, device=DEV).sort().values
    step = torch.randint(1, min(32, N), (E,), generator=g, device=DEV)
    return dict(w=w, send=send, recv=(send + step) % N,
                cut=torch.rand(E, 1, generator=g, device=DEV),
                nodes=_randn(g, N, ORB_C), edges=_randn(g, E, ORB_C),
                g_nodes=_randn(g, N, ORB_C), g_edges=_randn(g, E, ORB_C))


def _mlp_inputs(case, seed):
    g = _gen(seed)
    w = {}
    _mlp_norm(g, w, "m", case["n_in"])
    return dict(w=w, x=_randn(g, case["rows"], case["n_in"]), g=_randn(g, case["rows"], ORB_C))


def _edgewise_inputs(case, seed):
    from tt_atom import synthetic
    g = _gen(seed)
    N, E, C = case["nodes"], case["edges"], 128
    tgt = torch.randint(N, (E,), generator=g, device=DEV).sort().values
    src = (tgt + torch.randint(1, N, (E,), generator=g, device=DEV)) % N
    ev = F.normalize(_randn(g, E, 3), dim=1)
    ev = ev * (0.8 + 5.2 * torch.rand(E, 1, generator=g, device=DEV))
    return dict(w=synthetic.c2_weights(seed, C), jd=synthetic.jd_matrices(), src=src, tgt=tgt,
                ev=ev, x=_randn(g, N, 9, C), g=_randn(g, N, 9, C), C=C)


def _rotation_inputs(case, seed):
    from tt_atom import synthetic
    g = _gen(seed)
    N, E, W = case["nodes"], case["edges"], case["width"]
    wig = _wigner64(_randn(g, E, 3).double(), [j.double() for j in synthetic.jd_matrices()])
    return dict(wig=wig.float(), x=_randn(g, E, 9 * W), g=_randn(g, E, 9 * W),
                tgt=torch.randint(N, (E,), generator=g, device=DEV))


def _neighbor_inputs(case, seed):
    """One cluster per size, its atoms reordered and its axes reflected by the seed, so that every
    seed has as many edges."""
    rng = np.random.default_rng(seed)
    pos = _cluster(np.random.default_rng(case["atoms"]), case["atoms"])
    pos = pos[rng.permutation(case["atoms"])] * rng.choice([-1.0, 1.0], 3)
    return torch.from_numpy(pos.astype(np.float32))


# ------------------------------------------------------------------------- prepare and run
def prepare(case, seed):
    kind = case["kind"]
    if kind == "uma":
        from tt_atom import geometry, model, trace
        i = _uma_inputs(case, seed)
        bb = model.Backbone(i["w"], DEV, i["cfg"])
        geo = geometry.HostGeometry(i["w"], i["cfg"], i["host"]["to_m"], i["host"]["gauss_offset"],
                                    i["host"]["gauss_coeff"], device=DEV)
        eng = trace.TracedEngine(bb, geo, i["Z"], i["edges"], i["sys_emb"],
                                 edge_cell_shift=i["shift"])
        return dict(kind=kind, eng=eng, pos=i["pos"], stress=case["stress"])
    if kind == "orb":
        from tt_atom import orb
        i = _orb_inputs(case, seed)
        graph = orb.OrbGraph(DEV, senders=i["send"], receivers=i["recv"],
                             num_nodes=len(i["Z"]), atomic_numbers=i["Z"], natoms=i["natoms"])
        eng = orb.OrbEngine(orb.OrbModel(i["w"], i["cfg"], DEV), graph)
        return dict(kind=kind, eng=eng, pos=i["pos"])
    if kind == "orb_layer":
        from tt_atom import orb_model
        i = _layer_inputs(case, seed)
        layer = orb_model.AttentionInteractionLayer(i["w"], "l", DEV, latent_dim=ORB_C,
                                                    hidden_dim=ORB_H, fast=case["fast"])
        graph = orb_model.OrbGraphContext(DEV, senders=i["send"], receivers=i["recv"],
                                          cutoff=i["cut"], num_nodes=case["nodes"])
        return dict(i, kind=kind, layer=layer, graph=graph)
    if kind == "mlp":
        from tt_atom import orb_model
        i = _mlp_inputs(case, seed)
        mlp = orb_model.MLPNorm(i["w"], "m", DEV, case["n_in"], ORB_H, ORB_C, fast=case["fast"])
        return dict(i, kind=kind, mlp=mlp)
    if kind == "edgewise":
        from tt_atom import edgewise
        i = _edgewise_inputs(case, seed)
        step = edgewise.EdgewiseStep(i["w"], "c2", i["jd"], i["src"], i["tgt"], case["nodes"],
                                     C=i["C"], device=DEV, precision=case["precision"])
        return dict(i, kind=kind, step=step)
    if kind == "rotation":
        from tt_atom import rotation, scatter
        i = _rotation_inputs(case, seed)
        ij, coef = rotation.pack(i["wig"])
        table, width = scatter.build_gather(i["tgt"], case["nodes"], case["edges"])
        return dict(kind=kind, x=i["x"], g=i["g"], ij=ij, coef=coef, W=case["width"],
                    N=case["nodes"], table=torch.from_numpy(table).to(DEV), Dmax=width)
    return dict(kind=kind, pos=_neighbor_inputs(case, seed), cap=case["cap"] or None)


def run(state):
    s, kind = state, state["kind"]
    if kind == "uma":
        s["eng"].run(s["pos"], compute_stress=s["stress"])
        out = dict(energy=s["eng"].energy_buf, forces=s["eng"].forces)
        return dict(out, virial=s["eng"].virial_buf) if s["stress"] else out
    if kind == "orb":
        s["eng"].step(s["pos"])
        return dict(energies=s["eng"].raw, forces=s["eng"].forces)
    if kind == "orb_layer":
        from tt_atom import orb_forces
        n, e = s["layer"](s["nodes"], s["edges"], s["graph"])
        gn, ge, gc = orb_forces.attn_layer_bw(s["layer"], s["graph"], s["g_nodes"], s["g_edges"])
        return dict(nodes=n, edges=e, g_nodes=gn, g_edges=ge, g_cut=gc)
    if kind == "mlp":
        from tt_atom import orb_forces
        y = s["mlp"](s["x"])
        return dict(y=y, g_x=orb_forces.mlpnorm_bw(s["mlp"], s["g"]))
    if kind == "edgewise":
        out, g_ev = s["step"](s["x"], s["ev"], s["g"])
        return dict(out=out, g_ev=g_ev)
    if kind == "rotation":
        from tt_atom import rotation, scatter
        y = rotation.rotate(None, s["x"], s["ij"], s["coef"], 9, s["W"])
        gx, gc = rotation.rotate_bw(None, s["x"], s["g"], s["ij"], s["coef"], 9, s["W"])
        node = scatter.segment_sum(None, y, s["table"], s["Dmax"], s["N"], 9 * s["W"])
        return dict(y=y, g_x=gx, g_coef=gc, node=node)
    from tt_atom import geometry
    edges, shift = geometry.radius_graph_device(s["pos"], UMA_CUTOFF, max_neighbors=s["cap"])
    return dict(edges=edges, shift=shift)


# --------------------------------------------------------------------------- work, tolerance
def work(case):
    kind = case["kind"]
    if kind == "uma":
        N, C, H, ec, nb, L = case["atoms"], 128, 128, 128, 512, 4
        E = N * (UMA_CAP if N > 60 else max(1, min(UMA_CAP, int(0.8 * N))))
        k_in, rad = nb + 2 * ec, (L + 1) * ec
        out = 3 * C + L * 12 * C
        so2 = (6 * C) * (5 * H) + (8 * C) * (4 * H) + (4 * C) * (2 * H) + 9 * H * C + 16 * H * C \
            + 4 * H * C
        edge = k_in * rad + nb * rad + 2 * ((L + 1) * ec * ec + ec * out) + 2 * L * so2
        node = 2 * L * (2 * C * H + 18 * C * H) + 2 * (C * H + H * H)
        params = k_in * rad + (L + 1) * ec * ec + ec * out + L * (so2 + 8 * C * H)
        return dict(bytes=4.0 * params + 24.0 * N + 16.0 * E, flops=2.0 * (E * edge + N * node))
    if kind == "orb":
        N = 40 * case["systems"]
        E, C, H, L = 19 * N, ORB_C, ORB_H, 5
        mlp = H * H + H * C
        edge = 2 * (L * (C * H + mlp) + 128 * H + mlp)
        node = 2 * L * (2 * C * H + 3 * C * H + mlp) + C * H + mlp
        params = (2 * L + 2) * mlp + L * 6 * C * H + (128 + C) * H
        return dict(bytes=4.0 * params + 24.0 * N + 8.0 * E, flops=2.0 * (E * edge + N * node))
    if kind == "orb_layer":
        N, E, C, H = case["nodes"], case["edges"], ORB_C, ORB_H
        mlp = H * H + H * C
        flops = 4.0 * (E * (C * H + mlp) + N * (2 * C * H + 3 * C * H + mlp))
        return dict(bytes=4.0 * (4 * E * C + 4 * N * C + 3 * E + 2 * (mlp + 3 * C * H)),
                    flops=flops)
    if kind == "mlp":
        R, K = case["rows"], case["n_in"]
        params = K * ORB_H + ORB_H * ORB_H + ORB_H * ORB_C
        return dict(bytes=4.0 * (R * (2 * K + 2 * ORB_C) + params), flops=4.0 * R * params)
    if kind == "edgewise":
        N, E, C = case["nodes"], case["edges"], 128
        so2 = 29 * C * C
        return dict(bytes=4.0 * (3 * N * 9 * C + 6 * E + so2) + 16.0 * E, flops=4.0 * E * so2)
    if kind == "rotation":
        N, E, W = case["nodes"], case["edges"], case["width"]
        return dict(bytes=4.0 * (E * 4 * 9 * W + 70 * E + N * 9 * W), flops=2.0 * E * 106 * W)
    edges = case["atoms"] * (case["cap"] or 66)
    return dict(bytes=12.0 * case["atoms"] + 28.0 * edges, flops=0.0)


def tolerance(case):
    """About four times the largest error against ``exact`` over the listed cases and two dozen
    drawn ones."""
    kind = case["kind"]
    if kind == "neighbors":
        return "exact"
    if kind == "edgewise":
        # an edge close to the polar axis has an ill-conditioned azimuth: single values of its
        # adjoint are far further off than the norm
        if case["precision"] == "bf16":
            return dict(rel=1.6e-2, max=0.9)
        return dict(rel=5e-5, max=2.5e-2)
    if case.get("fast"):
        return dict(rel=1.6e-2, max=0.1)
    if kind == "uma":
        # the energy is a sum of node energies of both signs: its relative error is the fp32
        # error of the terms times the cancellation
        return dict(rel=5e-5, max=5e-4)
    if kind == "orb":
        return dict(rel=2e-5, max=1e-4)
    if kind == "rotation":
        return dict(rel=5e-7, max=3e-6)
    return dict(rel=5e-6, max=3e-5)


# ------------------------------------------------------------------------------------- exact
def _z_rotation(t, l):
    """[E, 2l+1, 2l+1]: cos(f t) on the diagonal, sin(f t) on the anti-diagonal, f = l .. -l."""
    f = torch.arange(l, -l - 1, -1, device=t.device, dtype=t.dtype) * t[:, None]
    return torch.diag_embed(torch.cos(f)) + torch.diag_embed(torch.sin(f)).flip(-1)


def _wigner64(vec, jd):
    """[E, 9, 9] rotations into the edge frame, rows in m-primed order."""
    u = F.normalize(vec, dim=1)
    beta, alpha = torch.acos(u[:, 1]), torch.atan2(u[:, 0], u[:, 2])
    out = vec.new_zeros(vec.shape[0], 9, 9)
    for l in range(3):
        J = jd[l].to(vec.device, vec.dtype)
        a = slice(l * l, (l + 1) * (l + 1))
        out[:, a, a] = J @ _z_rotation(-beta, l) @ J @ _z_rotation(-alpha, l)
    return out[:, list(PERM_M)]


def _lin(x, w, name):
    return F.linear(x, w[f"{name}.weight"], w.get(f"{name}.bias"))


def _so2_64(x, w, p):
    """SO(2) convolution of m-primed rows [E, 9, Cin] (the radial product already applied):
    (coefficients [E, 9, H], extra m = 0 columns)."""
    E, _, C = x.shape
    y0 = _lin(x[:, :3].reshape(E, 3 * C), w, f"{p}.fc_m0")
    rows = []
    for m, (lo, n) in enumerate(((3, 2), (7, 1))):
        W = w[f"{p}.so2_m_conv.{m}.fc.weight"]
        re, im = (x[:, lo + k * n:lo + (k + 1) * n].reshape(E, n * C) for k in (0, 1))
        Wa, Wb = W[:W.shape[0] // 2], W[W.shape[0] // 2:]
        rows += [re @ Wa.T - im @ Wb.T, im @ Wa.T + re @ Wb.T]
    H = rows[2].shape[1]
    extra = y0.shape[1] - 3 * H
    return torch.cat([y0[:, extra:]] + rows, 1).view(E, 9, H), y0[:, :extra]


def _radial64(x, w, p):
    for i in (0, 3):
        x = _lin(x, w, f"{p}.net.{i}")
        x = F.silu(F.layer_norm(x, x.shape[1:], w[f"{p}.net.{i + 1}.weight"],
                                w[f"{p}.net.{i + 1}.bias"], 1e-5))
    return _lin(x, w, f"{p}.net.6")


def _rms_sh64(x, w, p):
    degree = torch.tensor([0, 1, 1, 1, 2, 2, 2, 2, 2], device=x.device)
    x = torch.cat([x[:, :1] - x[:, :1].mean(2, keepdim=True), x[:, 1:]], 1)
    balance = (1.0 / (3.0 * (2.0 * degree + 1.0))).to(x.dtype)[None, :, None]
    inv = torch.rsqrt((x * x * balance).sum(1, keepdim=True).mean(2, keepdim=True) + 1e-5)
    y = x * inv * w[f"{p}.affine_weight"][degree][None]
    return torch.cat([y[:, :1] + w[f"{p}.affine_bias"], y[:, 1:]], 1)


def _so3_64(x, w, p):
    W = w[f"{p}.weight"]
    y = torch.cat([x[:, l * l:(l + 1) ** 2] @ W[l].T for l in range(3)], 1)
    return torch.cat([y[:, :1] + w[f"{p}.bias"], y[:, 1:]], 1)


def _uma64(i, stress):
    w = {k: v.to(DEV, torch.float64) for k, v in i["w"].items()}
    cfg, Z = i["cfg"], i["Z"].to(DEV)
    src, tgt = i["edges"]
    N, C, H = len(Z), cfg["sphere_channels"], cfg["hidden_channels"]
    pos = i["pos"].double().requires_grad_(True)
    strain = torch.zeros(3, 3, device=DEV, dtype=torch.float64, requires_grad=True)
    vec = pos[src] - pos[tgt]
    if i["shift"] is not None:
        vec = vec + i["shift"].double()
    vec = vec + vec @ (0.5 * (strain + strain.T))
    E = vec.shape[0]
    rot = _wigner64(vec, [w[f"Jd_{l}"] for l in range(3)])
    dist = vec.norm(dim=1)
    off = i["host"]["gauss_offset"].to(DEV, torch.float64)
    x_edge = torch.cat([torch.exp(float(i["host"]["gauss_coeff"][0]) * (dist[:, None] - off) ** 2),
                        w["source_embedding.weight"][Z[src]],
                        w["target_embedding.weight"][Z[tgt]]], 1)
    q = dist / cfg["cutoff"]
    env = torch.where(q < 1, 1 + q ** 5 * (-21.0 + q * (35.0 - 15.0 * q)), 0.0)[:, None, None]

    def scatter(rows):
        return rows.new_zeros(N, 9, C).index_add(0, tgt, rows)

    se = i["sys_emb"].double()[:, None]
    zero = torch.zeros(N, 8, C, device=DEV, dtype=torch.float64)
    x = torch.cat([w["sphere_embedding.weight"][Z][:, None] + se, zero], 1)
    deg = _radial64(x_edge, w, "edge_degree_embedding.rad_func").view(E, 3, C)
    x = x + scatter(rot[:, :3].transpose(1, 2) @ deg * env / 5.0)
    prime_degree, natural_degree = [0, 1, 0, 1, 0, 1, 1, 1], [0, 0, 0, 1, 1, 1, 1, 1]
    for b in range(cfg["num_layers"]):
        p = f"blocks.{b}"
        n = _rms_sh64(x, w, f"{p}.norm_1")
        n = torch.cat([n[:, :1] + se, n[:, 1:]], 1)
        m = rot @ torch.cat([n[src], n[tgt]], 2)
        r = _radial64(x_edge, w, f"{p}.edge_wise.so2_conv_1.rad_func").view(E, 6, 2 * C)
        m, gating = _so2_64(m * r[:, [0, 1, 2, 3, 4, 3, 4, 5, 5]], w, f"{p}.edge_wise.so2_conv_1")
        g = torch.sigmoid(gating).view(E, 2, H)[:, prime_degree]
        m = torch.cat([F.silu(m[:, :1]), m[:, 1:] * g], 1)
        m, _ = _so2_64(m, w, f"{p}.edge_wise.so2_conv_2")
        x = x + scatter(rot.transpose(1, 2) @ (m * env))
        n = _rms_sh64(x, w, f"{p}.norm_2")
        g = torch.sigmoid(F.silu(_lin(n[:, 0], w, f"{p}.atom_wise.scalar_mlp.0")))
        h = _so3_64(n, w, f"{p}.atom_wise.so3_linear_1")
        h = torch.cat([F.silu(h[:, :1]), h[:, 1:] * g.view(N, 2, H)[:, natural_degree]], 1)
        x = x + _so3_64(h, w, f"{p}.atom_wise.so3_linear_2")
    h = _rms_sh64(x, w, "norm")[:, 0]
    h = F.silu(_lin(F.silu(_lin(h, w, "energy_block.0")), w, "energy_block.2"))
    energy = _lin(h, w, "energy_block.4").sum()
    g_pos, g_strain = torch.autograd.grad(energy, [pos, strain])
    out = dict(energy=energy.detach().reshape(1), forces=-g_pos)
    return dict(out, virial=g_strain.reshape(9)) if stress else out


def _mlp64(x, w, p):
    h = F.silu(_lin(x, w, f"{p}.mlp.NN-0"))
    h = _lin(F.silu(_lin(h, w, f"{p}.mlp.NN-1")), w, f"{p}.mlp.NN-2")
    return h * torch.rsqrt((h * h).mean(1, keepdim=True) + 1e-6) * w[f"{p}.layer_norm.weight"]


def _layer64(nodes, edges, cut, send, recv, w, p):
    ra = torch.sigmoid(_lin(edges, w, f"{p}._receive_attn")) * cut
    sa = torch.sigmoid(_lin(edges, w, f"{p}._send_attn")) * cut
    ue = _mlp64(torch.cat([edges, nodes[send], nodes[recv]], 1), w, f"{p}._edge_mlp")
    sent = torch.zeros_like(nodes).index_add(0, send, ue * sa)
    got = torch.zeros_like(nodes).index_add(0, recv, ue * ra)
    return nodes + _mlp64(torch.cat([nodes, got, sent], 1), w, f"{p}._node_mlp"), edges + ue


def _harmonics64(u):
    """Real spherical harmonics to l = 3, each degree scaled by sqrt(2 l + 1)."""
    x, y, z = u.T
    r3, p = math.sqrt(3.0), x * x + z * z
    a, d = r3 * x * z, 0.5 * r3 * (z * z - x * x)
    s1, s2 = math.sqrt(5.0 / 6.0), math.sqrt(3.0 / 8.0)
    deg = [[torch.ones_like(x)], [x, y, z],
           [a, r3 * x * y, y * y - 0.5 * p, r3 * y * z, d],
           [s1 * (a * z + d * x), math.sqrt(5.0) * a * y, s2 * (4 * y * y - p) * x,
            0.5 * y * (2 * y * y - 3 * p), s2 * (4 * y * y - p) * z, math.sqrt(5.0) * d * y,
            s1 * (d * z - a * x)]]
    return torch.stack([math.sqrt(2 * l + 1) * c for l, cs in enumerate(deg) for c in cs], 1)


def _orb64(i):
    w = {k: v.to(DEV, torch.float64) for k, v in i["w"].items()}
    cfg, send, recv = i["cfg"], i["send"], i["recv"]
    pos = i["pos"].double().requires_grad_(True)
    vec = pos[recv] - pos[send]
    r = vec.norm(dim=1, keepdim=True)
    q = r / ORB_CUTOFF
    cut = (1 - 15 * q ** 4 + 24 * q ** 5 - 10 * q ** 6) * (r < ORB_CUTOFF)
    k = torch.arange(1, cfg["num_bases"] + 1, device=DEV) * (math.pi / ORB_CUTOFF)
    bessel = math.sqrt(2.0 / ORB_CUTOFF) * torch.sin(r * k) / r
    feat = cut * (bessel[:, :, None] * _harmonics64(vec / r)[:, None]).reshape(len(send), -1)
    nodes = _mlp64(w["atom_emb.embeddings.weight"][i["Z"].to(DEV)], w, "_encoder._node_fn")
    edges = _mlp64(feat, w, "_encoder._edge_fn")
    for l in range(cfg["num_message_passing_steps"]):
        nodes, edges = _layer64(nodes, edges, cut, send, recv, w, f"gnn_stacks.{l}")
    natoms = torch.tensor(i["natoms"], device=DEV)
    system = torch.repeat_interleave(torch.arange(len(natoms), device=DEV), natoms)
    mean = nodes.new_zeros(len(natoms), nodes.shape[1]).index_add(0, system, nodes)
    raw = _lin(F.silu(_lin(mean / natoms[:, None], w, "energy_head.mlp.NN-0")), w,
               "energy_head.mlp.NN-1")
    (g,) = torch.autograd.grad(raw.sum(), pos)
    return dict(energies=raw.detach(), forces=-g)


def exact(case, seed):
    kind = case["kind"]
    if kind == "neighbors":
        return None
    if kind == "uma":
        return _uma64(_uma_inputs(case, seed), case["stress"])
    if kind == "orb":
        return _orb64(_orb_inputs(case, seed))
    if kind == "orb_layer":
        i = _layer_inputs(case, seed)
        w = {k: v.double() for k, v in i["w"].items()}
        leaf = [i[k].double().requires_grad_(True) for k in ("nodes", "edges", "cut")]
        n, e = _layer64(*leaf, i["send"], i["recv"], w, "l")
        gn, ge, gc = torch.autograd.grad([n, e], leaf, [i["g_nodes"].double(),
                                                        i["g_edges"].double()])
        return dict(nodes=n.detach(), edges=e.detach(), g_nodes=gn, g_edges=ge, g_cut=gc)
    if kind == "mlp":
        i = _mlp_inputs(case, seed)
        w = {k: v.double() for k, v in i["w"].items()}
        x = i["x"].double().requires_grad_(True)
        y = _mlp64(x, w, "m")
        (g,) = torch.autograd.grad(y, x, i["g"].double())
        return dict(y=y.detach(), g_x=g)
    if kind == "edgewise":
        i = _edgewise_inputs(case, seed)
        w = {k: v.to(DEV, torch.float64) for k, v in i["w"].items()}
        ev = i["ev"].double().requires_grad_(True)
        rot = _wigner64(ev, i["jd"])
        m, _ = _so2_64(rot @ i["x"].double()[i["src"]], w, "c2")
        out = torch.zeros(case["nodes"], 9, i["C"], device=DEV, dtype=torch.float64)
        out = out.index_add(0, i["tgt"], rot.transpose(1, 2) @ m)
        (g,) = torch.autograd.grad(out, ev, i["g"].double())
        return dict(out=out.detach(), g_ev=g)
    i = _rotation_inputs(case, seed)
    E, W = case["edges"], case["width"]
    rot, x, g = i["wig"].double(), i["x"].double().view(E, 9, W), i["g"].double().view(E, 9, W)
    y = rot @ x
    node = y.new_zeros(case["nodes"], 9, W).index_add(0, i["tgt"], y)
    ii, jj = ((i["wig"].abs().amax(0) > 1e-6).nonzero()).T
    return dict(y=y.view(E, -1), g_x=(rot.transpose(1, 2) @ g).view(E, -1),
                g_coef=(g @ x.transpose(1, 2))[:, ii, jj], node=node.view(case["nodes"], -1))
