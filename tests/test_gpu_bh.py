"""GPU parity of the fused BH gradient (holotomocupy_amd.bh) against the FP64
oracle cascade and the per-operator cascade.  Tolerances as for the cascade:
relative L2 <= 1e-5 (object, probe), 1e-4 (positions, objective)."""
import numpy as np
import pytest
import torch

from test_gpu_rec import make_problem, dev, lst, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("geom", [(32, 40, 3, 4), (64, 48, 2, 3), (16, 24, 4, 5)])
def test_fused_gradient_vs_oracle(gpu, real, geom):
    n, nobj, ndist, B = geom
    print(f"[case] fused gradient n={n} nobj={nobj} ndist={ndist} B={B} real={real}", flush=True)
    rec, cas, x, v, w, d = make_problem(real, n=n, nobj=nobj, ndist=ndist, B=B, seed=20 + n)
    xd, dd = dev(x), torch.from_numpy(d).cuda()
    grads = {"prb": torch.zeros_like(xd["prb"]), "proj": torch.empty_like(xd["proj"]),
             "pos": torch.empty_like(xd["pos"])}
    obj = torch.zeros(1, dtype=torch.float64, device="cuda")
    rec.gradients_fused(xd, grads, dd, objective=obj)
    gprb, gproj, gpos = cas.gradients(*lst(x), d)
    assert rel(grads["prb"], gprb) < 1e-5
    assert rel(grads["proj"], gproj) < 1e-5
    assert rel(grads["pos"], gpos) < 1e-4
    assert obj.item() / rec.data_size == pytest.approx(cas.objective(*lst(x), d), rel=1e-4)
    # the per-operator cascade gives the same gradient
    g2 = {"prb": torch.zeros_like(xd["prb"]), "proj": torch.empty_like(xd["proj"]),
          "pos": torch.empty_like(xd["pos"])}
    rec.gradients_cascade(xd, g2, dd)
    assert rel(grads["proj"], g2["proj"].cpu().numpy()) < 1e-5
    assert rel(grads["prb"], g2["prb"].cpu().numpy()) < 1e-5


def test_fused_gradient_deterministic_and_accumulates(gpu):
    print("[case] fused gradient determinism", flush=True)
    rec, cas, x, v, w, d = make_problem(False, seed=31)
    xd, dd = dev(x), torch.from_numpy(d).cuda()
    outs = []
    for _ in range(2):
        g = {"prb": torch.zeros_like(xd["prb"]), "proj": torch.empty_like(xd["proj"]),
             "pos": torch.empty_like(xd["pos"])}
        rec.gradients_fused(xd, g, dd)
        outs.append(g)
    for k in outs[0]:
        assert torch.equal(outs[0][k], outs[1][k]), k
    # grads['prb'] is accumulated (the reference's +=, rec_mpi.py:347)
    g = {"prb": outs[0]["prb"].clone(), "proj": torch.empty_like(xd["proj"]), "pos": torch.empty_like(xd["pos"])}
    rec.gradients_fused(xd, g, dd)
    assert torch.allclose(g["prb"], 2 * outs[0]["prb"], rtol=1e-6, atol=1e-12)


def test_fused_gradient_two_probes(gpu):
    """Angles of two requests with different probes in one launch: each probe
    gradient equals the one computed separately."""
    print("[case] fused gradient two probes", flush=True)
    from holotomocupy_amd.bh import BHGradient
    rec, cas, x, v, w, d = make_problem(False, seed=41, B=4)
    bh = BHGradient(rec)
    xd, dd = dev(x), torch.from_numpy(d).cuda()
    B = xd["proj"].shape[0]
    prb2 = torch.stack([xd["prb"], xd["prb"] * (0.8 + 0.1j)])        # [2, ndist, nz, n]
    pidx = torch.tensor([0, 0, 1, 1], dtype=torch.int32, device="cuda")
    mag = rec.eff_demagnifications[:B].contiguous()
    gproj = torch.empty_like(xd["proj"])
    gpos = torch.empty_like(xd["pos"])
    gprb = torch.zeros_like(prb2)
    s, rp = bh.scales(B)
    bh(prb2, xd["proj"], xd["pos"], dd, mag, gproj, gpos, gprb, accumulate_prb=False,
       probe_index=pidx, scales=s, rho_prb=rp.repeat(2))
    for p, sl in ((0, slice(0, 2)), (1, slice(2, 4))):
        gp = torch.empty_like(xd["proj"][sl])
        gq = torch.empty_like(xd["pos"][sl])
        gr = torch.zeros_like(xd["prb"])
        bh(prb2[p].contiguous(), xd["proj"][sl].contiguous(), xd["pos"][sl].contiguous(), dd[sl].contiguous(),
           mag[sl].contiguous(), gp, gq, gr, accumulate_prb=False, scales=s[sl].contiguous(), rho_prb=rp)
        assert torch.allclose(gprb[p], gr, rtol=1e-5, atol=1e-7 * gr.abs().max().item())
        assert torch.allclose(gproj[sl], gp, rtol=1e-5, atol=1e-7 * gp.abs().max().item())
        assert torch.allclose(gpos[sl], gq, rtol=1e-5, atol=1e-7 * gq.abs().max().item())


def test_fused_gradient_address_table_equals_packed(gpu):
    """htamd_bh_gradient_tab (each angle's projection, data and object
    gradient and each probe slot's probe and probe gradient addressed through
    a table, as the serving loop calls it) equals htamd_bh_gradient on the
    same inputs packed, bit for bit: two requests of 3 and 1 angles with
    different probes, their arrays in separate allocations."""
    print("[case] fused gradient address table", flush=True)
    from holotomocupy_amd.bh import BHGradient
    rec, cas, x, v, w, d = make_problem(False, seed=43, B=4)
    bh = BHGradient(rec)
    xd, dd = dev(x), torch.from_numpy(d).cuda()
    B = 4
    prb2 = torch.stack([xd["prb"], xd["prb"] * (0.8 + 0.1j)])
    pidx = torch.tensor([0, 0, 0, 1], dtype=torch.int32, device="cuda")
    mag = rec.eff_demagnifications[:B].contiguous()
    s, rp = bh.scales(B)
    rho2 = rp.repeat(2)
    gproj, gpos, gprb = torch.empty_like(xd["proj"]), torch.empty_like(xd["pos"]), torch.empty_like(prb2)
    bh(prb2, xd["proj"], xd["pos"], dd, mag, gproj, gpos, gprb, accumulate_prb=False, probe_index=pidx, scales=s,
       rho_prb=rho2)
    # per-request copies in their own allocations
    reqs = [(slice(0, 3), 0), (slice(3, 4), 1)]
    proj_r = [xd["proj"][sl].clone() for sl, _ in reqs]
    data_r = [dd[sl].clone() for sl, _ in reqs]
    prb_r = [prb2[p].clone() for _, p in reqs]
    gproj_r = [torch.full_like(t, float("nan")) for t in proj_r]
    gprb_r = [torch.full_like(t, float("nan")) for t in prb_r]
    cols = [[], [], [], [], []]
    for k in range(2):
        for t, c in ((proj_r[k], 0), (data_r[k], 1), (gproj_r[k], 2)):
            step = t[0].numel() * t.element_size()
            cols[c].extend(t.data_ptr() + i * step for i in range(t.shape[0]))
        cols[3].append(prb_r[k].data_ptr())
        cols[4].append(gprb_r[k].data_ptr())
    tab = torch.tensor(sum(cols, []), dtype=torch.int64, device="cuda")
    gpos_t = torch.empty_like(gpos)
    ws = torch.empty(bh.workspace_bytes(B), dtype=torch.uint8, device="cuda")
    bh.call_tab(tab, B, 2, xd["pos"], mag, pidx, s, rho2, gpos_t, ws)
    torch.cuda.synchronize()
    assert torch.equal(gpos_t, gpos)
    for k, (sl, p) in enumerate(reqs):
        assert torch.equal(gproj_r[k], gproj[sl]), k
        assert torch.equal(gprb_r[k], gprb[p]), k


def test_fused_gradient_nonsquare_detector(gpu):
    """nz != n and magnified shifts."""
    print("[case] fused gradient non-square", flush=True)
    from types import SimpleNamespace
    from holotomocupy_amd.rec import Rec, physics
    from oracle import cascade as oc
    from oracle import propagation as op
    from oracle import shift as osh
    rng = np.random.default_rng(5)
    n, nz, nobj, nzobj, ndist, B = 64, 32, 72, 40, 2, 3
    args = SimpleNamespace(energy=17.1, detector_pixelsize=1.4760147601476e-6 * 16, focustodetectordistance=1.217,
                           z1=np.array([5.110, 6.879]) * 1e-3, ndist=ndist, ntheta=B, nz=nz, n=n, nzobj=nzobj,
                           nobj=nobj, obj_dtype="complex64", rho=[1, 0.5, 0.2])
    rec = Rec(args)
    ph = physics(args.energy, args.z1, args.focustodetectordistance, args.detector_pixelsize)
    cas = oc.Cascade(op.Propagation(n, nz, B, ndist, ph.wavelength, ph.voxelsize, ph.distance),
                     osh.Shift(n, nobj, nz, nzobj), ndist, nz, n, nzobj, nobj, rec.data_size,
                     np.tile(1 / ph.norm_magnifications, (B, 1)), rho=args.rho)
    prb = (1 + 0.1 * (rng.standard_normal((ndist, nz, n)) + 1j * rng.standard_normal((ndist, nz, n)))).astype(np.complex64)
    proj = (0.3 * (rng.standard_normal((B, nzobj, nobj)) + 1j * rng.standard_normal((B, nzobj, nobj)))).astype(np.complex64)
    pos = rng.uniform(-3, 3, (B, ndist, 2)).astype(np.float32)
    d = (np.abs(cas.forward(prb.astype(np.complex128), proj.astype(np.complex128), pos.astype(np.float64))) * 1.1).astype(np.float32)
    x = {"prb": prb, "proj": proj, "pos": pos}
    xd, dd = dev(x), torch.from_numpy(d).cuda()
    g = {"prb": torch.zeros_like(xd["prb"]), "proj": torch.empty_like(xd["proj"]), "pos": torch.empty_like(xd["pos"])}
    rec.gradients_fused(xd, g, dd)
    gprb, gproj, gpos = cas.gradients(*lst(x), d)
    assert rel(g["prb"], gprb) < 1e-5
    assert rel(g["proj"], gproj) < 1e-5
    assert rel(g["pos"], gpos) < 1e-4


@pytest.mark.parametrize("real", [False, True])
def test_fused_gradient_magnification_below_one(gpu, real):
    """A negative shrink puts some magnifications below 1 (wider candidate
    brackets in the gather-form Sadj); the rest stay at or above 1."""
    print(f"[case] fused gradient with magnifications below one real={real}", flush=True)
    B, nd = 3, 3
    shrink = np.array([[-0.3, 0.0, 0.1], [-0.15, -0.4, 0.0], [0.2, -0.05, -0.35]], dtype=np.float64)
    rec, cas, x, v, w, d = make_problem(real, n=32, nobj=40, ndist=nd, B=B, seed=31, shrink=shrink)
    assert float(rec.eff_demagnifications.min()) < 1.0 <= float(rec.eff_demagnifications.max())
    xd, dd = dev(x), torch.from_numpy(d).cuda()
    grads = {"prb": torch.zeros_like(xd["prb"]), "proj": torch.empty_like(xd["proj"]),
             "pos": torch.empty_like(xd["pos"])}
    rec.gradients_fused(xd, grads, dd)
    gprb, gproj, gpos = cas.gradients(*lst(x), d)
    assert rel(grads["prb"], gprb) < 1e-5
    assert rel(grads["proj"], gproj) < 1e-5
    assert rel(grads["pos"], gpos) < 1e-4


def test_fused_gradient_bench_size_properties(gpu):
    """Detector 2048^2, object plane 1024^2, 4 distances, 4 angles (the bench's
    shapes): the fused gradient agrees with the per-operator cascade (a second,
    independent implementation) to the operator bar, is deterministic, and its
    per-angle outputs do not depend on how the angles are split across
    launches (the probe gradient, a sum over angles, to 1e-6)."""
    print("[case] fused gradient 2048^2 properties", flush=True)
    from types import SimpleNamespace
    from holotomocupy_amd import phantom
    from holotomocupy_amd.rec import Rec
    n, nobj, nd, B = 2048, 1024, 4, 4
    rng = np.random.default_rng(19)
    args = SimpleNamespace(energy=17.1, detector_pixelsize=1.4760147601476e-6 * 2, focustodetectordistance=1.217,
                           z1=np.array([5.110, 5.464, 6.879, 9.817]) * 1e-3, ndist=nd, ntheta=B, nz=n, n=n,
                           nzobj=nobj, nobj=nobj, obj_dtype="complex64", rho=[1.0, 0.05, 0.02])
    rec = Rec(args)
    x = {"prb": torch.from_numpy(phantom.probe(rng, nd, n, n)).cuda(),
         "proj": torch.from_numpy(phantom.projections(rng, B, nobj, nobj)).cuda(),
         "pos": torch.from_numpy(phantom.positions(rng, B, nd)).cuda()}
    with torch.no_grad():
        data = (rec.forward(x).abs() * (1 + 0.05 * torch.randn((B, nd, n, n), device="cuda"))).float().contiguous()

    def zeros():
        return {"prb": torch.zeros_like(x["prb"]), "proj": torch.empty_like(x["proj"]),
                "pos": torch.empty_like(x["pos"])}

    g1, g2, gc = zeros(), zeros(), zeros()
    rec.gradients_fused(x, g1, data)
    rec.gradients_fused(x, g2, data)
    for k in g1:
        assert torch.equal(g1[k], g2[k]), k
    rec.gradients_cascade(x, gc, data)
    print({k: rel(g1[k], gc[k].cpu().numpy()) for k in g1}, flush=True)
    assert rel(g1["prb"], gc["prb"].cpu().numpy()) < 1e-5
    assert rel(g1["proj"], gc["proj"].cpu().numpy()) < 1e-5
    assert rel(g1["pos"], gc["pos"].cpu().numpy()) < 1e-4
    gs = zeros()
    for st in (0, 2):
        part = {"prb": x["prb"], "proj": x["proj"][st:st + 2], "pos": x["pos"][st:st + 2]}
        out = {"prb": gs["prb"], "proj": gs["proj"][st:st + 2], "pos": gs["pos"][st:st + 2]}
        rec.gradients_fused(part, out, data[st:st + 2], st=st)
    assert torch.equal(gs["proj"], g1["proj"]) and torch.equal(gs["pos"], g1["pos"])
    assert rel(gs["prb"], g1["prb"].cpu().numpy()) < 1e-6


@pytest.mark.parametrize("n,ndist,runs,real", [(64, 2, (1, 4, 5, 9, 3), False), (128, 3, (70, 1, 8), False),
                                               (32, 1, (2, 5), True), (256, 2, (3, 5), False), (256, 1, (4, 2), True),
                                               (512, 1, (1, 5), False), (512, 2, (2, 3), True),
                                               (1024, 1, (2, 5), False), (1024, 1, (1, 4), True)])
def test_probe_runs_alone_and_together(gpu, n, ndist, runs, real):
    """Groups of angles whose probe-gradient sums are formed apart and added:
    runs shorter than, equal to and longer than a group (and than the 64
    angles that one look back covers) give the same bits alone and in one
    launch, and the per-operator cascade's gradient."""
    print(f"[case] probe runs n={n} ndist={ndist} runs={runs} real={real}", flush=True)
    from holotomocupy_amd.bh import BHGradient
    B = sum(runs)
    rec, cas, x, v, w, d = make_problem(real, n=n, nobj=48, ndist=ndist, B=B, seed=61)
    xd, dd = dev(x), torch.from_numpy(d).cuda()
    bh = BHGradient(rec)
    mag = rec.eff_demagnifications[:B].contiguous()
    k = len(runs)
    prb = torch.stack([xd["prb"] * (1 + 0.1 * i) for i in range(k)]).contiguous()
    pidx = torch.tensor(sum(([i] * m for i, m in enumerate(runs)), []), dtype=torch.int32, device="cuda")
    s, rp = bh.scales(B)
    gproj, gpos, gprb = torch.empty_like(xd["proj"]), torch.empty_like(xd["pos"]), torch.empty_like(prb)
    bh(prb, xd["proj"], xd["pos"], dd, mag, gproj, gpos, gprb, accumulate_prb=False, probe_index=pidx, scales=s,
       rho_prb=rp.repeat(k))
    st = 0
    for i, m in enumerate(runs):
        sl = slice(st, st + m)
        one = {"prb": torch.zeros_like(xd["prb"]), "proj": torch.empty_like(gproj[sl]),
               "pos": torch.empty_like(gpos[sl])}
        var = {"prb": prb[i], "proj": xd["proj"][sl], "pos": xd["pos"][sl]}
        rec.gradients_fused(var, one, dd[sl], st=st)
        assert torch.equal(one["prb"], gprb[i]), i
        assert torch.equal(one["proj"], gproj[sl]) and torch.equal(one["pos"], gpos[sl]), i
        ref = {q: torch.zeros_like(t) for q, t in one.items()}
        rec.gradients_cascade(var, ref, dd[sl], st=st)
        assert rel(one["prb"], ref["prb"].cpu().numpy()) < 1e-5
        st += m


def test_angles_split_over_workgroups_with_a_remainder(gpu):
    """More angles than the row passes have workgroups for: each workgroup
    takes two, the last one one."""
    print("[case] row passes with two angles per workgroup", flush=True)
    B = 35
    rec, cas, x, v, w, d = make_problem(False, n=256, nobj=48, ndist=4, B=B, seed=62)
    xd, yd, dd = dev(x), dev(v), torch.from_numpy(d).cuda()
    g, ref = ({q: torch.zeros_like(t) for q, t in xd.items()} for _ in range(2))
    rec.gradients_fused(xd, g, dd)
    rec.gradients_cascade(xd, ref, dd)
    assert rel(g["prb"], ref["prb"].cpu().numpy()) < 1e-5
    assert rel(g["proj"], ref["proj"].cpu().numpy()) < 1e-5
    assert rel(g["pos"], ref["pos"].cpu().numpy()) < 1e-4
    for z in (yd, dev(w)):
        h = rec.hessian_fused(xd, yd, yd if z is yd else z, dd).item()
        assert h == pytest.approx(rec.hessian_cascade(xd, yd, yd if z is yd else z, dd), rel=1e-4)


def test_tab_call_with_scattered_probes(gpu):
    """A batch by address table whose angles take their probes in turn: more
    runs of equal probes than probes (only the probe gradients ask for one run
    each).  Every angle's object and position gradient is that of the angle
    alone, and no output is left from before."""
    print("[case] address table, probes in turn", flush=True)
    from holotomocupy_amd.bh import BHGradient
    B, k = 13, 2
    rec, cas, x, v, w, d = make_problem(False, n=64, nobj=48, ndist=2, B=B, seed=63)
    bh = BHGradient(rec)
    xd, dd = dev(x), torch.from_numpy(d).cuda()
    prb = [xd["prb"].clone(), xd["prb"] * (0.8 + 0.1j)]
    gprb = [torch.empty_like(p) for p in prb]
    gproj, gpos = torch.full_like(xd["proj"], float("nan")), torch.full_like(xd["pos"], float("nan"))
    pidx = torch.arange(B, dtype=torch.int32, device="cuda") % k
    mag = rec.eff_demagnifications[:B].contiguous()
    s, rp = bh.scales(B)
    tab = torch.tensor([t[b].data_ptr() for t in (xd["proj"], dd, gproj) for b in range(B)]
                       + [t.data_ptr() for t in prb + gprb], dtype=torch.int64, device="cuda")
    ws = torch.full((bh.workspace_bytes(B),), 0xff, dtype=torch.uint8, device="cuda")
    bh.call_tab(tab, B, k, xd["pos"], mag, pidx, s, rp.repeat(k), gpos, ws)
    for b in range(B):
        one = {"prb": torch.zeros_like(prb[0]), "proj": torch.empty_like(gproj[b:b + 1]),
               "pos": torch.empty_like(gpos[b:b + 1])}
        rec.gradients_fused({"prb": prb[b % k], "proj": xd["proj"][b:b + 1], "pos": xd["pos"][b:b + 1]}, one,
                            dd[b:b + 1], st=b)
        assert torch.equal(one["proj"][0], gproj[b]) and torch.equal(one["pos"][0], gpos[b]), b


@pytest.mark.parametrize("n,nobj,ndist,B", [(256, 256, 2, 48), (256, 128, 2, 48), (128, 128, 3, 9), (64, 48, 2, 300),
                                            (512, 64, 2, 500)])
def test_gradient_workspace_holds_no_second_work_field(gpu, n, nobj, ndist, B):
    """The group sums of the split row pass take the room of the object gradient,
    which is formed after them, and beyond it at most two slots to five angles
    (at least eight) where the work field has one per angle, nor more than a
    window of 8192 workgroups needs."""
    print(f"[case] gradient workspace n={n} nobj={nobj} ndist={ndist} B={B}", flush=True)
    from holotomocupy_amd.bh import BHGradient
    rec = make_problem(False, n=n, nobj=nobj, ndist=ndist, B=1, seed=64)[0]
    obj, slot = B * nobj * nobj * 8, ndist * n * n * 8
    base = 2 * obj + B * slot + B * ndist * n * 16  # coefficients, object gradient, work field, partial sums
    groups = min(B, max(8, min(-(-2 * B // 5), -(-8192 * 2048 // (ndist * n * n)))))
    assert BHGradient(rec).workspace_bytes(B) <= base + max(0, groups * slot - obj) + 8 * 256


@pytest.mark.parametrize("accumulate,nobj", [(False, 32), (True, 32), (False, 160)])
def test_probe_runs_over_several_windows(gpu, accumulate, nobj):
    """More groups of angles than their sums have slots (18 of 43 angles, 21
    groups): a run that begins in one window of groups and ends in the next, and
    runs of one angle on both sides, give the bits of each run alone.  Also with
    object rows that are too wide to be staged (and room for all groups)."""
    print(f"[case] probe runs over windows accumulate={accumulate} nobj={nobj}", flush=True)
    from holotomocupy_amd.bh import BHGradient
    runs = (1,) * 10 + (30,) + (1,) * 3
    B, k = sum(runs), len(runs)
    rec, cas, x, v, w, d = make_problem(False, n=64, nobj=nobj, ndist=2, B=B, seed=65)
    xd, dd = dev(x), torch.from_numpy(d).cuda()
    bh = BHGradient(rec)
    mag = rec.eff_demagnifications[:B].contiguous()
    prb = torch.stack([xd["prb"] * (1 + 0.1 * i) for i in range(k)]).contiguous()
    pidx = torch.tensor(sum(([i] * m for i, m in enumerate(runs)), []), dtype=torch.int32, device="cuda")
    s, rp = bh.scales(B)
    before = 0.01 * prb.flip(0)
    gproj, gpos, gprb = torch.empty_like(xd["proj"]), torch.empty_like(xd["pos"]), before.clone()
    bh(prb, xd["proj"], xd["pos"], dd, mag, gproj, gpos, gprb, accumulate_prb=accumulate, probe_index=pidx, scales=s,
       rho_prb=rp.repeat(k))
    tprb = torch.empty_like(prb) if not accumulate else before.clone()
    tproj, tpos = torch.empty_like(gproj), torch.empty_like(gpos)
    tab = torch.tensor([t[b].data_ptr() for t in (xd["proj"], dd, tproj) for b in range(B)]
                       + [t[i].data_ptr() for t in (prb, tprb) for i in range(k)], dtype=torch.int64, device="cuda")
    ws = torch.full((bh.workspace_bytes(B),), 0xff, dtype=torch.uint8, device="cuda")
    bh.call_tab(tab, B, k, xd["pos"], mag, pidx, s, rp.repeat(k), tpos, ws, accumulate_prb=accumulate)
    assert torch.equal(tproj, gproj) and torch.equal(tpos, gpos) and torch.equal(tprb, gprb)
    st = 0
    for i, m in enumerate(runs):
        sl = slice(st, st + m)
        one = {"prb": before[i].clone() if accumulate else torch.zeros_like(prb[i]),
               "proj": torch.empty_like(gproj[sl]), "pos": torch.empty_like(gpos[sl])}
        rec.gradients_fused({"prb": prb[i], "proj": xd["proj"][sl], "pos": xd["pos"][sl]}, one, dd[sl], st=st)
        assert torch.equal(one["prb"], gprb[i]), i
        assert torch.equal(one["proj"], gproj[sl]) and torch.equal(one["pos"], gpos[sl]), i
        st += m


def test_one_run_over_two_windows(gpu):
    """80 angles of one probe at 1024^2: 20 groups in windows of 15.  Object and
    position gradients are those of the angles by fives, the probe gradient their
    sum (up to its rounding)."""
    print("[case] one run over two windows", flush=True)
    from types import SimpleNamespace
    from holotomocupy_amd.rec import Rec
    n, nobj, B = 1024, 64, 80
    rec = Rec(SimpleNamespace(energy=17.1, detector_pixelsize=1.4760147601476e-6 * 4, focustodetectordistance=1.217,
                              z1=np.array([5.110]) * 1e-3, ndist=1, ntheta=B, nz=n, n=n, nzobj=nobj, nobj=nobj,
                              obj_dtype="complex64", rho=[1, 0.5, 0.2]))
    g = torch.Generator(device="cuda").manual_seed(66)
    c = lambda *s: torch.randn(s, dtype=torch.complex64, device="cuda", generator=g)  # noqa: E731
    x = {"prb": 1 + 0.1 * c(1, n, n), "proj": 0.1 * c(B, nobj, nobj),
         "pos": torch.randn((B, 1, 2), device="cuda", generator=g)}
    d = 1 + 0.1 * torch.rand((B, 1, n, n), device="cuda", generator=g)
    one = {k: torch.zeros_like(t) for k, t in x.items()}
    rec.gradients_fused(x, one, d)
    part = {k: torch.zeros_like(t) for k, t in x.items()}
    for st in range(0, B, 5):
        sl = slice(st, st + 5)
        rec.gradients_fused({"prb": x["prb"], "proj": x["proj"][sl], "pos": x["pos"][sl]},
                            {"prb": part["prb"], "proj": part["proj"][sl], "pos": part["pos"][sl]}, d[sl], st=st)
    assert torch.equal(one["proj"], part["proj"]) and torch.equal(one["pos"], part["pos"])
    assert rel(one["prb"], part["prb"].cpu().numpy()) < 1e-6
