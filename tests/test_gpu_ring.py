"""The kernels with a compile-time ring length against the runtime-size kernels and the oracle.

The plain search of an FFT-friendly ring length runs two-pass transforms (k_corr_ring: per-pair and
staged-reference variants, shells split over work-groups where the search is small, k_ring_finish).
PFTCC_GENERIC=1 keeps a handle on the runtime-size kernels (k_corr_generic), which take every form.
Tolerance: both sides are FP32 transforms whose error against FP64 is within 1e-5 of the peak (the
bound of the other FP32 tests), so vectors agree within 2e-5 of the peak.
"""
import numpy as np
import pytest

from cases import make_case
from gpu_helpers import peak_rel_err, say, to_lib
from pftcc import SRCH_SHC3D

pytestmark = pytest.mark.gpu

FP32_TOL = 1e-5

# one length of each radix pair and parity class: B odd or even, 3, 5, 7, 11 and 13 in either pass,
# A with and without a factor 4, the Good-Thomas and the general form, the smallest and largest
LENGTHS = [16, 24, 36, 48, 52, 66, 70, 100, 130, 150, 162, 182, 220, 256, 308, 324, 338, 364, 400, 450, 462, 486, 500,
           512, 546, 588, 600]


def both(monkeypatch, pf, cps):
    monkeypatch.setenv("PFTCC_GENERIC", "1")
    gen = to_lib(pf, cps)
    monkeypatch.delenv("PFTCC_GENERIC")
    return to_lib(pf, cps), gen


def shift_list(ns):
    rng = np.random.default_rng(ns)
    return rng.uniform(-2.5, 2.5, (ns, 2)).astype(np.float32) if ns else None


FORMS = [
    dict(),
    dict(ctf=False, kstop=5),
    dict(match_filt=True),
    dict(euclid=True),
]


@pytest.mark.parametrize("n", LENGTHS)
def test_ring_kernels_equal_the_generic_kernel(n, monkeypatch):
    for form in FORMS:
        kw = dict(ctf=True, kstop=7)
        kw.update(form)
        pf, cps = make_case(seed=n, n=n, kfrom=2, kto=8, nrefs=3, nptcls=5, ldim=max(40, n), eo_mixed=True, **kw)
        lib, gen = both(monkeypatch, pf, cps)
        ids = np.array([2, 5, 1, 3, 4])
        for ns in (0, 1, 5, 41):                # 41 shifts: the staged-reference variant (CC, no filter)
            say(f"ring kernels: n={n} {form} ns={ns}")
            tile, staged = lib.get_corr_tile(ns)
            plain = not form.get("match_filt") and not form.get("euclid")
            assert tile > 0 and staged == (plain and ns >= lib.get_corr_min_shifts())
            assert staged == plain or ns != 41
            got = lib.gencorrs_batch(ids, None, shift_list(ns))
            ref = gen.gencorrs_batch(ids, None, shift_list(ns))
            assert np.all(np.isfinite(got))
            v, w = got.reshape(-1, got.shape[-1]), ref.reshape(-1, ref.shape[-1])
            worst = max(peak_rel_err(a, b) for a, b in zip(v, w))
            assert worst < 2 * FP32_TOL, (form, ns, worst)
        lib.kill()
        gen.kill()


@pytest.mark.parametrize("n,ns", [(36, 5), (150, 41), (308, 4), (308, 41), (486, 9)])
def test_split_search_equals_the_whole_one(n, ns):
    """One particle per call splits the shells over work-groups; the batch of all does not."""
    nptcls = 800
    pf, cps = make_case(seed=n + ns, n=n, kfrom=2, kto=8, nrefs=3, nptcls=nptcls, ldim=max(40, n), eo_mixed=True)
    lib = to_lib(pf, cps)
    say(f"split search: n={n} ns={ns}")
    sh = shift_list(ns)
    ids = np.arange(1, nptcls + 1)
    whole = lib.gencorrs_batch(ids, None, sh)
    cc, ir, ish, rot = lib.search(ids, None, sh)
    for i in (0, 399, nptcls - 1):
        part = lib.gencorrs_batch(ids[i:i + 1], None, sh)
        v, w = part.reshape(-1, part.shape[-1]), whole[i].reshape(-1, part.shape[-1])
        assert max(peak_rel_err(a, b) for a, b in zip(v, w)) < 2 * FP32_TOL
        for r in range(3):
            for s, o in enumerate(pf.gencorrs_shifts(r, i, sh)):
                assert peak_rel_err(part[0, r, s], o) < FP32_TOL
                assert peak_rel_err(whole[i, r, s], o) < FP32_TOL
        # a search's winner is the first maximum of the same call's vectors
        c1, i1, s1, t1 = lib.search(ids[i:i + 1], None, sh)
        r, s, t = np.unravel_index(int(np.argmax(part[0])), part[0].shape)
        assert (i1[0], s1[0], t1[0]) == (r + 1, s, t + 1) and c1[0] == part[0, r, s, t]
        r, s, t = np.unravel_index(int(np.argmax(whole[i])), whole[i].shape)
        assert (ir[i], ish[i], rot[i]) == (r + 1, s, t + 1) and cc[i] == whole[i, r, s, t]
    lib.kill()


@pytest.mark.parametrize("n", LENGTHS)
def test_ring_spectra_and_inverse_stage(n):
    """Ring spectra of listed references (k_ring_spec, 8 rings per work-group) and of particles
    (k_memoize) against FP64 transforms; packing, contraction and inverse stage (k_ring_zifft) of the
    precision form against the plain search, for ring-constant |CTF|.
    Tolerance: 1e-5 of a ring's peak; the split-BF16 bar of 1e-4 of the peak and the plain search's 1e-5."""
    say(f"ring spectra and inverse stage: n={n}")
    pf, cps = make_case(seed=7 * n, n=n, kfrom=2, kto=8, kstop=7, ctf=True, astig=0.0, nrefs=23, nptcls=9,
                        ldim=max(40, n), eo_mixed=True)
    lib = to_lib(pf, cps)

    def spectra(rings):                 # rfft_2n(Re p + Im p | Re p - Im p), memoize_ffts
        p = rings.astype(np.complex128)
        return np.fft.rfft(np.concatenate([p.real + p.imag, p.real - p.imag], axis=-1), axis=-1)

    for iseven, refs in ((True, [23, 1, 7, 7, 2]), (False, [5]), (False, np.arange(1, 24))):
        exact = spectra((pf.refs_even if iseven else pf.refs_odd)[np.array(refs) - 1]).reshape(-1, n + 1)
        got = lib.get_ref_spectra(refs, iseven).reshape(-1, n + 1)
        assert max(peak_rel_err(a, b) for a, b in zip(got, exact)) < FP32_TOL, (iseven, refs)
    for i in (1, 9):
        exact = spectra(pf.ptcls[i - 1])
        assert max(peak_rel_err(a, b) for a, b in zip(lib.get_memo(i), exact)) < FP32_TOL
    ids = np.array([9, 2, 5, 1, 3])
    refs = np.concatenate([np.arange(23, 1, -2), np.arange(2, 23, 3)]).astype(np.int32)
    for ns in (0, 4):
        plain = lib.gencorrs_batch(ids, refs, shift_list(ns))
        got = lib.gencorrs_mfma_batch(ids, refs, shifts=shift_list(ns))
        v, w = got.reshape(-1, got.shape[-1]), plain.reshape(-1, got.shape[-1])
        worst = max(peak_rel_err(a, b) for a, b in zip(v, w))
        assert worst < 1e-4 + FP32_TOL, (ns, worst)
    lib.kill()


@pytest.mark.parametrize("nptcls,ns", [(637, 0), (638, 0), (5, 32), (5, 33)])
def test_call_lists_as_arguments_or_copies(nptcls, ns):
    """Lists of 640 entries and 32 shifts go to the device as kernel arguments, longer ones as copies."""
    say(f"call lists: {nptcls} particles, 3 references, {ns} shifts")
    pf, cps = make_case(seed=nptcls + ns, n=16, kfrom=2, kto=7, ctf=True, nrefs=3, nptcls=nptcls, ldim=32, eo_mixed=True)
    lib = to_lib(pf, cps)
    ids = np.random.default_rng(3).permutation(nptcls) + 1
    refs = np.array([3, 1, 2], np.int32)
    sh = shift_list(ns)
    full = lib.gencorrs_batch(ids, refs, sh).reshape(nptcls, 3, max(ns, 1), -1)
    cc, ir, ish, rot = lib.search(ids, refs, sh)
    for i in range(nptcls):
        r, s, t = np.unravel_index(int(np.argmax(full[i])), full[i].shape)
        assert (ir[i], ish[i], rot[i]) == (refs[r], s, t + 1) and cc[i] == full[i, r, s, t]
    for i in (0, nptcls - 1):
        for r in range(3):
            exact = pf.gencorrs_shifts(refs[r] - 1, ids[i] - 1, sh) if ns else [pf.gencorrs(refs[r] - 1, ids[i] - 1, None)]
            for s in range(max(ns, 1)):
                assert peak_rel_err(full[i, r, s], exact[s]) < FP32_TOL
    lib.kill()


@pytest.mark.parametrize("n", [16, 24, 32, 40, 48, 64, 100, 192, 240, 308, 400, 500, 600])
def test_shift_search_callback_equals_the_generic_kernel(n, monkeypatch):
    """The shift search's callback (k_corr_items: eight or four shells at a time, 13 and 11 of them here)
    against the runtime-size kernel: the same rotations, cc within 2e-5.  The FP64 objective is the
    same kernel on both handles, so the shifts agree far below the search's own tolerance."""
    kto = min(14, n // 2)
    for form in FORMS:
        kw = dict(ctf=True, kstop=kto - 2)
        kw.update(form)
        if "kstop" in form:
            kw["kstop"] = min(form["kstop"], kto)
        say(f"callback: n={n} {form}")
        pf, cps = make_case(seed=3 * n, n=n, kfrom=2, kto=kto, nrefs=3, nptcls=12, ldim=max(40, n), **kw)
        for i in range(12):
            pf.ptcls[i] = (pf.refs_even[i % 3] * (1.0 if pf.ctfmats is None else pf.ctfmats[i]) +
                           0.3 * pf.ptcls[i]).astype(np.complex64)
        lib, gen = both(monkeypatch, pf, cps)
        ir, ip = np.arange(12, dtype=np.int32) % 3 + 1, np.arange(1, 13, dtype=np.int32)
        cxy, rot = lib.shsrch_grad_batch(ir, ip, trs=3.0)
        ref, rrot = gen.shsrch_grad_batch(ir, ip, trs=3.0)
        assert np.array_equal(rot, rrot), (form, rot, rrot)
        assert np.max(np.abs(cxy[:, 0] - ref[:, 0])) < 2 * FP32_TOL
        assert np.max(np.abs(cxy[:, 1:] - ref[:, 1:])) < 1e-2
        lib.kill()
        gen.kill()


@pytest.mark.parametrize("n", [132, 176, 220, 364, 450, 546])
@pytest.mark.parametrize("ns", [0, 25])
def test_ring_kernel_keeps_the_generic_kernel_s_accuracy(n, ns, monkeypatch):
    """Lengths whose searches ran on the runtime-size kernel: the relative error of whole vectors against
    FP64, over searches large enough that no shells are split, is not larger than that kernel's.  0.15
    covers the scatter of the two estimates (48 pairs and more, each over 2 n rotations)."""
    nptcls, nrefs = 480, 3 if ns else 12
    say(f"accuracy of the ring kernel: n={n} ns={ns}")
    pf, cps = make_case(seed=n + ns, n=n, kfrom=2, kto=n // 5, ctf=True, astig=0.3, nrefs=nrefs, nptcls=nptcls,
                        ldim=2 * (n // 3))
    for i in range(nptcls):
        pf.ptcls[i] = (pf.refs_even[i % nrefs] + pf.ptcls[i]).astype(np.complex64)
    sh = shift_list(ns)
    err = []
    for h in both(monkeypatch, pf, cps):
        got = h.gencorrs_batch(np.arange(1, nptcls + 1), None, sh).reshape(nptcls, nrefs, max(ns, 1), -1)
        h.kill()
        num = den = 0.0
        for i in range(0, nptcls, 120 if ns else 60):
            for r in range(min(nrefs, 6)):
                exact = pf.gencorrs_shifts(r, i, sh) if ns else [pf.gencorrs(r, i, None, method="fft")]
                num += np.sum((got[i, r] - np.stack(exact)) ** 2)
                den += np.sum(np.square(exact))
        err.append(np.sqrt(num / den))
    say(f"  relative error {err[0]:.2e}, runtime-size kernel {err[1]:.2e}")
    assert err[0] < 1.15 * err[1]


@pytest.mark.parametrize("form", [dict(), dict(match_filt=True), dict(euclid=True)])
def test_objective_of_an_item_is_the_same_in_every_batch(form):
    """The FP64 objective and gradient of an item have the same bits alone, among a few and among many
    (1024 and 1025 items of three wavefronts lie on both sides of k_rot8's variants)."""
    say(f"objective in batches: {form}")
    pf, cps = make_case(seed=29, n=192, kfrom=2, kto=40, ctf=True, nrefs=3, nptcls=8, ldim=128, eo_mixed=True, **form)
    lib = to_lib(pf, cps)
    rng = np.random.default_rng(4)
    n = 1025
    r, p, o = rng.integers(1, 4, n), rng.integers(1, 9, n), rng.integers(1, 385, n)
    sh = rng.uniform(-4, 4, (n, 2))
    f, g = lib.grad_batch(r, p, sh, o)
    for k in (1, 3, 40, 1024):
        fk, gk = lib.grad_batch(r[:k], p[:k], sh[:k], o[:k])
        assert np.array_equal(fk, f[:k]) and np.array_equal(gk, g[:k]), k
    for i in range(5):
        f1, g1 = lib.gencorr_grad_for_rot_8(r[i], p[i], sh[i], o[i])
        assert f1 == f[i] and np.array_equal(g1, g[i, :2])
    lib.kill()


@pytest.mark.parametrize("n", LENGTHS)
def test_pair_is_the_same_in_every_launch(n):
    """A pair's vector has the same bits alone (its shells spread over work-groups, k_ring_finish), among a
    few and among 400 particles x 3 references (not spread: more than half of 768 work-groups)."""
    for form in FORMS:
        kw = dict(ctf=True, kstop=11)
        kw.update(form)
        pf, cps = make_case(seed=2 * n, n=n, kfrom=2, kto=13, nrefs=3, nptcls=400, ldim=max(40, n), eo_mixed=True, **kw)
        lib = to_lib(pf, cps)
        ids = np.arange(1, 401)
        for ns in (0, 1, 41):
            say(f"one pair, few pairs, many pairs: n={n} {form} ns={ns}")
            sh = shift_list(ns)
            many = lib.gencorrs_batch(ids, None, sh).reshape(400, 3, max(ns, 1), -1)
            few = lib.gencorrs_batch(ids[5:8], None, sh).reshape(3, 3, max(ns, 1), -1)
            one = lib.gencorrs_batch(ids[9:10], np.array([2], np.int32), sh).reshape(max(ns, 1), -1)
            assert np.array_equal(few, many[5:8]), (form, ns, np.mean(few != many[5:8]))
            assert np.array_equal(one, many[9, 1]), (form, ns, np.mean(one != many[9, 1]))
            if ns < 2:
                assert np.array_equal(lib.gencorrs(3, 11, sh[0] if ns else None), many[10, 2, 0])
        lib.kill()


def test_stochastic_walk_does_not_depend_on_the_batch():
    """A particle's stochastic search ends at the same reference with the same bits among 400 particles and
    among 7 (few enough that late rounds spread their shells over work-groups)."""
    say("stochastic walks: n 176, 400 and 7 particles x 90 references")
    pf, cps = make_case(seed=176, n=176, kfrom=2, kto=30, ctf=True, nrefs=90, nptcls=400, ldim=144, eo_mixed=True)
    lib = to_lib(pf, cps)
    rng = np.random.default_rng(9)
    order = np.stack([rng.permutation(90) + 1 for _ in range(400)])
    top = lib.gencorrs_batch(np.arange(1, 401)).max(axis=(1, 2, 3))
    prev = (top * rng.uniform(0.7, 1.0, 400)).astype(np.float32)
    many = lib.strategy_srch(SRCH_SHC3D, np.arange(1, 401), srch_order=order, prev_corr=prev, ref_corrs=True)
    sel = np.arange(3, 400, 61)
    few = lib.strategy_srch(SRCH_SHC3D, sel + 1, srch_order=order[sel], prev_corr=prev[sel], ref_corrs=True)
    for key in ("best_ref", "best_rot", "best_corr", "nrefs_eval", "found_better", "ref_corrs"):
        assert np.array_equal(many[key][sel], few[key]), key
    lib.kill()
