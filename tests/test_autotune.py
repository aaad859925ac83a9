"""What the autotuner builds is what it names: tile forms, at every grid size."""
import pytest

from paraiso_amd import autotune, generator, variants


@pytest.fixture
def built(monkeypatch):
    """{library name: Setup} of the machines that would be compiled."""
    out = {}

    def build_machine(setup, om, name, precise=False, force=False):
        out[name] = (setup, [k.name for k in om.kernels])
        return name
    monkeypatch.setattr(generator, "build_machine", build_machine)
    return out


def one_form(setup, kernels):
    return all(setup.form_of(k)["lane"] is None and not setup.form_of(k)["tiny"] for k in kernels)


@pytest.mark.parametrize("variant,candidate", [("hydro_f32", ((64, 16), 512)),
                                               ("life_i32", ((64, 32), 1024)),
                                               ("wave3d_f32", ((64, 8, 128), 512, 48, 2))])
def test_candidates_are_tiles_at_every_size(built, variant, candidate):
    _, lib = autotune._build_candidate(variant, candidate)
    setup, kernels = built[lib]
    assert setup.tile == candidate[0] and one_form(setup, kernels)
    # the variant itself has other forms on some grids
    assert not one_form(variants.VARIANTS[variant][1], kernels)


def test_flips_and_their_baseline_are_tiles_at_every_size(built):
    variant, kernel = "hydro_f32", "proceed_pipelined"
    flips = [None] + autotune.alloc_candidates(variant, kernel, 2)
    for fl in flips:
        autotune._build_flip(variant, kernel, fl)
    assert len(built) == 3
    assert all(one_form(*x) for x in built.values())
    forms = [s.form_of(kernel) for s, _ in built.values()]
    assert len(set(str(f) for f in forms)) == 3          # only the flipped choice differs
    assert len(set(f["tile"] for f in forms)) == 1


def test_recorded_forms_keep_the_variants_own(monkeypatch):
    """A recorded tile or flip of one kernel leaves every kernel its streaming form."""
    rec = {"proceed_x8": {"tile": [32, 32], "threads": 512}, "proceed": {"manifest": [4]}}
    monkeypatch.setattr(autotune, "tuned", lambda: {"life_i32": {"kernel_forms": rec}})
    setup, own = variants.setup_of("life_i32"), variants.VARIANTS["life_i32"][1]
    for k in ("proceed", "proceed_x4", "proceed_x8", "proceed_x16"):
        assert setup.form_of(k)["lane"] == own.form_of(k)["lane"] is not None
    assert setup.form_of("proceed_x8")["tile"] == (32, 32)
    assert setup.form_of("proceed")["manifest"] == (4,)
