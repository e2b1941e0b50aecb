"""Setup-string fidelity (CPU): the library parses SimulationBuilder JSON as serde does
(simulation_builder.rs:21-66, line_force_model/builder/mod.rs:20-46,
builder/single_wing.rs:31-47, dynamic_wake/builder.rs:28-120, wake/settings.rs:11-58,
solvers/*.rs, section_models/foil.rs:14-117).

* the fixtures in tests/golden/setups/ were written by the reference's own setup package
  (interfaces/stormbird_setup, tests/golden/make_setup_fixtures.py): every one loads unchanged
  and gives the oracle's strip, point and panel counts;
* structs with deny_unknown_fields reject unknown keys; ForceCalculationSettings and the
  SpatialVector record (no such attribute) ignore them;
* usize fields take integer literals only; Option fields take null; required fields are
  required; duplicate keys, malformed numbers and unknown enum variants are errors;
* valid setups outside this library (other section models, circulation corrections) are
  rejected with a message naming the feature.
"""
import copy
import glob
import json
import os

import pytest

import stormbird_amd as sb
from stormbird_amd import setups as S

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "setups")
# SimulationBuilder strings; csm_*.json hold CompleteSailModelBuilder strings
FIXTURES = sorted(p for p in glob.glob(os.path.join(GOLDEN, "*.json")) if not os.path.basename(p).startswith("csm_"))


def test_fixtures_exist():
    assert len(FIXTURES) >= 5


@pytest.mark.parametrize("path", FIXTURES, ids=[os.path.basename(p) for p in FIXTURES])
def test_reference_setup_package_output_loads(oracle, path):
    text = open(path).read()
    info = sb.setup_info(text)
    o = oracle.Simulation(text, "pm")
    assert info["nr_ctrl_points"] == o.nr_ctrl_points
    assert info["nr_freestream_points"] == o.nr_freestream_points()
    assert info["nr_panels"] == o.nr_panels
    assert info["quasi_steady"] == (1 if "QuasiSteady" in json.loads(text)["simulation_settings"] else 0)


CSM_FIXTURES = sorted(glob.glob(os.path.join(GOLDEN, "csm_*.json")))


@pytest.mark.parametrize("path", CSM_FIXTURES, ids=[os.path.basename(p) for p in CSM_FIXTURES])
def test_reference_complete_sail_model_output_loads(oracle, path):
    from stormbird_amd.complete_sail_model import csm_setup_info

    text = open(path).read()
    d = json.loads(text)
    info = csm_setup_info(text)
    o = oracle.Simulation(json.dumps(d["lifting_line_simulation"]), "pm")
    assert info["nr_ctrl_points"] == o.nr_ctrl_points
    assert info["nr_freestream_points"] == o.nr_freestream_points()
    assert info["nr_set_points"] == len(d["controller"]["set_points"])


def base():
    return json.loads(open(os.path.join(GOLDEN, "two_sails_dynamic_all_settings.json")).read())


def parses(d):
    sb.setup_info(json.dumps(d) if not isinstance(d, str) else d)


def rejects(d, match):
    with pytest.raises(ValueError, match=match):
        parses(d)


def wake(d):
    return d["simulation_settings"]["Dynamic"]["wake"]


def solver(d):
    return d["simulation_settings"]["Dynamic"]["solver"]["SimpleIterative"]


@pytest.mark.parametrize("where", ["root", "lfm", "wing", "foil", "wake", "solver", "dynamic", "sin"])
def test_unknown_fields_rejected(where):
    d = base()
    target = {"root": d, "lfm": d["line_force_model"], "wing": d["line_force_model"]["wing_builders"][0],
              "foil": d["line_force_model"]["wing_builders"][0]["section_model"]["Foil"], "wake": wake(d),
              "solver": solver(d), "dynamic": d["simulation_settings"]["Dynamic"],
              "sin": wake(d)["viscous_core_length_evolution"]["SinIncrease"]}[where]
    target["not_a_field"] = 1
    rejects(d, "unknown field")


def test_quasi_steady_structs_reject_unknown_fields():
    d = json.loads(open(os.path.join(GOLDEN, "two_sails_quasi_steady_iterative.json")).read())
    # use_raw_circulation_during_iterations exists in SimpleIterative, not in the quasi-steady builder
    d["simulation_settings"]["QuasiSteady"]["solver"]["SimpleIterative"]["use_raw_circulation_during_iterations"] = True
    rejects(d, "unknown field")
    d = json.loads(open(os.path.join(GOLDEN, "two_sails_quasi_steady_linearized.json")).read())
    d["simulation_settings"]["QuasiSteady"]["wake"]["nr_panels_per_line_element"] = 10
    rejects(d, "unknown field")
    d = json.loads(open(os.path.join(GOLDEN, "two_sails_quasi_steady_linearized.json")).read())
    d["simulation_settings"]["QuasiSteady"]["solver"]["Linearized"]["damping_factor"] = 0.1
    rejects(d, "unknown field")


def test_unknown_fields_ignored_where_serde_ignores_them():
    d = base()
    d["line_force_model"]["force_calculation_settings"]["something_else"] = 3
    d["line_force_model"]["rotation"]["w"] = 1.0
    parses(d)


def test_vector_forms():
    d = base()
    d["line_force_model"]["translation"] = [1.0, 2.0, 3.0]
    parses(d)
    d["line_force_model"]["translation"] = {"x": 1.0, "y": 2.0}
    rejects(d, "vector")
    d["line_force_model"]["translation"] = [1.0, 2.0]
    rejects(d, "vector")


@pytest.mark.parametrize("value", [32.0, 1e2, -4, "32"])
def test_usize_fields_take_integer_literals(value):
    for setter in (lambda d: d["line_force_model"].__setitem__("nr_sections", value),
                   lambda d: d["line_force_model"]["wing_builders"][0].__setitem__("nr_sections", value),
                   lambda d: wake(d).__setitem__("nr_panels_per_line_element", value),
                   lambda d: solver(d).__setitem__("max_iterations_per_time_step", value)):
        d = base()
        setter(d)
        rejects(d, "integer")


def test_integer_literals_are_floats_where_floats_are_expected():
    d = base()
    d["line_force_model"]["density"] = 1
    wake(d)["first_panel_relative_length"] = 1
    parses(d)


def test_option_fields_take_null_and_others_do_not():
    d = base()
    d["line_force_model"]["wing_builders"][0]["nr_sections"] = None
    d["line_force_model"]["wing_builders"][0]["line_segment_is_virtual"] = None
    parses(d)
    for setter in (lambda d: d["line_force_model"].__setitem__("density", None),
                   lambda d: wake(d).__setitem__("shape_damping_factor", None),
                   lambda d: d["line_force_model"]["wing_builders"][0].__setitem__("non_zero_circulation_at_ends", None)):
        d = base()
        setter(d)
        with pytest.raises(ValueError):
            parses(d)


def test_required_fields():
    for key in ("section_points", "chord_vectors", "section_model"):
        d = base()
        del d["line_force_model"]["wing_builders"][0][key]
        with pytest.raises(ValueError):
            parses(d)
    d = base()
    del d["line_force_model"]["nr_sections"]
    rejects(d, "nr_sections")
    d = base()
    del d["line_force_model"]
    rejects(d, "line_force_model")


def test_defaults_when_fields_are_absent():
    """Absent simulation_settings is QuasiSteady; absent solver/wake take their defaults."""
    d = base()
    del d["simulation_settings"]
    assert sb.setup_info(json.dumps(d))["quasi_steady"] == 1
    d = base()
    d["simulation_settings"] = {"Dynamic": {}}
    info = sb.setup_info(json.dumps(d))
    assert info["quasi_steady"] == 0 and info["nr_wake_rows"] == 100
    d["simulation_settings"] = {"QuasiSteady": {}}
    assert sb.setup_info(json.dumps(d))["nr_freestream_points"] == info["nr_ctrl_points"]


@pytest.mark.parametrize("text", [
    '{"line_force_model": {"nr_sections": 4, "nr_sections": 5, "wing_builders": []}}',
    '{"line_force_model": {"nr_sections": 04}}',
    '{"line_force_model": {"nr_sections": +4}}',
    '{"line_force_model": {"density": .5}}',
    '{"line_force_model": {"density": 1.}}',
    '{"line_force_model": {"density": NaN}}',
    '{"line_force_model": {"density": Infinity}}',
    '{"line_force_model": {"density": 0x10}}',
    '{"line_force_model": {"nr_sections": 4}} trailing',
])
def test_malformed_json(text):
    with pytest.raises(ValueError):
        sb.setup_info(text)


def test_string_escapes_and_enum_forms():
    d = base()
    wake(d)["symmetry_condition"] = "Z"  # "Z" written as an escape
    text = json.dumps(d, ensure_ascii=True).replace('"Z"', '"\\u005a"')
    sb.setup_info(text)
    d = base()
    wake(d)["symmetry_condition"] = "Q"
    rejects(d, "SymmetryCondition")
    d = base()
    wake(d)["viscous_core_length"] = {"Relative": 0.1, "Absolute": 0.2}
    rejects(d, "enum variant")
    d = base()
    d["simulation_settings"] = {"Dynamic": {}, "QuasiSteady": {}}
    rejects(d, "enum variant")


@pytest.mark.parametrize("model, msg", [
    ({"RotatingCylinder": {"revolutions_per_second": 1.0}}, "RotatingCylinder"),
    ({"VaryingFoil": {"internal_state_data": [0.0], "foils_data": [{}]}}, "VaryingFoil"),
    ("EffectiveWindSensor", "EffectiveWindSensor"),
])
def test_valid_setups_outside_this_library_name_the_feature(model, msg):
    d = base()
    d["line_force_model"]["wing_builders"][0]["section_model"] = model
    rejects(d, msg)
    d = base()
    d["line_force_model"]["circulation_correction"] = {"Prescribed": {}}
    rejects(d, "circulation correction")


def test_wings_without_strips_at_either_end_are_rejected():
    """A wing of zero length between others is taken (no strips, one span point); first or last there is no
    strip that its span point could take its values from.  In a process of its own: reading them
    anyway ends it."""
    import subprocess
    import sys

    code = """
import json
import stormbird_amd as sb
from stormbird_amd import setups as S
for dynamic in (False, True):
    for at in (0, 1, 2):
        d = json.loads(S.wing_sails_quasi_steady(nr_strips=4))
        if dynamic:
            d["simulation_settings"] = S.dynamic_settings(nr_panels=5)
        w = d["line_force_model"]["wing_builders"][at]
        w["section_points"][1] = dict(w["section_points"][0])
        try:
            i = sb.setup_info(json.dumps(d))
            print(at, i["nr_ctrl_points"], i["nr_wings"], i["nr_span_points"])
        except ValueError as e:
            print(at, e)
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100,
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    want = ["0 wing 0 has no strips (zero length) and no wing with strips on both sides", "1 8 3 11",
            "2 wing 2 has no strips (zero length) and no wing with strips on both sides"]
    assert r.returncode == 0 and r.stdout.splitlines() == want * 2, (r.returncode, r.stdout, r.stderr[-500:])
