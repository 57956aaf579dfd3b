"""When the tests of programs linked with the reference's sources are skipped, and when they run."""
import pytest

from conftest import REFERENCE_PROGRAMS, why_skipped


@pytest.mark.parametrize("built", [False, True])
@pytest.mark.parametrize("checkout", [False, True])
@pytest.mark.parametrize("key", sorted(REFERENCE_PROGRAMS))
def test_only_without_program_and_sources(tmp_path, key, checkout, built):
    source = tmp_path / "paged_kv.cpp"
    if checkout:
        source.write_text("")
    if built:
        out = tmp_path / "oracle" / "_ref" / "integration"
        out.mkdir(parents=True)
        (out / REFERENCE_PROGRAMS[key]).write_text("")
    file_name, test_name = (key, "test_any") if key.endswith(".py") else ("test_any.py", key)
    reason = why_skipped(file_name, test_name, str(tmp_path), str(source))
    assert (reason is not None) == (not checkout and not built)


def test_other_tests_are_never_skipped(tmp_path):
    assert why_skipped("test_abi_cpu.py", "test_any", str(tmp_path), str(tmp_path / "none")) is None
