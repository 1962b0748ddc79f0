"""Which tests run where."""


def test_tests_of_the_gpu_are_marked(request):
    """A test that takes the `gpu` fixture runs with `-m gpu` and not without."""
    unmarked = [i.nodeid for i in request.session.items if "gpu" in i.fixturenames and not i.get_closest_marker("gpu")]
    assert not unmarked, unmarked
