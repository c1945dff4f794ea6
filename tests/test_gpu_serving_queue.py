"""Requests that queue: more of them at once than slots, so that all but the first have to
wait for one.  `admitted` is when a slot holds the request: none is before its arrival, no
more requests than slots are ever held, and each that waited was admitted after another
request had finished."""
import pytest

from casmcode_monte_amd import serving

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots,requests", [(1, 5), (3, 10)])
def test_waiting_requests_follow_finished_ones(slots, requests):
    print("serving queue", slots, requests, flush=True)
    reqs = [serving.Request(rid=i, edge=20 + 4 * i, temperature=900.0 + 100.0 * i,
                            exchange_potential=0.05, seed=300 + i, arrival=0.0,
                            max_passes=1000, precision=1e-9) for i in range(requests)]
    srv = serving.Server(classes=((64, slots, True),), chunk=100, check_period=500)
    res, stats = srv.serve(reqs)
    srv.close()
    assert len(res) == requests and stats["n_requests"] == requests
    done = [res[i] for i in range(requests)]
    assert all(0.0 <= r.arrival <= r.admitted < r.finished for r in done)
    assert all(a.admitted < b.admitted for a, b in zip(done, done[1:]))  # in their order
    for r in done:
        held = sum(q.admitted <= r.admitted < q.finished for q in done)
        assert held <= slots, r
    for i, r in enumerate(done[slots:], start=slots):
        before = sum(q.finished < r.admitted for q in done)
        assert before >= i - slots + 1, r
