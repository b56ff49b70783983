"""Control handed from thread to thread (native, without a GPU)."""
import threading
import time

import pytest

from pfeife_amd.hip import Baton


def test_one_thread_runs_at_a_time_in_the_order_of_the_hand_overs():
    n, rounds = 4, 200
    baton, log, running = Baton(2 * n), [], []

    def loop(i):
        baton.switch(None, i)
        while True:
            running.append(i)
            log.append(i)
            assert running == [i]
            running.pop()
            if len(log) >= n * rounds - (n - 1 - i):
                return baton.switch(n + i, -1)
            baton.switch(n + i, i)

    threads = [threading.Thread(target=loop, args=(i,), daemon=True) for i in range(n)]
    for t in threads:
        t.start()
    for r in range(rounds):
        for i in range(n):
            if (r + i) % 3 == 0:
                baton.alert((i + 1) % n)         # (whether or not it sleeps, whether or not it is next)
            baton.switch(i, n + i, patience=50000)
            assert log[-1] == i and len(log) == r * n + i + 1
    for t in threads:
        t.join(10)
        assert not t.is_alive()


@pytest.mark.parametrize("patience", [-1, 0, 5000])
def test_an_alert_or_a_time_limit_is_no_token(patience):
    baton, got = Baton(1), []
    t = threading.Thread(target=lambda: (baton.switch(None, 0, patience), got.append(1)), daemon=True)
    t.start()
    for _ in range(3):
        baton.alert(0)
        time.sleep(0.02)
        assert not got
    baton.switch(0, -1)
    t.join(10)
    assert got


def test_tokens_given_before_the_wait_are_kept():
    baton = Baton(2)
    for _ in range(3):
        baton.switch(1, -1)
    for _ in range(3):
        baton.switch(None, 1)


def test_bad_slots_are_errors():
    with pytest.raises(RuntimeError):
        Baton(0)
    baton = Baton(2)
    for call in (lambda: baton.alert(2), lambda: baton.alert(-1), lambda: baton.switch(2, -1), lambda: baton.switch(0, 2)):
        with pytest.raises(RuntimeError):
            call()
