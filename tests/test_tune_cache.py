"""The tuner's cache belongs to a build of the library: a choice timed with other
kernels is not taken.  No device."""
import hashlib
import json

from eagleimp_amd import tune

from test_tune_host import _Engine, _Targets


def test_choice_of_other_kernels_is_not_taken(tmp_path, monkeypatch):
    monkeypatch.setattr(tune, "CACHE", str(tmp_path / "tune.json"))
    tg, batches = _Targets(300, 10000), (128, 256)
    # an entry as kept for the same panel, K, window and shapes by a library with
    # other kernels
    vs = tune.candidates(10000)
    sig = json.dumps([_Engine.Nad, _Engine.Ncorr, _Engine.M, 10000, 1000, list(batches),
                      [(v["threads"], v["chunks_per_wave"]) for v in vs]])
    key = hashlib.sha1(sig.encode()).hexdigest()[:16]
    (tmp_path / "tune.json").write_text(json.dumps({key: dict(variant=4, batch=128)}))
    eng = _Engine()
    best = tune.tune(eng, tg, range(300), batches=batches)
    assert not best["cached"] and best["variant"] == 3 and eng.submits > 0
    # and one of this library is, until the library changes
    assert tune.tune(_Engine(), tg, range(300), batches=batches)["cached"]
    other = tmp_path / "lib.so"
    other.write_bytes(b"another build")
    monkeypatch.setattr(tune, "LIB_PATH", str(other))
    assert not tune.tune(_Engine(), tg, range(300), batches=batches)["cached"]
