"""The words of a worker's job slot (requests' tags, answers, refusals), on the
CPU: whatever came before, and in whatever order an answer's words land, the
slot is complete only when the whole answer is there."""
from tests import hostcc

MODEL = r"""
    uint64_t w[kJobWords];
    auto complete = [&](uint32_t tag) {
        for (uint64_t x : w)
            if (!slot_word_of(x, tag)) return false;
        return true;
    };
    unsigned rnd = 1;
    auto land = [&](uint32_t tag, int n, bool refusal, int seq) {
        // the first n words of the answer in a random order of landing
        int order[kJobWords];
        for (int i = 0; i < n; i++) order[i] = i;
        for (int i = n - 1; i > 0; i--) {
            rnd = rnd * 1664525u + 1013904223u;
            const int j = (rnd >> 8) % (i + 1), t = order[i];
            order[i] = order[j], order[j] = t;
        }
        for (int i = 0; i < n; i++) {
            if (complete(tag)) { printf("torn at request %d, word %d\n", seq, i); exit(0); }
            w[order[i]] = slot_word(tag, refusal ? refusal_value(order[i]) : seq + i);
        }
        if (!complete(tag)) { printf("lost at request %d\n", seq); exit(0); }
    };
    for (int refusals : {0, 1, 2, 253, 254, 255, 508, 509}) {
        const uint32_t epoch = 7;
        for (int i = 0; i < kJobWords; i++) w[i] = 0;  // as the init kernel leaves it
        int seq = 0;
        for (int round = 0; round < 4; round++) {
            land(request_tag(epoch, seq), kJobWords, false, seq), seq++;
            for (int i = 0; i < refusals; i++) land(request_tag(epoch, seq), kRefusalWords, true, seq), seq++;
        }
    }
    for (uint32_t e : {0u, 1u, 0xffffffu, 0x1000000u, 0xffffffffu})
        for (uint32_t s = 0; s < 600; s++)
            if (request_tag(e, s) == 0 || request_tag(e, s) == request_tag(e, s + 1)) { printf("tag\n"); exit(0); }
    if (refusal_value(0) != kNoJob) printf("refusal\n");
    printf("sound\n");
"""


def test_no_torn_answer_after_any_number_of_refusals(tmp_path):
    assert hostcc.run(tmp_path, MODEL) == "sound\n"


def test_a_refusal_of_one_word_would_be_torn(tmp_path):
    # the model finds it: 254 refusals that leave words 1.. with an old tag
    one = MODEL.replace("land(request_tag(epoch, seq), kRefusalWords, true, seq), seq++",
                        "w[0] = slot_word(request_tag(epoch, seq), refusal_value(0)), seq++")
    assert hostcc.run(tmp_path, one).startswith("torn")
