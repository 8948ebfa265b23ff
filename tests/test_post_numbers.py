"""Sequence numbers of posted results: one is taken only where a kernel will post it, so that the latest number can be
waited for at any time."""
import host_cpp

BODY = r"""
  Device d;                      // no device memory: only the numbering is looked at
  double host[64];
  unsigned long long word = 0;
  d.hpostDev = host;
  d.hseqDev = &word;
  unsigned int tickets[TICKETS] = {};
  d.tickets = tickets;
  for (int blocks : { 1, FINISH_BLOCKS, FINISH_BLOCKS + 1, 4096 })
    for (int sums : { 0, 1 }) {
      const unsigned long long before = d.seq;
      const Post p = dev_post(&d, POST_TRIG, TICKET_TRIG, blocks, sums != 0);
      printf("%d %d %d %llu %llu\n", blocks, sums, p.ticket != nullptr, d.seq - before, p.seq - before);
    }
"""


def test_numbers_are_posted(tmp_path):
    rows = [tuple(map(int, line.split())) for line in host_cpp.run(tmp_path, BODY)]
    assert len(rows) == 8
    for blocks, sums, ticket, taken, number in rows:
        assert ticket == (blocks <= 32)
        # a grid that finishes its sums posts the number itself; sums of a larger one are posted by the reduction
        # launched behind it; nothing posts a larger trigger grid's number
        posted = bool(ticket or sums)
        assert taken == posted, (blocks, sums)
        if posted:
            assert number == 1
