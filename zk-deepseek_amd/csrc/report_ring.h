// Reports that launches leave in pinned host memory, taken in by later calls: a ring of slots of PARTS words each.  A
// launch's workgroups store its number into the upper half of every one of its words; it has arrived when all carry it.
// Host code only, no GPU runtime.
#pragma once

namespace zk {

template <class Tag, unsigned SLOTS, int PARTS>
struct ReportRing {
    volatile unsigned long long *words = nullptr;      // [SLOTS][PARTS], cleared once
    Tag tag[SLOTS];
    unsigned seq_of[SLOTS];
    int parts_of[SLOTS];
    unsigned head = 0, tail = 0;                        // slots used and taken in so far; head - tail are on their way
    unsigned seq = 0;

    // The words of the next report and its number; null while every slot is on its way.
    unsigned long long *open(unsigned *number)
    {
        if (!words || head - tail >= SLOTS) return nullptr;
        if (++seq == 0) seq = 1;
        *number = seq;
        return const_cast<unsigned long long *>(words) + (unsigned long)(head % SLOTS) * PARTS;
    }
    // The launch that stores `parts` words under `number` is on the stream.
    void push(const Tag &t, unsigned number, int parts)
    {
        tag[head % SLOTS] = t;
        seq_of[head % SLOTS] = number;
        parts_of[head % SLOTS] = parts;
        head++;
    }
    bool arrived(unsigned n) const
    {
        const volatile unsigned long long *w = words + (unsigned long)(n % SLOTS) * PARTS;
        for (int i = 0; i < parts_of[n % SLOTS]; i++)
            if ((unsigned)(w[i] >> 32) != seq_of[n % SLOTS]) return false;
        return true;
    }
    // take(tag, words, parts) for every report that has arrived, oldest first.  The stream delivers them in order, so one
    // that is still missing when a later one is there will never come (its launch failed): it is dropped, or the ring
    // would wait for it for good.
    template <class F>
    void drain(F &&take)
    {
        while (tail != head) {
            if (arrived(tail)) {
                take(tag[tail % SLOTS], words + (unsigned long)(tail % SLOTS) * PARTS, parts_of[tail % SLOTS]);
                tail++;
                continue;
            }
            unsigned later = tail + 1;
            while (later != head && !arrived(later)) later++;
            if (later == head) return;
            if (!arrived(tail)) tail++;                 // (looked at once more: it may have come in between)
        }
    }
};

}  // namespace zk
