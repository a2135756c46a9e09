// The copies into LDS of one wave of prefill_rows64.hip with four key parts: their
// order and the waits that its reads rely on, as plain constants, checked below
// against a model of the wave's copy queue (copies land in the order of issue; a
// wait leaves at most its count of them in flight).  Host code: no HIP here.
#pragma once

namespace rows64 {

// A wave's K units go round a ring of three in LDS, its V units round one of two.
constexpr int kRingK = 3, kRingV = 2;

// Copies issued before the first unit: K 0 is waited for alone, and K 1, which
// the first iteration reads, stands before V 0.
struct First {
    bool k[4];  // in order: the next unit of K, or of V
};
constexpr First kFirst = {{true, true, false, true}};  // K 0, K 1, V 0, K 2

// Units of K and V that may be in flight
constexpr int kLeftFirst = 3;  // when K 0 is read
constexpr int kLeftK = 3;      // when K i + 1 is read, K i + 3 being the last issued
constexpr int kLeftV = 1;      // when V i is read: K i + 3

// Iteration i: issue K i + 3, wait (left_k), read K i + 1, wait (left_v), read V i,
// issue V i + 1.  True if every unit read has landed and no unit is overwritten
// before it has been read.
constexpr bool copies_ok(const First& first, int left_first, int left_k, int left_v, int units) {
    struct Queue {
        int issued = 0, landed = 0;       // both operands, in order of issue
        int k = 0, v = 0;                 // units issued
        int at_k[64] = {}, at_v[64] = {};  // place of a unit in the queue, from 1
        int read_k = 0, read_v = 0;       // units read
        bool ok = true;
        constexpr void issue(bool is_k) {
            if (is_k) {
                if (k >= read_k + kRingK) ok = false;
                at_k[k++] = ++issued;
            } else {
                if (v >= read_v + kRingV) ok = false;
                at_v[v++] = ++issued;
            }
        }
        constexpr void wait(int left) {
            if (issued - left > landed) landed = issued - left;
        }
        constexpr void read(bool is_k, int unit) {
            const int at = is_k ? at_k[unit] : at_v[unit];
            if (at == 0 || at > landed) ok = false;
            (is_k ? read_k : read_v) = unit + 1;
        }
    };
    if (units > 56) return false;  // the model's arrays
    Queue q;
    for (bool is_k : first.k) q.issue(is_k);
    q.wait(left_first);
    q.read(true, 0);
    for (int i = 0; i < units; ++i) {
        q.issue(true);
        q.wait(left_k);
        q.read(true, i + 1);
        q.wait(left_v);
        q.read(false, i);
        q.issue(false);
    }
    return q.ok;
}
static_assert(copies_ok(kFirst, kLeftFirst, kLeftK, kLeftV, 1));
static_assert(copies_ok(kFirst, kLeftFirst, kLeftK, kLeftV, 2));
static_assert(copies_ok(kFirst, kLeftFirst, kLeftK, kLeftV, 40));

}  // namespace rows64
