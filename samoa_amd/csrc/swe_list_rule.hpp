// swe_list_rule.hpp -- when a remeshed mesh's edge lists are stored (plain C++,
// also compiled for the host).
#pragma once

#include <stdint.h>

namespace swe {

// Steps that pay for the lists.  Storing them takes a launch and its gap (7-8 us)
// and 8 us per million cells; a step with them saves 0.6-0.9 us and 2.5 us per
// million cells.  us a step without / with lists stored before the first of 4, 6,
// 8, 10, 12 and 16 steps between remeshings:
//     8 k cells   22.4 / 23.6, 18.7 / 19.6, 17.5 / 18.1, 16.3 / 16.3, 14.8 / 14.9, 14.1 / 14.0
//     44 k        22.7 / 23.9, 19.1 / 19.5, 16.8 / 16.9, 16.0 / 16.1, 15.3 / 15.1, 13.7 / 13.5
//     220 k       29.3 / 30.1, 24.5 / 25.0, 22.3 / 22.4, 21.2 / 21.1, 20.3 / 20.2, 19.2 / 19.0
//     310 k       32.4 / 33.0, 28.1 / 28.0, 26.6 / 26.4, 25.1 / 24.6, 24.4 / 23.8, 23.0 / 22.2
//     1 M         57.2 / 57.1, 52.4 / 51.5, 49.5 / 48.8, 48.0 / 46.5, 47.7 / 45.9, 46.4 / 44.1
//     4 M         184 / 183, 170 / 165, 163 / 157, 159 / 153, 156 / 148, 153 / 144
constexpr int64_t lists_break_even(int64_t cells) { return cells < (1 << 18) ? 12 : 6; }

// Before `steps` traversals of a mesh that had `uses` so far: whether to store its
// lists now.  A mesh is taken to last as long as the one before it (`before`
// traversals); one that has had twice its break-even by now gets them anyway.
inline bool lists_pay(int64_t cells, int64_t uses, int64_t steps, int64_t before) {
    const int64_t pay = lists_break_even(cells);
    const int64_t left = before - uses > steps ? before - uses : steps;
    return left >= pay || uses + steps > 2 * pay;
}

}  // namespace swe
