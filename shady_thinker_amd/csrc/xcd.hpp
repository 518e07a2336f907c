// Order of workgroups over the 8 XCDs (plain C++: also compiled for the host).
#pragma once

namespace st {

// Workgroups go to the XCDs round-robin: XCD x runs workgroups x, x + 8, ... of
// a grid of n. The place of workgroup b when each XCD takes consecutive places
// (as many as it has workgroups): a bijection of [0, n) for every n.
constexpr int xcd_order(int b, int n) {
    const int x = b % 8, rest = n % 8;
    return x * (n / 8) + (x < rest ? x : rest) + b / 8;
}

}  // namespace st
