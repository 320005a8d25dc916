// q3h_passes.h - which prompts of a batched start share a pass of the talker
// (host code, no device dependencies).
#pragma once

#include <vector>

namespace q3h {

// The passes over prompts of rows[0 .. n - 1] rows, at most `limit` rows each
// (none longer than that): the prompts of each in order. A pass takes every
// prompt left that still fits, so one that fills a pass by itself does not keep
// the ones after it from sharing theirs.
inline std::vector<std::vector<int>> start_passes(const int *rows, int n, int limit) {
  std::vector<std::vector<int>> passes;
  std::vector<int> left(n);
  for (int i = 0; i < n; i++) left[i] = i;
  while (!left.empty()) {
    std::vector<int> pass, rest;
    int sum = 0;
    for (int i : left) {
      const bool fits = pass.empty() || rows[i] <= limit - sum;
      (fits ? pass : rest).push_back(i);
      if (fits) sum += rows[i];
    }
    passes.push_back(std::move(pass));
    left = std::move(rest);
  }
  return passes;
}

}  // namespace q3h
