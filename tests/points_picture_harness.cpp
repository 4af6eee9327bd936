// SparseGridMap on the CPU: entries appended without the index, then looked up (test_points_picture.py).
#include "SparseGrid.h"

// n entries appended as new, at[] of them again by insert, operator[] and find; the entries in order of key.  Returns how
// many look-ups went wrong.
extern "C" int appended(const int64_t *keys, int n, int split, int64_t *sortedKeys, int *sortedRows) {
  SparseGridMap m;
  std::vector<SparseGridMap::value_type> kv;
  for (int i = 0; i < n; ++i)
    kv.emplace_back(keys[i], i);
  m.appendNew(kv.data(), (size_t)split);
  int wrong = 0;
  if (split < n) // one through the index, the others behind it without
    wrong += !m.insert(kv[split]).second;
  if (split + 1 < n)
    m.appendNew(kv.data() + split + 1, (size_t)(n - split - 1));
  wrong += (int)m.size() != n || m.find(-5) != m.end();
  for (int i = 0; i < n; ++i) {
    wrong += m.insert(SparseGridMap::value_type(keys[i], -1)).second;
    wrong += m[keys[i]] != i;
    auto it = m.find(keys[i]);
    wrong += it == m.end() || it->second != i;
  }
  int k = 0;
  for (auto it = m.begin(); it != m.end(); ++it, ++k)
    sortedKeys[k] = it->first, sortedRows[k] = it->second;
  m.clear();
  wrong += m.size() != 0 || (n && m.find(keys[0]) != m.end());
  return wrong;
}
