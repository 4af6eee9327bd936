// A max-pooling's backward pass over interfaces that are not the batch's own, on the CPU (test_foreign_interface.py): nothing
// wants a gradient, so that no kernel runs, and what lies before the caller's interface is not its to read.
#include <new>
#include <sys/mman.h>
#include <unistd.h>
#include "SpatiallySparseLayer.h"

int main() {
  const size_t page = (size_t)sysconf(_SC_PAGESIZE), room = (sizeof(SpatiallySparseBatchInterface) + page - 1) / page * page;
  char *const at = (char *)mmap(nullptr, 2 * room, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  if (at == MAP_FAILED || mprotect(at + room, room, PROT_READ | PROT_WRITE) != 0)
    return 1;
  SpatiallySparseBatchSubInterface sub;
  auto *const input = new (at + room) SpatiallySparseBatchInterface(&sub);
  SpatiallySparseBatchInterface output(&sub);
  SpatiallySparseBatch batch(&sub);
  alignas(cudaMemStream) static char noStream[sizeof(cudaMemStream)];
  MaxPoolingLayer pool(*reinterpret_cast<cudaMemStream *>(noStream), 3, 2, 2);
  pool.backwards(batch, *input, output, 0.1f, 0.9f);
  input->~SpatiallySparseBatchInterface();
  return 0;
}
