// Host/device vector with the reference's vectorCUDA<T> surface
// (vectorCUDA.h:6-40): the data lives either in a std::vector (onGPU ==
// false) or in HBM (onGPU == true); hVector() and dPtr() migrate it on demand
// and device storage only ever grows (vectorCUDA.cu:171-185).  Device memory
// and copies go through the C ABI of libscn_hip.so.  The type keeps the
// reference's name so that driver code compiles unchanged.
#pragma once
#include <vector>
#include "scn_hip.h"

// The stream object layer constructors take (utilities.h:105-112).  Every
// instance owns one library context, i.e. one HIP stream on the GPU.
class cudaMemStream {
public:
  scn_ctx *ctx;
  // layers: the stream runs layers, and not only the producers' rule books
  // (16 MB for each of those would be memory that nothing uses, and 1 ms of a
  // new net's first batch)
  explicit cudaMemStream(bool layers = true, size_t imageRoom = ROOM);
  ~cudaMemStream();
  cudaMemStream(const cudaMemStream &) = delete;
  cudaMemStream &operator=(const cudaMemStream &) = delete;
  void *stream() const;
  void synchronize() const;
  // Room for the weights of a pass over a batch as its contractions read them, in
  // the order of the stream: a net's own stream has ROOM of it from the start, which
  // holds those of a net of some 5 M weights (and so the first batch does not wait
  // for allocations: an allocation a layer was 0.1 ms of the first 1.6 of a net with
  // up to 800 channels), the other lanes' streams, which a net may never use, make
  // it with their first batch (0.1 ms of a new net for each), and all make more as
  // soon as it is asked for.
  static constexpr size_t ROOM = (size_t)32 << 20;
  void *imageRoom(size_t bytes);

private:
  void *images = nullptr;
  size_t imageBytes = 0;
};

// the context vectorCUDA objects use when no stream is named: the one of the
// oldest live cudaMemStream (the net's own memStream)
scn_ctx *scnDefaultContext();
void scnCheck(int rc, const char *file, int line);
void scnExit(int code); // flush, then leave without static destructors
#define SCN_CHECKED(expr) scnCheck((expr), __FILE__, __LINE__)

template <typename t> class vectorCUDA {
private:
  t *d_vec;
  size_t dsize;       // size while on the GPU
  size_t dAllocated;  // elements allocated on the GPU (>= dsize)
  std::vector<t> vec;
  void toCPU(scn_ctx *ctx);
  void toGPU(scn_ctx *ctx);

public:
  vectorCUDA(bool onGPU = true, size_t dsize = 0);
  ~vectorCUDA();
  vectorCUDA(const vectorCUDA &) = delete;
  vectorCUDA &operator=(const vectorCUDA &) = delete;
  vectorCUDA(vectorCUDA &&o);
  bool onGPU;
  void copyToCPU();
  void copyToGPU();
  void copyToCPUAsync(cudaMemStream &memStream);
  void copyToGPUAsync(cudaMemStream &memStream);
  t *&dPtr();
  std::vector<t> &hVector();
  unsigned int size();
  void setZero();
  void setZero(cudaMemStream &memStream);
  void setConstant(float a = 0);
  void setUniform(float a = 0, float b = 1);
  void resize(int n);
  // 64-bit clean variants: the reference's int sizes overflow on feature
  // matrices beyond 2^31 elements (large 3-D batches).  An allocation leaves
  // room for a quarter more and `head` elements.
  void resize64(size_t n, size_t head = 0);
  size_t size64();
};
