// Net runtime, batch production, public facades and canned architectures.
#include <typeinfo>
#include <cstring>
#include <algorithm>
#include <atomic>
#include <cassert>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include "BatchProducer.h"
#include "NetworkArchitectures.h"
#include "SparseConvNet.h"
#include "SparseConvNetCUDA.h"

#define FEATURE_QUANTUM 32 // KERNELBLOCKSIZE of the reference (utilities.h:73)

// ================================================================ runtime
SparseConvNetCUDA::SparseConvNetCUDA(int dimension, int nInputFeatures,
                                     int nClasses, int pciBusID, int nTop,
                                     int nBatchProducerThreads)
    : dimension(dimension), nClasses(nClasses), nTop(nTop),
      inputSpatialSize(0), nInputFeatures(nInputFeatures),
      nOutputFeatures(nInputFeatures), deviceID(0),
      nBatchProducerThreads(nBatchProducerThreads), producerStreamsWanted(0) {
  (void)pciBusID; // one GPU per process: the context picks device 0
  assert(nBatchProducerThreads >= 1 &&
         nBatchProducerThreads <= N_MAX_BATCH_PRODUCER_THREADS);
  std::cout << "Sparse CNN - dimension=" << dimension
            << " nInputFeatures=" << nInputFeatures << " nClasses=" << nClasses
            << std::endl;
  // (lane streams first: streams take hardware queues in order of creation,
  // and the forward passes should not share theirs with producer streams)
  nForwardLanes = nBatchProducerThreads >= 4 ? 2 : 1;
  for (int lane = 1; lane < nForwardLanes; ++lane)
    laneStreams.emplace_back(new cudaMemStream(true, 0));
  batchPool.reserve(nBatchProducerThreads);
  const int nStreams = std::min(nBatchProducerThreads, N_PRODUCER_STREAMS);
  for (int c = 0; c < nStreams; c++) {
    batchMemStreams.emplace_back(new cudaMemStream(false));
    freeProducerStreams.push_back(batchMemStreams.back().get());
  }
  for (int c = 0; c < nBatchProducerThreads; c++) {
    initialSubInterfaces.push_back(new SpatiallySparseBatchSubInterface());
    batchPool.emplace_back(initialSubInterfaces.back());
    batchPool.back().preprocessStream = batchMemStreams[c % nStreams].get();
  }
}
// (between passes: no producer thread holds a stream)
void SparseConvNetCUDA::setProducerStreams(int n) {
  std::lock_guard<std::mutex> lock(streamPoolMutex);
  producerStreamsWanted = n;
  const int all = (int)batchMemStreams.size();
  const int use = n < 1 || n > all ? all : n;
  freeProducerStreams.clear();
  for (int c = 0; c < use; c++)
    freeProducerStreams.push_back(batchMemStreams[c].get());
}
int SparseConvNetCUDA::producerStreamsInUse() {
  std::lock_guard<std::mutex> lock(streamPoolMutex);
  const int all = (int)batchMemStreams.size();
  return producerStreamsWanted < 1 || producerStreamsWanted > all ? all : producerStreamsWanted;
}
cudaMemStream *SparseConvNetCUDA::acquireProducerStream(int batchNumber) {
  std::unique_lock<std::mutex> lock(streamPoolMutex);
  auto mine = waitingBatches.insert(batchNumber);
  streamPoolChanged.wait(lock, [&] {
    return !freeProducerStreams.empty() && *waitingBatches.begin() == batchNumber;
  });
  waitingBatches.erase(mine);
  cudaMemStream *s = freeProducerStreams.front(); // the longest idle one
  freeProducerStreams.erase(freeProducerStreams.begin());
  if (!freeProducerStreams.empty() && !waitingBatches.empty())
    streamPoolChanged.notify_all(); // the next waiter may go too
  return s;
}
void SparseConvNetCUDA::releaseProducerStream(cudaMemStream *stream) {
  {
    std::lock_guard<std::mutex> lock(streamPoolMutex);
    freeProducerStreams.push_back(stream);
  }
  streamPoolChanged.notify_all();
}
cudaMemStream &SparseConvNetCUDA::laneStream(int lane) {
  return lane == 0 ? memStream : *laneStreams[lane - 1];
}
void SparseConvNetCUDA::synchronizeLanes() {
  memStream.synchronize();
  for (auto &s : laneStreams)
    s->synchronize();
}
void SparseConvNetCUDA::limitBatchProducerThreads(int n) {
  if (n < 1 || n >= nBatchProducerThreads)
    return;
  nBatchProducerThreads = n;
  if (n < 4)
    nForwardLanes = 1;
  while ((int)batchPool.size() > n)
    batchPool.pop_back();
  const int nStreams = std::min(n, N_PRODUCER_STREAMS);
  while ((int)batchMemStreams.size() > nStreams)
    batchMemStreams.pop_back();
  setProducerStreams(producerStreamsWanted);
  for (int c = 0; c < n; c++)
    batchPool[c].preprocessStream = batchMemStreams[c % nStreams].get();
}
SparseConvNetCUDA::~SparseConvNetCUDA() {
  for (auto &s : batchMemStreams)
    s->synchronize();
  synchronizeLanes();
  batchPool.clear();
  for (auto p : layers)
    delete p;
  for (auto p : initialSubInterfaces)
    delete p;
  for (auto p : sharedSubInterfaces)
    delete p;
  for (auto &lane : laneSubInterfaces)
    for (auto p : lane)
      delete p;
}
// SparseConvNetCUDA.cu:50-70
void SparseConvNetCUDA::addLearntLayer(int nFeatures,
                                       ActivationFunction activationFn,
                                       float dropout, float alpha) {
  // every learnt layer but the classifier is rounded to a multiple of 32
  if (activationFn != SOFTMAX)
    nFeatures = std::max(FEATURE_QUANTUM, intRound(nFeatures, FEATURE_QUANTUM));
  if (dropout > 0)
    dropout = 1 - (intRound(nFeatures * (1 - dropout), FEATURE_QUANTUM) + 0.01f) *
                      1.0f / nFeatures;
  if (dropout < 0)
    dropout = 0;
  std::cout << layers.size() << ":";
  if (activationFn == PRELU)
    layers.push_back(new NetworkInNetworkPReLULayer(
        memStream, nOutputFeatures, nFeatures, dropout, alpha));
  else
    layers.push_back(new NetworkInNetworkLayer(memStream, nOutputFeatures,
                                               nFeatures, dropout,
                                               activationFn, alpha));
  nOutputFeatures = nFeatures;
}
void SparseConvNetCUDA::addNetworkInNetworkLayer(
    int nFeatures, ActivationFunction activationFn, float dropout) {
  addLearntLayer(nFeatures, activationFn, dropout, 1.0f);
}
// SparseConvNetCUDA.cu:75-98: filterSize 1 adds no gather layer
void SparseConvNetCUDA::addConvolutionalLayer(int nFeatures, int filterSize,
                                              int filterStride,
                                              ActivationFunction activationFn,
                                              float dropout,
                                              int minActiveInputs,
                                              float poolingToFollow) {
  if (filterSize > 1) {
    std::cout << layers.size() << ":";
    layers.push_back(new ConvolutionalLayer(memStream, filterSize, filterStride,
                                            dimension, nOutputFeatures,
                                            minActiveInputs));
    nOutputFeatures *= ipow(filterSize, dimension);
  }
  addLearntLayer(nFeatures, activationFn, dropout,
                 powf(filterSize * 1.0 / filterStride / poolingToFollow, 2));
}
// addLeNetLayerPOFMP / PDFMP / ROFMP / RDFMP (SparseConvNetCUDA.cu:112-163)
void SparseConvNetCUDA::addLeNetLayerFMP(int kind, int nFeatures,
                                         int filterSize, int filterStride,
                                         int poolSize, float fmpShrink,
                                         ActivationFunction activationFn,
                                         float dropout, int minActiveInputs) {
  addConvolutionalLayer(nFeatures, filterSize, filterStride, activationFn,
                        dropout, minActiveInputs, fmpShrink);
  if (fmpShrink > 1) {
    std::cout << layers.size() << ":";
    layers.push_back(new FractionalMaxPoolingLayer(
        memStream, (FmpKind)kind, poolSize, fmpShrink, dimension));
  }
}
void SparseConvNetCUDA::addLeNetLayerMP(int nFeatures, int filterSize,
                                        int filterStride, int poolSize,
                                        int poolStride,
                                        ActivationFunction activationFn,
                                        float dropout, int minActiveInputs) {
  addConvolutionalLayer(nFeatures, filterSize, filterStride, activationFn,
                        dropout, minActiveInputs, poolSize);
  if (poolSize > 1) {
    std::cout << layers.size() << ":";
    layers.push_back(
        new MaxPoolingLayer(memStream, poolSize, poolStride, dimension));
  }
}
void SparseConvNetCUDA::addTriangularConvolutionalLayer(
    int nFeatures, int filterSize, int filterStride,
    ActivationFunction activationFn, float dropout, int minActiveInputs,
    float poolingToFollow) {
  if (filterSize > 1) {
    std::cout << layers.size() << ":";
    layers.push_back(new ConvolutionalTriangularLayer(
        memStream, filterSize, filterStride, dimension, nOutputFeatures,
        minActiveInputs));
    nOutputFeatures *= triangleSize(filterSize, dimension);
  }
  addLearntLayer(nFeatures, activationFn, dropout,
                 powf(filterSize * 1.0 / filterStride / poolingToFollow, 2));
}
// The reference hands (.., dropout, poolSize, minActiveInputs) to a callee
// whose parameters are (.., dropout, minActiveInputs, poolingToFollow)
// (SparseConvNetCUDA.cu:165-168 against :183-185): through this builder the
// convolution's minActiveInputs is the pool size.  Kept, because nets built
// with the reference behave that way.
void SparseConvNetCUDA::addTriangularLeNetLayerMP(
    int nFeatures, int filterSize, int filterStride, int poolSize,
    int poolStride, ActivationFunction activationFn, float dropout,
    int minActiveInputs) {
  addTriangularConvolutionalLayer(nFeatures, filterSize, filterStride,
                                  activationFn, dropout, poolSize,
                                  minActiveInputs);
  if (poolSize > 1) {
    std::cout << layers.size() << ":";
    layers.push_back(new MaxPoolingTriangularLayer(memStream, poolSize,
                                                   poolStride, dimension));
  }
}
void SparseConvNetCUDA::addTerminalPoolingLayer(int poolSize, int S) {
  std::cout << layers.size() << ":";
  layers.push_back(new TerminalPoolingLayer(memStream, poolSize, S));
}
// SparseConvNetCUDA.cu:198-210: classifier, then the spatial sizes are worked
// out from the top (size 1) down to the input field
void SparseConvNetCUDA::addSoftmaxLayer() {
  addLearntLayer(nClasses, SOFTMAX, 0.0f, 1);
  inputSpatialSize = 1;
  std::cout << "Spatially sparse CNN with layer sizes: " << inputSpatialSize;
  for (int i = (int)layers.size() - 1; i >= 0; i--)
    inputSpatialSize = layers[i]->calculateInputSpatialSize(inputSpatialSize);
  std::cout << std::endl;
  std::cout << "Input-field dimensions = " << inputSpatialSize;
  for (int i = 1; i < dimension; ++i)
    std::cout << "x" << inputSpatialSize;
  std::cout << std::endl;
}
void SparseConvNetCUDA::setFusedConvolutions(bool on) {
  for (size_t i = 0; i + 1 < layers.size(); ++i) {
    int nOut = 0;
    if (auto *n = dynamic_cast<NetworkInNetworkLayer *>(layers[i + 1]))
      nOut = n->nFeaturesOut;
    else if (auto *n = dynamic_cast<NetworkInNetworkPReLULayer *>(layers[i + 1]))
      nOut = n->nFeaturesOut;
    if (auto *c = dynamic_cast<ConvolutionalLayer *>(layers[i]))
      c->deferGather =
          on && nOut > 0 &&
          scn_conv_nin_supported(c->nFeaturesOut / c->nFeaturesIn,
                                 c->nFeaturesIn, nOut);
    if (auto *c = dynamic_cast<ConvolutionalTriangularLayer *>(layers[i]))
      c->deferGather =
          on && nOut > 0 &&
          scn_conv_nin_supported(c->nFeaturesOut / c->nFeaturesIn,
                                 c->nFeaturesIn, nOut);
  }
}
void SparseConvNetCUDA::ensureInterfaces() {
  // one shared sub-interface per depth, one interface per depth and slot
  // (BatchProducer.cu:28-33)
  while (batchPool[0].interfaces.size() <= layers.size()) {
    sharedSubInterfaces.push_back(new SpatiallySparseBatchSubInterface());
    for (auto &slot : batchPool)
      slot.interfaces.emplace_back(sharedSubInterfaces.back());
  }
  // ... and one more set per forward lane beyond the first
  laneSubInterfaces.resize(laneStreams.size());
  for (auto &lane : laneSubInterfaces)
    while (lane.size() < sharedSubInterfaces.size())
      lane.push_back(new SpatiallySparseBatchSubInterface());
}
// every grids object the slot owns, emptied in one launch at the start of a batch
static void clearDeviceGrids(scn_ctx *ctx, SpatiallySparseBatch &b) {
  std::vector<scn_grids *> owned;
  for (auto &iface : b.interfaces)
    if (iface.deviceGrids && iface.ownsDeviceGrids)
      owned.push_back(iface.deviceGrids);
  if (!owned.empty())
    SCN_CHECKED(scn_grids_clear_many(ctx, owned.data(), (int)owned.size()));
}
// Every layer's rule book for the batch in slot b, on ctx's stream.  First with
// deferred counts: no host round trip per layer, sizes are upper bounds until
// one scn_rules_settle at the end, after which the real sizes are put in
// place.  A batch that outgrows the bounds (or the first batch of a slot, which
// has no bounds yet: its plans simply wait) is planned again the exact way.
static void planAllLayers(SparseConvNetCUDA &cnn, scn_ctx *ctx,
                          SpatiallySparseBatch &b) {
  for (size_t i = 0; i < cnn.layers.size(); i++) {
    scn_prof_tag(ctx, (int)i);
    cnn.layers[i]->preprocess(b, b.interfaces[i], b.interfaces[i + 1]);
  }
}
static void buildRuleBooks(SparseConvNetCUDA &cnn, scn_ctx *ctx,
                           SpatiallySparseBatch &b, bool mayRunAhead = false) {
  // (plans that continue from one another are recorded and run together)
  SCN_CHECKED(scn_ctx_defer_counts(ctx, 1));
  SCN_CHECKED(scn_ctx_chain_rules(ctx, cnn.chainRuleBooks ? 1 : 0));
  planAllLayers(cnn, ctx, b);
  SCN_CHECKED(scn_ctx_chain_rules(ctx, 0));
  SCN_CHECKED(scn_ctx_defer_counts(ctx, 0));
  // Running ahead: every layer's rows can be read on the device, the result has
  // a row per sample whatever the counts turn out to be, and no bound is refused
  // where the rows there are might not be (32-bit pooling choices).
  bool ahead = mayRunAhead && b.interfaces.back().nSpatialSites == b.batchSize;
  for (size_t i = 1; ahead && i < b.interfaces.size(); ++i) {
    SpatiallySparseBatchInterface &f = b.interfaces[i];
    ahead = (int64_t)f.nSpatialSites * (int64_t)f.featuresPresent.size() <= 2147483647ll &&
            (!f.ownsDeviceGrids || scn_ctx_rows_from(ctx, f.deviceGrids) == SCN_OK);
  }
  SCN_CHECKED(scn_ctx_rows_from(ctx, nullptr));
  if (ahead)
    b.countsPending = true;
  else
    cnn.settleRuleBooks(b);
}
bool SparseConvNetCUDA::settleRuleBooks(SpatiallySparseBatch &b) {
  SparseConvNetCUDA &cnn = *this;
  scn_ctx *ctx = b.preprocessStream ? b.preprocessStream->ctx : memStream.ctx;
  const bool ahead = b.countsPending;
  b.countsPending = false;
  const int rc = scn_rules_settle(ctx);
  if (rc == SCN_ERR_CAPACITY) {
    planAllLayers(cnn, ctx, b); // every plan empties its own output tables again
    return false;
  }
  SCN_CHECKED(rc);
  int held = 1;
  if (ahead)
    SCN_CHECKED(scn_ctx_rows_held(ctx, &held));
  // real sizes: a layer that owns its grids asks them, the others inherit
  for (size_t i = 0; i < cnn.layers.size(); i++) {
    SpatiallySparseBatchInterface &in = b.interfaces[i], &out = b.interfaces[i + 1];
    if (out.ownsDeviceGrids && out.deviceGrids) {
      int32_t nSites = 0;
      int64_t width = 0;
      SCN_CHECKED(scn_grids_info(out.deviceGrids, nullptr, nullptr, nullptr,
                                 nullptr, &nSites));
      SCN_CHECKED(scn_rules_width(out.deviceGrids, &width));
      out.nSpatialSites = nSites;
      out.rules.resize64((size_t)nSites * (size_t)width);
    } else {
      out.nSpatialSites = in.nSpatialSites;
    }
    if (!ahead)
      continue;
    // what the forward pass sized and counted by the bounds
    const size_t n = (size_t)out.nSpatialSites;
    if (out.sub->features.size64() > 0)
      out.sub->features.resize64(n * out.featuresPresent.size());
    if (out.sub->poolingChoices.size64() > 0)
      out.sub->poolingChoices.resize64(n * out.featuresPresent.size());
    int nIn = 0, nOut = 0;
    if (auto *l = dynamic_cast<NetworkInNetworkLayer *>(layers[i]))
      nIn = l->nFeaturesIn, nOut = l->nFeaturesOut;
    else if (auto *l = dynamic_cast<NetworkInNetworkPReLULayer *>(layers[i]))
      nIn = l->nFeaturesIn, nOut = l->nFeaturesOut;
    if (held)
      addMultiplyAdds((__int128_t)n * nIn * nOut);
  }
  return held != 0;
}
// Host-resident input of at least this many bytes is uploaded by the copy
// engine rather than read over the bus by the kernels that use it.
static const size_t kCopyEngineBytes = 4u << 20;
void SparseConvNetCUDA::preprocessResident(int cc, const ResidentBatch &input,
                                           bool mayRunAhead) {
  SpatiallySparseBatch &b = batchPool[cc];
  scn_ctx *ctx = b.preprocessStream ? b.preprocessStream->ctx : memStream.ctx;
  b.reset();
  b.type = UNLABELEDBATCH;
  b.batchSize = input.batchSize;
  SpatiallySparseBatchInterface &in = b.interfaces[0];
  in.nFeatures = nInputFeatures;
  in.spatialSize = inputSpatialSize;
  in.nSpatialSites = input.nSpatialSites;
  in.featuresPresent.hVector() = range(nInputFeatures);
  if (!in.deviceGrids) {
    SCN_CHECKED(scn_grids_create(ctx, &in.deviceGrids));
    in.ownsDeviceGrids = true;
  }
  scn_prof_tag(ctx, -1);
  clearDeviceGrids(ctx, b);
  const int32_t *d_sample = input.d_sample, *d_row = input.d_row,
                *d_background = input.d_background;
  const int64_t *d_key = input.d_key;
  // input.onHost: the arrays are pinned host memory (the upload of
  // BatchProducer.cu:127-134, on this slot's stream).  A small batch is read
  // over the bus by the grid-building kernel and the copy below themselves,
  // which costs no launch of its own.  A large one goes through the copy
  // engine into this slot's staging first: kernels that wait for the bus
  // would hold the wavefront slots that the other batches' layers need for as
  // long as the transfer takes.
  size_t nElems = (size_t)input.nSpatialSites * nInputFeatures;
  const bool byCopyEngine =
      input.onHost &&
      (size_t)input.nActive * 16 + nElems * sizeof(float) >= kCopyEngineBytes;
  if (byCopyEngine) {
    const size_t n = (size_t)input.nActive;
    b.stagingSample.resize64(n);
    b.stagingKey.resize64(2 * n);
    b.stagingRow.resize64(n);
    SCN_CHECKED(scn_h2d_async(ctx, b.stagingSample.dPtr(), d_sample, n * 4));
    SCN_CHECKED(scn_h2d_async(ctx, b.stagingKey.dPtr(), d_key, n * 8));
    SCN_CHECKED(scn_h2d_async(ctx, b.stagingRow.dPtr(), d_row, n * 4));
    d_sample = b.stagingSample.dPtr();
    d_key = (const int64_t *)b.stagingKey.dPtr();
    d_row = b.stagingRow.dPtr();
  }
  in.sub->features.copyToGPU();
  in.sub->features.resize64(nElems);
  SCN_CHECKED(scn_grids_build_copy(
      ctx, in.deviceGrids, input.batchSize, dimension, in.spatialSize, d_sample,
      d_key, d_row, input.nActive, d_background, input.nSpatialSites,
      in.sub->features.dPtr(), input.d_features,
      byCopyEngine ? 0 : nElems * sizeof(float)));
  if (byCopyEngine)
    SCN_CHECKED(scn_h2d_async(ctx, in.sub->features.dPtr(), input.d_features,
                              nElems * sizeof(float)));
  buildRuleBooks(*this, ctx, b, mayRunAhead);
  if (!b.countsPending)
    SCN_CHECKED(scn_sync(ctx));
}
void SparseConvNetCUDA::setPrecision(int precision) {
  for (auto *l : layers) {
    if (auto *n = dynamic_cast<NetworkInNetworkLayer *>(l))
      n->precision = precision;
    if (auto *n = dynamic_cast<NetworkInNetworkPReLULayer *>(l))
      n->precision = precision;
  }
}
// SparseConvNetCUDA.cu:227-271, forward branch
void SparseConvNetCUDA::processBatch(SpatiallySparseBatch &batch,
                                     float learningRate, float momentum,
                                     std::ofstream &f, std::ofstream &g) {
  forwardBatch(batch);
  if (batch.type == TRAINBATCH)
    backwardBatch(batch, learningRate, momentum);
  finishBatch(batch, f, g);
}
// What a backward pass begins with, in one launch: the gradients that layers add to are
// cleared (a dozen launches of 4 us between the others otherwise) and the filters
// turned round.
void SparseConvNetCUDA::startOfBackward(SpatiallySparseBatch &batch, BackwardStart &start) {
  for (size_t i = 0; i < layers.size(); i++) {
    SpatiallySparseBatchInterface &input = batch.interfaces[i];
    const size_t nf = input.featuresPresent.size();
    // (rows of a left out convolution that was gathered all the same are not used)
    if (i == 0 || !batch.interfaces[i - 1].deferredGatherFrom)
      input.gradientSums = 0;
    const size_t own = (size_t)input.nSpatialSites * nf, sums = input.gradientSums * nf;
    // (a pooling whose rules are turned round writes the whole gradient, and the sums
    // where it takes the activation's derivative)
    const bool writes = batch.interfaces[i + 1].poolInverse;
    input.gradientCleared = layers[i]->addsInputGradient() && input.backpropErrors && !writes &&
                            !batch.interfaces[i + 1].deferredGatherFrom;
    input.sumsDone = false;
    input.sumsCleared = sums && !writes;
    if (!input.gradientCleared && !sums)
      continue;
    input.sub->dfeatures.resize64(own + sums);
    if (writes)
      continue;
    start.words.push_back(input.gradientCleared ? own + sums : sums);
    start.clear.push_back(input.sub->dfeatures.dPtr() + (input.gradientCleared ? 0 : own));
  }
  for (size_t i = 0; i < layers.size(); i++)
    layers[i]->transposedFilters(batch.interfaces[i], start.filters);
}
// The training half of processBatch (SparseConvNetCUDA.cu:248-252): the
// classifier has left d cost / d soft-max input in the top interface; every
// layer, last to first, hands the gradient down and updates its weights.
void SparseConvNetCUDA::backwardBatch(SpatiallySparseBatch &batch,
                                      float learningRate, float momentum) {
  // (done already where the forward pass ended in a launch that takes it along)
  if (!batch.backwardStarted) {
    BackwardStart start;
    startOfBackward(batch, start);
    size_t n = start.clear.size();
    for (; n > SCN_FILL_MAX; n -= SCN_FILL_MAX)
      SCN_CHECKED(scn_fill32_many(memStream.ctx, start.clear.data() + n - SCN_FILL_MAX,
                                  start.words.data() + n - SCN_FILL_MAX, SCN_FILL_MAX, 0u));
    for (size_t i = 0; i == 0 || i < start.filters.size(); i += SCN_FILTERS_MAX) {
      SCN_CHECKED(scn_gradients_begin(memStream.ctx, start.clear.data(), start.words.data(), (int)n,
                                      start.filters.data() + i,
                                      (int)std::min<size_t>(SCN_FILTERS_MAX, start.filters.size() - i)));
      n = 0;
    }
  }
  batch.backwardStarted = false;
  batch.updates.clear();
  batch.products.clear();
  batch.collectUpdates = true;
  for (int i = (int)layers.size() - 1; i >= 0; i--) {
    scn_prof_tag(memStream.ctx, i);
    if (i >= 2 && i + 1 == (int)layers.size() &&
        backwardTerminalClassifier(batch, layers[i - 2], layers[i - 1], layers[i], batch.interfaces[i - 2],
                                   batch.interfaces[i - 1], batch.interfaces[i], batch.interfaces[i + 1], memStream,
                                   learningRate, momentum)) {
      --i; // (the pooling, too)
      continue;
    }
    if (i > 0 && layers[i]->choosesInputs())
      layers[i - 1]->activationAhead(batch, batch.interfaces[i - 1],
                                     batch.interfaces[i], batch.interfaces[i + 1]);
    layers[i]->backwards(batch, batch.interfaces[i], batch.interfaces[i + 1],
                         learningRate, momentum);
  }
  batch.collectUpdates = false;
  for (size_t i = 1; i < batch.interfaces.size(); i++)
    batch.interfaces[i].sub->turnedImage = nullptr;
  SCN_CHECKED(scn_weight_images_later(memStream.ctx, nullptr, 0));
  scn_prof_tag(memStream.ctx, -1); // (no layer's)
  for (size_t i = 0; i < batch.products.size(); i += SCN_ATB_MAX)
    SCN_CHECKED(scn_AtB_many(memStream.ctx, batch.products.data() + i,
                             (int)std::min<size_t>(SCN_ATB_MAX, batch.products.size() - i)));
  for (size_t i = 0; i < batch.updates.size(); i += SCN_NAG_MAX)
    SCN_CHECKED(scn_nag_update_many(
        memStream.ctx, batch.updates.data() + i,
        (int)std::min<size_t>(SCN_NAG_MAX, batch.updates.size() - i),
        learningRate, momentum, 1));
  // the backward kernels read the slot's rule books and features: the slot
  // stays with the consumer until the stream has passed this point
  BatchResultStage &r = *batch.result;
  if (!r.consumed)
    SCN_CHECKED(scn_event_create(memStream.ctx, &r.consumed));
  SCN_CHECKED(scn_event_record(memStream.ctx, r.consumed));
  r.consumedPending = true;
}
// The weights as the contractions of this pass read them, all layers' in one
// launch (by themselves 3 to 5 us a layer), side by side in the stream's room: one
// pass at a time reads them.  Made for every batch: nothing is kept that a change
// of the weights could leave behind.
void SparseConvNetCUDA::makeWeightImages(SpatiallySparseBatch &batch, cudaMemStream &ms) {
  std::vector<WeightImage> images;
  for (size_t i = 0; i < layers.size(); i++) {
    SpatiallySparseBatchInterface &input = batch.interfaces[i], &output = batch.interfaces[i + 1];
    output.sub->weightImage = output.sub->turnedImage = nullptr;
    output.sub->roundedToo = output.sub->rounded = false;
    if (batch.type == RESCALEBATCH) // (whose weights change on the way)
      continue;
    if (batch.countsPending)
      SCN_CHECKED(scn_ctx_rows_from(ms.ctx, output.deviceGrids));
    const bool gathers = i > 0 && layers[i - 1]->defersGather(batch, input);
    layers[i]->weightImages(batch, input, output, gathers ? &batch.interfaces[i - 1] : nullptr, images);
  }
  if (batch.countsPending)
    SCN_CHECKED(scn_ctx_rows_from(ms.ctx, nullptr));
  size_t total = 0;
  auto room = [](int64_t bytes) { return ((size_t)bytes + 255) & ~(size_t)255; };
  for (auto &x : images)
    total += room(x.bytes);
  char *at = total ? (char *)ms.imageRoom(total) : nullptr;
  std::vector<scn_image_item> items;
  for (auto &x : images) {
    x.item.d_image = *x.image = at;
    items.push_back(x.item);
    at += room(x.bytes);
  }
  scn_prof_tag(ms.ctx, -1); // (no layer's)
  // (the last of them beside the first layer, where that takes them along)
  size_t i = 0;
  for (; i + SCN_IMAGES_MAX < items.size(); i += SCN_IMAGES_MAX)
    SCN_CHECKED(scn_weight_images_many(ms.ctx, items.data() + i, SCN_IMAGES_MAX));
  SCN_CHECKED(scn_weight_images_later(ms.ctx, items.data() + i, (int)(items.size() - i)));
}
// A convolution whose matrix stays, of channels in other than fours (a net's first
// layer): the layer behind it makes the matrix and reads it in one launch.  Not where
// there is something to do between the two, or channels that a batch leaves out.
bool SparseConvNetCUDA::matrixWithNext(SpatiallySparseBatch &batch, size_t i) const {
  SpatiallySparseBatchInterface &input = batch.interfaces[i], &output = batch.interfaces[i + 1];
  const int nIn = input.nFeatures;
  if (nIn % 4 == 0 || batch.type == TRAINBATCH || batch.type == RESCALEBATCH || i + 1 >= layers.size() ||
      layers[i]->defersGather(batch, output) || (int)input.featuresPresent.size() != nIn ||
      (int)output.featuresPresent.size() != output.nFeatures ||
      !(dynamic_cast<ConvolutionalLayer *>(layers[i]) || dynamic_cast<ConvolutionalTriangularLayer *>(layers[i])))
    return false;
  int nOut = 0;
  if (auto *n = dynamic_cast<NetworkInNetworkLayer *>(layers[i + 1]))
    nOut = n->nFeaturesOut;
  else if (auto *n = dynamic_cast<NetworkInNetworkPReLULayer *>(layers[i + 1]))
    nOut = n->nFeaturesOut;
  return nOut > 0 && scn_conv_nin_supported(output.nFeatures / nIn, nIn, nOut);
}
// The two halves of processBatch.  forwardBatch only queues work on the net's
// stream (every layer, then the copy of the probabilities to the host);
// finishBatch waits for that copy and does the host-side statistics.  The
// dataset loops queue batch i + 1 before finishing batch i, so the stream never
// runs dry while the host is busy.
void SparseConvNetCUDA::forwardBatch(SpatiallySparseBatch &batch, int lane) {
  assert(lane >= 0 && lane < nForwardLanes);
  assert(lane == 0 || (batch.type != TRAINBATCH && batch.type != RESCALEBATCH));
  // the lane's stream and feature buffers
  cudaMemStream &ms = laneStream(lane);
  batch.forwardStream = lane == 0 ? nullptr : &ms;
  for (size_t i = 0; i < layers.size(); i++)
    batch.interfaces[i + 1].sub =
        lane == 0 ? sharedSubInterfaces[i] : laneSubInterfaces[lane - 1][i];
  makeWeightImages(batch, ms);
  // a RESCALEBATCH rescales every layer's weights right after its forward
  // pass (SparseConvNetCUDA.cu:230-241)
  float scalingUnderneath = 1;
  batch.result->copied = batch.result->graded = false;
  batch.backwardStarted = false;
  for (size_t i = 0; i < layers.size(); i++) {
    batch.interfaces[i + 1].sub->reset();
    scn_prof_tag(ms.ctx, (int)i);
    if (batch.countsPending)
      SCN_CHECKED(scn_ctx_rows_from(ms.ctx, batch.interfaces[i + 1].deviceGrids));
    if (i + 2 == layers.size() && isTerminalClassifier(batch, layers[i], layers[i + 1], batch.interfaces[i + 1],
                                                       batch.interfaces[i + 2])) {
      // (of those two layers the backward pass begins with nothing that their forward
      // calls would set; counts that are pending may be other ones by then)
      BackwardStart start;
      const bool begins = batch.type == TRAINBATCH && !batch.countsPending;
      if (begins)
        startOfBackward(batch, start);
      batch.backwardStarted = begins && start.clear.size() <= SCN_FILL_MAX && start.filters.size() <= SCN_FILTERS_MAX;
      forwardTerminalClassifier(batch, layers[i + 1], batch.interfaces[i], batch.interfaces[i + 1],
                                batch.interfaces[i + 2], ms, (int)i + 1, batch.backwardStarted ? &start : nullptr);
      break;
    }
    batch.interfaces[i + 1].matrixWithNext = matrixWithNext(batch, i);
    layers[i]->forwards(batch, batch.interfaces[i], batch.interfaces[i + 1]);
    if (batch.type == RESCALEBATCH) {
      std::cout << i << ":"
                << batch.interfaces[i].sub->features.size64() * sizeof(float) /
                       (1 << 20)
                << "MB ";
      layers[i]->scaleWeights(batch.interfaces[i], batch.interfaces[i + 1],
                              scalingUnderneath, i == layers.size() - 1);
    }
  }
  if (batch.countsPending)
    SCN_CHECKED(scn_ctx_rows_from(ms.ctx, nullptr));
  for (size_t i = 1; i < batch.interfaces.size(); i++) { // (what no layer has taken)
    batch.interfaces[i].sub->weightImage = nullptr;
    batch.interfaces[i].sub->roundedToo = batch.interfaces[i].sub->rounded = false;
  }
  // what no launch has made (a batch of no rows) does not outlast the pass
  if (batch.type != TRAINBATCH)
    SCN_CHECKED(scn_weight_images_later(ms.ctx, nullptr, 0));
  SoftmaxClassifierLaunch(batch.interfaces.back(), batch, ms);
}
void SparseConvNetCUDA::finishBatch(SpatiallySparseBatch &batch,
                                    std::ofstream &f, std::ofstream &g) {
  SoftmaxClassifierCollect(batch.interfaces.back(), batch, nTop);
  if (batch.result->consumedPending) {
    SCN_CHECKED(scn_event_wait(batch.result->consumed));
    batch.result->consumedPending = false;
  }
  if (f.is_open())
    for (auto &p : batch.predictions) {
      for (size_t k = 0; k < p.size(); k++)
        f << (k ? " " : "") << p[k];
      f << std::endl;
    }
  if (g.is_open())
    for (auto &p : batch.probabilities) {
      for (size_t k = 0; k < p.size(); k++)
        g << (k ? " " : "") << p[k];
      g << std::endl;
    }
}
static void printThroughput(long long nanoseconds, size_t nPictures) {
  std::cout << " MegaMultiplyAdds/sample:"
            << roundf(multiplyAddCount / nPictures / 1000000)
            << " time:" << nanoseconds / 1000000000L
            << "s GigaMultiplyAdds/s:" << roundf(multiplyAddCount / nanoseconds)
            << " rate:" << roundf(nPictures * 1000000000.0f / nanoseconds)
            << "/s" << std::endl;
}
ForwardQueue::ForwardQueue(SparseConvNetCUDA &cnn, BatchProducer &bp,
                           bool training)
    : cnn(cnn), count(0) {
  lanes = training ? 1 : cnn.nForwardLanes;
  // a batch stays queued while up to `depth` younger ones are queued behind
  // it; each of them holds a slot, and the producers need one to work in
  depth = std::min(lanes, cnn.nBatchProducerThreads - 1);
  if (depth < lanes)
    lanes = std::max(1, depth);
  bp.keepAlive = depth;
  if (lanes > 1)
    for (int lane = 0; lane < lanes; ++lane) {
      workers.emplace_back(new Worker());
      workers.back()->thread = std::thread(&ForwardQueue::work, this, lane);
    }
}
ForwardQueue::~ForwardQueue() {
  for (auto &w : workers) {
    {
      std::lock_guard<std::mutex> lock(w->m);
      w->stop = true;
    }
    w->cv.notify_all();
    w->thread.join();
  }
}
void ForwardQueue::work(int lane) {
  Worker &w = *workers[lane];
  for (;;) {
    SpatiallySparseBatch *b = nullptr;
    {
      std::unique_lock<std::mutex> lock(w.m);
      w.cv.wait(lock, [&] { return w.stop || !w.todo.empty(); });
      if (w.todo.empty())
        return; // (stop is only set once everything queued has been popped)
      b = w.todo.front();
      w.todo.erase(w.todo.begin());
    }
    cnn.forwardBatch(*b, lane);
    b->result->enqueued.store(true, std::memory_order_release);
  }
}
SpatiallySparseBatch *ForwardQueue::push(SpatiallySparseBatch *b) {
  const int lane = count++ % lanes;
  if (workers.empty()) {
    cnn.forwardBatch(*b, lane);
  } else {
    b->result->enqueued.store(false, std::memory_order_relaxed);
    Worker &w = *workers[lane];
    {
      std::lock_guard<std::mutex> lock(w.m);
      w.todo.push_back(b);
    }
    w.cv.notify_one();
  }
  inFlight.push_back(b);
  if ((int)inFlight.size() > depth)
    return pop();
  return nullptr;
}
SpatiallySparseBatch *ForwardQueue::pop() {
  if (inFlight.empty())
    return nullptr;
  SpatiallySparseBatch *b = inFlight.front();
  inFlight.erase(inFlight.begin());
  // its forward pass may still be on its way into the lane's stream
  while (!b->result->enqueued.load(std::memory_order_acquire))
    std::this_thread::yield();
  return b;
}
// SparseConvNetCUDA.cu:272-326
float SparseConvNetCUDA::processDataset(SpatiallySparseDataset &dataset,
                                        int batchSize, float learningRate,
                                        float momentum) {
  assert(dataset.pictures.size() > 0);
  float errorRate = 0, nll = 0;
  multiplyAddCount = 0;
  auto start = std::chrono::system_clock::now();
  std::ofstream f, g;
  BatchProducer bp(*this, dataset, inputSpatialSize, batchSize, dataset.type == TRAINBATCH);
  if (dataset.type == UNLABELEDBATCH) {
    f.open("unlabelledData.predictions");
    g.open("unlabelledData.probabilities");
  }
  const bool oneLane = dataset.type == TRAINBATCH || dataset.type == RESCALEBATCH;
  ForwardQueue queue(*this, bp, oneLane);
  SpatiallySparseBatch *trainQueued = nullptr; // training batch queued, not yet read
  auto finish = [&](SpatiallySparseBatch *batch) {
    finishBatch(*batch, f, g);
    errorRate += batch->mistakes * 1.0 / dataset.pictures.size();
    nll += batch->negativeLogLikelihood * 1.0 / dataset.pictures.size();
  };
  while (SpatiallySparseBatch *batch = bp.nextBatch()) {
    SpatiallySparseBatch *due = nullptr;
    if (batch->type == TRAINBATCH) {
      forwardBatch(*batch);
      backwardBatch(*batch, learningRate, momentum);
      // (one training batch may stay queued while the next is produced)
      due = trainQueued;
      trainQueued = batch;
      if (!bp.keepAlive) {
        due = batch;
        trainQueued = nullptr;
      }
    } else {
      due = queue.push(batch);
    }
    if (due)
      finish(due);
  }
  if (trainQueued)
    finish(trainQueued);
  while (SpatiallySparseBatch *batch = queue.pop())
    finish(batch);
  auto end = std::chrono::system_clock::now();
  auto diff =
      std::chrono::duration_cast<std::chrono::nanoseconds>(end - start).count();
  if (dataset.type != RESCALEBATCH) { // SparseConvNetCUDA.cu:311
    std::cout << dataset.name;
    if (dataset.type != UNLABELEDBATCH)
      std::cout << " Mistakes:" << 100.0 * errorRate << "% NLL:" << nll;
    printThroughput(diff, dataset.pictures.size());
  }
  return nll;
}
// SparseConvNetCUDA.cu:507-538
void SparseConvNetCUDA::processDatasetDumpTopLevelFeatures(
    SpatiallySparseDataset &dataset, int batchSize, int reps) {
  assert(dataset.pictures.size() > 0);
  assert(dataset.type != TRAINBATCH);
  std::ofstream f((dataset.name + ".features").c_str());
  const size_t n = layers.size();
  for (int rep = 0; rep < reps; rep++) {
    BatchProducer bp(*this, dataset, inputSpatialSize, batchSize);
    while (SpatiallySparseBatch *batch = bp.nextBatch()) {
      for (size_t i = 0; i + 1 < n; i++) {
        batch->interfaces[i + 1].sub->reset();
        layers[i]->forwards(*batch, batch->interfaces[i], batch->interfaces[i + 1]);
      }
      SpatiallySparseBatchInterface &top = batch->interfaces[n - 1];
      assert(top.nFeatures == (int)top.featuresPresent.size());
      assert(!top.deferredGatherFrom); // (a convolution is never the last-but-one layer's output here)
      std::vector<float> &v = top.sub->features.hVector(); // waits for the stream
      std::vector<int> &labels = batch->labels.hVector();
      for (int i = 0; i < batch->batchSize; i++) {
        f << batch->sampleNumbers[i] << " " << labels[i];
        for (int j = 0; j < top.nFeatures; j++)
          f << " " << v[(size_t)i * top.nFeatures + j];
        f << std::endl;
      }
    }
  }
}
// SparseConvNetCUDA.cu:540-566
void SparseConvNetCUDA::calculateInputRegularizingConstants(
    SpatiallySparseDataset dataset) { // a copy of the dataset
  inputNormalizingConstants.resize(0); // no rescaling while measuring
  std::cout << "Using " << std::min(10000, (int)dataset.pictures.size())
            << " out of " << dataset.pictures.size()
            << " training samples to calculate regularizing constants."
            << std::endl;
  if (dataset.pictures.size() > 10000)
    dataset.pictures.resize(10000);
  dataset.type = TESTBATCH; // no dropout, no augmentation
  std::vector<float> c(nInputFeatures, 0);
  {
    BatchProducer bp(*this, dataset, inputSpatialSize, 100);
    while (SpatiallySparseBatch *batch = bp.nextBatch()) {
      std::vector<float> &features = batch->interfaces[0].sub->features.hVector();
      for (size_t i = 0; i < features.size(); ++i)
        c[i % nInputFeatures] =
            std::max(c[i % nInputFeatures], std::fabs(features[i]));
    }
  }
  for (int i = 0; i < nInputFeatures; ++i) {
    inputNormalizingConstants.push_back(c[i] > 0 ? 1.0f / c[i] : 0);
    std::cout << inputNormalizingConstants.back() << " ";
  }
  std::cout << std::endl;
}
// SparseConvNetCUDA.cu:327-405: nReps forward passes, probabilities averaged
void SparseConvNetCUDA::processDatasetRepeatTest(
    SpatiallySparseDataset &dataset, int batchSize, int nReps,
    std::string predictionsFilename, std::string confusionMatrixFilename) {
  assert(dataset.pictures.size() > 0);
  multiplyAddCount = 0;
  auto start = std::chrono::system_clock::now();
  const size_t nPictures = dataset.pictures.size();
  std::vector<std::vector<int>> votes(nPictures,
                                      std::vector<int>(dataset.nClasses));
  std::vector<std::vector<float>> probs(nPictures,
                                        std::vector<float>(dataset.nClasses));
  for (int rep = 1; rep <= nReps; ++rep) {
    {
      BatchProducer bp(*this, dataset, inputSpatialSize, batchSize);
      ForwardQueue queue(*this, bp, false);
      auto finish = [&](SpatiallySparseBatch *batch) {
        std::ofstream f, g;
        finishBatch(*batch, f, g);
        for (int i = 0; i < batch->batchSize; ++i) {
          int ii = batch->sampleNumbers[i];
          votes[ii][batch->predictions[i][0]]++;
          for (int j = 0; j < dataset.nClasses; ++j)
            probs[ii][j] += batch->probabilities[i][j];
        }
      };
      while (SpatiallySparseBatch *batch = bp.nextBatch())
        if (SpatiallySparseBatch *due = queue.push(batch))
          finish(due);
      while (SpatiallySparseBatch *batch = queue.pop())
        finish(batch);
    }
    int errors = (int)nPictures;
    float nll = 0;
    if (dataset.type != UNLABELEDBATCH)
      for (size_t i = 0; i < nPictures; ++i) {
        std::vector<int> predictions = vectorTopIndices(probs[i], nTop);
        for (int j = 0; j < nTop; j++)
          if (predictions[j] == dataset.pictures[i]->label)
            errors--;
        nll -= log(std::max(probs[i][dataset.pictures[i]->label] / rep,
                            (float)1.0e-15));
      }
    if (!predictionsFilename.empty()) {
      std::cout << predictionsFilename << std::endl;
      std::ofstream f(predictionsFilename.c_str());
      if (!dataset.header.empty())
        f << dataset.header << std::endl;
      for (size_t i = 0; i < nPictures; ++i) {
        f << dataset.pictures[i]->identify();
        if (dataset.type != UNLABELEDBATCH)
          f << "," << dataset.pictures[i]->label;
        for (int j = 0; j < dataset.nClasses; ++j)
          f << "," << probs[i][j] / rep;
        f << std::endl;
      }
    }
    if (!confusionMatrixFilename.empty() && dataset.type != UNLABELEDBATCH) {
      std::vector<float> cm((size_t)dataset.nClasses * dataset.nClasses);
      for (size_t i = 0; i < nPictures; ++i)
        for (int j = 0; j < dataset.nClasses; ++j)
          cm[dataset.pictures[i]->label * dataset.nClasses + j] +=
              probs[i][j] / rep;
      std::ofstream f(confusionMatrixFilename.c_str());
      for (int i = 0; i < dataset.nClasses; ++i) {
        for (int j = 0; j < dataset.nClasses; ++j)
          f << cm[i * dataset.nClasses + j] << " ";
        f << std::endl;
      }
    }
    auto end = std::chrono::system_clock::now();
    auto diff = std::chrono::duration_cast<std::chrono::nanoseconds>(end - start)
                    .count();
    std::cout << dataset.name << " rep " << rep << "/" << nReps;
    if (dataset.type != UNLABELEDBATCH)
      std::cout << " Mistakes: " << 100.0 * errors / nPictures << "% NLL "
                << nll / nPictures;
    printThroughput(diff, nPictures);
  }
}
// raw little-endian fp32, no header (SparseConvNetCUDA.cu:406-442)
void SparseConvNetCUDA::loadWeights(std::string baseName, int epoch,
                                    bool momentum, int firstNlayers) {
  std::string filename = baseName + "_epoch-" + std::to_string(epoch) + ".cnn";
  std::ifstream f(filename.c_str(), std::ios::in | std::ios::binary);
  if (!f) {
    std::cout << "Cannot find " << filename << std::endl;
    scnExit(EXIT_FAILURE);
  }
  std::cout << "Loading network parameters from " << filename << std::endl;
  for (int i = 0; i < std::min((int)layers.size(), firstNlayers); i++)
    layers[i]->loadWeightsFromStream(f, momentum);
  if (inputNormalizingConstants.size() > 0)
    f.read((char *)&inputNormalizingConstants[0],
           sizeof(float) * inputNormalizingConstants.size());
}
void SparseConvNetCUDA::saveWeights(std::string baseName, int epoch,
                                    bool momentum) {
  std::string filename = baseName + "_epoch-" + std::to_string(epoch) + ".cnn";
  std::ofstream f(filename.c_str(), std::ios::binary);
  if (!f) {
    std::cout << "Cannot write " << filename << std::endl;
    scnExit(EXIT_FAILURE);
  }
  for (auto *l : layers)
    l->putWeightsToStream(f, momentum);
  if (inputNormalizingConstants.size() > 0)
    f.write((char *)&inputNormalizingConstants[0],
            sizeof(float) * inputNormalizingConstants.size());
}

// ========================================================== batch producer
SpatiallySparseDataset BatchProducer::emptyDataset;

BatchProducer::BatchProducer(SparseConvNetCUDA &cnn,
                             SpatiallySparseDataset &dataset, int spatialSize,
                             int batchSize, bool unseen)
    : cnn(cnn), batchCounter(-1), dataset(dataset), batchSize(batchSize),
      spatialSize(spatialSize), unseen(unseen), stopping(false) {
  assert(batchSize > 0);
  nBatches = ((int)dataset.pictures.size() + batchSize - 1) / batchSize;
  permutation = range((int)dataset.pictures.size());
  if (dataset.type == TRAINBATCH && cnn.shuffleTrainingData) {
    RNG rng; // BatchProducer.cu:23-26
    rng.vectorShuffle(permutation);
  }
  start();
}
BatchProducer::BatchProducer(SparseConvNetCUDA &cnn,
                             const ResidentBatch &residentBatch, int nBatches)
    : BatchProducer(cnn, std::vector<ResidentBatch>(1, residentBatch), nBatches) {}
BatchProducer::BatchProducer(SparseConvNetCUDA &cnn,
                             const std::vector<ResidentBatch> &residentBatches,
                             int nBatches)
    : cnn(cnn), batchCounter(-1), nBatches(nBatches), dataset(emptyDataset),
      batchSize(residentBatches.at(0).batchSize),
      spatialSize(cnn.inputSpatialSize), residents(residentBatches),
      stopping(false) {
  start();
}
void BatchProducer::start() {
  cnn.ensureInterfaces();
  slotFull.assign(cnn.nBatchProducerThreads, 0);
  slotOpen.assign(cnn.nBatchProducerThreads, 0);
  // (pictures that are coded without random numbers, each for itself; a class derived
  // from theirs may do otherwise)
  inParts = residents.empty() && cnn.nBatchProducerThreads > 1;
  for (size_t i = 0; inParts && i < dataset.pictures.size(); ++i)
    inParts = typeid(*dataset.pictures[i]) == typeid(SparsePointsPicture);
  for (int c = 0; c < cnn.nBatchProducerThreads; c++)
    cnn.batchPool[c].batchSize = 0;
  for (int nThread = 0; nThread < cnn.nBatchProducerThreads; ++nThread)
    workers.emplace_back(inParts ? &BatchProducer::sharedProducerThread : &BatchProducer::batchProducerThread, this,
                         nThread);
}
BatchProducer::~BatchProducer() {
  {
    std::lock_guard<std::mutex> lock(slotMutex);
    stopping = true;
  }
  slotChanged.notify_all();
  for (auto &w : workers)
    if (w.joinable())
      w.join();
}
// CPU half of BatchProducer.cu:40-87: distort, codify, normalise
void BatchProducer::openBatch(int c, int cc) {
  SpatiallySparseBatch &b = cnn.batchPool[cc];
  SpatiallySparseBatchInterface &in = b.interfaces[0];
  in.keepGrids(batchSize);
  b.reset();
  b.type = dataset.type;
  b.unseen = unseen;
  in.nFeatures = dataset.nFeatures;
  in.spatialSize = spatialSize;
  in.featuresPresent.hVector() = range(dataset.nFeatures);
  const int last = std::min((c + 1) * batchSize, (int)dataset.pictures.size());
  for (int i = c * batchSize; i < last; i++) {
    b.sampleNumbers.push_back(permutation[i]);
    b.batchSize++;
    if (in.spareGrids.empty()) {
      in.grids.push_back(SparseGrid());
    } else {
      in.grids.push_back(std::move(in.spareGrids.back()));
      in.spareGrids.pop_back();
    }
  }
}
void BatchProducer::normalise(std::vector<float> &features) {
  if (cnn.inputNormalizingConstants.size() > 0)
    for (size_t i = 0; i < features.size(); ++i)
      features[i] *= cnn.inputNormalizingConstants[i % dataset.nFeatures];
}
void BatchProducer::preprocessBatch(int c, int cc, RNG &rng) {
  openBatch(c, cc);
  SpatiallySparseBatch &b = cnn.batchPool[cc];
  SpatiallySparseBatchInterface &in = b.interfaces[0];
  b.parts.resize(std::max<size_t>(b.parts.size(), 1));
  std::vector<float> &features = b.parts[0].features;
  std::vector<int> &labels = b.parts[0].labels;
  features.clear();
  labels.clear();
  for (int i = 0; i < b.batchSize; i++) {
    Picture *const own = dataset.pictures[b.sampleNumbers[i]], *pic = own->distort(rng, dataset.type);
    labels.push_back(pic->label);
    pic->codifyInputData(in.grids[i], features, in.nSpatialSites, in.spatialSize);
    if (pic != own)
      delete pic;
  }
  assert(features.size() == (size_t)in.nFeatures * (size_t)in.nSpatialSites);
  normalise(features);
  b.parts[0].rows = in.nSpatialSites;
  stageBatch(cc, 1);
}
// The pictures of part `part` of batch c, their rows numbered from 0
void BatchProducer::preprocessPart(int c, int cc, int part) {
  SpatiallySparseBatch &b = cnn.batchPool[cc];
  SpatiallySparseBatchInterface &in = b.interfaces[0];
  SpatiallySparseBatch::Part &p = b.parts[part];
  p.features.clear();
  p.rows = 0;
  p.labels.clear();
  for (int i = firstOfPart(b.batchSize, part); i < firstOfPart(b.batchSize, part + 1); ++i) {
    Picture *const pic = dataset.pictures[permutation[c * batchSize + i]];
    p.labels.push_back(pic->label);
    pic->codifyInputData(in.grids[i], p.features, p.rows, in.spatialSize);
  }
  assert(p.features.size() == (size_t)in.nFeatures * (size_t)p.rows);
  normalise(p.features);
}
// The grids as the four arrays scn_grids_build takes, and the features, in
// the slot's pinned staging: still on the CPU's time, no stream is held yet.
void BatchProducer::stageBatch(int cc, int nParts) {
  SpatiallySparseBatch &b = cnn.batchPool[cc];
  SpatiallySparseBatchInterface &in = b.interfaces[0];
  size_t n = 0, nFeatures = 0;
  for (auto &g : in.grids)
    n += g.mp.size();
  for (int part = 0; part < nParts; ++part)
    nFeatures += b.parts[part].features.size();
  b.hostSample.reserve(n * sizeof(int32_t));
  b.hostKey.reserve(n * sizeof(int64_t));
  b.hostRow.reserve(n * sizeof(int32_t));
  b.hostBackground.reserve((size_t)b.batchSize * sizeof(int32_t));
  b.hostFeatures.reserve(nFeatures * sizeof(float));
  int32_t *sample = b.hostSample.as<int32_t>(), *row = b.hostRow.as<int32_t>(),
          *bg = b.hostBackground.as<int32_t>();
  int64_t *key = b.hostKey.as<int64_t>();
  size_t at = 0, to = 0;
  int base = 0; // the rows of the parts before
  for (int part = 0; part < nParts; ++part) {
    const int end = nParts == 1 ? b.batchSize : firstOfPart(b.batchSize, part + 1);
    for (int item = nParts == 1 ? 0 : firstOfPart(b.batchSize, part); item < end; ++item) {
      SparseGrid &g = in.grids[item];
      if (base) {
        g.backgroundCol += g.backgroundCol < 0 ? 0 : base;
        g.mp.addToRows(base);
      }
      bg[item] = g.backgroundCol;
      for (auto &e : g.mp.entries()) {
        sample[at] = item;
        key[at] = e.first;
        row[at] = e.second;
        ++at;
      }
    }
    const SpatiallySparseBatch::Part &p = b.parts[part];
    b.labels.hVector().insert(b.labels.hVector().end(), p.labels.begin(), p.labels.end());
    if (!p.features.empty())
      std::memcpy(b.hostFeatures.as<float>() + to, p.features.data(), p.features.size() * sizeof(float));
    to += p.features.size();
    base += p.rows;
  }
  in.nSpatialSites = base;
  b.hostSites = n;
  b.hostFeatureCount = nFeatures;
}
// Of an unseen training batch the convolutions whose gathered matrix, and that
// matrix's gradient, the layer behind can do without: no dropout on either side,
// and shapes that the fused kernels take, forwards and (turned round) backwards.
static void leaveOutConvolutions(SparseConvNetCUDA &cnn, scn_ctx *ctx, SpatiallySparseBatch &b) {
  std::vector<scn_inverse_item> items;
  for (size_t i = 0; i + 2 < cnn.layers.size(); ++i) { // (the classifier's gradient has no rows for sums)
    SpatiallySparseBatchInterface &in = b.interfaces[i], &middle = b.interfaces[i + 1], &out = b.interfaces[i + 2];
    if ((!dynamic_cast<ConvolutionalLayer *>(cnn.layers[i]) &&
         !dynamic_cast<ConvolutionalTriangularLayer *>(cnn.layers[i])) ||
        (!dynamic_cast<NetworkInNetworkLayer *>(cnn.layers[i + 1]) &&
         !dynamic_cast<NetworkInNetworkPReLULayer *>(cnn.layers[i + 1])))
      continue;
    const int nIn = in.nFeatures, N = out.nFeatures, fs = middle.nFeatures / nIn;
    if ((int)middle.featuresPresent.size() != middle.nFeatures || (int)out.featuresPresent.size() != N ||
        nIn > 4096 || N > 4096 || !scn_conv_nin_supported_p(fs, nIn, N, SCN_FP32) ||
        (in.backpropErrors && !scn_conv_nin_supported_p(fs, N, nIn, SCN_FP32)))
      continue;
    middle.leftOut = true;
    const size_t rows = (size_t)middle.nSpatialSites;
    middle.positions.resize64(scn_positions_pitch(rows) * fs);
    if (in.backpropErrors) {
      out.gradientSums = (size_t)b.batchSize * fs;
      middle.inverse.resize64((size_t)in.nSpatialSites * fs);
      middle.background.resize64(rows + 2 * (size_t)b.batchSize);
    }
    items.push_back({in.deviceGrids, middle.rules.dPtr(), in.backpropErrors ? middle.inverse.dPtr() : nullptr,
                     in.backpropErrors ? middle.background.dPtr() : nullptr, middle.positions.dPtr(),
                     (int64_t)rows, in.nSpatialSites, fs});
  }
  for (size_t i = 0; i < items.size(); i += SCN_INVERSE_MAX)
    SCN_CHECKED(scn_rules_inverse_many(ctx, items.data() + i, (int)std::min<size_t>(SCN_INVERSE_MAX, items.size() - i)));
}
// ... and its poolings' rules turned round, where their windows overlap little: a
// gradient that is read by rows and written once.  A sample's windows are walked by one
// workgroup for its background row, 256 of them in 2 us, so that the longest sample
// decides, not the average: us, turned round and scattered (clearing, adding), of 63800 x
// 32 in 100 samples with one of 2000 25.8, 36.5, of 3000 33.8, 36.4, of 4850 47, 37, of
// 39200 (of 100087) 320, 53; of 63800 x 96 with one of 4800 70, 88, of 8000 95, 92; of 14700
// x 32 with one of 9550 79, 14; of 4 x 2970 x 32 25, 12; of 101700 x 32 voxels, one of
// 13600, 115, 71.  With sums over the background of the convolution before, which the
// scatter leaves to scn_background_sums: of the first of these with one of 8000 85, 91, of
// 21800 215, 149; the voxels 153, 138; 4 x 2970 x 32 31, 20.
static int64_t longestTurned(SpatiallySparseBatchInterface &in, SpatiallySparseBatchInterface &out) {
  const int64_t all = out.nSpatialSites * (int64_t)out.featuresPresent.size();
  return in.gradientSums ? 1000 + 24 * all / 10000 : 600 + 17 * all / 10000;
}
static void turnPoolings(SparseConvNetCUDA &cnn, scn_ctx *ctx, SpatiallySparseBatch &b) {
  std::vector<scn_pool_inverse_item> items;
  std::vector<SpatiallySparseBatchInterface *> outs;
  auto room = [](size_t n) { return (n + 3) & ~(size_t)3; };
  size_t total = 0;
  for (size_t i = 0; i < cnn.layers.size(); ++i) {
    MaxPoolingLayer *const pool = dynamic_cast<MaxPoolingLayer *>(cnn.layers[i]);
    SpatiallySparseBatchInterface &in = b.interfaces[i], &out = b.interfaces[i + 1];
    if (!pool || !in.backpropErrors)
      continue;
    const int slots = scn_pool_inverse_slots(pool->dimension, pool->poolSize, pool->poolStride);
    const int64_t nf = (int64_t)out.featuresPresent.size();
    if (slots == 0 || nf % 4 != 0 || nf == 0 || in.nSpatialSites * std::max<int64_t>(nf, slots) > 0x7fffffffll ||
        out.nSpatialSites * nf > 0x7fffffffll ||
        out.nSpatialSites > longestTurned(in, out) * b.batchSize) // (one is as long as the average)
      continue;
    out.poolSlots = slots;
    items.push_back({in.deviceGrids, out.deviceGrids, out.rules.dPtr(), nullptr, nullptr, out.nSpatialSites,
                     in.nSpatialSites, pool->poolSize, pool->poolStride});
    outs.push_back(&out);
    total += room((size_t)in.nSpatialSites * slots) + room(2 * (size_t)b.batchSize + 1);
  }
  if (items.empty())
    return;
  b.poolInverses.resize64(total);
  int *at = b.poolInverses.dPtr();
  for (size_t k = 0; k < items.size(); ++k) {
    items[k].d_inverse = at;
    at += room((size_t)items[k].inputRows * outs[k]->poolSlots);
    items[k].d_samples = at;
    at += room(2 * (size_t)b.batchSize + 1);
    outs[k]->poolInverse = items[k].d_inverse;
    outs[k]->poolSamples = items[k].d_samples;
  }
  const size_t starts = (size_t)b.batchSize + 1;
  b.poolStarts.reserve(items.size() * starts * sizeof(int32_t));
  for (size_t i = 0; i < items.size(); i += SCN_INVERSE_MAX)
    SCN_CHECKED(scn_pool_inverse_many_copy(ctx, items.data() + i, (int)std::min<size_t>(SCN_INVERSE_MAX, items.size() - i),
                                           b.poolStarts.as<int32_t>() + i * starts));
}
// (when the stream is through: the poolings with a sample too long are scattered)
static void keepTurnedPoolings(SparseConvNetCUDA &cnn, SpatiallySparseBatch &b) {
  const int32_t *first = b.poolStarts.as<int32_t>();
  for (size_t i = 1; i < b.interfaces.size(); ++i) {
    SpatiallySparseBatchInterface &out = b.interfaces[i];
    if (!out.poolInverse)
      continue;
    int64_t longest = 0;
    for (int s = 0; s < b.batchSize; ++s)
      longest = std::max<int64_t>(longest, first[s + 1] - first[s]);
    first += b.batchSize + 1;
    if (longest > longestTurned(b.interfaces[i - 1], out))
      out.poolInverse = out.poolSamples = nullptr;
    else
      ++cnn.poolingsTurned;
  }
}
// GPU half: the input grids go to HBM, then every layer builds its rule book,
// all on the slot's stream
void BatchProducer::preprocessBatchOnDevice(int cc) {
  SpatiallySparseBatch &b = cnn.batchPool[cc];
  SpatiallySparseBatchInterface &in = b.interfaces[0];
  cudaMemStream &ms = b.preprocessStream ? *b.preprocessStream : cnn.memStream;
  scn_ctx *ctx = ms.ctx;
  // (flattened into pinned memory by stageBatch; read from there or copied first as in
  // preprocessResident: five queued copies of a megabyte kept a thread for 100 to 160 us
  // beside nine others)
  const size_t n = b.hostSites, bytes = b.hostFeatureCount * sizeof(float);
  const bool byCopyEngine = n * 16 + bytes >= kCopyEngineBytes;
  const int32_t *sample = b.hostSample.as<int32_t>(), *row = b.hostRow.as<int32_t>();
  const int64_t *key = b.hostKey.as<int64_t>();
  if (byCopyEngine) {
    b.stagingSample.resize64(n);
    b.stagingKey.resize64(2 * n);
    b.stagingRow.resize64(n);
    SCN_CHECKED(scn_h2d_async(ctx, b.stagingSample.dPtr(), sample, n * 4));
    SCN_CHECKED(scn_h2d_async(ctx, b.stagingKey.dPtr(), key, n * 8));
    SCN_CHECKED(scn_h2d_async(ctx, b.stagingRow.dPtr(), row, n * 4));
    sample = b.stagingSample.dPtr();
    key = (const int64_t *)b.stagingKey.dPtr();
    row = b.stagingRow.dPtr();
  }
  if (!in.deviceGrids) {
    SCN_CHECKED(scn_grids_create(ctx, &in.deviceGrids));
    in.ownsDeviceGrids = true;
  }
  scn_prof_tag(ctx, -1);
  clearDeviceGrids(ctx, b);
  in.sub->features.copyToGPU(); // (its host vector is empty: nothing moves)
  in.sub->features.resize64(b.hostFeatureCount);
  SCN_CHECKED(scn_grids_build_copy(ctx, in.deviceGrids, b.batchSize, cnn.dimension, in.spatialSize, sample, key, row,
                                   (int64_t)n, b.hostBackground.as<int32_t>(), in.nSpatialSites,
                                   in.sub->features.dPtr(), b.hostFeatures.p, byCopyEngine ? 0 : bytes));
  if (byCopyEngine)
    SCN_CHECKED(scn_h2d_async(ctx, in.sub->features.dPtr(), b.hostFeatures.p, bytes));
  if (b.type == TRAINBATCH) {
    // the classifier's gradient reads the labels on the device: uploaded here,
    // on this slot's stream, so that the net's stream is never waited for
    b.result->labels = b.labels.hVector();
    b.labels.copyToGPUAsync(ms);
  }
  buildRuleBooks(cnn, ctx, b);
  if (b.unseen) {
    leaveOutConvolutions(cnn, ctx, b);
    turnPoolings(cnn, ctx, b);
  }
  SCN_CHECKED(scn_sync(ctx));
  keepTurnedPoolings(cnn, b);
}
void BatchProducer::batchProducerThread(int nThread) {
  RNG rng;
  for (int c = nThread; c < nBatches; c += cnn.nBatchProducerThreads) {
    {
      std::unique_lock<std::mutex> lock(slotMutex);
      slotChanged.wait(lock, [&] { return stopping || !slotFull[nThread]; });
      if (stopping)
        return;
    }
    {
      std::lock_guard<std::mutex> slot(cnn.batchLock[nThread]);
      const bool resident = !residents.empty();
      if (!resident)
        preprocessBatch(c, nThread, rng); // CPU half
      // GPU half, on a stream borrowed for it
      cudaMemStream *stream = cnn.acquireProducerStream(c);
      cnn.batchPool[nThread].preprocessStream = stream;
      if (resident)
        cnn.preprocessResident(nThread, residents[c % residents.size()]);
      else
        preprocessBatchOnDevice(nThread);
      cnn.releaseProducerStream(stream);
    }
    {
      std::lock_guard<std::mutex> lock(slotMutex);
      slotFull[nThread] = 1;
    }
    slotChanged.notify_all();
  }
}
int BatchProducer::firstOfPart(int size, int part) const {
  return (int)((int64_t)size * part / cnn.nBatchProducerThreads);
}
// The threads take the pictures in the order of the batches, a part of a batch at a
// time, and the one that ends a batch's last part does its GPU half: the first batch of
// an epoch, for which the net waits, is coded by all of them in a tenth of the time (400
// us beside nine others that code the next ones), and is alone in launching its rule
// books' kernels.
void BatchProducer::sharedProducerThread(int) {
  RNG rng; // (not drawn from: with SCN_SEED set, the generators made later have the numbers that they had)
  const int nSlots = cnn.nBatchProducerThreads;
  for (;;) {
    int c, cc, part;
    {
      std::unique_lock<std::mutex> lock(slotMutex);
      slotChanged.wait(lock, [&] {
        return stopping || nextOpen >= nBatches || nextPart || (!opening && !slotOpen[nextOpen % nSlots]);
      });
      if (stopping || nextOpen >= nBatches)
        return;
      c = nextOpen;
      cc = c % nSlots;
      if (nextPart == 0) { // (this thread's batch until it has parts to take)
        slotOpen[cc] = 1;
        opening = true;
        lock.unlock();
        SpatiallySparseBatch &b = cnn.batchPool[cc];
        openBatch(c, cc);
        b.parts.resize(std::max<size_t>(b.parts.size(), nSlots));
        b.partsLeft = nSlots;
        lock.lock();
        opening = false;
      }
      part = nextPart++;
      if (nextPart == nSlots) {
        ++nextOpen;
        nextPart = 0;
        if (nextOpen >= nBatches)
          slotChanged.notify_all();
      }
    }
    if (part == 0)
      slotChanged.notify_all(); // (who waited for the slot has parts to take)
    preprocessPart(c, cc, part);
    {
      std::lock_guard<std::mutex> lock(slotMutex);
      if (--cnn.batchPool[cc].partsLeft > 0)
        continue;
    }
    stageBatch(cc, nSlots);
    cudaMemStream *stream = cnn.acquireProducerStream(c);
    cnn.batchPool[cc].preprocessStream = stream;
    preprocessBatchOnDevice(cc);
    cnn.releaseProducerStream(stream);
    {
      std::lock_guard<std::mutex> lock(slotMutex);
      slotFull[cc] = 1;
    }
    slotChanged.notify_all();
  }
}
int BatchProducer::slotsReady() {
  std::lock_guard<std::mutex> lock(slotMutex);
  int n = 0;
  for (char full : slotFull)
    n += full != 0;
  // (slots of batches already handed out stay marked until they are given back)
  const int out = std::min(batchCounter + 1, keepAlive + 1);
  return std::max(0, n - std::max(0, out));
}
SpatiallySparseBatch *BatchProducer::nextBatch() {
  if (batchCounter - keepAlive >= 0) { // hand a finished slot back to its worker
    int cc = (batchCounter - keepAlive) % cnn.nBatchProducerThreads;
    const BatchResultStage &r = *cnn.batchPool[cc].result;
    if (r.pending || r.consumedPending) {
      std::fprintf(stderr, "BatchProducer: slot %d handed back while the net's "
                           "stream may still read it\n", cc);
      scnExit(EXIT_FAILURE);
    }
    cnn.batchPool[cc].batchSize = 0;
    {
      std::lock_guard<std::mutex> lock(slotMutex);
      slotFull[cc] = slotOpen[cc] = 0;
    }
    slotChanged.notify_all();
  }
  batchCounter++;
  if (batchCounter >= nBatches) {
    for (auto &w : workers)
      if (w.joinable())
        w.join();
    return NULL;
  }
  int cc = batchCounter % cnn.nBatchProducerThreads;
  {
    std::unique_lock<std::mutex> lock(slotMutex);
    slotChanged.wait(lock, [&] { return slotFull[cc] != 0; });
  }
  return &cnn.batchPool[cc];
}

// ================================================================= facades
SparseConvNet::SparseConvNet(int dimension, int nInputFeatures, int nClasses,
                             int pciBusID, int nTop)
    : cnn(new SparseConvNetCUDA(dimension, nInputFeatures, nClasses, pciBusID,
                                nTop)) {}
SparseConvNet::~SparseConvNet() {}
void SparseConvNet::addLeNetLayerMP(int nFeatures, int filterSize,
                                    int filterStride, int poolSize,
                                    int poolStride,
                                    ActivationFunction activationFn,
                                    float dropout, int minActiveInputs) {
  cnn->addLeNetLayerMP(nFeatures, filterSize, filterStride, poolSize,
                       poolStride, activationFn, dropout, minActiveInputs);
}
void SparseConvNet::addLeNetLayerPOFMP(int nFeatures, int filterSize,
                                       int filterStride, int poolSize,
                                       float fmpShrink,
                                       ActivationFunction activationFn,
                                       float dropout, int minActiveInputs) {
  cnn->addLeNetLayerFMP(FMP_PSEUDORANDOM_OVERLAPPING, nFeatures, filterSize, filterStride, poolSize,
                        fmpShrink, activationFn, dropout, minActiveInputs);
}
void SparseConvNet::addLeNetLayerROFMP(int nFeatures, int filterSize,
                                       int filterStride, int poolSize,
                                       float fmpShrink,
                                       ActivationFunction activationFn,
                                       float dropout, int minActiveInputs) {
  cnn->addLeNetLayerFMP(FMP_RANDOM_OVERLAPPING, nFeatures, filterSize, filterStride, poolSize,
                        fmpShrink, activationFn, dropout, minActiveInputs);
}
void SparseConvNet::addLeNetLayerPDFMP(int nFeatures, int filterSize,
                                       int filterStride, int poolSize,
                                       float fmpShrink,
                                       ActivationFunction activationFn,
                                       float dropout, int minActiveInputs) {
  cnn->addLeNetLayerFMP(FMP_PSEUDORANDOM_NONOVERLAPPING, nFeatures, filterSize, filterStride, poolSize,
                        fmpShrink, activationFn, dropout, minActiveInputs);
}
void SparseConvNet::addLeNetLayerRDFMP(int nFeatures, int filterSize,
                                       int filterStride, int poolSize,
                                       float fmpShrink,
                                       ActivationFunction activationFn,
                                       float dropout, int minActiveInputs) {
  cnn->addLeNetLayerFMP(FMP_RANDOM_NONOVERLAPPING, nFeatures, filterSize, filterStride, poolSize,
                        fmpShrink, activationFn, dropout, minActiveInputs);
}
void SparseConvNet::addTerminalPoolingLayer(int poolSize) {
  cnn->addTerminalPoolingLayer(poolSize, ipow(poolSize, cnn->dimension));
}
void SparseConvNet::addSoftmaxLayer() { cnn->addSoftmaxLayer(); }
float SparseConvNet::processDataset(SpatiallySparseDataset &dataset,
                                    int batchSize, float learningRate,
                                    float momentum) {
  return cnn->processDataset(dataset, batchSize, learningRate, momentum);
}
void SparseConvNet::processDatasetRepeatTest(
    SpatiallySparseDataset &dataset, int batchSize, int nReps,
    std::string predictionsFilename, std::string confusionMatrixFilename) {
  cnn->processDatasetRepeatTest(dataset, batchSize, nReps, predictionsFilename,
                                confusionMatrixFilename);
}
void SparseConvNet::processDatasetDumpTopLevelFeatures(
    SpatiallySparseDataset &dataset, int batchSize, int reps) {
  cnn->processDatasetDumpTopLevelFeatures(dataset, batchSize, reps);
}
void SparseConvNet::calculateInputRegularizingConstants(
    SpatiallySparseDataset dataset) {
  cnn->calculateInputRegularizingConstants(dataset);
}
void SparseConvNet::loadWeights(std::string baseName, int epoch, bool momentum,
                                int firstNlayers) {
  cnn->loadWeights(baseName, epoch, momentum, firstNlayers);
}
void SparseConvNet::saveWeights(std::string baseName, int epoch,
                                bool momentum) {
  cnn->saveWeights(baseName, epoch, momentum);
}

SparseConvTriangLeNet::SparseConvTriangLeNet(int dimension, int nInputFeatures,
                                             int nClasses, int pciBusID,
                                             int nTop)
    : cnn(new SparseConvNetCUDA(dimension, nInputFeatures, nClasses, pciBusID,
                                nTop)) {}
SparseConvTriangLeNet::~SparseConvTriangLeNet() {}
void SparseConvTriangLeNet::addLeNetLayerMP(int nFeatures, int filterSize,
                                            int filterStride, int poolSize,
                                            int poolStride,
                                            ActivationFunction activationFn,
                                            float dropout,
                                            int minActiveInputs) {
  cnn->addTriangularLeNetLayerMP(nFeatures, filterSize, filterStride, poolSize,
                                 poolStride, activationFn, dropout,
                                 minActiveInputs);
}
void SparseConvTriangLeNet::addTerminalPoolingLayer(int poolSize) {
  cnn->addTerminalPoolingLayer(poolSize,
                               triangleSize(poolSize, cnn->dimension));
}
void SparseConvTriangLeNet::addSoftmaxLayer() { cnn->addSoftmaxLayer(); }
float SparseConvTriangLeNet::processDataset(SpatiallySparseDataset &dataset,
                                            int batchSize, float learningRate,
                                            float momentum) {
  return cnn->processDataset(dataset, batchSize, learningRate, momentum);
}
void SparseConvTriangLeNet::processDatasetRepeatTest(
    SpatiallySparseDataset &dataset, int batchSize, int nReps,
    std::string predictionsFilename, std::string confusionMatrixFilename) {
  cnn->processDatasetRepeatTest(dataset, batchSize, nReps, predictionsFilename,
                                confusionMatrixFilename);
}
void SparseConvTriangLeNet::processDatasetDumpTopLevelFeatures(
    SpatiallySparseDataset &dataset, int batchSize, int reps) {
  cnn->processDatasetDumpTopLevelFeatures(dataset, batchSize, reps);
}
void SparseConvTriangLeNet::calculateInputRegularizingConstants(
    SpatiallySparseDataset dataset) {
  cnn->calculateInputRegularizingConstants(dataset);
}
void SparseConvTriangLeNet::loadWeights(std::string baseName, int epoch,
                                        bool momentum, int firstNlayers) {
  cnn->loadWeights(baseName, epoch, momentum, firstNlayers);
}
void SparseConvTriangLeNet::saveWeights(std::string baseName, int epoch,
                                        bool momentum) {
  cnn->saveWeights(baseName, epoch, momentum);
}

// ============================================================ architectures
// NetworkArchitectures.cpp:3-68
DeepCNet::DeepCNet(int dimension, int l, int k, ActivationFunction fn,
                   int nInputFeatures, int nClasses, float p, int cudaDevice,
                   int nTop)
    : SparseConvNet(dimension, nInputFeatures, nClasses, cudaDevice, nTop) {
  for (int i = 0; i <= l; i++)
    addLeNetLayerMP((i + 1) * k, i == 0 ? 3 : 2, 1, i < l ? 3 : 1,
                    i < l ? 2 : 1, fn, p * i * 1.0f / l);
  addSoftmaxLayer();
}
DeepC2::DeepC2(int dimension, int l, int k, ActivationFunction fn,
               int nInputFeatures, int nClasses, float p, int cudaDevice,
               int nTop)
    : SparseConvNet(dimension, nInputFeatures, nClasses, cudaDevice, nTop) {
  for (int i = 0; i <= l; i++)
    addLeNetLayerMP((i + 1) * k, 2, 1, i < l ? 3 : 1, i < l ? 2 : 1, fn,
                    p * i * 1.0f / l);
  addSoftmaxLayer();
}
DeepCNiN::DeepCNiN(int dimension, int l, int k, ActivationFunction fn,
                   int nInputFeatures, int nClasses, float p, int cudaDevice,
                   int nTop)
    : SparseConvNet(dimension, nInputFeatures, nClasses, cudaDevice, nTop) {
  for (int i = 0; i <= l; i++) {
    addLeNetLayerMP((i + 1) * k, 2, 1, i < l ? 3 : 1, i < l ? 2 : 1, fn,
                    p * i * 1.0f / l);
    addLeNetLayerMP((i + 1) * k, 1, 1, 1, 1, fn, p * i * 1.0f / l);
  }
  addSoftmaxLayer();
}
DeepC2C2::DeepC2C2(int dimension, int l, int k, ActivationFunction fn,
                   int nInputFeatures, int nClasses, float p, int cudaDevice,
                   int nTop)
    : SparseConvNet(dimension, nInputFeatures, nClasses, cudaDevice, nTop) {
  for (int i = 0; i < l; i++) {
    addLeNetLayerMP((i + 1) * k, 2, 1, 1, 1, fn, p * i * 1.0f / l);
    addLeNetLayerMP((i + 1) * k, 2, 1, 3, 2, fn, p * i * 1.0f / l);
  }
  addLeNetLayerMP((l + 1) * k, 2, 1, 1, 1, fn, p);
  addLeNetLayerMP((l + 1) * k, 1, 1, 1, 1, fn, p);
  addSoftmaxLayer();
}
DeepC3C3::DeepC3C3(int dimension, int l, int k, ActivationFunction fn,
                   int nInputFeatures, int nClasses, float p, int cudaDevice,
                   int nTop)
    : SparseConvNet(dimension, nInputFeatures, nClasses, cudaDevice, nTop) {
  for (int i = 0; i < l; i++) {
    addLeNetLayerMP((i + 1) * k, 3, 1, 1, 1, fn, p * i * 1.0f / l);
    addLeNetLayerMP((i + 1) * k, 3, 1, 3, 2, fn, p * i * 1.0f / l);
  }
  addLeNetLayerMP((l + 1) * k, 3, 1, 1, 1, fn, p);
  addLeNetLayerMP((l + 1) * k, 1, 1, 1, 1, fn, p);
  addSoftmaxLayer();
}
DeepC3C3Valid::DeepC3C3Valid(int dimension, int l, int k,
                             ActivationFunction fn, int nInputFeatures,
                             int nClasses, float p, int cudaDevice, int nTop)
    : SparseConvNet(dimension, nInputFeatures, nClasses, cudaDevice, nTop) {
  for (int i = 0; i < l; i++) {
    addLeNetLayerMP((i + 1) * k, 3, 1, 1, 1, fn, p * i * 1.0f / l, -1);
    addLeNetLayerMP((i + 1) * k, 3, 1, 3, 2, fn, p * i * 1.0f / l, -1);
  }
  // one ordinary convolution at the end, in case no site survived
  addLeNetLayerMP((l + 1) * k, 3, 1, 1, 1, fn, p, +1);
  addLeNetLayerMP((l + 1) * k, 1, 1, 1, 1, fn, p);
  addSoftmaxLayer();
}

// NetworkArchitectures.cpp:72-122: l levels of C2 + fractional max-pooling,
// then C2 and a 1x1 NiN, dropout rising to p
#define SCN_FMP_ARCHITECTURE(Name, Builder)                                    \
  Name::Name(int dimension, int l, int k, float fmpShrink,                     \
             ActivationFunction fn, int nInputFeatures, int nClasses, float p, \
             int cudaDevice, int nTop)                                         \
      : SparseConvNet(dimension, nInputFeatures, nClasses, cudaDevice, nTop) { \
    for (int i = 0; i < l; i++)                                                \
      Builder(k * (i + 1), 2, 1, 2, fmpShrink, fn, p * i / (l + 1));           \
    addLeNetLayerMP(k * (l + 1), 2, 1, 1, 1, fn, p * l / (l + 1));             \
    addLeNetLayerMP(k * (l + 2), 1, 1, 1, 1, fn, p);                           \
    addSoftmaxLayer();                                                         \
  }
SCN_FMP_ARCHITECTURE(POFMPSparseConvNet, addLeNetLayerPOFMP)
SCN_FMP_ARCHITECTURE(ROFMPSparseConvNet, addLeNetLayerROFMP)
SCN_FMP_ARCHITECTURE(PDFMPSparseConvNet, addLeNetLayerPDFMP)
SCN_FMP_ARCHITECTURE(RDFMPSparseConvNet, addLeNetLayerRDFMP)
#undef SCN_FMP_ARCHITECTURE
