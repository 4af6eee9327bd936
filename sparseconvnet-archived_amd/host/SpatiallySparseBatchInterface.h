// Data carried between layers (SpatiallySparseBatchInterface.h:8-46).
#pragma once
#include <vector>
#include "SparseGrid.h"
#include "vectorCUDA.h"

// The large vectors of one depth; they stay in HBM and are shared by every
// batch slot (BatchProducer.cu:28-33).
class SpatiallySparseBatchSubInterface {
public:
  vectorCUDA<float> features;
  vectorCUDA<float> dfeatures; // gradient of the cost, training batches only
  vectorCUDA<float> dactivated; // of a pooling's output: that, times the derivative of the layer below
  vectorCUDA<int> poolingChoices;
  // room for a bf16 copy of `features` (two bytes an element), for a following fused
  // convolution with bf16 operands: made by it, where its window is large enough for
  // the rows to be read many times over, or
  vectorCUDA<float> features16;
  // by the pooling that makes the features: is to be, and has been in this pass, in the
  // room behind them, from that element on (allocations of its own were two of a new
  // wide net's first pass)
  bool roundedToo = false, rounded = false;
  size_t roundedAt = 0;
  float *roundedRows() { return features.dPtr() + roundedAt; }
  // the weights of the layer whose output this is, laid out for its forward pass
  // and, turned round, for the gradient of its input: made for one batch by
  // SparseConvNetCUDA::makeWeightImages, in the stream's room for them, and used up
  // by the layer (null: none)
  void *weightImage = nullptr, *turnedImage = nullptr;
  SpatiallySparseBatchSubInterface();
  void reset();
};

class SpatiallySparseBatchInterface {
public:
  SpatiallySparseBatchSubInterface *sub;
  int nFeatures;                   // features per spatial location
  vectorCUDA<int> featuresPresent; // all of them, except under dropout in a training batch
  int nSpatialSites; // active rows of the whole batch, background rows included
  int spatialSize;
  bool backpropErrors;
  // sub->dfeatures has been cleared for the layer that adds to it next
  // (SparseConvNetCUDA::backwardBatch clears those of a whole pass at once)
  bool gradientCleared = false;
  // a layer's output: the activation's derivative is in dfeatures already (taken
  // over the outputs of the pooling behind it), and, with activationAhead, the bias
  // gradient has been summed; a pooling's: sub->dactivated holds what it is to
  // spread (activationAhead), or it takes the derivative of `through` itself
  bool activationDone = false, activationAhead = false;
  int through = -1;
  // A convolution's output in a batch nobody looks into (SpatiallySparseBatch::
  // unseen) whose matrix and gradient are left out: the rules turned round
  // (scn_rules_inverse_many; all but the positions empty where no gradient of its
  // input is wanted).
  bool leftOut = false;
  vectorCUDA<int> inverse, background, positions;
  // rows of sub->dfeatures behind the layer's own: sums over the background of
  // such a convolution's input; they are there, or cleared for scn_background_sums
  // to add to
  size_t gradientSums = 0;
  bool sumsDone = false, sumsCleared = false;
  // A pooling's output in such a batch: its rules turned round (scn_pool_inverse_many;
  // in the batch's room for them, for as long as it is this batch), null: the
  // gradient is scattered
  const int *poolInverse = nullptr, *poolSamples = nullptr;
  int poolSlots = 0;
  // Host view of the sparse grids.  Filled by the Pictures for the input
  // interface; for deeper interfaces the grids are built in HBM
  // (deviceGrids) and this view is only materialised by downloadGrids().
  std::vector<SparseGrid> grids;
  // A picture batch's input: the last batch's grids, empty, for the next one's to be
  // built in (keepGrids, by the producer that fills them; no more than a batch has).
  // Ten producers that allocate and free a hundred grids each hold one another up (a
  // batch's half on the CPU 0.6 to 1.7 ms, and 0.45 to 0.65 for most of them without).
  std::vector<SparseGrid> spareGrids;
  scn_grids *deviceGrids;
  bool ownsDeviceGrids;
  vectorCUDA<int> rules;
  // Output of a fractional max-pooling layer: the regions drawn for this
  // batch, inputL then inputR, each [batchSize][dimension][spatialSize].
  std::vector<int> regionTicks;
  // Set by a convolutional layer that left its gather to the following NiN
  // layer (fused kernel): the interface whose features the rules index.  The
  // feature matrix of THIS interface is then not materialised.
  SpatiallySparseBatchInterface *deferredGatherFrom;
  // ... and that layer leaves the matrix here as well (a pass over the net says
  // so: SparseConvNetCUDA::forwardBatch)
  bool matrixWithNext = false;
  SpatiallySparseBatchInterface(SpatiallySparseBatchSubInterface *s);
  SpatiallySparseBatchInterface(SpatiallySparseBatchInterface &&o);
  ~SpatiallySparseBatchInterface();
  void downloadGrids(int batchSize);
  void keepGrids(size_t most); // grids become spare ones
  void summary();
  void reset();
};
