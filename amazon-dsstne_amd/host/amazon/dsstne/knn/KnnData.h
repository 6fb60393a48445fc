// KnnData.h — device-resident item table and result buffers of the exact KNN search (reference: knn/KnnData.h:33-140).
// One GPU: numGpus must be 1.  The item table is stored column-major [rowsPadded x D] as the reference builds it.
#ifndef DSSTNE_AMD_KNN_KNNDATA_H
#define DSSTNE_AMD_KNN_KNNDATA_H

#include <cstdint>
#include <map>
#include <string>
#include <vector>

#include "DataReader.h"

namespace astdl {
namespace knn {

// FP32 and FP16 as in the reference (knn/KnnData.h).  FP32Split ("fp32-split") has no counterpart there: fp32 storage whose
// inner products are formed from bf16 matrix instructions (dsx_knn_search_split): fp32-accurate scores, not bit-identical to
// FP32's, about 1.5 times as fast; the table is kept as bf16 planes, 1.5 times its fp32 size.
enum class DataType { FP32 = 0, FP16 = 1, FP32Split = 2 };

std::string getDataTypeString(DataType dataType);
DataType getDataTypeFromString(const std::string& dataTypeLiteral);

enum class MemoryType { Host = 1, Device = 2 };

struct Matrix {
    void* data;
    uint32_t numRows;
    int numColumns;
    size_t elementSize;
    MemoryType memoryType;

    Matrix();
    Matrix(void* data, uint32_t numRows, int numColumns, size_t elementSize, MemoryType memoryType);
    size_t getSizeInBytes();
    size_t getLength();
};

Matrix loadDataOnHost(DataReader* dataReader);

// Matrices of which something else is kept (copies of the table, in the workspace), to be used like the vector of them that they are. A program
// that has asked for one may write to it, or put another in its place, at any time from then on: handedOut says so, and what is kept is not
// relied on any more.
class WatchedMatrices {
public:
    explicit WatchedMatrices(size_t count) : all(count) {}
    operator std::vector<Matrix>&() const { return handOut(); }
    WatchedMatrices& operator=(const std::vector<Matrix>& other) { handOut() = other; return *this; }
    Matrix& operator[](size_t i) const { return handOut()[i]; }
    Matrix& at(size_t i) const { return handOut().at(i); }
    Matrix& front() const { return handOut().front(); }
    Matrix& back() const { return handOut().back(); }
    Matrix* data() const { return handOut().data(); }
    std::vector<Matrix>::iterator begin() const { return handOut().begin(); }
    std::vector<Matrix>::iterator end() const { return handOut().end(); }
    size_t size() const { return all.size(); }
    bool empty() const { return all.empty(); }

private:
    friend struct KnnData;
    friend class KnnExactGpu;
    std::vector<Matrix>& handOut() const
    {
        handedOut = true;
        return all;
    }
    mutable std::vector<Matrix> all;
    mutable bool handedOut = false;
};

struct KnnData {
    const int numGpus;
    const int batchSize;
    const int maxK;

    WatchedMatrices dCollectionPartitions;       // column major
    std::vector<Matrix> dInputBatches;
    std::vector<Matrix> dResultScores;
    std::vector<Matrix> dResultIndexes;
    std::vector<Matrix> hResultScores;
    std::vector<Matrix> hResultIndexes;
    std::vector<std::vector<std::string>> hKeys;
    WatchedMatrices dWorkspaces;                 // score blocks + partial lists of the search (instead of a full product matrix)
    std::vector<uint32_t> collectionRowsPadded;  // pad rows per device (rows are padded to a multiple of 8)
    // FP32, FP16: not 0 if the workspace holds copies of the table that load made (dsx_knn_prepare, _f16: with which storage); searches use them unless the program
    // has asked for the table or the workspace itself, and as long as this is not set to 0
    std::vector<int> workspacePrepared;
    std::vector<float> elapsedSgemm;             // milliseconds of the last search, per device
    std::vector<float> elapsedTopK;
    const DataType dataType;

    KnnData(int numGpus, int batchSize, int maxK, DataType dataType);
    void load(int device, DataReader* dataReader);
    void load(const std::map<int, DataReader*>& deviceToData);
    void load(const std::map<int, std::string>& deviceToFile, char keyValDelim, char vecDelim);
    int getFeatureSize() const;
    ~KnnData();

private:
    friend class KnnExactGpu;
    // Searches that are to go without screening (unscreenedStorage: or without bytes), and how many were to when one last had to be repeated: every repetition
    // doubles the number (64 at most), every search that went well halves it.
    uint32_t unscreened = 0, unscreenedNext = 0;
    int unscreenedStorage = 0;
    // the pinned memory that load put into hResultScores and hResultIndexes
    void* pinnedScores = nullptr;
    void* pinnedIndexes = nullptr;
};

Matrix allocateMatrixOnHost(uint32_t numRows, int numColumns, size_t elementSize);
Matrix allocateMatrixOnDevice(uint32_t numRows, int numColumns, size_t elementSize);
void freeMatrix(const Matrix& matrix);

}  // namespace knn
}  // namespace astdl

#endif
