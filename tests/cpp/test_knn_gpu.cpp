// KnnData as a program that works on its public matrices itself sees it.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <numeric>
#include <vector>

#include "amazon/dsstne/knn/KnnExactGpu.h"
#include "check.h"
#include "dsx.h"

using namespace astdl::knn;

static const uint32_t ROWS = 20003;
static const int DIM = 32, BATCH = 40, K = 10;

// whole numbers from -3 to 3, whose sums are exact in any order
static std::vector<float> numbers(size_t count, uint32_t seed)
{
    std::vector<float> v(count);
    for (auto& x : v) {
        seed = seed * 1664525u + 1013904223u;
        x = (float)((int)(seed >> 24) % 7 - 3);
    }
    return v;
}

// Whether a search of data finds the K best of `items`, ties by ascending row.
static bool finds(KnnData& data, const std::vector<float>& items, const std::vector<float>& queries)
{
    KnnExactGpu knn(&data);
    std::vector<uint32_t> rows(BATCH * K);
    std::vector<float> scores(BATCH * K);
    knn.searchRows(K, queries.data(), BATCH, rows.data(), scores.data());
    for (int q = 0; q < BATCH; q++) {
        std::vector<float> s(ROWS, 0.0f);
        for (uint32_t r = 0; r < ROWS; r++)
            for (int d = 0; d < DIM; d++) s[r] += queries[q * DIM + d] * items[(size_t)r * DIM + d];
        std::vector<uint32_t> order(ROWS);
        std::iota(order.begin(), order.end(), 0u);
        std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return s[a] > s[b]; });
        for (int j = 0; j < K; j++)
            if (rows[q * K + j] != order[j] || scores[q * K + j] != s[order[j]]) return false;
    }
    return true;
}

// The items in the order of the device table: [DIM][rows padded].
static std::vector<float> columnMajor(const std::vector<float>& items, uint32_t padded)
{
    std::vector<float> t((size_t)padded * DIM, 0.0f);
    for (uint32_t r = 0; r < ROWS; r++)
        for (int d = 0; d < DIM; d++) t[(size_t)d * padded + r] = items[(size_t)r * DIM + d];
    return t;
}

int main()
{
    const std::vector<float> items = numbers((size_t)ROWS * DIM, 1), other = numbers((size_t)ROWS * DIM, 2), queries = numbers(BATCH * DIM, 3);
    const uint32_t padded = (ROWS + 7) / 8 * 8;

    printf("items written into the device table after load\n");
    fflush(stdout);
    {
        KnnData data(1, BATCH, K, DataType::FP32);
        ArrayDataReader reader(items.data(), ROWS, DIM);
        data.load(0, &reader);
        CHECK(finds(data, items, queries));
        const std::vector<float> t = columnMajor(other, padded);
        CHECK_EQ(dsx_memcpy_h2d(data.dCollectionPartitions[0].data, t.data(), t.size() * sizeof(float)), DSX_OK);
        CHECK(finds(data, other, queries));
        // (and again through the pointer of before)
        Matrix& table = data.dCollectionPartitions[0];
        const std::vector<float> back = columnMajor(items, padded);
        CHECK_EQ(dsx_memcpy_h2d(table.data, back.data(), back.size() * sizeof(float)), DSX_OK);
        CHECK(finds(data, items, queries));
        // a table loaded anew, written through a reference that was taken before
        ArrayDataReader again(other.data(), ROWS, DIM);
        data.load(0, &again);
        CHECK(finds(data, other, queries));
        CHECK_EQ(dsx_memcpy_h2d(table.data, back.data(), back.size() * sizeof(float)), DSX_OK);
        CHECK(finds(data, items, queries));
    }

    printf("a workspace that the program uses between searches\n");
    fflush(stdout);
    {
        KnnData data(1, BATCH, K, DataType::FP32);
        ArrayDataReader reader(items.data(), ROWS, DIM);
        data.load(0, &reader);
        CHECK(finds(data, items, queries));
        std::vector<Matrix>& spaces = data.dWorkspaces;
        const std::vector<float> numbersToo = numbers((size_t)ROWS * DIM, 4);
        CHECK(spaces[0].elementSize > numbersToo.size() * sizeof(float));
        CHECK_EQ(dsx_memcpy_h2d(spaces[0].data, numbersToo.data(), numbersToo.size() * sizeof(float)), DSX_OK);
        CHECK(finds(data, items, queries));
    }
    printf("result buffers of the program's own\n");
    fflush(stdout);
    {
        KnnData data(1, BATCH, K, DataType::FP32);
        ArrayDataReader reader(items.data(), ROWS, DIM);
        data.load(0, &reader);
        freeMatrix(data.hResultScores[0]);
        data.hResultScores[0] = allocateMatrixOnHost(BATCH, K, sizeof(float));
        CHECK_EQ(dsx_host_is_pinned(data.hResultScores[0].data, BATCH * K * sizeof(float)), 0);
        CHECK(finds(data, items, queries));
        Matrix before = data.hResultIndexes[0];
        CHECK_EQ(dsx_host_is_pinned(before.data, BATCH * K * sizeof(float)), 1);
        data.hResultIndexes[0] = allocateMatrixOnHost(BATCH, K, sizeof(uint32_t));
        CHECK(finds(data, items, queries));
        CHECK_EQ(((uint32_t*)data.hResultIndexes[0].data)[BATCH * K - 1] < ROWS, true);
        // the call itself refuses what the device cannot write to
        CHECK_EQ(dsx_knn_search_host(DSX_KNN_FP32, data.dCollectionPartitions[0].data, padded, padded - ROWS, DIM, (const float*)data.dInputBatches[0].data, BATCH, K,
                                     (float*)data.dResultScores[0].data, (uint32_t*)data.dResultIndexes[0].data, (float*)data.hResultScores[0].data,
                                     (uint32_t*)data.hResultIndexes[0].data, nullptr, 0, nullptr),
                 DSX_EINVAL);
        freeMatrix(before);
    }
    printf("tables that outlive the device\n");
    fflush(stdout);
    {
        KnnData data(1, BATCH, K, DataType::FP32);
        ArrayDataReader reader(items.data(), ROWS, DIM);
        data.load(0, &reader);
        while (dsx_is_initialized()) dsx_shutdown();
    }
    return finish("test_knn_gpu");
}
