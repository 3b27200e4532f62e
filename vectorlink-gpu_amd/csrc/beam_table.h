// The beam step of calls that have the distances of all their queries and vectors at hand (beam_table.hip).
#pragma once
#include "beam_ctrl.h"
#include "beam_row.h"

struct TableStepArgs {
    MergeArgs m;
    const int32_t *beams;
    int64_t n_vectors;
    int width;
    uint32_t width_magic;  // as in StepArgs
    uint32_t *table;       // distances as bits, one row per query; entries of queued and visited ids are kTableTaken
    int64_t columns;
    const int *unordered;  // set: some distance is not an ordinary number, and the loop goes on without the table
    int enter;             // the first launch with this table: what the row has queued or visited is not marked yet
    int window;            // iterations of the launch
    int raise_fill;        // the launch after it may be one that asks how full the visited lists are (BeamCtrl::first)
    int count_wanted;
    BeamReport *report;
};

// What the table kernel is built for; the rest runs without a table.
constexpr int kTableMaxQueue = 192, kTableMaxCandidates = 512, kTableMaxVisit = 8, kTableMaxExcluded = 64;

int vl_launch_table_step(const TableStepArgs &s, hipStream_t st);
