/*
 * oskar_evaluate_jones_E(): the station beam of every station into one
 * Jones array (oskar/interferometer/src/oskar_evaluate_jones_E.c:88-192):
 * one oskar_station_beam() per station model, or, with station beam
 * duplication, one per distinct model of the type map and a device copy for
 * every later station of that model.  Flat stations of one dipole type with
 * plain weights are evaluated up to 16 to a launch, by the kernel that
 * oskar_station_beam() uses for one.
 */
#include <math.h>
#include <stdlib.h>

#include "private.h"
#include "oskar_evaluate_jones_E.h"

/* Beams waiting to be evaluated by one launch: members of the same kind,
 * over the same directions. */
typedef struct Group
{
    oskar_AaStation member[OSKAR_AA_GROUP];
    int count, size, is_3d, normalise, num_points;
    const oskar_Mem* const* dirs;
    double frequency_hz;
    oskar_Mem* beam;
} Group;

static void group_flush(Group* g, int* status)
{
    const int n = g->count;
    g->count = 0;
    if (n == 0 || *status) return;
    *status = oskar_amd_hip_status(oskar_amd_aa_beam_launch(
            oskar_mem_precision(g->beam), oskar_mem_is_matrix(g->beam),
            g->is_3d, g->normalise, g->member, n,
            2.0 * M_PI * g->frequency_hz / 299792458.0, g->num_points,
            oskar_mem_void_const(g->dirs[0]),
            oskar_mem_void_const(g->dirs[1]),
            oskar_mem_void_const(g->dirs[2]), oskar_mem_void(g->beam),
            oskar_amd_current_stream()));
}

/* Members of a launch: as many (up to OSKAR_AA_GROUP) as leave the least of
 * the last round of workgroups idle, a round being four on each of 256 CUs
 * (16 stations x 65 workgroups ran as two rounds, 37 us; 15 as one). */
static int group_size(int num_points)
{
    const long long blocks = ((long long) num_points + 255) / 256;
    int m = 0, best = 1;
    double most = 0.0;
    for (m = 1; m <= OSKAR_AA_GROUP; ++m)
    {
        const long long rounds = (m * blocks + 1023) / 1024;
        const double full = (double) (m * blocks) / (1024.0 * rounds);
        if (full >= most)
        {
            most = full;
            best = m;
        }
    }
    return best;
}

/* The beam of one station model into row offset_out of the Jones array:
 * added to the group if it can be evaluated with others, else evaluated
 * now (rows are independent, so the order does not matter). */
static void station_row(Group* g, oskar_Station* station,
        oskar_StationWork* work, int coord_type, int num_points,
        const oskar_Mem* const source_coords[3], double ref_lon_rad,
        double ref_lat_rad, const oskar_Telescope* tel, int time_index,
        double time_start_mjd_utc, double time_mjd_utc, double frequency_hz,
        int offset_out, oskar_Mem* out, int* status)
{
    int is_3d = 0, normalise = 0;
    oskar_AaStation member;
    const int norm_type = oskar_telescope_phase_centre_coord_type(tel);
    const double norm_lon = oskar_telescope_phase_centre_longitude_rad(tel);
    const double norm_lat = oskar_telescope_phase_centre_latitude_rad(tel);
    if (*status) return;
    if (station && oskar_amd_station_beam_member(station, work, coord_type,
            num_points, source_coords, norm_type, norm_lon, norm_lat,
            time_index, time_mjd_utc, frequency_hz, offset_out, out,
            &member, &is_3d, &normalise))
    {
        if (g->count == g->size || (g->count > 0 &&
                (is_3d != g->is_3d || normalise != g->normalise)))
            group_flush(g, status);
        g->is_3d = is_3d;
        g->normalise = normalise;
        g->num_points = num_points;
        g->dirs = source_coords;
        g->frequency_hz = frequency_hz;
        g->beam = out;
        g->member[g->count++] = member;
        return;
    }
    oskar_station_beam(station, work, coord_type, num_points, source_coords,
            ref_lon_rad, ref_lat_rad, norm_type, norm_lon, norm_lat,
            time_index, time_start_mjd_utc, time_mjd_utc, frequency_hz,
            offset_out, out, status);
}

void oskar_evaluate_jones_E(oskar_Jones* E, int coord_type, int num_points,
        const oskar_Mem* const source_coords[3], double ref_lon_rad,
        double ref_lat_rad, oskar_Telescope* tel, int time_index,
        double time_start_mjd_utc, double time_mjd_utc, double frequency_hz,
        oskar_StationWork* work, int* status)
{
    int i = 0, j = 0;
    if (*status) return;
    const int num_stations = oskar_telescope_num_stations(tel);
    const int num_sources = oskar_jones_num_sources(E);
    if (num_stations == 0)
    {
        *status = OSKAR_ERR_MEMORY_NOT_ALLOCATED;
        return;
    }
    if (num_stations != oskar_jones_num_stations(E))
    {
        *status = OSKAR_ERR_DIMENSION_MISMATCH;
        return;
    }
    if (num_points > num_sources || num_points < 0)
    {
        *status = OSKAR_ERR_DIMENSION_MISMATCH;
        return;
    }
    oskar_Mem* out = oskar_jones_mem(E);
    Group group;
    group.count = 0;
    group.size = group_size(num_points);
    if (!oskar_telescope_allow_station_beam_duplication(tel))
    {
        if (oskar_telescope_num_station_models(tel) < num_stations)
        {
            *status = OSKAR_ERR_OUT_OF_RANGE;
            return;
        }
        for (i = 0; i < num_stations && !*status; ++i)
            station_row(&group, oskar_telescope_station(tel, i), work,
                    coord_type, num_points, source_coords, ref_lon_rad,
                    ref_lat_rad, tel, time_index, time_start_mjd_utc,
                    time_mjd_utc, frequency_hz, i * num_sources, out,
                    status);
        group_flush(&group, status);
        return;
    }
    {
        /* Models evaluated so far and the first station that holds each. */
        const int* type_map = (const int*) oskar_mem_void_const(
                oskar_telescope_station_type_map_const(tel));
        int* model_done = (int*) malloc((size_t) num_stations * sizeof(int));
        int* model_row = (int*) malloc((size_t) num_stations * sizeof(int));
        int num_done = 0;
        if (!model_done || !model_row)
        {
            free(model_done);
            free(model_row);
            *status = OSKAR_ERR_MEMORY_ALLOC_FAILURE;
            return;
        }
        for (i = 0; i < num_stations && !*status; ++i)
        {
            const int model = type_map[i];
            int row = -1;
            if (model < 0 || model >= oskar_telescope_num_station_models(tel))
            {
                *status = OSKAR_ERR_OUT_OF_RANGE;
                break;
            }
            for (j = 0; j < num_done; ++j)
                if (model_done[j] == model) { row = model_row[j]; break; }
            if (row >= 0)
            {
                group_flush(&group, status);
                oskar_mem_copy_contents(out, out,
                        (size_t) i * (size_t) num_sources,
                        (size_t) row * (size_t) num_sources,
                        (size_t) num_sources, status);
            }
            else
            {
                station_row(&group, oskar_telescope_station(tel, model),
                        work, coord_type, num_points, source_coords,
                        ref_lon_rad, ref_lat_rad, tel, time_index,
                        time_start_mjd_utc, time_mjd_utc, frequency_hz,
                        i * num_sources, out, status);
                model_done[num_done] = model;
                model_row[num_done++] = i;
            }
        }
        group_flush(&group, status);
        free(model_done);
        free(model_row);
    }
}
