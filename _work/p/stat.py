# kernel trace csv -> per kernel durations for the last half
import csv, sys, glob, collections
for f in sorted(glob.glob(sys.argv[1] + '/**/*kernel_trace.csv', recursive=True)):
    rows = list(csv.DictReader(open(f)))
    rows.sort(key=lambda r: int(r['Start_Timestamp']))
    n = int(sys.argv[2]) if len(sys.argv) > 2 else 100
    print(f, len(rows))
    prev = None
    for r in rows[-n:]:
        a, b = int(r['Start_Timestamp']), int(r['End_Timestamp'])
        gap = (a - prev) / 1e3 if prev else 0
        prev = b
        g = int(r['Grid_Size_X'])*int(r['Grid_Size_Y'])*int(r['Grid_Size_Z']) // max(1, int(r['Workgroup_Size_X'])*int(r['Workgroup_Size_Y'])*int(r['Workgroup_Size_Z']))
        print(f"{(b-a)/1e3:8.2f} gap {gap:7.2f} wg {g:6d}x{r['Workgroup_Size_X']:4s} lds {r.get('LDS_Block_Size','?'):>7s} vgpr {r.get('VGPR_Count','?')}/{r.get('Accum_VGPR_Count','?')} {r['Kernel_Name'][:100]}")
